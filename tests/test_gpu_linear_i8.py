"""The int8 x int8 linear on its kernels' edges, against the product of the
operands' own values in 64 bits.

Per output the kernels round the scaled sum of each K block, add it and round,
and multiply by a scale once or twice: at most KB + 4 roundings of 2^-24 of
the sum of the blocks' magnitudes.
"""
import pytest
import torch

import qtpytorch_amd as qa

pytestmark = pytest.mark.gpu


def _values(t, M, K):
    n = t._mx_n
    bits, block = t._mx_dtype.bits, t._mx_block
    by = t._mx_packed.reshape(-1).view(torch.uint8).to(torch.int64)
    codes = torch.stack([(by >> s) & ((1 << bits) - 1) for s in range(0, 8, bits)], 1).reshape(-1)[:n]
    codes = torch.where(codes >= 1 << (bits - 1), codes - (1 << bits), codes)
    scale = t._mx_scales.double().repeat_interleave(block)[:n]
    return codes.double().reshape(M, K), scale.reshape(M, K)


def _check(M, K, N, xd, wd, xb, wb, bias):
    g = torch.Generator(device="cuda").manual_seed(M * 31 + K * 7 + N)
    x = torch.randn(M, K, generator=g, device="cuda") * torch.exp2(torch.randint(-8, 8, (M, 1), generator=g,
                                                                                  device="cuda").float())
    w = torch.randn(N, K, generator=g, device="cuda")
    b = torch.randn(N, generator=g, device="cuda") if bias else None
    xq, wq = qa.mx_tensor.quantize(x, xd, xb), qa.mx_tensor.quantize(w, wd, wb)
    got = qa.fused_int8_linear(xq, wq, b).double()
    (cx, sx), (cw, sw) = _values(xq, M, K), _values(wq, N, K)
    kb = 128 if all(v % 128 == 0 for v in (K, xb, wb)) else 64
    want, size = torch.zeros_like(got), torch.zeros_like(got)
    for k in range(0, K, kb):
        part = (cx[:, k:k + kb] @ cw[:, k:k + kb].t()) * sx[:, k, None] * sw[None, :, k]
        want += part
        size += part.abs()
    if b is not None:
        want += b.double()
        size += b.double().abs()
    assert ((got - want).abs() <= (K // kb + 4) * 2.0 ** -24 * size + 1e-40).all()


# the 256 x 128 loop: per-token scales as they are, one scale for two rows, and per block
@pytest.mark.parametrize("xb", [256, 512, 128])
@pytest.mark.parametrize("M,N,wd,wb", [(2049, 4000, "int8d", 128), (4096, 2113, "int4d", 256)])
def test_large(M, N, wd, wb, xb):
    _check(M, 256, N, "int8d", wd, xb, wb, bias=N % 2 == 0)
