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


# 64-tiles: the smallest, ragged tiles, a last half stage, K split with and
# without a short last part, blocks of 64, both widths, each form of the scales
@pytest.mark.parametrize("M,K,N,dt,xb,wb", [
    (1, 64, 1, "int8d", 64, 64), (3, 128, 65, "int8d", 128, 128), (65, 192, 63, "int4d", 192, 64),
    (8, 768, 512, "int8d", 768, 128), (8, 1536, 70, "int8d", 1536, 128), (17, 3264, 200, "int8d", 64, 64),
    (64, 4096, 256, "int4d", 4096, 4096), (63, 1792, 129, "int4d", 128, 128), (129, 320, 2000, "int8d", 320, 64),
    (40, 512, 96, "int8d", 256, 128), (40, 512, 96, "int8d", 1024, 128), (1100, 1024, 4096, "int8d", 1024, 128),
    (2049, 128, 4000, "int4d", 128, 128), (1090, 192, 4100, "int8d", 192, 64),
    (57, 704, 816, "int8d", 704, 128), (33, 192, 70, "int4d", 128, 256), (9, 320, 129, "int8d", 128, 1024),
    (9, 384, 129, "int8d", 128, 384), (9, 384, 129, "int8d", 768, 1152)])
def test_tiles(M, K, N, dt, xb, wb):
    _check(M, K, N, dt, dt, xb, wb, bias=M % 2 == 1)


def test_no_room_for_partial_sums():
    """A workspace that ends before the partial sums: K is not split, and the
    result is the unsplit one's; shorter ones are refused as before."""
    from qtpytorch_amd import _lib as L
    M, K, N = 8, 4096, 256
    g = torch.Generator(device="cuda").manual_seed(3)
    xq = qa.mx_tensor.quantize(torch.randn(M, K, generator=g, device="cuda"), "int8d", K)
    wq = qa.mx_tensor.quantize(torch.randn(N, K, generator=g, device="cuda"), "int8d", 128)
    full = L.lib().mxk_linear_i8_workspace(M, K, N, 8, 8, K, 128)
    base = (4 * 32 * M + 255) // 256 * 256 + (4 * 32 * N + 255) // 256 * 256
    assert full > base
    ws = torch.empty(full, dtype=torch.uint8, device="cuda")

    def run(nbytes):
        out = torch.full((M, N), float("nan"), device="cuda")
        rc = L.lib().mxk_linear_i8(xq._mx_packed.data_ptr(), M * K, xq._mx_scales.data_ptr(), M, K, 8,
                                   wq._mx_packed.data_ptr(), N * K, wq._mx_scales.data_ptr(), N * K // 128, 128, 8,
                                   M, K, N, 0, out.data_ptr(), ws.data_ptr(), nbytes, L.stream_of(ws))
        return rc, out

    (r0, a), (r1, b), (r2, _) = run(full), run(base), run(base - 1)
    assert r0 == 0 and r1 == 0 and r2 != 0
    (cx, sx), (cw, sw) = _values(xq, M, K), _values(wq, N, K)
    size = (cx * sx).abs() @ (cw * sw).abs().t()
    want = (cx * sx) @ (cw * sw).t()
    for got in (a, b):
        assert ((got.double() - want).abs() <= 36 * 2.0 ** -24 * size).all()
