"""Scales at and past the limits of the large packed GEMM's three-instruction
epilogue (2^-51 <= |SA| < 2^54 or zero, |SB| < 2^53): bit for bit against the
oracle on sampled rows, on either side of each limit, with infinities and NaN."""
import pytest
import torch

from tests.test_gpu_parity import _large_gemm_vs_oracle

pytestmark = pytest.mark.gpu

M, K, N = 4096, 384, 2048
ROWS = [0, 1, 2, 3, 5, 250, 2047, 4095]


@pytest.fixture(scope="module")
def qa():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import qtpytorch_amd
    return qtpytorch_amd


@pytest.mark.parametrize("dt", ["int8d", "int4d"])
@pytest.mark.parametrize("which,factor", [
    ("a", 2.0 ** -51), ("a", 2.0 ** -52), ("a", 0.0), ("a", -1.0), ("a", 1.9 * 2.0 ** 53), ("a", 2.0 ** 54),
    ("a", 2.0 ** -130), ("b", 1.9 * 2.0 ** 52), ("b", 2.0 ** 53), ("b", 2.0 ** -140), ("b", -2.0), ("b", 0.0)])
def test_scale_limits(qa, dt, which, factor):
    g = torch.Generator(device="cuda").manual_seed(5)
    pa, sa, _ = qa.ops.quantize(torch.randn(M, K, generator=g, device="cuda"), dt, 128)
    pb, sb, _ = qa.ops.quantize(torch.randn(K, N, generator=g, device="cuda"), dt, 128)
    # one operand's scales at the limit (powers of two times the limit's own
    # significand), in every third block and in all of row 0
    t = (sa if which == "a" else sb).clone()
    t[::3] = factor
    t[: K // 128] = factor
    sa, sb = (t, sb) if which == "a" else (sa, t)
    _large_gemm_vs_oracle(qa, dt, M, K, N, pa, sa, pb, sb, ROWS)


@pytest.mark.parametrize("dt", ["int8d", "int4d"])
def test_non_finite_scales(qa, dt):
    g = torch.Generator(device="cuda").manual_seed(6)
    pa, sa, _ = qa.ops.quantize(torch.randn(M, K, generator=g, device="cuda"), dt, 128)
    pb, sb, _ = qa.ops.quantize(torch.randn(K, N, generator=g, device="cuda"), dt, 128)
    kb = K // 128
    sa, sb = sa.clone(), sb.clone()
    sa[1 * kb], sa[2 * kb + 1] = float("inf"), float("nan")
    sb[7], sb[N + 9] = float("inf"), float("nan")
    bits = qa.get_mx_dtype(dt).bits
    c = qa.ops.qscale_gemm(pa, sa, pb, sb, M, K, N, bits, 128, 0, want_packed=False, want_c=True, want_acc=True)
    ref = torch.zeros(M, N, device="cuda")
    for i in range(kb):  # the same fp32 operations, in order
        ref = ref + (c["acc"][i].float() * sa.view(M, kb)[:, i, None]) * sb.view(kb, N)[i]
    assert torch.equal(c["c"].isnan(), ref.isnan())
    ok = ~ref.isnan()
    assert torch.equal(c["c"][ok], ref[ok])
