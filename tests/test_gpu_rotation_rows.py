"""'h' dtypes over rows of 129 .. 8192 elements (and the short and long rows
next to that range): codes, scales and dequantized values bit for bit against
the oracle, over every row length class of the register transform (rows of
whole blocks take the fused kernels, others the rotation to fp32)."""
import pytest
import torch

from oracle import mx_oracle as orc
from tests import _golden as G

pytestmark = pytest.mark.gpu

SEED = 77
#           n = 256 (d < n, d = n), 512, 1024 .. 8192 with and without padding, d % 128 != 0, d % 4 != 0
SHAPES = [(33, 256), (5, 129), (7, 200), (40, 384), (3, 512), (9, 640), (6, 1000), (17, 1024), (4, 2048), (3, 3001),
          (2, 3072), (5, 4096), (2, 5120), (3, 8192), (9, 96), (2, 9000)]


@pytest.fixture(scope="module")
def qa():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import qtpytorch_amd
    return qtpytorch_amd


def _check(qa, x, dt):
    q = qa.mx_tensor.quantize(x.cuda(), dt, 128, seed=SEED)
    p, s, n = orc.quantize(x, dt, 128, seed=SEED)
    assert G.bits_equal(q.packed.cpu(), p), (dt, tuple(x.shape))
    assert G.bits_equal(q.mx_scales.cpu(), s), (dt, tuple(x.shape))
    ref = orc.dequant(p, s, dt, n, 128, seed=SEED, orig_shape=tuple(x.shape), hadamard_mode="rows").reshape(x.shape)
    y = q.dequantize().cpu()
    both = y.isnan() & ref.isnan()
    assert torch.equal(y.masked_fill(both, 0).view(torch.int32), ref.masked_fill(both, 0).view(torch.int32)), \
        (dt, tuple(x.shape))


@pytest.mark.parametrize("dt", ["int1dh", "int2dh", "int4dh", "int8dh", "float4dh", "float8dh"])
def test_rows(qa, dt):
    for i, (r, d) in enumerate(SHAPES):
        g = torch.Generator().manual_seed(d)
        x = torch.randn(r, d, generator=g)
        x[torch.rand(r, d, generator=g) < 1e-2] *= 30
        if r > 2:
            x[1] = 0
        _check(qa, x.to((torch.float32, torch.bfloat16, torch.float16)[i % 3]), dt)


@pytest.mark.parametrize("dt", ["int4dh", "float8dh"])
def test_many_rows(qa, dt):
    """More rows than the grid holds at once, and a last workgroup that is not full."""
    _check(qa, torch.randn(70001, 256, generator=torch.Generator().manual_seed(1)), dt)


def test_tiny_and_non_finite(qa):
    x = torch.randn(6, 1024, generator=torch.Generator().manual_seed(2))
    x[0] *= 1e-38
    x[1, 5] = float("inf")
    x[2, 9] = float("nan")
    x[3] *= 2.0 ** -100
    for dt in ("int4dh", "float4dh", "int1dh"):
        q = qa.mx_tensor.quantize(x.cuda(), dt, 128, seed=SEED)
        p, s, _ = orc.quantize(x, dt, 128, seed=SEED)
        fin = torch.tensor([0, 3, 4, 5])
        assert torch.equal(q.packed.cpu().view(6, -1)[fin], p.view(6, -1)[fin])
        assert torch.equal(q.mx_scales.cpu().view(6, -1)[fin], s.view(6, -1)[fin])
        assert torch.equal(q.mx_scales.cpu().isfinite(), s.isfinite())
