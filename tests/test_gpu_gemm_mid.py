"""The packed GEMM's middle sizes: ragged rows and columns, rows that start
inside a dword or a byte, K no multiple of the block, blocks of 64 and 128,
64- and 128-tiles, with the requantization in the epilogue and as a pass of
its own; all bit for bit against the oracle."""
import pytest
import torch

from oracle import mx_oracle as orc
from tests import _golden as G

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def qa():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import qtpytorch_amd
    return qtpytorch_amd


def _check(qa, M, K, N, dt, block, want_acc=False):
    g = torch.Generator().manual_seed(M + 3 * K + 7 * N)
    a, b = torch.randn(M, K, generator=g), torch.randn(K, N, generator=g)
    a[torch.rand(M, K, generator=g) < 1e-2] *= 40
    pa, sa, na = orc.quantize(a, dt, block)
    pb, sb, nb = orc.quantize(b, dt, block)
    pc, sc, name = orc.dispatch_qgemm(pa, sa, dt, (M, K), na, pb, sb, dt, (K, N), nb, block)
    bits = qa.get_mx_dtype(dt).bits
    r = qa.ops.qscale_gemm(pa.cuda(), sa.cuda(), pb.cuda(), sb.cuda(), M, K, N, bits, block,
                           qa.get_mx_dtype(name).bits, want_c=want_acc, want_acc=want_acc)
    tag = (M, K, N, dt, block)
    assert G.bits_equal(r["packed"].cpu(), pc), tag
    assert G.bits_equal(r["scales"].cpu(), sc), tag
    if want_acc:
        ca = orc.unpack_auto(pa, bits, M * K).reshape(M, K)
        cb = orc.unpack_auto(pb, bits, K * N).reshape(K, N)
        assert torch.equal(r["acc"].cpu(), orc.int_accumulators(ca, cb, M, K, N, block)), tag


# tile edges; N and K odd (int4: a row starts inside a byte), multiples of 2, 4, 8, 16
SHAPES = [(1, 64, 64), (63, 100, 65), (64, 128, 72), (130, 130, 70), (65, 201, 129), (129, 72, 260), (300, 1000, 258),
          (520, 384, 640), (200, 129, 900)]


@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("dt", ["int8d", "int4d"])
def test_shapes(qa, dt, block):
    for i, (M, K, N) in enumerate(SHAPES):
        _check(qa, M, K, N, dt, block, want_acc=i % 3 == 1)


@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("dt", ["int8d", "int4d"])
@pytest.mark.parametrize("N", [1600, 1664, 1650])
def test_large_tiles(qa, N, dt, block):
    """208 or 210 128-tiles: fused requantization (N whole blocks) and not, an odd number of stages."""
    _check(qa, 2040, 320, N, dt, block)


@pytest.mark.parametrize("dt", ["int8d", "int4d"])
def test_scale_counts(qa, dt):
    """Scale arrays of another length are read as ones."""
    M, K, N = 200, 256, 300
    a, b = torch.randn(M, K), torch.randn(K, N)
    pa, sa, _ = orc.quantize(a, dt, 128)
    pb, sb, _ = orc.quantize(b, dt, 128)
    bits = qa.get_mx_dtype(dt).bits
    ca, cb = orc.unpack_auto(pa, bits, M * K).reshape(M, K), orc.unpack_auto(pb, bits, K * N).reshape(K, N)
    ref = orc.int_accumulators(ca, cb, M, K, N, 128).sum(0).float()
    c = qa.ops.qscale_gemm(pa.cuda(), sa[:-1].cuda(), pb.cuda(), sb[:-1].cuda(), M, K, N, bits, 128, 0,
                           want_packed=False, want_c=True)["c"].cpu()
    assert torch.equal(c, ref)
