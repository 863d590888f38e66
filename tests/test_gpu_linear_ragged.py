"""The weight-only linear over weights whose blocks do not line up with
128-column tiles: out_features (mx_linear) or in_features ([out, in] weights)
no multiple of 128, or blocks other than 128.

Checked against x.double() @ dequant(W).double() with the oracle's dequantized
weight.  The kernel carries x and c * s as f16 pairs hi + lo and leaves out lo
* lo: each term is off by at most 3 * 2^-22 of itself, and the fp32 sums add at
most one rounding of 2^-24 per 32 terms and partial.  Rows of x and columns of W
(of [in, out] weights: groups of 8 columns, or of 32 in blocks of 128 and more)
are scaled by powers of two that put their largest value at 2^13 or more, where f16 keeps
2^-25: a value far below that largest is off by 2^-38 of it (of weights: of the
largest value that the blocks of its columns can hold)."""
import pytest
import torch

from oracle import mx_oracle as orc

pytestmark = pytest.mark.gpu

FMTS = ["int1d", "int2d", "int4d", "int8d", "float4d", "float8d"]


@pytest.fixture(scope="module")
def qa():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import qtpytorch_amd
    return qtpytorch_amd


def _case(M, K, N, dt, block, nt, src, seed=0):
    g = torch.Generator().manual_seed(1000 * M + 10 * K + N + seed)
    x = torch.randn(M, K, generator=g).to(src)
    w = 0.02 * torch.randn(*((N, K) if nt else (K, N)), generator=g)
    w[torch.rand(w.shape, generator=g) < 1e-2] *= 20
    packed, scales, n = orc.quantize(w, dt, block)
    return x, packed, scales, orc.dequant(packed, scales, dt, n, block).reshape(w.shape)


def _run(qa, x, packed, scales, dt, K, N, block, nt, bias=None):
    d = "cuda:0"
    fn = qa.ops.linear_wq_nt if nt else qa.ops.linear_wq
    sizes = (N, K) if nt else (K, N)
    return fn(x.to(d), packed.to(d), scales.to(d), dt, *sizes, block, bias=None if bias is None else bias.to(d)).cpu()


def _check(y, x, wd, nt, bias=None, top=None, block=128):
    """top: the largest value each weight's block can hold (else |wd|)."""
    xd, w = x.double(), (wd.t() if nt else wd).double()
    ref = xd @ w + (0 if bias is None else bias.double())
    K, N = w.shape
    terms = xd.abs() @ w.abs()
    wmax = (w.abs() if top is None else top.t() if nt else top).double().amax(0)
    if not nt:
        g = 32 if block >= 128 else 8
        wmax = torch.nn.functional.pad(wmax, (0, -N % g)).view(-1, g).amax(1).repeat_interleave(g)[:N]
    floor = 2.0 ** -38 * (xd.abs().amax(1, keepdim=True) * w.abs().sum(0) + xd.abs().sum(1, keepdim=True) * wmax)
    tol = (3 * 2.0 ** -22 + (K / 32 + 16) * 2.0 ** -24) * terms + floor + 2.0 ** -23 * ref.abs() + 1e-37
    err = (y.double() - ref).abs()
    assert bool((err <= tol).all()), f"worst {float((err / tol).max()):.3g} x the bound"


SHAPES = [  # rows: edges of the 16-, 32- and 64-row tiles and of the waves along rows; columns around a tile; K around a step
    (1, 33, 1), (16, 64, 127), (17, 95, 129), (32, 200, 1000), (33, 31, 257), (64, 1000, 130), (65, 129, 259),
    (129, 257, 300), (300, 96, 391), (5, 4096, 203), (16, 1, 7), (3, 2049, 1001),
]


@pytest.mark.parametrize("nt", [False, True], ids=["kn", "nk"])
@pytest.mark.parametrize("dt", FMTS)
def test_shapes(qa, dt, nt):
    for i, (M, K, N) in enumerate(SHAPES):
        if nt:
            K, N = N, K
        src = (torch.float32, torch.bfloat16, torch.float16)[i % 3]
        x, p, s, wd = _case(M, K, N, dt, 128, nt, src)
        bias = torch.randn(N) if i % 2 else None
        _check(_run(qa, x, p, s, dt, K, N, 128, nt, bias), x, wd, nt, bias)


@pytest.mark.parametrize("nt", [False, True], ids=["kn", "nk"])
@pytest.mark.parametrize("block", [8, 20, 64, 96, 200, 1000])
def test_blocks(qa, block, nt):
    for dt in ("int4d", "int8d", "float8d"):
        for M, K, N in ((4, 160, 256), (70, 133, 77)):
            x, p, s, wd = _case(M, K, N, dt, block, nt, torch.float32)
            _check(_run(qa, x, p, s, dt, K, N, block, nt), x, wd, nt, block=block)


@pytest.mark.parametrize("nt", [False, True], ids=["kn", "nk"])
def test_magnitudes(qa, nt):
    """Rows of x of very different magnitudes, a zero row, and small and large W."""
    M, K, N = 40, 513, 321
    x, _, _, _ = _case(M, K, N, "int8d", 128, nt, torch.float32)
    x *= 10.0 ** torch.linspace(-7, 7, M)[:, None]
    x[3] = 0
    for e in (1e-6, 1e6):
        w = e * torch.randn(*((N, K) if nt else (K, N)), generator=torch.Generator().manual_seed(5))
        p, s, n = orc.quantize(w, "int8d", 128)
        wd = orc.dequant(p, s, "int8d", n, 128).reshape(w.shape)
        y = _run(qa, x, p, s, "int8d", K, N, 128, nt)
        _check(y, x, wd, nt)
        assert not y[3].any()


@pytest.mark.parametrize("nt", [False, True], ids=["kn", "nk"])
@pytest.mark.parametrize("M,src", [(8, torch.float32), (70, torch.float32), (70, torch.bfloat16)])
@pytest.mark.parametrize("dt", FMTS)
def test_mixed_k_magnitudes(qa, dt, M, src, nt):
    """x large where W is small along K and the other way round: every term counts."""
    K, N = (1000, 77) if nt else (2048, 203)
    x, _, _, _ = _case(M, K, N, dt, 8, nt, src)
    w = 0.02 * torch.randn(*((N, K) if nt else (K, N)), generator=torch.Generator().manual_seed(7))
    small = torch.arange(K) // 8 % 2 == 0
    x = torch.where(small, x.float() * 1e5, x.float()).to(src)
    w *= torch.where(small, 1e-5, 1.0)[None, :] if nt else torch.where(small, 1e-5, 1.0)[:, None]
    p, s, n = orc.quantize(w, dt, 8 if nt else 128)
    _check(_run(qa, x, p, s, dt, K, N, 8 if nt else 128, nt), x, orc.dequant(p, s, dt, n, 8 if nt else 128).reshape(w.shape), nt)


@pytest.mark.parametrize("nt", [False, True], ids=["kn", "nk"])
@pytest.mark.parametrize("M", [3, 70])
@pytest.mark.parametrize("dt", FMTS)
def test_columns_do_not_see_what_lies_past_k(qa, dt, M, nt):
    """K no multiple of a step: the last step also loads the next row of an [out,
    in] weight, or the padding of the last block.  A column keeps its bits when
    the scales there grow by 2^20 (a rescued NaN would be another sum)."""
    for K, N, block in (((1000, 40, 8), (1001, 60, 8), (133, 200, 128), (4100, 24, 128)) if nt
                        else ((1001, 391, 128), (4100, 203, 64))):
        x, p, s, _ = _case(M, K, N, dt, block, nt, torch.float32)
        q = torch.arange(s.numel()) * block
        if nt:  # blocks inside the odd rows
            loud = (q // K % 2 == 1) & ((q + block - 1) // K == q // K)
            keep = torch.arange(N) % 2 == 0
        else:  # the last block; the tiles before it
            loud = torch.arange(s.numel()) == s.numel() - 1
            keep = torch.arange(N) < (int(q[-1]) - (K - 1) * N) // 128 * 128
        assert loud.any() and keep.any()
        a = _run(qa, x, p, s, dt, K, N, block, nt)
        b = _run(qa, x, p, torch.where(loud, s * 2.0 ** 20, s), dt, K, N, block, nt)
        assert torch.equal(a[:, keep], b[:, keep]), (K, N, block)


@pytest.mark.parametrize("nt", [False, True], ids=["kn", "nk"])
@pytest.mark.parametrize("M,src", [(3, torch.float32), (20, torch.bfloat16), (70, torch.float32), (70, torch.bfloat16)])
@pytest.mark.parametrize("dt", FMTS)
def test_ends_of_k(qa, dt, M, src, nt):
    """K around whole steps of 32 (the last step takes the last 32 rows of K, and those
    that the step before has count once), and below one step."""
    for K in (31, 32, 33, 40, 63, 64, 65, 95, 164):
        for N, block in ((40, 8), (131, 128)):
            x, p, s, wd = _case(M, K, N, dt, block, nt, src)
            _check(_run(qa, x, p, s, dt, K, N, block, nt), x, wd, nt, block=block)


@pytest.mark.parametrize("nt", [False, True], ids=["kn", "nk"])
@pytest.mark.parametrize("M", [3, 70])
@pytest.mark.parametrize("dt", FMTS)
def test_column_magnitudes(qa, dt, M, nt):
    """Columns far smaller than the ones beside them, and one scale that is not
    finite: every other column keeps its own precision."""
    for block, K, N in ((8, 300, 264), (8, 77, 131), (64, 333, 391), (128, 600, 203), (256, 1025, 300), (128, 4100, 140)):
        if nt:
            K, N = N, K
        x, p, s, _ = _case(M, K, N, dt, block, nt, torch.float32)
        g = torch.Generator().manual_seed(K)
        flat = torch.arange(s.numel()) * block
        # a magnitude for each row of [out, in] weights, for each place of a block's start of [in, out] ones
        mag = torch.exp2(-30 * torch.rand(N, generator=g))
        s = s * (mag[flat // K] if nt else mag[(flat % N) // 16 * 16])
        q = 5 if nt else s.numel() // 2
        s[q] = (float("inf"), float("nan"))[M % 2]
        wd = orc.dequant(p, s, dt, K * N, block).reshape((N, K) if nt else (K, N))
        y = _run(qa, x, p, s, dt, K, N, block, nt)
        vmax = 1.0 if dt[0] == "f" or dt == "int1d" else float(2 ** (int(dt[3]) - 1) - 1)
        top = (vmax * torch.where(s.isfinite(), s, 0.0)).repeat_interleave(block)[:K * N].reshape(wd.shape)
        ok = wd.isfinite().all(1 if nt else 0)
        assert 0 < int(ok.sum()) < N
        assert not y[:, ~ok].isfinite().any()
        # (groups of columns keep their place: what is left out counts as zero)
        wd = torch.where(ok[:, None] if nt else ok[None, :], wd, 0.0)
        _check(torch.where(ok[None, :], y, 0.0), x, wd, nt, top=top, block=block)


@pytest.mark.parametrize("nt", [False, True], ids=["kn", "nk"])
@pytest.mark.parametrize("M", [3, 70])
def test_non_finite(qa, nt, M):
    """Infinities and NaN in x and in the scales come out where an fp32 product has them."""
    K, N = 300, 203
    x, p, s, wd = _case(M, K, N, "int8d", 128, nt, torch.float32)
    x[0, 7] = float("inf")
    x[1, 9] = float("nan")
    s[5] = float("inf")
    wd = orc.dequant(p, s, "int8d", K * N, 128).reshape(wd.shape)
    y = _run(qa, x, p, s, "int8d", K, N, 128, nt)
    ref = x.double() @ (wd.t() if nt else wd).double()
    assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isinf(), ref.isinf())
    assert torch.equal(y[y.isinf()].sign().double(), ref[ref.isinf()].sign())
    fin = ref.isfinite()
    assert float(((y.double() - ref)[fin]).abs().max()) <= 1e-3 * float(ref[fin].abs().max())


@pytest.mark.parametrize("nt", [False, True], ids=["kn", "nk"])
@pytest.mark.parametrize("dt", FMTS)
@pytest.mark.parametrize("M,K,N", [(6, 300, 203), (70, 301, 140), (20, 4100, 77)])
def test_non_finite_rows_and_columns(qa, M, K, N, dt, nt):
    """Whole rows and single values of NaN and of infinities of one and both
    signs, beside a scale that is infinite and one that is NaN, with and without
    K split: NaN, infinities and finite values where a 64-bit product has them."""
    for src in (torch.float32, torch.bfloat16):
        x, p, s, _ = _case(M, K, N, dt, 128, nt, src)
        x[0, :], x[1, 7], x[2, 5], x[2, 6] = float("inf"), float("nan"), float("inf"), -float("inf")
        x[3, :], x[4, K - 1] = float("nan"), -float("inf")
        s[3], s[-1] = float("inf"), float("nan")
        wd = orc.dequant(p, s, dt, K * N, 128).reshape((N, K) if nt else (K, N))
        bias = torch.randn(N)
        y = _run(qa, x, p, s, dt, K, N, 128, nt, bias)
        # (one product after the other: a library's sum may meet its operands padded)
        t = x.double()[:, :, None] * (wd.t() if nt else wd).double()[None]
        ref = t.sum(1) + bias
        assert torch.equal(y.isnan(), ref.isnan()) and torch.equal(y.isinf(), ref.isinf())
        assert torch.equal(y[y.isinf()].sign().double(), ref[ref.isinf()].sign())
        fin = ref.isfinite()
        assert not fin.any() or float((y.double() - ref)[fin].abs().max()) <= 1e-5 * float(ref[fin].abs().max())


@pytest.mark.parametrize("nt", [False, True], ids=["kn", "nk"])
def test_non_finite_rows_take_no_longer_than_the_scalar_kernel(qa, nt):
    """A NaN in x costs nothing, infinities at most a small multiple of the fp32
    kernel that runs without a workspace (the sum of one output after the other
    took 30 times the product for a single NaN)."""
    M, K, N = 64, 2048, 1001
    if nt:
        K, N = N, K
    x, p, s, _ = _case(M, K, N, "int8d", 128, nt, torch.float32)
    x, p, s = x.cuda(), p.cuda(), s.cuda()
    lib, L = qa._lib.lib(), qa._lib
    out = torch.empty(M, N, device="cuda")

    def scalar():
        if nt:
            return lib.mxk_linear_wq_nt(x.data_ptr(), 0, M, K, p.data_ptr(), p.numel() * p.element_size(), s.data_ptr(),
                                        s.numel(), 0, N, 0, 8, 128, 0, out.data_ptr(), 0, 0, L.stream_of(x))
        return lib.mxk_linear_wq(x.data_ptr(), 0, M, K, p.data_ptr(), s.data_ptr(), 0, N, 0, 8, 128, 0, out.data_ptr(),
                                 0, 0, L.stream_of(x))

    def us(fn):
        best = float("inf")
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            fn()
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) * 1e3)
        return best

    fn = qa.ops.linear_wq_nt if nt else qa.ops.linear_wq
    call = lambda v: fn(v, p, s, "int8d", *((N, K) if nt else (K, N)), 128)
    assert scalar() == 0
    one, rows, inf = x.clone(), x.clone(), x.clone()
    one[5, 9] = rows[::2, 3] = float("nan")
    inf[::3, 4] = float("inf")
    base, fp32 = us(lambda: call(x)), us(scalar)
    t = [us(lambda: call(v)) for v in (one, rows, inf)]
    print(f"{nt} finite {base:.0f} us, scalar kernel {fp32:.0f}; a NaN {t[0]:.0f}, NaN rows {t[1]:.0f}, infinities {t[2]:.0f}")
    assert max(t[:2]) < 3 * base and t[2] < 8 * fp32


def test_small_blocks_take_little_longer(qa):
    """Few rows, few columns: the largest scales of blocks of 8 to 64 are found about as
    fast as those of 128 (one load after the other: 1.7 to 2.8 times the call)."""
    M, K, N = 16, 4096, 1000

    def us(block):
        x, p, s, _ = _case(M, K, N, "int8d", block, False, torch.float32)
        x, p, s = x.cuda(), p.cuda(), s.cuda()
        best = float("inf")
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                qa.ops.linear_wq(x, p, s, "int8d", K, N, block)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b) * 1e3 / 20)
        return best

    t = {block: us(block) for block in (128, 8, 32, 64)}
    print(t)
    assert max(t.values()) < 1.4 * t[128]


@pytest.mark.parametrize("nt", [False, True], ids=["kn", "nk"])
def test_keeps_no_workspace(qa, nt):
    """A call's scratch memory (x again, and the partial sums) goes back with it."""
    M, K, N = 16, 8192, 1001
    if nt:
        K, N = N, K
    x, p, s, _ = _case(M, K, N, "int4d", 128, nt, torch.float32)
    x, p, s = x.cuda(), p.cuda(), s.cuda()
    fn = qa.ops.linear_wq_nt if nt else qa.ops.linear_wq
    assert qa._lib.lib().mxk_linear_ragged_workspace(M, K, N, 4, 128) >= 4 * M * K
    side = torch.cuda.Stream()  # a stream of its own: nothing kept for it yet
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        before = torch.cuda.memory_allocated()
        y = fn(x, p, s, "int4d", *((N, K) if nt else (K, N)), 128)
        held = torch.cuda.memory_allocated() - before
    torch.cuda.current_stream().wait_stream(side)
    assert held <= y.numel() * 4 + 512


def test_module_and_gradient(qa):
    """mx_linear with an odd width: forward, input gradient and a captured replay."""
    g = torch.Generator().manual_seed(3)
    lin = torch.nn.Linear(160, 203, bias=False)
    with torch.no_grad():
        lin.weight.copy_(0.05 * torch.randn(203, 160, generator=g))
    m = qa.mx_linear.from_linear(lin.cuda(), "int4d")
    x = torch.randn(24, 160, generator=g).cuda().requires_grad_(True)
    y = m(x)
    go = torch.randn(24, 203, generator=g).cuda()
    (gx,) = torch.autograd.grad(y, x, go)
    wd = m.weight.cpu()
    _check(y.detach().cpu(), x.detach().cpu(), wd, False)
    _check(gx.cpu(), go.cpu(), wd, True)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.no_grad(), torch.cuda.stream(s):
        m(x)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            yg = m(x)
    torch.cuda.current_stream().wait_stream(s)
    for _ in range(3):
        yg.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(yg, y)
        m(x)
