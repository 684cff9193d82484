"""The GPU kernels at the sizes where their tilings can go wrong: edges of
tiles and K steps, remainders, empty and uneven spin runs, small scratch.
Against exact integers, FP64 matrix products on the host or the oracle."""
import numpy
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from oracle import ftcc as oracle  # noqa: E402
from oracle import fock_space as fs  # noqa: E402
from test_gpu_adjoint import antisym  # noqa: E402
from test_gpu_parity import _spin_problem, dev, rel, to_np  # noqa: E402

U64, U32 = 2.0 ** -53, 2.0 ** -24


def _gemm(M, N, K, batch, layout, precision, alpha, beta, ints=0):
    """C = alpha A B + beta C on the engine, the host's, |A| |B| and |C|."""
    from kelvin_amd.engine import FTEngine
    d = dev()
    g = torch.Generator().manual_seed(M + 3 * N + 7 * K)

    def draw(*s):
        if ints:
            return torch.randint(-ints, ints + 1, s, generator=g).double()
        return torch.randn(*s, generator=g, dtype=torch.float64)

    def lay(x, c):
        x = x.to(d)
        return x if c == 'n' else \
            x.transpose(1, 2).contiguous().transpose(1, 2)
    A, B, C = draw(batch, M, K), draw(batch, K, N), draw(batch, M, N)
    Cd = C.to(d)
    eng = FTEngine(2, 2, 1)
    eng.gemm(lay(A, layout[0]), lay(B, layout[1]), Cd, alpha=alpha, beta=beta,
             precision=precision)
    out = to_np(Cd)
    eng.close()
    return (out, (alpha * (A @ B) + beta * C).numpy(),
            (abs(alpha) * (A.abs() @ B.abs())).numpy(),
            (abs(beta) * C.abs()).numpy())


@pytest.mark.parametrize("layout", ["nn", "tn", "nt", "tt"])
@pytest.mark.parametrize("M,N,K,batch", [
    (1, 1, 1, 1), (15, 130, 4, 2), (31, 65, 32, 1), (33, 64, 33, 3),
    (48, 129, 48, 1), (49, 63, 49, 2), (64, 31, 64, 1), (130, 16, 31, 2),
    (127, 33, 47, 1), (66, 48, 64, 3), (200, 50, 1, 1), (65, 66, 63, 2),
    (65, 66, 65, 2),                     # K one past the short-K kernel
    (4096, 4100, 5, 1),                  # more 64x64 tiles than it takes
    (20, 30, 3000, 1), (300, 260, 900, 2)])   # split K, many and few sums
def test_gemm_tile_and_k_edges(M, N, K, batch, layout):
    """Rounding of two FP64 sums of K products: 2 (K + 3) u |A| |B|."""
    out, ref, ab, c = _gemm(M, N, K, batch, layout, "fp64", 0.75, -0.5)
    assert (numpy.abs(out - ref) <= 2 * (K + 3) * U64 * (ab + c)).all()


@pytest.mark.parametrize("M,N,K,batch", [
    (1, 1, 1, 1), (32, 257, 16, 2), (33, 256, 17, 1), (64, 300, 32, 1),
    (65, 512, 33, 3), (96, 96, 64, 1), (128, 289, 80, 1), (129, 257, 96, 1),
    (160, 300, 95, 1), (192, 520, 160, 2), (193, 257, 48, 1),
    (224, 224, 64, 1), (225, 300, 31, 1), (255, 511, 128, 1),
    (256, 256, 161, 1), (257, 64, 64, 1), (300, 128, 40, 1),
    (520, 192, 200, 9), (300, 32, 96, 2), (511, 416, 64, 9)])
def test_split_product_tile_and_k_edges(M, N, K, batch):
    """Integers below 2^8 are exact in bf16 and their sums in FP32: equal to
    the last bit.  Normal numbers: the split leaves 2^-18 of an operand, the
    dropped lo*lo 2^-18 of a product, FP32 sums of 3 K terms."""
    out, ref, ab, c = _gemm(M, N, K, batch, "nt", "bf16x3", 1.0, 0.0, ints=9)
    assert numpy.array_equal(out, ref)
    out, ref, ab, c = _gemm(M, N, K, batch, "nt", "bf16x3", 0.5, 2.0)
    bound = (3 * 2.0 ** -17 + 3 * (K + 1) * U32) * ab + 4 * U64 * c
    assert (numpy.abs(out - ref) <= bound).all()


def test_engine_goes_on_after_a_failed_growth(monkeypatch):
    """A split product whose partial sums find no room fails with ENOMEM; the
    buffer that was there serves the next one."""
    from kelvin_amd._lib import FTCCError
    from kelvin_amd.engine import FTEngine
    d = dev()
    eng = FTEngine(2, 2, 1)

    def product(M, K):
        A = torch.randn(M, K, dtype=torch.float64, device=d)
        B = torch.randn(K, M, dtype=torch.float64, device=d)
        C = torch.zeros(M, M, dtype=torch.float64, device=d)
        eng.gemm(A, B, C, precision="fp64")
        assert bool(((C - A @ B).abs() <=
                     2 * (K + 3) * U64 * (A.abs() @ B.abs())).all())
    held = eng.workspace_bytes()
    monkeypatch.setenv("FTCC_CONTEXT_GB", repr((held + 4096) / 2.0 ** 30))
    with pytest.raises(FTCCError, match="FTCC_CONTEXT_GB"):
        product(512, 16384)
    assert eng.workspace_bytes() == held
    product(30, 3000)
    monkeypatch.delenv("FTCC_CONTEXT_GB")
    product(512, 16384)
    assert eng.workspace_bytes() > held
    eng.close()


@pytest.mark.parametrize("precision,K", [("fp64", 1023), ("fp64", 1030),
                                         ("fp32", 1030)])
@pytest.mark.parametrize("layout", ["nn", "tt"])
def test_gemm_of_1024_wide_tiles(layout, precision, K):
    """One product of 1024 128x128 tiles, which long K takes: rounding of
    two FP64 sums as above; FP32: of the operands and of a sum of K."""
    from kelvin_amd.engine import FTEngine
    d = dev()
    M, N = 4090, 4081
    A = torch.randn(M, K, dtype=torch.float64, device=d)
    B = torch.randn(K, N, dtype=torch.float64, device=d)
    C = torch.randn(M, N, dtype=torch.float64, device=d)
    ref = 0.75 * (A @ B) - 0.5 * C
    bound = 0.75 * (A.abs() @ B.abs()) + 0.5 * C.abs()
    if layout == "tt":
        A, B = A.t().contiguous().t(), B.t().contiguous().t()
    eng = FTEngine(2, 2, 1)
    eng.gemm(A, B, C, alpha=0.75, beta=-0.5, precision=precision)
    u = 2 * U64 if precision == "fp64" else U32
    assert bool(((C - ref).abs() <= (K + 3) * u * bound).all())
    eng.close()


@pytest.mark.parametrize("precision", ["fp64", "bf16x3"])
@pytest.mark.parametrize("spin", [True, False])
def test_engine_goes_on_after_any_failed_allocation(spin, precision,
                                                    monkeypatch):
    """Integrals, residual and a propagation step with memory that ends
    somewhere on the way, then again with enough: what was allocated before
    the failure is complete or taken again."""
    from kelvin_amd._lib import FTCCError
    from kelvin_amd.engine import FTEngine
    from kelvin_amd.ov_blocks import one_e_blocks, two_e_blocks
    d = dev()
    ng = 3
    rng = numpy.random.default_rng(8)
    no, nv, (F, I, t1, t2, lo, lv) = _run_problem(((2, 3), (5, 4)), ng, rng)
    T1, T2 = (torch.as_tensor(x, device=d) for x in (t1, t2))
    one = one_e_blocks(**{k: F[k] for k in ('oo', 'ov', 'vo', 'vv')})
    two = two_e_blocks(**{k: I[k] for k in I})

    def use(eng):
        eng.set_blocks(one, two)
        eng.set_denominators(numpy.ones((nv, no)),
                             numpy.ones((nv, nv, no, no)))
        eng.set_grid(numpy.zeros(ng), numpy.zeros((ng, ng)))
        if spin:
            eng.set_spin(lo, lv)
        out = [torch.empty_like(T1), torch.empty_like(T2)]
        eng.residual(T1, T2, *out)
        out += [T1.clone(), T2.clone()]
        eng.td_step(out[2], out[3], 0.01, order=4)
        return [to_np(x) for x in out]
    eng = FTEngine(no, nv, ng, precision=precision)
    least = eng.workspace_bytes()
    ref = use(eng)
    most = eng.workspace_bytes()
    eng.close()
    for part in numpy.linspace(0.01, 0.99, 25):
        eng = FTEngine(no, nv, ng, precision=precision)
        with monkeypatch.context() as m:
            m.setenv("FTCC_CONTEXT_GB",
                     repr((least + part * (most - least)) / 2.0 ** 30))
            with pytest.raises(FTCCError, match="FTCC_CONTEXT_GB"):
                use(eng)
        for x, y in zip(use(eng), ref):
            assert rel(x, y) < 1e-13, part
        eng.close()


@pytest.mark.parametrize("M,N,K", [(3, 2, 2 ** 22 + 5),
                                   (2, 35, 2 ** 22 - 64)])
def test_split_product_of_long_rows(M, N, K):
    """Rows of 2^22 elements and more (and the longest below them): sums of
    few ones and twos, exact."""
    from kelvin_amd.engine import FTEngine
    d = dev()
    g = torch.Generator().manual_seed(K)
    A = torch.randint(-1, 2, (M, K), generator=g, dtype=torch.int8)
    B = torch.randint(-1, 2, (N, K), generator=g, dtype=torch.int8)
    A[:, 0], B[:, 0], A[:, -1], B[:, -1] = 2, 1, 1, 2
    A, B = A.to(d).double(), B.to(d).double()
    ref = A @ B.t()
    assert float(ref.abs().max()) < 2 ** 22
    C = torch.zeros(M, N, dtype=torch.float64, device=d)
    eng = FTEngine(2, 2, 1)
    eng.gemm(A, B.t(), C, precision="bf16x3")
    assert torch.equal(C, ref)
    eng.close()


@pytest.mark.parametrize("layout", ["nn", "tn", "nt", "tt"])
@pytest.mark.parametrize("M,N,K,batch", [(70, 65, 127, 1), (64, 64, 129, 2),
                                         (33, 130, 4100, 1),
                                         (260, 300, 1000, 3)])
def test_fp32_products_add_up_in_fp64(M, N, K, batch, layout):
    """Products of 1 and 1 + 2^-17: sums of 128 of them are exact in FP32 and
    of any number in FP64, while one FP32 sum loses the 2^-17 from 256 terms
    on.  Equal to the last bit."""
    from kelvin_amd.engine import FTEngine
    d = dev()
    x = 1.0 + 2.0 ** -17

    def ones(r, c, t):
        a = torch.ones(batch, c, r, dtype=torch.float64, device=d)
        return a.transpose(1, 2) if t == "t" else a.reshape(batch, r, c)
    eng = FTEngine(2, 2, 1)
    for plan in ((0, 1024), (1, 1024), (2, 2048)):
        eng.set_gemm_plan(*plan)
        C = torch.zeros(batch, M, N, dtype=torch.float64, device=d)
        eng.gemm(ones(M, K, layout[0]), x * ones(K, N, layout[1]), C,
                 precision="fp32")
        assert bool((C == K * x).all()), plan
    eng.close()


def test_fp32_residual_adds_up_in_fp64():
    """The same through a ring product of the spin-blocked residual: only
    <mb||ej> of four beta indices (1 + 2^-17) and opposite-spin amplitudes
    (1), so that R2 is a sum of 1024 equal terms."""
    from kelvin_amd.engine import FTEngine
    from kelvin_amd.engine import ONE_E, TWO_E
    from kelvin_amd.ov_blocks import one_e_blocks, two_e_blocks
    d = dev()
    n, h = 64, 32
    x = 1.0 + 2.0 ** -17
    F = {k: torch.zeros(n, n, dtype=torch.float64, device=d) for k in ONE_E}
    I = {k: torch.zeros(n, n, n, n, dtype=torch.float64, device=d)
         for k in TWO_E}
    I["vovo"][h:, h:, h:, h:] = -x
    t1 = torch.zeros(1, n, n, dtype=torch.float64, device=d)
    t2 = torch.zeros(1, n, n, n, n, dtype=torch.float64, device=d)
    for a, b, s in ((0, h, 1.0), (h, 0, -1.0)):
        t2[:, a:a + h, b:b + h, :h, h:] = s
        t2[:, a:a + h, b:b + h, h:, :h] = -s
    eng = FTEngine(n, n, 1, precision="fp32")
    eng.set_blocks(one_e_blocks(**F), two_e_blocks(**I))
    eng.set_denominators(torch.ones(n, n, dtype=torch.float64, device=d),
                         torch.ones(n, n, n, n, dtype=torch.float64,
                                    device=d))
    eng.set_grid(numpy.zeros(1), numpy.zeros((1, 1)))
    lab = numpy.repeat([0, 1], h)
    eng.set_spin(lab, lab)
    b1, b2 = torch.empty_like(t1), torch.empty_like(t2)
    eng.residual(t1, t2, b1, b2)
    r = b2[0, :h, h:, :h, h:]
    assert bool((r.abs() == h * h * x).all())
    eng.close()


# (alpha, beta) occupied and virtual orbitals: (v, o) classes of 31, 32, 33,
# 64, 65 pairs, runs of 31 to 33 orbitals, unequal and empty runs
_RUNS = [((1, 2), (31, 16)), ((3, 4), (11, 8)), ((5, 5), (13, 13)),
         ((2, 8), (4, 8)), ((3, 0), (5, 4)), ((33, 2), (2, 3)),
         ((2, 1), (33, 32)), ((4, 4), (8, 8)), ((1, 1), (1, 1)),
         ((0, 3), (5, 4)), ((3, 2), (0, 4)), ((0, 2), (0, 5))]


def _run_problem(runs, ng, rng):
    (oa, ob), (va, vb) = runs
    lab = numpy.repeat([0, 1, 0, 1], [oa, ob, va, vb])
    return (oa + ob, va + vb,
            _spin_problem(oa + ob, va + vb, ng, lab, rng))


def _run_engine(F, I, no, nv, ng, lo, lv, prec):
    from kelvin_amd.engine import FTEngine
    from kelvin_amd.ov_blocks import one_e_blocks, two_e_blocks
    eng = FTEngine(no, nv, ng, precision=prec)
    eng.set_blocks(one_e_blocks(**{k: F[k] for k in ('oo', 'ov', 'vo', 'vv')}),
                   two_e_blocks(**{k: I[k] for k in I}))
    eng.set_denominators(numpy.ones((nv, no)), numpy.ones((nv, nv, no, no)))
    eng.set_grid(numpy.zeros(ng), numpy.zeros((ng, ng)))
    eng.set_spin(lo, lv)
    return eng


@pytest.mark.parametrize("workspace", [None, "0.0001"])
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-5),
                                      ("bf16x3", 2e-4)])
@pytest.mark.parametrize("runs", _RUNS)
def test_blocked_residual_at_class_and_run_edges(prec, tol, runs, workspace,
                                                 monkeypatch):
    """Products, grouped contractions and the doubles assembly of the
    spin-blocked residual, all grid points at once and one at a time; the
    tolerances of the residual tests of these precisions."""
    d = dev()
    ng = 2
    if workspace:
        monkeypatch.setenv("FTCC_WORKSPACE_GB", workspace)
    rng = numpy.random.default_rng(sum(map(sum, runs)))
    no, nv, (F, I, t1, t2, lo, lv) = _run_problem(runs, ng, rng)
    ref1, ref2 = oracle.residual_tbar(F, I, t1, t2)
    eng = _run_engine(F, I, no, nv, ng, lo, lv, prec)
    T1, T2 = (torch.as_tensor(x, device=d) for x in (t1, t2))
    b1, b2 = torch.empty_like(T1), torch.empty_like(T2)
    eng.residual(T1, T2, b1, b2)
    assert rel(to_np(b1), ref1) < tol
    assert rel(to_np(b2), ref2) < tol
    eng.close()


def test_propagation_after_a_longer_grid():
    """Propagation steps with one slice and then, on the same engine, with
    five: every slice like the single one, to rounding."""
    d = dev()
    rng = numpy.random.default_rng(2)
    no, nv, (F, I, t1, t2, lo, lv) = _run_problem(((2, 3), (5, 4)), 1, rng)
    eng = _run_engine(F, I, no, nv, 1, lo, lv, "fp64")
    one = [torch.as_tensor(x, device=d) for x in (t1, t2)]
    five = [torch.cat([x] * 5) for x in one]
    eng.td_step(*one, 0.01, order=4)
    eng.set_grid(numpy.zeros(5), numpy.zeros((5, 5)))
    eng.td_step(*five, 0.01, order=4)
    for x, y in zip(one, five):
        for k in range(5):
            assert rel(to_np(y[k]), to_np(x[0])) < 1e-13
    eng.close()


# compositions of one (no, nv): the classes of the second need longer operand
# slots than those of the first, a longer operand set in the third pair
_RELABEL = [[((3, 4), (11, 8)), ((3, 4), (10, 9))],
            [((7, 7), (12, 12)), ((8, 6), (11, 13)), ((7, 7), (12, 12))],
            [((2, 2), (4, 4)), ((4, 0), (3, 5)), ((1, 3), (6, 2))]]


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-5),
                                      ("bf16x3", 2e-4)])
@pytest.mark.parametrize("runs", _RELABEL)
def test_one_engine_takes_other_compositions(prec, tol, runs):
    """One engine given system after system of the same (no, nv) that divide
    differently between the spins, then other labels of the same blocks (the
    spins exchanged: no runs any more); the tolerances of the residual."""
    from kelvin_amd.ov_blocks import one_e_blocks, two_e_blocks
    d = dev()
    ng = 2
    rng = numpy.random.default_rng(sum(map(sum, runs[0])))
    eng = None
    for k, r in enumerate(runs):
        no, nv, (F, I, t1, t2, lo, lv) = _run_problem(r, ng, rng)
        if eng is None:
            eng = _run_engine(F, I, no, nv, ng, lo, lv, prec)
        else:
            eng.set_blocks(
                one_e_blocks(**{k: F[k] for k in ('oo', 'ov', 'vo', 'vv')}),
                two_e_blocks(**{k: I[k] for k in I}))
            eng.set_spin(lo, lv)
        ref1, ref2 = oracle.residual_tbar(F, I, t1, t2)
        T1, T2 = (torch.as_tensor(x, device=d) for x in (t1, t2))
        for labels in ((lo, lv), (1 - lo, 1 - lv)):
            eng.set_spin(*labels)
            b1, b2 = torch.empty_like(T1), torch.empty_like(T2)
            eng.residual(T1, T2, b1, b2)
            assert rel(to_np(b1), ref1) < tol, (k, labels)
            assert rel(to_np(b2), ref2) < tol, (k, labels)
    eng.close()


@pytest.mark.parametrize("first", ["fp64", "fp32"])
def test_precision_switches_keep_the_chunk(first):
    """FP32 and FP64 residuals in turn on one engine: the chunk stays (all
    grid points here) and every result is that of its precision; tolerances
    of the residual."""
    d = dev()
    ng = 6
    rng = numpy.random.default_rng(3)
    no, nv, (F, I, t1, t2, lo, lv) = _run_problem(((5, 5), (13, 13)), ng, rng)
    ref1, ref2 = oracle.residual_tbar(F, I, t1, t2)
    eng = _run_engine(F, I, no, nv, ng, lo, lv, first)
    T1, T2 = (torch.as_tensor(x, device=d) for x in (t1, t2))
    b1, b2 = torch.empty_like(T1), torch.empty_like(T2)
    for prec in (first, "fp64", "fp32", "fp64", "bf16x3", "fp32", "fp64"):
        eng.set_precision(prec)
        eng.residual(T1, T2, b1, b2)
        tol = {"fp64": 1e-12, "fp32": 1e-5, "bf16x3": 2e-4}[prec]
        assert rel(to_np(b1), ref1) < tol, prec
        assert rel(to_np(b2), ref2) < tol, prec
        if prec != "bf16x3":
            assert eng.chunk() == ng, prec
    eng.close()


@pytest.mark.parametrize("workspace,cache", [(None, "64"), (None, "0"),
                                             ("0.0001", "0")])
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("bf16x3", 2e-4)])
@pytest.mark.parametrize("runs", [r for r in _RUNS if sum(r[1]) < 60])
def test_blocked_adjoint_at_class_and_run_edges(prec, tol, runs, workspace,
                                                cache, monkeypatch):
    """The transposed residual over spin blocks against the oracle's, with
    the intermediates kept and rebuilt, and with little scratch; tolerances
    as for the residual.  The bf16x3 form takes every product whatever its
    size."""
    d = dev()
    ng = 3
    monkeypatch.setenv("FTCC_ADJOINT_CACHE_GB", cache)
    monkeypatch.setenv("FTCC_ADJOINT_LOWP_MIN_GFLOP", "0")
    if workspace:
        monkeypatch.setenv("FTCC_WORKSPACE_GB", workspace)
    rng = numpy.random.default_rng(7 + sum(map(sum, runs)))
    no, nv, (F, I, t1, t2, lo, lv) = _run_problem(runs, ng, rng)
    v1 = rng.normal(size=t1.shape) * (lv[:, None] == lo[None, :])
    v2 = antisym(rng.normal(size=t2.shape)) * (
        (lv[:, None, None, None] + lv[None, :, None, None]) ==
        (lo[None, None, :, None] + lo[None, None, None, :]))
    ref1, ref2 = _adjoint_reference(F, I, t1, t2, v1, v2)
    eng = _run_engine(F, I, no, nv, ng, lo, lv, "fp64")
    T1, T2, V1, V2 = (torch.as_tensor(x, device=d) for x in (t1, t2, v1, v2))
    eng.adjoint_begin(T1, T2)
    eng.adjoint_precision(prec)
    G1, G2 = eng.empty_amplitudes()
    eng.adjoint_apply(V1, V2, G1, G2)
    eng.adjoint_end()
    assert rel(to_np(G1), ref1) < tol
    assert rel(to_np(G2), ref2) < tol
    if prec == "bf16x3":
        assert max(rel(to_np(G1), ref1), rel(to_np(G2), ref2)) > 1e-12
    eng.close()


def _adjoint_reference(F, I, t1, t2, v1, v2):
    ref1, ref2 = numpy.empty_like(v1), numpy.empty_like(v2)
    for y in range(len(v1)):
        g1, g2 = oracle.stanton_rhs_transpose(F, I, t1[y], t2[y], v1[y],
                                              v2[y])
        ref1[y], ref2[y] = g1, oracle.antisymmetrize(g2)
    return ref1, ref2


@pytest.mark.parametrize("cache", ["64", "0"])
def test_adjoint_after_other_labels(cache, monkeypatch):
    """Three kinds of orbitals that every block conserves; the second kind
    counts as beta or as alpha, so that the pair classes of one problem have
    two sets of lengths (128 and 192 ring pairs).  J^T after each relabelling
    and with blocking off, against the oracle; tolerance of the adjoint."""
    d = dev()
    ng, o, v = 3, (4, 2, 1), (7, 4, 2)
    monkeypatch.setenv("FTCC_ADJOINT_CACHE_GB", cache)
    rng = numpy.random.default_rng(11)
    no, nv = sum(o), sum(v)
    kind = numpy.repeat([0, 1, 2, 0, 1, 2], o + v)
    # equal sums of 4^kind: the same kinds on both sides of a block
    F, I, t1, t2, _, _ = _spin_problem(no, nv, ng, 4 ** kind, rng)
    ko, kv = 4 ** kind[:no], 4 ** kind[no:]
    v1 = rng.normal(size=t1.shape) * (kv[:, None] == ko[None, :])
    v2 = antisym(rng.normal(size=t2.shape)) * (
        (kv[:, None, None, None] + kv[None, :, None, None]) ==
        (ko[None, None, :, None] + ko[None, None, None, :]))
    ref1, ref2 = _adjoint_reference(F, I, t1, t2, v1, v2)
    as_beta, as_alpha = (kind >= 1).astype(int), (kind >= 2).astype(int)
    eng = _run_engine(F, I, no, nv, ng, as_beta[:no], as_beta[no:], "fp64")
    T1, T2, V1, V2 = (torch.as_tensor(x, device=d) for x in (t1, t2, v1, v2))
    eng.adjoint_begin(T1, T2)
    for lab in (as_beta, as_alpha, None, as_beta, 1 - as_alpha):
        if lab is None:
            eng.set_spin(None, None)
        else:
            eng.set_spin(lab[:no], lab[no:])
        G1, G2 = eng.empty_amplitudes()
        eng.adjoint_apply(V1, V2, G1, G2)
        assert rel(to_np(G1), ref1) < 1e-12, lab
        assert rel(to_np(G2), ref2) < 1e-12, lab
    # kept intermediates stay FP64 when rebuilt by a low-precision application
    monkeypatch.setenv("FTCC_ADJOINT_LOWP_MIN_GFLOP", "0")
    eng.adjoint_end()
    eng.set_spin(as_beta[:no], as_beta[no:])
    eng.adjoint_begin(T1, T2)
    eng.set_spin(as_alpha[:no], as_alpha[no:])
    for prec, tol in (("bf16x3", 2e-4), ("fp64", 1e-12)):
        eng.adjoint_precision(prec)
        eng.adjoint_apply(V1, V2, G1, G2)
        assert rel(to_np(G1), ref1) < tol, prec
        assert rel(to_np(G2), ref2) < tol, prec
    eng.adjoint_end()
    eng.close()


@pytest.mark.parametrize("cache", ["64", "0"])
@pytest.mark.parametrize("prec", ["fp64", "bf16x3"])
def test_adjoint_in_little_memory(prec, cache, monkeypatch):
    """J^T wherever one grid point at a time has room: with memory between
    what one point at a time and what all of them take, begin and apply go on
    with fewer points (the operand copies and partial sums of an application
    are allocated at its first launch).  Equal to the unbounded result up to
    the order of sums."""
    d = dev()
    ng = 7
    monkeypatch.setenv("FTCC_ADJOINT_CACHE_GB", cache)
    monkeypatch.setenv("FTCC_ADJOINT_LOWP_MIN_GFLOP", "0")
    rng = numpy.random.default_rng(5)
    no, nv, (F, I, t1, t2, lo, lv) = _run_problem(((6, 6), (12, 12)), ng, rng)
    v1 = rng.normal(size=t1.shape) * (lv[:, None] == lo[None, :])
    v2 = antisym(rng.normal(size=t2.shape)) * (
        (lv[:, None, None, None] + lv[None, :, None, None]) ==
        (lo[None, None, :, None] + lo[None, None, None, :]))
    T1, T2, V1, V2 = (torch.as_tensor(x, device=d) for x in (t1, t2, v1, v2))

    def apply():
        eng = _run_engine(F, I, no, nv, ng, lo, lv, "fp64")
        eng.adjoint_begin(T1, T2)
        eng.adjoint_precision(prec)
        G1, G2 = eng.empty_amplitudes()
        eng.adjoint_apply(V1, V2, G1, G2)
        eng.adjoint_apply(V1, V2, G1, G2)
        held = eng.workspace_bytes()
        eng.adjoint_end()
        eng.close()
        return held, to_np(G1), to_np(G2)
    every, ref1, ref2 = apply()
    with monkeypatch.context() as m:
        m.setenv("FTCC_WORKSPACE_GB", "0.0001")
        one, g1, g2 = apply()
    assert one < every
    for part in (0.001, 0.05, 0.2, 0.4, 0.6, 0.8, 0.9, 0.95, 0.99):
        with monkeypatch.context() as m:
            m.setenv("FTCC_CONTEXT_GB",
                     repr((one + part * (every - one)) / 2.0 ** 30))
            held, g1, g2 = apply()
        assert held < every
        assert rel(g1, ref1) < 1e-13 and rel(g2, ref2) < 1e-13, part


@pytest.mark.parametrize("quad", ['lin', 'mid', 'L'])
@pytest.mark.parametrize("ng", [3, 5, 7, 9, 17, 33])
def test_adjoint_recurrence_lengths(quad, ng):
    """Batches of eight slices, remainders and grids shorter than one:
    sums of ng terms of at most unit weight, a few ng u."""
    from kelvin_amd import quadrature
    from kelvin_amd.engine import FTEngine
    d = dev()
    rng = numpy.random.default_rng(ng)
    n = 3
    ti, g, G = quadrature.ft_quad(ng, 4.0, quad)
    en = numpy.sort(rng.uniform(-1, 1, n))
    eng = FTEngine(n, n, ng)
    eri = fs.random_antisym(n, rng, hermitian=True) * 0.1
    eng.set_system(en, numpy.diag(en), eri, 4.0, 0.0)
    eng.set_grid(ti, G)
    l1, l2 = rng.normal(size=(ng, n, n)), rng.normal(size=(ng, n, n, n, n))
    L1, L2 = (torch.as_tensor(x, device=d) for x in (l1, l2))
    O1, O2 = eng.empty_amplitudes()
    eng.integrate_adjoint(L1, L2, O1, O2)
    assert rel(to_np(O1), oracle.int_adjoint(
        ng, l1, ti, oracle.D1(en, en), G)) < 1e-13
    assert rel(to_np(O2), oracle.int_adjoint(
        ng, l2, ti, oracle.D2(en, en), G)) < 1e-13
    eng.close()
