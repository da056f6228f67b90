"""The plain recurrence with the vectors resident on the chip
(TBTKX_OPT_RESIDENT): bitwise the moments of the per-step kernels and of the
oracle's restatement of the reference's CPU recurrence
(Lib/src/Solver/ChebyshevExpander.cpp:65-82, 103-199), over models in one
workgroup and in chunks with halos, at the edges of rows per thread, with
every count of entries beside the diagonal, rows without a diagonal, real and
complex H, with and without the value palette.
"""
import numpy as np
import pytest

from tbtk_amd import engine as X
from tbtk_amd import lattice as L

pytestmark = pytest.mark.gpu


@pytest.fixture
def res(engine):
    yield engine
    for opt, v in ((X.OPT_RESIDENT, 1), (X.OPT_PALETTE, 1), (X.OPT_REAL, 1)):
        engine.set_option(opt, v)


def banded(n, offsets, seed, cplx=False, diag=True, distinct=True):
    """A hermitian band matrix with the given positive offsets; rows beyond
    the middle have no diagonal entry unless `diag`."""
    rng = np.random.default_rng(seed)
    r, c, v = [], [], []
    for o in offsets:
        if o >= n:
            continue
        i = np.arange(n - o)
        a = rng.uniform(-1, 1, n - o) if distinct else np.full(n - o, -0.7)
        a = a.astype(np.complex128)
        if cplx:
            a = a * np.exp(1j * rng.uniform(0, 6, n - o))
        r += [i, i + o]
        c += [i + o, i]
        v += [a, np.conj(a)]
    i = np.arange(n if diag else n // 2)
    r.append(i)
    c.append(i)
    v.append(rng.uniform(-1, 1, i.size).astype(np.complex128))
    return L.coo_to_csr(np.concatenate(r), np.concatenate(c), np.concatenate(v), n)


def check(eng, oracle_mod, csr, s, frm, to, M, oracle=True):
    n = csr[0].size - 1
    print(f"N={n} Z={csr[1].size} M={M}", flush=True)
    eng.set_csr(csr, s)
    got = eng.moments(frm, to, M)
    ran = eng.get_option(X.OPT_RESIDENT)
    eng.set_option(X.OPT_RESIDENT, 0)
    ref = eng.moments(frm, to, M)
    assert eng.get_option(X.OPT_RESIDENT) == 0
    eng.set_option(X.OPT_RESIDENT, 1)
    assert np.array_equal(got, ref)
    if oracle:
        assert np.array_equal(got, oracle_mod.moments(csr, s, frm, to, M))
    return ran


@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("half", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 1023, 1024, 1025, 2049, 3073])
def test_one_workgroup(res, oracle_mod, n, half, cplx):
    csr = banded(n, [1, 30, 31][:half], seed=n + half, cplx=cplx, diag=half != 2)
    to = sorted({0, n - 1, n // 2, min(n - 1, n // 2 + 31)})
    for M in (1, 2, 3, 40):
        ran = check(res, oracle_mod, csr, 8.0, n // 2, to, M)
    assert ran == 1 or n > 1024


@pytest.mark.parametrize("palette", [1, 0])
@pytest.mark.parametrize("cplx", [False, True], ids=["real", "complex"])
@pytest.mark.parametrize("n,offsets", [
    (20000, [1, 40]),            # several steps per exchange
    (20011, [1, 2, 97]),         # odd length, a short last chunk
    (9000, [3, 500]),            # chunks of a few halo widths
    (60000, [1]),
    (70003, [400, 401]),
    (30000, [1, 2, 3, 60]),      # 4 entries on either side
])
def test_chunks(res, oracle_mod, n, offsets, cplx, palette):
    csr = banded(n, offsets[:3], seed=n, cplx=cplx, distinct=not palette)
    res.set_option(X.OPT_PALETTE, palette)
    to = sorted({0, 1, n - 1, n // 2, n // 2 - offsets[-1], n // 3, *range(n // 2, n // 2 + 50)})
    for M in (2, 9, 133):
        check(res, oracle_mod, csr, 8.0, n // 2, to, M, oracle=M < 133 or n <= 30000)


def test_chunked_models_run_resident(res, oracle_mod):
    """The rule sends medium lattices to the chunked kernel and large bands
    back to the per-step kernels; graph replay and chosen step forms too."""
    m = L.square_spin(120, 70, disorder=1.0, seed=3)
    assert check(res, oracle_mod, m.csr(), 6.0, 8000, [0, 8000, 8001, 16799], 300) == 1
    m = L.square(100, 110, disorder=0.5, seed=3, flux=0.013)
    assert check(res, oracle_mod, m.csr(), 5.0, 5000, [0, 5000, 5110, 10999], 300) == 1
    m = L.ring(40000)   # periodic: the band is the whole matrix
    assert check(res, oracle_mod, m.csr(), 2.5, 7, [7, 8], 50, oracle=False) == 0
    m = L.square_spin(20, 20, disorder=1.0, seed=3)
    res.set_csr(m.csr(), 6.0)
    res.moments(3, [3], 30)
    assert res.get_option(X.OPT_RESIDENT) == 1
    for opt, v, back in ((X.OPT_GRAPH, 1, 0), (X.OPT_PLAIN_KERNEL, 0, 2), (X.OPT_SLOT_ROWS, 2, 0),
                         (X.OPT_ROW_PATTERNS, 2, 1)):
        res.set_option(opt, v)
        res.moments(3, [3], 30)
        assert res.get_option(X.OPT_RESIDENT) == 0
        res.set_option(opt, back)


def test_real_model_in_complex_arithmetic(res, oracle_mod):
    res.set_option(X.OPT_REAL, 0)
    m = L.nambu_swave(14, 13, disorder=0.5, seed=3)
    assert check(res, oracle_mod, m.csr(), 7.0, 300, [300, 301, 303, 0], 200) == 1


def test_many_targets_and_repeats(res, oracle_mod):
    m = L.honeycomb_ribbon(30, 12, disorder=0.5, seed=5)
    n = m.basis_size
    to = list(range(n)) + [5, 7]
    assert check(res, oracle_mod, m.csr(), 9.2, 700, to, 60) == 1


@pytest.mark.parametrize("flux", [0.0, 0.07])
def test_multi_in_one_launch(res, oracle_mod, flux):
    """tbtkx_moments_multi with a workgroup per start vector: more vectors
    than compute units, empty, repeated and unordered to-lists."""
    m = L.square(23, 19, disorder=0.5, seed=4, flux=flux)
    csr, n, M = m.csr(), m.basis_size, 77
    rng = np.random.default_rng(1)
    froms = rng.integers(0, n, 300)
    tos = [[int(f)] + [int(x) for x in rng.integers(0, n, rng.integers(0, 4))] for f in froms]
    tos[3] = []
    tos[10] = [9, 4, 9]
    res.set_csr(csr, 5.0)
    got = res.moments_multi(froms, tos, M)
    assert res.get_option(X.OPT_RESIDENT) == 1
    res.set_option(X.OPT_RESIDENT, 0)
    ref = res.moments_multi(froms, tos, M)
    for j in range(300):
        assert np.array_equal(got[j], ref[j]), j
    for j in (0, 10, 299):
        assert np.array_equal(got[j], oracle_mod.moments(csr, 5.0, int(froms[j]), tos[j], M))


def test_nan_and_infinite_entries(res):
    """A row that is not finite spreads as in the per-step kernels."""
    for bad in (np.nan, np.inf):
        for n in (900, 12000):
            rp, col, val = banded(n, [1, 33], seed=7)
            val = val.copy()
            val[rp[n // 2 + 200]] = bad
            res.set_csr((rp, col, val), 8.0)
            a = res.moments(n // 2, [n // 2, n // 2 + 60], 40)
            res.set_option(X.OPT_RESIDENT, 0)
            b = res.moments(n // 2, [n // 2, n // 2 + 60], 40)
            res.set_option(X.OPT_RESIDENT, 1)
            assert np.array_equal(a, b, equal_nan=True)


def cylinder(la, lb, orb, seed):
    """A square lattice that wraps within its layers of lb cells, with a
    diagonal bond, of `orb` states per cell: bonds beyond the layer's end."""
    rng = np.random.default_rng(seed)
    a, b, o = (x.ravel() for x in np.meshgrid(np.arange(la), np.arange(lb), np.arange(orb),
                                              indexing="ij"))
    here = (a * lb + b) * orb + o
    r, c, v = [here], [here], [rng.uniform(-1, 1, here.size).astype(np.complex128)]
    for da, db, t in ((0, 1, -1.0), (1, 0, -0.75), (1, 1, 0.25)):
        ok = a + da < la
        there = ((a + da) * lb + (b + db) % lb) * orb + o
        r += [here[ok], there[ok]]
        c += [there[ok], here[ok]]
        v += [np.full(ok.sum(), t, dtype=np.complex128)] * 2
    n = la * lb * orb
    return L.coo_to_csr(np.concatenate(r), np.concatenate(c), np.concatenate(v), n)


@pytest.mark.parametrize("real", [1, 0], ids=["real", "complex"])
@pytest.mark.parametrize("name,n,ran", [
    ("square_spin", (173, 61), 1), ("square_spin", (40, 701), 1), ("square_spin", (7, 3001), None),
    ("square_spin", (611, 613), 1), ("nambu", (97, 101), 1), ("nambu", (257, 260), 1),
    ("honeycomb", (40, 997), 1), ("honeycomb", (5, 2003), None), ("cubic", (31, 29, 37), 1),
    ("cubic", (93, 89, 71), None), ("square", (1021, 1019), None), ("cylinder", (61, 83), None),
    ("cylinder", (3, 5000), None), ("cylinder", (301, 700), None)])
def test_tiles(res, oracle_mod, name, n, ran, real):
    """Tiles of a lattice's layers, narrow and wide, with short last tiles and
    bonds that wrap: bitwise the per-step kernels; targets across the tiles."""
    f = {"square_spin": L.square_spin, "nambu": L.nambu_swave, "honeycomb": L.honeycomb_ribbon,
         "cubic": L.cubic, "square": L.square}
    csr = cylinder(*n, 2, seed=3) if name == "cylinder" else f[name](*n, disorder=0.5, seed=2).csr()
    N = csr[0].size - 1
    res.set_option(X.OPT_REAL, real)
    to = sorted({0, 1, N - 1, N // 2, N // 3, *range(N // 2, min(N, N // 2 + 3000), 2)})
    for M in (2, 3, 41):
        got = check(res, oracle_mod, csr, 9.2, N // 2 + 1, to, M, oracle=N < 100000 and M == 41)
        assert ran is None or not real or got == ran


def test_tiles_without_palette(res, oracle_mod):
    """Distinct values: the narrow tiles, or a launch per step where only the
    wide ones would fit."""
    m = L.square(300, 211, disorder=0.5, seed=3, flux=0.013)
    to = [0, 30000, 30001, 63299]
    assert check(res, oracle_mod, m.csr(), 5.0, 30000, to, 60) == 1
    csr = cylinder(211, 190, 1, seed=4)
    res.set_option(X.OPT_PALETTE, 0)
    assert check(res, oracle_mod, csr, 5.0, 9, [0, 9, 189, 190, 40089], 60) == 1


def test_two_handles_at_once(oracle_mod):
    """Threads with handles of their own whose workgroups exchange, narrow tiles
    beside wide ones and blocks: every call bitwise the handle's first."""
    import threading
    wrong, done = [], []

    def work(make, s, call):
        eng = X.Engine(0)
        m = make()
        eng.set_csr(m.csr(), s)
        first = call(eng, m.basis_size)
        for _ in range(20):
            if not np.array_equal(call(eng, m.basis_size), first):
                wrong.append(m.name)
        done.append(eng.get_option(X.OPT_RESIDENT))
        eng.close()

    plain = lambda eng, N: eng.moments(N // 2, [0, N // 2, N - 1], 300)
    block = lambda eng, N: eng.moments_block(np.arange(0, N, N // 37), 60, 0)
    jobs = [(lambda: L.square_spin(173, 61, disorder=0.5, seed=2), 6.0, plain),
            (lambda: L.square_spin(611, 613, disorder=0.5, seed=2), 6.0, plain),
            (lambda: L.honeycomb_ribbon(40, 997, disorder=0.5, seed=4), 9.2, block)]
    threads = [threading.Thread(target=work, args=j) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert wrong == [] and done == [1, 1, 1]
