"""FP32 blocks of a real H resident on the chip: unit vectors with gathered and
doubled moments, random phases and batches, against the step kernels
(TBTKX_OPT_RESIDENT 0) and the oracle, at models of one workgroup, of several
tiles, at the edges of 8 columns per team and of rows per thread, and models
that need several launches.

Tolerance: values are stored as FP32 after every step on both sides (2^-24
relative to the largest, 6e-8), and rounding errors of a Chebyshev recurrence
of M steps add to at most M of them, in practice to sqrt(M): 6e-8 sqrt(M) times 4.
"""
import numpy as np
import pytest

from tbtk_amd import engine as X
from tbtk_amd import lattice as L

pytestmark = pytest.mark.gpu


@pytest.fixture
def res(engine):
    yield engine
    engine.set_option(X.OPT_RESIDENT, 1)


def model(name, n):
    f = {"spin": L.square_spin, "nambu": L.nambu_swave, "honeycomb": L.honeycomb_ribbon,
         "square": L.square, "cubic": L.cubic}[name]
    s = {"spin": 6.0, "nambu": 7.0, "honeycomb": 9.2, "square": 5.0, "cubic": 7.5}[name]
    return f(*n, disorder=0.5, seed=4), s


def close(a, b, M, scale=1.0):
    assert np.isfinite(a).all()
    assert np.abs(a - b).max() <= 4 * 6e-8 * np.sqrt(M) * scale


SHAPES = [("square", (9, 7), 3), ("square", (512, 1), 8), ("spin", (16, 16), 9),
          ("nambu", (31, 33), 17), ("square", (64, 64), 65), ("honeycomb", (33, 32), 1),
          ("spin", (57, 61), 37), ("honeycomb", (7, 501), 12), ("cubic", (21, 23, 19), 20),
          ("nambu", (120, 131), 100), ("honeycomb", (40, 997), 37), ("spin", (520, 530), 16)]


@pytest.mark.parametrize("name,n,cols", SHAPES)
def test_blocks(res, oracle_mod, name, n, cols):
    m, s = model(name, n)
    N = m.basis_size
    print(name, N, cols, flush=True)
    res.set_csr(m.csr(), s)
    sites = np.random.default_rng(3).integers(0, N, cols)
    sites[0], sites[-1] = 0, N - 1
    for M, flags in ((2, 0), (3, X.DOUBLING), (41, 0), (64, X.DOUBLING), (63, X.DOUBLING)):
        a = res.moments_block(sites, M, flags)
        res.set_option(X.OPT_RESIDENT, 0)
        b = res.moments_block(sites, M, flags)
        res.set_option(X.OPT_RESIDENT, 1)
        close(a, b, M)
    if N < 20000:
        for j in (0, cols - 1):
            f = int(sites[j])
            close(a[j], oracle_mod.moments(m.csr(), s, f, [f], 63)[0], 63)


@pytest.mark.parametrize("name,n,R", [("square", (9, 7), 1), ("cubic", (21, 23, 19), 5),
                                      ("honeycomb", (40, 97), 32), ("square", (300, 301), 33),
                                      ("cubic", (60, 61, 62), 9)])
def test_random_phases(res, name, n, R):
    m, s = model(name, n)
    N = m.basis_size
    print(name, N, R, flush=True)
    res.set_csr(m.csr(), s)
    a = res.moments_trace(R, 11, 50)
    res.set_option(X.OPT_RESIDENT, 0)
    b = res.moments_trace(R, 11, 50)
    close(a, b, 50, N * R)


@pytest.mark.parametrize("doubling", [True, False])
def test_batch(res, doubling):
    rng = np.random.default_rng(5)
    specs, scales, sites, moments = [], [], [], []
    for i, (f, a, s) in enumerate([(L.square_spec, (20, 50), 5.0), (L.honeycomb_ribbon_spec, (23, 211), 9.2),
                                   (L.square_spec, (70, 901), 5.0), (L.honeycomb_ribbon_spec, (3, 5), 9.2)]):
        sp = f(*a, disorder=0.5, seed=i)
        specs.append(sp)
        scales.append(s)
        sites.append(np.sort(rng.choice(sp.basis_size, (8, 33, 64, 1)[i], replace=False)))
        moments.append((40, 61, 33, 20)[i])
    res.multi_set_lattices(specs, scales)
    a = res.multi_moments(sites, moments, X.DOUBLING if doubling else 0)
    res.set_option(X.OPT_RESIDENT, 0)
    b = res.multi_moments(sites, moments, X.DOUBLING if doubling else 0)
    for x, y, M in zip(a, b, moments):
        close(x, y, M)


def test_many_values_and_zero_entries(res):
    """Distinct bond values (no palette) keep the step kernels; explicit zeros
    and rows without a diagonal run resident."""
    n = 3000
    rng = np.random.default_rng(8)
    for distinct in (True, False):
        i = np.arange(n - 1)
        v = rng.uniform(-1, 1, n - 1) if distinct else np.where(i % 3 == 0, 0.0, -0.8)
        d = np.arange(n // 2)
        csr = L.coo_to_csr(np.concatenate([i, i + 1, d]), np.concatenate([i + 1, i, d]),
                           np.concatenate([v, v, rng.uniform(-1, 1, d.size)]).astype(complex), n)
        res.set_csr(csr, 4.0)
        a = res.moments_block([0, 5, n // 2, n - 1], 60, X.DOUBLING)
        res.set_option(X.OPT_RESIDENT, 0)
        b = res.moments_block([0, 5, n // 2, n - 1], 60, X.DOUBLING)
        res.set_option(X.OPT_RESIDENT, 1)
        close(a, b, 60)


# The two sides hold the same FP32 values (gathered moments are equal bit for
# bit); their dots differ in the order of N FP64 sums of products whose magnitudes
# add to at most 1 (|T_n| <= 1), twice in 2 <n|n> - mu_0: 4 N 2^-53.
def dots(N):
    return 4 * N * 2.0 ** -53


def sides(eng, call):
    """The resident result, which must have run so, and the step kernels'."""
    a = call()
    assert eng.get_option(X.OPT_RESIDENT) == 1
    eng.set_option(X.OPT_RESIDENT, 0)
    b = call()
    assert eng.get_option(X.OPT_RESIDENT) == 0
    eng.set_option(X.OPT_RESIDENT, 1)
    return a, b


MANY = ((41, 0), (64, X.DOUBLING), (63, X.DOUBLING))
FEW = ((3, 0), (3, X.DOUBLING), (4, X.DOUBLING))   # two steps


@pytest.mark.parametrize("name,n,cols,moments", [
    ("square", (9, 7), 3, MANY), ("cubic", (9, 8, 7), 40, MANY), ("nambu", (31, 33), 17, MANY),
    ("square", (64, 64), 65, MANY), ("spin", (57, 61), 37, MANY), ("honeycomb", (7, 501), 12, MANY),
    ("nambu", (120, 131), 100, MANY), ("honeycomb", (40, 997), 37, MANY),
    ("spin", (520, 530), 16, MANY), ("honeycomb", (500, 500), 9, MANY),
    ("honeycomb", (32, 32), 2048, FEW), ("nambu", (32, 32), 2048, FEW),
    ("square", (63, 65), 2041, FEW), ("spin", (1024, 500), 16, ((11, 0), (21, X.DOUBLING)))])
def test_blocks_that_run_resident(res, name, n, cols, moments):
    """One workgroup, tiles of few and of all rows per thread, one and two passes,
    many steps and two."""
    m, s = model(name, n)
    N = m.basis_size
    print(name, N, cols, flush=True)
    res.set_csr(m.csr(), s)
    sites = np.random.default_rng(3).integers(0, N, cols)
    sites[0], sites[-1] = 0, N - 1
    for M, flags in moments:
        a, b = sides(res, lambda: res.moments_block(sites, M, flags))
        if flags == 0:
            assert np.array_equal(a, b), M
        else:
            assert np.abs(a - b).max() <= dots(N), M


@pytest.mark.parametrize("name,n,R", [
    ("square", (9, 7), 1), ("cubic", (9, 8, 7), 40), ("nambu", (120, 131), 50),
    ("spin", (200, 211), 24), ("square", (300, 301), 33)])
def test_random_phases_that_run_resident(res, name, n, R):
    m, s = model(name, n)
    N = m.basis_size
    print(name, N, R, flush=True)
    res.set_csr(m.csr(), s)
    a, b = sides(res, lambda: res.moments_trace(R, 11, 50))
    assert np.abs(a - b).max() <= dots(N) * N * R


def test_which_matrices_run_resident(res):
    """Bond values of more than a palette don't, few with explicit zeros do."""
    n = 3000
    i, d = np.arange(n - 1), np.arange(n // 2)
    rng = np.random.default_rng(8)
    for v, ran in ((rng.uniform(-1, 1, n - 1), 0), (np.where(i % 3 == 0, 0.0, -0.8), 1)):
        csr = L.coo_to_csr(np.concatenate([i, i + 1, d]), np.concatenate([i + 1, i, d]),
                           np.concatenate([v, v, rng.uniform(-1, 1, d.size)]).astype(complex), n)
        res.set_csr(csr, 4.0)
        res.moments_block([0, 5, n // 2, n - 1], 60, X.DOUBLING)
        assert res.get_option(X.OPT_RESIDENT) == ran


def test_calls_that_would_lose_keep_the_steps(res):
    """Eight passes of four steps with dots, and a batch whose steps are fewer than
    its launches are worth."""
    m, s = model("spin", (1024, 500))
    res.set_csr(m.csr(), s)
    res.moments_block(np.arange(64), 8, X.DOUBLING)
    assert res.get_option(X.OPT_RESIDENT) == 0
    specs = [L.square_spec(*z, disorder=0.5, seed=i) for i, z in enumerate([(600, 600), (500, 400), (30, 30)])]
    res.multi_set_lattices(specs, [5.0] * 3)
    res.multi_moments([np.arange(64)] * 3, [3, 13, 23], X.DOUBLING)
    assert res.get_option(X.OPT_RESIDENT) == 0
