"""Blocks of few columns at their own width (the uneven batch's step on the
single model) against the 64-wide block step, which a fixed block width
selects: gather-mode moments bitwise, doubling moments and traces up to the
order of their FP64 dot sums (2 n rows eps, with |mu| <= 1: 1e-11 here). Also
the dot sums gathered over several steps between reductions.
"""
import numpy as np
import pytest

from tbtk_amd import engine as X
from tbtk_amd import lattice as L

pytestmark = pytest.mark.gpu

MODELS = {
    4: (lambda: L.honeycomb_ribbon(9, 14, disorder=0.5, seed=1), 9.2),
    6: (lambda: L.square_spin(17, 13, disorder=1.0, seed=2), 6.0),
    7: (lambda: L.cubic(9, 8, 7, disorder=1.0, seed=3), 7.5),
    "complex": (lambda: L.square(19, 23, disorder=0.5, seed=4, flux=0.03), 5.0),
}


@pytest.fixture
def eng(engine):
    yield engine
    engine.set_option(X.OPT_BLOCK_WIDTH, 0)


def both(eng, call):
    got = call()
    eng.set_option(X.OPT_BLOCK_WIDTH, 64)
    ref = call()
    eng.set_option(X.OPT_BLOCK_WIDTH, 0)
    return got, ref


@pytest.mark.parametrize("n", [1, 2, 3, 5, 13, 26, 37, 64, 65, 130, 190, 193, 261, 300])
@pytest.mark.parametrize("model", list(MODELS))
def test_narrow_block(eng, model, n):
    make, s = MODELS[model]
    m = make()
    eng.set_csr(m.csr(), s)
    sites = np.random.default_rng(n).integers(0, m.basis_size, n)
    print(f"{m.name}: N={m.basis_size} sites={n}", flush=True)
    got, ref = both(eng, lambda: eng.moments_block(sites, 41, 0))
    assert np.array_equal(got, ref)
    for M in (1, 2, 70, 77):
        got, ref = both(eng, lambda: eng.moments_block(sites, M, X.DOUBLING))
        assert np.abs(got - ref).max() < 1e-11


@pytest.mark.parametrize("R", [1, 7, 32, 50, 64, 70, 96, 97, 133])
def test_narrow_trace(eng, R):
    m = L.cubic(9, 8, 7, disorder=1.0, seed=3)
    eng.set_csr(m.csr(), 7.5)
    got, ref = both(eng, lambda: eng.moments_trace(R, 11, 63, X.DOUBLING))
    assert np.abs(got - ref).max() < 1e-11 * R * m.basis_size


def test_batch_survives_narrow_blocks(eng):
    """The uneven batch and the single model share the step's work buffers."""
    a, b = L.square(20, 31, disorder=0.5, seed=1), L.honeycomb_ribbon(8, 11, disorder=0.5, seed=2)
    eng.multi_set([a.csr(), b.csr()], [5.0, 9.2])
    sites, moments = [np.arange(9), np.arange(3, 40)], [90, 41]
    first = eng.multi_moments(sites, moments, X.DOUBLING)
    big = L.cubic(12, 11, 10, disorder=1.0, seed=3)
    eng.set_csr(big.csr(), 7.5)
    eng.moments_block(np.arange(60), 50, X.DOUBLING)
    again = eng.multi_moments(sites, moments, X.DOUBLING)
    for x, y in zip(first, again):
        assert np.abs(x - y).max() < 1e-11
    for (x, m, s, st, M) in zip(first, (a, b), (5.0, 9.2), sites, moments):
        eng.set_csr(m.csr(), s)
        assert np.abs(x - eng.moments_block(st, M, X.DOUBLING)).max() < 1e-11


# The same of a real H with the step kernels chosen: by default such blocks run
# resident on both sides of the comparisons above.
@pytest.fixture
def steps(engine):
    engine.set_option(X.OPT_RESIDENT, 0)
    yield engine
    engine.set_option(X.OPT_BLOCK_WIDTH, 0)
    engine.set_option(X.OPT_RESIDENT, 1)


@pytest.mark.parametrize("n", [1, 2, 3, 5, 13, 26, 37, 64, 65, 130, 190, 193, 261, 300])
@pytest.mark.parametrize("model", [4, 6, 7])
def test_narrow_block_steps(steps, model, n):
    make, s = MODELS[model]
    m = make()
    steps.set_csr(m.csr(), s)
    sites = np.random.default_rng(n).integers(0, m.basis_size, n)
    print(f"{m.name}: N={m.basis_size} sites={n}", flush=True)
    got, ref = both(steps, lambda: steps.moments_block(sites, 41, 0))
    assert np.array_equal(got, ref)
    for M in (70, 77):
        got, ref = both(steps, lambda: steps.moments_block(sites, M, X.DOUBLING))
        assert np.abs(got - ref).max() < 1e-11


@pytest.mark.parametrize("R", [1, 7, 50, 64, 97])
def test_narrow_trace_steps(steps, R):
    m = L.cubic(9, 8, 7, disorder=1.0, seed=3)
    steps.set_csr(m.csr(), 7.5)
    got, ref = both(steps, lambda: steps.moments_trace(R, 11, 63, X.DOUBLING))
    assert np.abs(got - ref).max() < 1e-11 * R * m.basis_size


def test_batch_survives_narrow_block_steps(steps):
    test_batch_survives_narrow_blocks(steps)


def test_real_batch_steps(steps, oracle_mod):
    """The uneven batch's step on real models, two vectors per column, with a
    row count per group of its own each: bitwise the block step, and the oracle
    within the FP32 storage's 4 x 6e-8 sqrt(M)."""
    specs = [(L.square(9, 7, disorder=0.5, seed=1), 5.0, 3, 41), (L.square_spin(13, 11, disorder=1.0, seed=2), 6.0, 64, 64),
             (L.honeycomb_ribbon(12, 9, disorder=0.5, seed=4), 9.2, 33, 50),
             (L.square(30, 40, disorder=0.5, seed=6), 5.0, 1, 60)]
    sites = [np.random.default_rng(1).integers(0, m.basis_size, n) for m, _, n, _ in specs]
    moments = [x[3] for x in specs]
    steps.multi_set([x[0].csr() for x in specs], [x[1] for x in specs])
    got = {f: steps.multi_moments(sites, moments, f) for f in (0, X.DOUBLING)}
    for i, ((m, s, _, M), st) in enumerate(zip(specs, sites)):
        steps.set_csr(m.csr(), s)
        assert np.array_equal(got[0][i], steps.moments_block(st, M, 0))
        exact = np.array([oracle_mod.moments(m.csr(), s, int(b), [int(b)], M)[0] for b in st])
        for f in got:
            assert np.abs(got[f][i] - exact).max() <= 4 * 6e-8 * np.sqrt(M)
