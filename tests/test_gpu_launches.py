"""How many launches a call makes, counted between the engine and the HIP runtime."""
import pytest

from shim import run_shimmed

pytestmark = pytest.mark.gpu


def test_narrow_blocks_are_tuned_once(tmp_path):
    """A block of few columns times its launch shapes on the first call only: not
    again for the same call, where the columns run in two parts of different
    widths (65 and 91), nor for another number of moments. A part makes 2
    launches for the start vectors, one per step and 2 per 16 steps; a trial of
    6 shapes makes 48."""
    run_shimmed(tmp_path, """
m = L.square(300, 301, disorder=0.5, seed=4, flux=0.03)
eng.set_csr(m.csr(), 5.0)
count = value("shim_launches")
for n, parts in ((37, 1), (65, 2), (91, 2)):
    sites = np.arange(n)
    eng.moments_block(sites, 60, X.DOUBLING)
    for M in (60, 62, 64):
        count.value = 0
        eng.moments_block(sites, M, X.DOUBLING)
        print(n, M, count.value, flush=True)
        assert eng.last_timing()[1] == parts * (M // 2)
        assert 0 < count.value <= parts * 40, (n, M, count.value)
""")


def test_many_small_models_are_not_scanned(tmp_path):
    """A batch whose models could never pay for a resident launch each isn't
    looked over for one: the first call's launches are the step path's."""
    run_shimmed(tmp_path, """
specs = [L.square_spec(5, 4 + i % 3, disorder=0.5, seed=i) for i in range(300)]
count, got = value("shim_launches"), []
for resident in (1, 0):
    eng = X.Engine(0)
    eng.set_option(X.OPT_RESIDENT, resident)
    eng.multi_set_lattices(specs, [5.0] * 300)
    count.value = 0
    got.append(eng.multi_moments([np.arange(3)] * 300, [40] * 300, X.DOUBLING))
    got.append(count.value)
assert got[1] == got[3], (got[1], got[3])
for a, b in zip(got[0], got[2]):
    assert np.abs(a - b).max() < 1e-12
""")


def test_blocks_that_narrow_parts_would_slow_down(tmp_path):
    """A few steps, or few rows and more than 64 columns, run in one wide block: no
    second part's launches. Resident blocks are off, columns complex."""
    run_shimmed(tmp_path, """
eng.set_option(X.OPT_RESIDENT, 0)
m = L.square(60, 60, disorder=0.5, seed=4, flux=0.03)
eng.set_csr(m.csr(), 5.0)
for n, M, flags in ((1, 2, 0), (64, 4, X.DOUBLING), (65, 200, X.DOUBLING), (96, 101, 0),
                    (224, 200, X.DOUBLING)):
    eng.moments_block(np.arange(n), M, flags)
    S = (M + 1) // 2 if flags else M - 1
    steps, width = eng.last_timing()[1], eng.get_option(X.OPT_BLOCK_WIDTH)
    print(n, M, steps, width, flush=True)
    assert steps == S * -(-n // width), (n, M)
""")
