"""How many launches a call makes, counted between the engine and the HIP runtime."""
import pytest

from shim import run_shimmed

pytestmark = pytest.mark.gpu


def test_narrow_blocks_are_tuned_once(tmp_path):
    """A block of few columns times its launch shapes on the first call only: not
    again for the same call, where the columns run in two parts of different
    widths (65 and 91), nor for another number of moments. A part makes 2
    launches for the start vectors, one per step and 2 per 16 steps; a trial of
    12 shapes makes 96."""
    run_shimmed(tmp_path, """
m = L.square(19, 23, disorder=0.5, seed=4, flux=0.03)
eng.set_csr(m.csr(), 5.0)
count = value("shim_launches")
for n, parts in ((37, 1), (65, 2), (91, 2)):
    sites = np.arange(n)
    eng.moments_block(sites, 60, X.DOUBLING)
    for M in (60, 62, 64):
        count.value = 0
        eng.moments_block(sites, M, X.DOUBLING)
        print(n, M, count.value, flush=True)
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
