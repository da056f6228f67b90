"""What the engine reports of the last call (options read back, steps timed) is
what that call ran, with resident recurrences and blocks of few columns among the
forms."""
import numpy as np
import pytest

from tbtk_amd import engine as X
from tbtk_amd import lattice as L

pytestmark = pytest.mark.gpu


@pytest.fixture
def eng():
    e = X.Engine(0)
    yield e
    e.close()


def test_resident_is_of_the_last_call(eng):
    """After a resident call of any kind, a call that can't run so reads 0."""
    m = L.square_spin(16, 16, disorder=0.5, seed=2)
    flux = L.square(19, 23, disorder=0.5, seed=4, flux=0.03)
    read = lambda: eng.get_option(X.OPT_RESIDENT)
    eng.set_csr(m.csr(), 6.0)
    eng.moments(5, [5], 40)
    assert read() == 1
    eng.moments_block(np.arange(9), 40, X.VEC_FP64)
    assert read() == 0
    eng.moments_block(np.arange(9), 40, X.DOUBLING)
    assert read() == 1
    eng.set_option(X.OPT_MULTI, 2)
    eng.moments_multi([1, 2], [[1], [2]], 40)
    assert read() == 0
    eng.set_option(X.OPT_MULTI, 0)
    eng.moments_multi([1, 2], [[1], [2]], 40)
    assert read() == 1
    eng.set_csr(flux.csr(), 5.0)
    eng.moments_block(np.arange(9), 40, X.DOUBLING)
    assert read() == 0
    eng.moments(5, [5], 40)
    assert read() == 1
    eng.multi_set([flux.csr()], [5.0])
    eng.multi_moments([np.arange(3)], [40], X.DOUBLING)
    assert read() == 0


def test_moments_multi_reports_together(eng):
    eng.set_csr(L.square_spin(16, 16, disorder=0.5, seed=2).csr(), 6.0)
    eng.set_option(X.OPT_PALETTE, 0)
    eng.moments(3, [3], 10)
    assert eng.get_option(X.OPT_PALETTE) == 0
    eng.set_option(X.OPT_PALETTE, 1)
    eng.moments_multi([1, 2], [[1], [2]], 40)
    assert (eng.get_option(X.OPT_MULTI), eng.get_option(X.OPT_RESIDENT)) == (2, 1)
    assert eng.get_option(X.OPT_PALETTE) == 1
    eng.moments_multi([1], [[1]], 40)
    assert eng.get_option(X.OPT_MULTI) == 1


@pytest.mark.parametrize("doubling,S", [(True, 20), (False, 39)])
def test_steps_of_resident_blocks(eng, doubling, S):
    """Steps of a launch's columns: all 200 of a model of one workgroup at once."""
    eng.set_csr(L.square_spin(16, 16, disorder=0.5, seed=2).csr(), 6.0)
    eng.moments_block(np.arange(200), 40, X.DOUBLING if doubling else 0)
    assert eng.get_option(X.OPT_RESIDENT) == 1
    assert eng.last_timing()[1] == S


def test_steps_and_shape_of_blocks_with_a_narrow_rest(eng):
    """128 columns in full blocks and 65 in two parts: the steps of each, and the
    shape of the full blocks. The uneven batch's tile is not a narrow block's."""
    flux = L.square(300, 301, disorder=0.5, seed=4, flux=0.03)
    eng.multi_set([flux.csr()] * 2, [5.0] * 2)
    eng.multi_moments([np.arange(40)] * 2, [40] * 2, X.DOUBLING)
    tile = eng.get_option(X.OPT_TILE_ROWS)
    eng.set_csr(flux.csr(), 5.0)
    eng.moments_block(np.arange(128), 40, X.DOUBLING)
    shape = [eng.get_option(o) for o in (X.OPT_BLOCK_WIDTH, X.OPT_STRIP_ROWS, X.OPT_GRID_SHARE)]
    full = eng.last_timing()[1]
    assert full == 20 * -(-128 // shape[0])
    for n in (193, 129):
        eng.moments_block(np.arange(n), 40, X.DOUBLING)
        assert [eng.get_option(o) for o in (X.OPT_BLOCK_WIDTH, X.OPT_STRIP_ROWS,
                                            X.OPT_GRID_SHARE)] == shape
        assert eng.last_timing()[1] == full + 20 * (2 if n == 193 else 1)
    assert eng.get_option(X.OPT_TILE_ROWS) == tile


def test_shape_of_a_resident_batch(eng):
    """No tiles and no grid of the step kernel, also after a call that had them."""
    specs = [L.square_spec(200, 211, disorder=0.5, seed=1),
             L.square_spec(170, 201, disorder=0.5, seed=2)]
    eng.multi_set_lattices(specs, [5.0, 5.0])
    for resident in (0, 1):
        eng.set_option(X.OPT_RESIDENT, resident)
        eng.multi_moments([np.arange(64), np.arange(40)], [120, 90], X.DOUBLING)
        assert eng.get_option(X.OPT_RESIDENT) == resident
        assert (eng.get_option(X.OPT_TILE_ROWS) == 0) == bool(resident)
    assert eng.get_option(X.OPT_GRID_SHARE) == 0


def test_first_moment_alone_takes_no_cooperative_launch(eng):
    m = L.square_spin(173, 61, disorder=0.5, seed=2)
    eng.set_csr(m.csr(), 6.0)
    assert np.array_equal(eng.moments(7, [3, 7], 1)[:, 0], [0, 1])
    assert eng.get_option(X.OPT_RESIDENT) == 0
    eng.moments(7, [3, 7], 20)
    assert eng.get_option(X.OPT_RESIDENT) == 1
