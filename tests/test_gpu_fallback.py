"""Where a resident recurrence can't run, the step kernels run instead, with their
results: a cooperative launch that the runtime refuses, no memory for the
scratch that only the resident path needs, and a wait given up on the device.
Each is brought about on the host by a shim between the library and the runtime.
"""
import subprocess
import sys

import numpy as np
import pytest

from tbtk_amd import engine as X
from tbtk_amd import lattice as L
from shim import ROOT, run_shimmed

pytestmark = pytest.mark.gpu

CALLS = """
def plain(f, n, s):
    m = f(*n, disorder=0.5, seed=2)
    N = m.basis_size
    eng.set_csr(m.csr(), s)
    return lambda: eng.moments(N // 2, [0, N // 2, N // 2 + 1, N - 1], 60)

def block(flags):
    m = L.honeycomb_ribbon(40, 997, disorder=0.5, seed=4)
    sites = np.random.default_rng(3).integers(0, m.basis_size, 37)
    eng.set_csr(m.csr(), 9.2)
    return lambda: eng.moments_block(sites, 80, flags)

def trace():
    eng.set_csr(L.square(300, 301, disorder=0.5, seed=4).csr(), 5.0)
    return lambda: eng.moments_trace(33, 11, 80)

def batch():
    specs = [L.square_spec(200, 211, disorder=0.5, seed=1), L.square_spec(170, 201, disorder=0.5, seed=2)]
    eng.multi_set_lattices(specs, [5.0, 5.0])
    return lambda: np.concatenate([x.ravel() for x in eng.multi_moments(
        [np.arange(64), np.arange(40)], [120, 90], X.DOUBLING)])

CASES = [("tiles", lambda: plain(L.square_spin, (173, 61), 6.0)),
         ("wide tiles", lambda: plain(L.square_spin, (611, 613), 6.0)),
         ("gathered block", lambda: block(0)), ("doubled block", lambda: block(X.DOUBLING)),
         ("trace", trace), ("batch", batch)]
"""

BODY = CALLS + """
trouble, how = value("{name}"), {how}
for name, make in CASES:
    eng = X.Engine(0)
    call = make()
    eng.set_option(X.OPT_RESIDENT, 0)
    ref = call()
    eng.set_option(X.OPT_RESIDENT, 1)
    trouble.value = how
    print(name, flush=True)
    got = call()
    trouble.value = 0
    assert eng.get_option(X.OPT_RESIDENT) == 0, name
    assert np.array_equal(got, ref), name
    if {settled}:
        value("shim_cooperative").value = 0
        assert np.array_equal(call(), ref), name
        assert value("shim_cooperative").value == 0, name
    else:
        call()
        assert eng.get_option(X.OPT_RESIDENT) == 1, name
"""


@pytest.mark.parametrize("name,how,settled", [
    ("shim_refuse", 1, True), ("shim_malloc_limit", 100000, False), ("shim_give_up", 1, False),
    ("shim_drop", 1, False)])
def test_step_kernels_take_over(tmp_path, name, how, settled):
    """A refused launch is not tried again at once; memory and waits are. Without
    its last workgroup (shim_drop) a launch's waits for that one's rows end after a
    second, the others' when they see it, and every workgroup leaves the kernel."""
    run_shimmed(tmp_path, BODY.format(name=name, how=how, settled=settled))


def test_second_process_on_the_gpu(engine, tmp_path):
    """Only one process at a time has cooperative launches on a GPU: another one
    runs the step kernels, bitwise the same."""
    m = L.square_spin(173, 61, disorder=0.5, seed=2)
    N = m.basis_size
    engine.set_csr(m.csr(), 6.0)
    here = engine.moments(N // 2, [0, N // 2, N - 1], 60)
    assert engine.get_option(X.OPT_RESIDENT) == 1
    out = str(tmp_path / "there.npy")
    code = f"""
import sys
sys.path.insert(0, {ROOT!r})
import numpy as np
from tbtk_amd import engine as X, lattice as L
eng, m = X.Engine(0), L.square_spin(173, 61, disorder=0.5, seed=2)
eng.set_csr(m.csr(), 6.0)
N = m.basis_size
np.save({out!r}, [eng.moments(N // 2, [0, N // 2, N - 1], 60) for _ in range(3)])
"""
    subprocess.run([sys.executable, "-u", "-c", code], check=True, timeout=60)
    for there in np.load(out):
        assert np.array_equal(there, here)


def test_exact_blocks_need_no_slot_values(tmp_path):
    """Vectors that run in exact blocks: without the palette the plain step reads
    values in slots (2 x 5 x 16 B a row), which aren't built for them."""
    run_shimmed(tmp_path, """
m = L.square(101, 97, disorder=0.5, seed=3)
eng.set_csr(m.csr(), 5.0)
eng.set_option(X.OPT_PALETTE, 0)
froms = np.arange(0, 9000, 150)
call = lambda: np.concatenate(eng.moments_multi(froms, [[int(f)] for f in froms], 30))
eng.set_option(X.OPT_MULTI, 2)
eng.set_option(X.OPT_PLAIN_KERNEL, 0)
ref = call()
eng.set_option(X.OPT_PLAIN_KERNEL, 2)
value("shim_malloc_limit").value = 500000
for mode in (2, 0):
    eng.set_option(X.OPT_MULTI, mode)
    assert np.array_equal(call(), ref)
    assert eng.get_option(X.OPT_MULTI) == 2
""")


def test_matrix_contraction_without_pinned_memory(tmp_path):
    """Results through a pageable buffer, bitwise, in several parts of it."""
    run_shimmed(tmp_path, """
rng = np.random.default_rng(2)
eng.lut_generate(64, 1500, -5.0, 5.0, 6.0)
eng.coeffs_upload(rng.normal(size=(900, 64)) + 1j * rng.normal(size=(900, 64)))
value("shim_no_pinned").value = 1
pageable = eng.contract_mfma(X.RETARDED)
value("shim_no_pinned").value = 0
assert np.array_equal(pageable, eng.contract_mfma(X.RETARDED))
""")


def test_batch_with_little_memory_for_dot_slots(tmp_path):
    """Memory for one step's dot slots (20 MB), not for several (266 MB): reduced
    every step, bitwise the same sums."""
    run_shimmed(tmp_path, """
m = L.square(100, 200, disorder=0.5, seed=3, flux=0.01)
got = []
for limit in (0, 100000000):
    eng = X.Engine(0)
    eng.multi_set([m.csr()], [5.0])
    eng.set_option(X.OPT_TILE_ROWS, 2)
    value("shim_malloc_limit").value = limit
    got.append(eng.multi_moments([np.arange(40)], [60], X.DOUBLING)[0])
    value("shim_malloc_limit").value = 0
assert np.array_equal(*got)
""")
