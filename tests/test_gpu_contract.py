"""The FP64 contraction's three kernels (few, each, many vectors): bitwise the
oracle's lookup contraction with the uploaded table, and its direct form, at the sizes where the
split changes (energies and vectors beside multiples of a tile, moments beside
multiples of a chunk).
"""
import numpy as np
import pytest

from tbtk_amd import engine as X

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gtype", range(4))
@pytest.mark.parametrize("K,M,E", [
    (1, 1, 2), (1, 2, 15), (2, 31, 16), (3, 33, 17), (5, 511, 65), (1, 513, 130), (2, 1030, 300),
    (70, 40, 1000), (90, 16, 1001), (200, 15, 1001), (203, 17, 1000), (515, 33, 1025), (9, 20, 20000),
])
def test_contraction_bitwise(engine, oracle_mod, K, M, E, gtype):
    rng = np.random.default_rng(K + M + E)
    c = rng.normal(size=(K, M)) + 1j * rng.normal(size=(K, M))
    s, lo, hi = 6.0, -5.7, 5.8
    table = oracle_mod.lookup_table(M, E, lo, hi, s)
    engine.lut_upload(table)
    got = engine.contract(c, gtype)
    de = (hi - lo) / (E - 1)
    direct = engine.contract_direct(c, gtype, E, lo, de, s)
    for k in sorted({0, K // 2, K - 1}):
        assert np.array_equal(got[k], oracle_mod.gf_lookup(gtype, table, c[k])), k
        assert np.array_equal(direct[k], oracle_mod.gf_direct(gtype, c[k], lo, hi, E, s)), k
    engine.lut_destroy()
