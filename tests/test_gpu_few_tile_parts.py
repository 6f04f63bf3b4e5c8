"""Split-K parts of FP64 products with few tiles, which may be as short as 128 columns: K ranges
shorter than a part, just over two, and many parts of one small product, against the grouped path."""
import numpy as np
import pytest

from tamm_amd import configs

pytestmark = pytest.mark.gpu
TOL = 1e-13  # FP64 sums of at most 1e4 products, relative Frobenius


@pytest.mark.parametrize("o,v,ot,vt,spin", [(18, 10, 6, 5, False), (9, 30, 3, 10, False), (10, 46, 5, 23, False),
                                            (20, 30, 7, 11, False), (18, 60, 6, 15, True)])
@pytest.mark.parametrize("term", [configs.LADDER, configs.RING], ids=lambda t: t.name)
def test_matches_grouped(eng, o, v, ot, vt, spin, term):
    wl = configs.scaled_spin(o, v, ot, vt)
    if not spin:
        for t in wl.tensors.values():
            t.spin = None
    ew = eng.EngineWorkload(wl, configs.DEFAULT_SEED)
    out = {}
    for mode in (eng.EXEC_GROUPED_F64, eng.EXEC_SECTOR_F64):
        R = ew.tensors["R"]
        R.fill(1.0)
        ew.contraction(term, mode).execute()
        out[mode] = R.download()
    ref, got = out[eng.EXEC_GROUPED_F64], out[eng.EXEC_SECTOR_F64]
    assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)
