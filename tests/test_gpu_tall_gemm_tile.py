"""FP64 sector GEMMs whose columns fill tiles of 80 rather than of 128 or 160 (256-row tiles): one
tile and less, exactly one, several with a remainder, split-K parts, and an operand packed for its
odd blocks, against the grouped path."""
import numpy as np
import pytest

from tamm_amd import configs

pytestmark = pytest.mark.gpu
TOL = 1e-13  # FP64 sums of at most 1e4 products, relative Frobenius


# rows v*v = 144, 256, 576, 1156 (odd blocks), 3136; columns o*o = 400, 72 of padded 80 (spin)
@pytest.mark.parametrize("o,v,ot,vt,spin", [(20, 12, 5, 12, False), (20, 16, 5, 8, False), (20, 24, 5, 12, False),
                                            (20, 34, 7, 17, False), (20, 56, 10, 14, False), (12, 40, 6, 10, True)])
@pytest.mark.parametrize("parts", [0, 1, 3])
def test_matches_grouped(eng, o, v, ot, vt, spin, parts):
    wl = configs.scaled_spin(o, v, ot, vt)
    if not spin:
        for t in wl.tensors.values():
            t.spin = None
    ew = eng.EngineWorkload(wl, configs.DEFAULT_SEED)
    out = {}
    for mode in (eng.EXEC_GROUPED_F64, eng.EXEC_SECTOR_F64):
        R = ew.tensors["R"]
        R.fill(1.0)
        eng.check(eng.lib().tmx_set_parallel_split(parts))
        try:
            c = ew.contraction(configs.LADDER, mode)
        finally:
            eng.check(eng.lib().tmx_set_parallel_split(0))
        c.execute()
        out[mode] = R.download()
    ref, got = out[eng.EXEC_GROUPED_F64], out[eng.EXEC_SECTOR_F64]
    assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)
