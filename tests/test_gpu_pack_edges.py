"""Packing and scatter passes of sector plans at the edges of their tiles: blocks of odd and even
rows and columns around 32, 64 and 128 (rows that do and do not allow 16-byte loads), fewer and more
tiles than one per XCD, and source data at an odd multiple of 8 bytes, against the grouped path."""
import numpy as np
import pytest

from tamm_amd import configs

pytestmark = pytest.mark.gpu
# relative Frobenius: FP64 sums of at most 1e4 products; 35-bit operands, 2^-34 of the row maximum
# (about 4 times the rms of normal data) in each factor
TOL = {"EXEC_SECTOR_F64": 1e-13, "EXEC_SPLIT_I8": 1e-9}


@pytest.mark.parametrize("o,v,ot,vt", [(2, 4, 1, 2), (6, 12, 3, 6), (6, 22, 3, 11), (10, 24, 5, 12),
                                       (14, 26, 7, 13), (6, 46, 3, 23), (12, 44, 6, 22), (16, 50, 8, 7)])
@pytest.mark.parametrize("mode", sorted(TOL))
def test_tile_edges(eng, o, v, ot, vt, mode):
    wl = configs.scaled_spin(o, v, ot, vt)
    ew = eng.EngineWorkload(wl, configs.DEFAULT_SEED)
    for term in (configs.LADDER, configs.RING, configs.HOLE_HOLE):
        C, A = ew.tensors[term.c[0]], ew.tensors[term.a[0]]
        shifted = eng.DeviceBuffer(8 * A.size + 8)
        eng.check(eng.lib().tmx_memcpy(shifted.ptr + 8, A.ptr, 8 * A.size, eng.D2D, None))
        got = []
        for m, kw in ((eng.EXEC_GROUPED_F64, {}), (getattr(eng, mode), {}), (getattr(eng, mode), {"A": shifted.ptr + 8})):
            C.fill(1.0)
            ew.contraction(term, m).execute(**kw)
            got.append(C.download())
        for x in got[1:]:
            assert np.linalg.norm(x - got[0]) <= TOL[mode] * np.linalg.norm(got[0]), term.name
