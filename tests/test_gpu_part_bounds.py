"""Split-K parts of FP64 products of few tiles over K blocks of 4 and 9 columns: no part is shorter
than the 64 columns that the launch model may go down to.  Against the grouped path."""
import numpy as np
import pytest

from tamm_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("o,v,ot,vt", [(20, 24, 10, 2), (18, 27, 9, 3), (20, 16, 5, 2)])
def test_tiny_blocks(eng, o, v, ot, vt):
    wl = configs.scaled_spin(o, v, ot, vt)
    for t in wl.tensors.values():
        t.spin = None
    ew = eng.EngineWorkload(wl, configs.DEFAULT_SEED)
    R, out = ew.tensors["R"], []
    for mode in (eng.EXEC_GROUPED_F64, eng.EXEC_SECTOR_F64):
        c = ew.contraction(configs.LADDER, mode)
        R.fill(1.0)
        c.execute()
        out.append(R.download())
    # K blocks are padded to 4 columns: 4 stay 4, 9 become 12
    klen = v * v * (12 if vt == 3 else 4) // (vt * vt)
    assert 1 <= c.schedule_info()[0] <= max(1, klen // 64)
    assert np.linalg.norm(out[1] - out[0]) <= 1e-13 * np.linalg.norm(out[0])
