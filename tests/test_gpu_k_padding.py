"""K blocks of sector plans, padded to 16 (split) or 4 (FP64) columns, and K classes, padded to whole
stages: ragged blocks of 1 to 49 columns in several classes, parts that begin inside a class, and
workspace that held NaNs before, against the grouped path."""
import numpy as np
import pytest

from tamm_amd import configs

pytestmark = pytest.mark.gpu
# relative Frobenius: FP64 sums of at most 1e3 products; 35-bit operands, 2^-34 of the row maximum
# (about 4 times the rms of normal data) in each factor
TOL = {"EXEC_SECTOR_F64": 1e-13, "EXEC_SPLIT_I8": 1e-9}


@pytest.mark.parametrize("o,v,lo,hi", [(12, 24, 1, 4), (8, 32, 1, 7), (10, 30, 3, 5), (6, 18, 2, 2)])
@pytest.mark.parametrize("mode", sorted(TOL))
@pytest.mark.parametrize("parts", [0, 3])
def test_ragged_classes(eng, o, v, lo, hi, mode, parts):
    step = configs._cc_step("step", o, v, lo, hi, 7, "ragged tiles in spin and irrep ranges")
    wl = configs.with_loss_and_grads(configs.Workload("ragged", "", step.spaces, configs._cc_tensors("O", "V", True),
                                                      [configs.LADDER, configs.RING, configs.HOLE_HOLE], ["R"]))
    ew = eng.EngineWorkload(wl, configs.DEFAULT_SEED)
    for term in wl.terms + wl.extra["adjoint_terms"]:
        C, out = ew.tensors[term.c[0]], []
        for m in (eng.EXEC_GROUPED_F64, getattr(eng, mode)):
            poison = eng.DeviceBuffer(1 << 26)  # the plan's workspace comes from here
            eng.check(eng.lib().tmx_fill(poison.ptr, (1 << 26) // 8, float("nan"), None))
            eng.synchronize()
            poison.free()
            eng.check(eng.lib().tmx_set_parallel_split(parts))
            try:
                c = ew.contraction(term, m)
            finally:
                eng.check(eng.lib().tmx_set_parallel_split(0))
            C.fill(1.0)
            c.execute()
            out.append(C.download())
        assert np.linalg.norm(out[1] - out[0]) <= TOL[mode] * np.linalg.norm(out[0]), term.name
