"""Small products that AUTO takes off the sector path: marking an operand constant moves them there
where the kept packed copy makes it faster, with the same results; a tiny one stays."""
import ctypes

import numpy as np
import pytest

from tamm_amd import configs

pytestmark = pytest.mark.gpu
# relative Frobenius against the grouped path: FP64 sums of at most 1e4 products; 35-bit operands,
# 2^-34 of the row maximum (about 4 times the rms of normal data) in each factor
TOL = {"EXEC_AUTO": 1e-13, "EXEC_AUTO_SPLIT": 1e-9}


def _workload(eng, o, v, ot, vt):
    wl = configs.scaled_spin(o, v, ot, vt)
    del wl.tensors["X"]
    return eng.EngineWorkload(wl, configs.DEFAULT_SEED)


def _run(ew, c):
    C = ew.tensors["R"]
    C.fill(1.0)
    c.execute()
    return C.download()


@pytest.mark.parametrize("mode", sorted(TOL))
def test_constant_operand_moves_small_product(eng, mode):
    ew = _workload(eng, 10, 100, 5, 25)
    V = ew.tensors["V"]
    ref = _run(ew, ew.contraction(configs.LADDER, eng.EXEC_GROUPED_F64))
    c = ew.contraction(configs.LADDER, getattr(eng, mode))
    level = eng.Level([c])  # its reference does not matter to the move
    assert c.mode == eng.EXEC_GROUPED_F64
    c.set_constant(False, True)  # T: too little to gain
    assert c.mode == eng.EXEC_GROUPED_F64
    c.set_constant(True, False)
    assert c.mode == (eng.EXEC_SECTOR_F64 if mode == "EXEC_AUTO" else eng.EXEC_SPLIT_I8)
    for rep in range(2):  # packs, then reuses the packed copy
        got = _run(ew, c)
        assert np.linalg.norm(got - ref) <= TOL[mode] * np.linalg.norm(ref)
    V.scale(-2.0)
    c.set_constant(True, False)  # its values changed
    ref = _run(ew, ew.contraction(configs.LADDER, eng.EXEC_GROUPED_F64))
    ew.tensors["R"].fill(1.0)
    level.execute()
    assert np.linalg.norm(ew.tensors["R"].download() - ref) <= TOL[mode] * np.linalg.norm(ref)
    c.set_constant(False, False)
    got = _run(ew, c)
    assert np.linalg.norm(got - ref) <= TOL[mode] * np.linalg.norm(ref)


@pytest.mark.parametrize("mode", sorted(TOL))
def test_no_move_during_a_capture(eng, mode):
    # building a plan copies and synchronises, which another stream's capture may not survive
    hip = eng.lib()  # its runtime
    stream = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
    ew = _workload(eng, 10, 100, 5, 25)
    C = ew.tensors["R"]
    ref = _run(ew, ew.contraction(configs.LADDER, eng.EXEC_GROUPED_F64))
    c = ew.contraction(configs.LADDER, getattr(eng, mode))

    def record():
        c.set_constant(True, False)
        assert c.mode == eng.EXEC_GROUPED_F64
        c.execute(stream=stream.value)

    g = eng.Graph(record, stream=stream.value)
    for rep in range(3):
        C.fill(1.0)
        eng.synchronize()
        g.launch()
        assert hip.hipStreamSynchronize(stream) == 0
        assert np.array_equal(C.download(), ref)
    del g
    assert hip.hipStreamDestroy(stream) == 0
    c.set_constant(True, False)
    assert c.mode == (eng.EXEC_SECTOR_F64 if mode == "EXEC_AUTO" else eng.EXEC_SPLIT_I8)
    assert np.linalg.norm(_run(ew, c) - ref) <= TOL[mode] * np.linalg.norm(ref)


@pytest.mark.parametrize("mode", sorted(TOL))
def test_tiny_product_stays(eng, mode):
    ew = _workload(eng, 4, 16, 2, 4)
    ref = _run(ew, ew.contraction(configs.LADDER, eng.EXEC_GROUPED_F64))
    c = ew.contraction(configs.LADDER, getattr(eng, mode))
    c.set_constant(True, True)
    assert c.mode == eng.EXEC_GROUPED_F64
    assert np.array_equal(_run(ew, c), ref)
