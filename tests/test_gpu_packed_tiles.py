"""Launches of FP64 plans that can read A in place, for executions that pack it: a constant operand
or an unaligned address in the narrow tiles that packed operands take, odd blocks (always packed), and
the autotuner on either, against the grouped path."""
import numpy as np
import pytest

from tamm_amd import configs

pytestmark = pytest.mark.gpu
TOL = 1e-13  # FP64 sums of at most 1e4 products, relative Frobenius
LADDER = configs.LADDER


def _workload(eng, o, v, ot, vt):
    wl = configs.scaled_spin(o, v, ot, vt)
    del wl.tensors["X"], wl.tensors["W"]
    ew = eng.EngineWorkload(wl, configs.DEFAULT_SEED)
    return ew, _run(ew, ew.contraction(LADDER, eng.EXEC_GROUPED_F64))


def _run(ew, c, **kw):
    ew.tensors["R"].fill(1.0)
    c.execute(**kw)
    return ew.tensors["R"].download()


def _check(got, ref):
    assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)


@pytest.mark.parametrize("o,ot", [(6, 3), (8, 4)])  # 9 and 18, 16 and 32 columns a sector
def test_few_columns(eng, o, ot):
    ew, ref = _workload(eng, o, 100, ot, 50)
    c = ew.contraction(LADDER, eng.EXEC_SECTOR_F64)
    assert c.kernel_info() == (256, 80, False, True)
    _check(_run(ew, c), ref)
    V = ew.tensors["V"]
    shifted = eng.DeviceBuffer(8 * V.size + 8)
    eng.check(eng.lib().tmx_memcpy(shifted.ptr + 8, V.ptr, 8 * V.size, eng.D2D, None))
    _check(_run(ew, c, A=shifted.ptr + 8), ref)
    c.set_constant(True, False)
    assert c.kernel_info() == (32, 32, False, False)
    for _ in range(2):
        _check(_run(ew, c), ref)
    assert len(c.execute_stages()) == 5  # as many GEMM launches as the execution has
    c.set_constant(False, True)
    assert c.kernel_info() == (256, 80, False, True)
    _check(_run(ew, c), ref)


def test_few_columns_odd_blocks(eng):
    ew, ref = _workload(eng, 6, 100, 3, 25)
    c = ew.contraction(LADDER, eng.EXEC_SECTOR_F64)
    assert c.kernel_info() == (32, 32, False, False)
    _check(_run(ew, c), ref)


@pytest.mark.parametrize("o,v,ot,vt", [(10, 40, 5, 10), (6, 60, 3, 30), (12, 60, 6, 10)])
def test_autotune_in_place_and_packed(eng, o, v, ot, vt):
    ew, ref = _workload(eng, o, v, ot, vt)
    c = ew.contraction(LADDER, eng.EXEC_SECTOR_F64)
    for const in (False, True, False):
        c.set_constant(const, False)
        assert c.kernel_info()[3] == (not const)
        _check(_run(ew, c), ref)
        c.autotune()
        assert c.kernel_info()[3] == (not const)  # whatever shapes won
        _check(_run(ew, c), ref)
    # a plan created after the tuning takes the recorded shapes
    d = ew.contraction(LADDER, eng.EXEC_SECTOR_F64)
    assert d.kernel_info()[3]
    _check(_run(ew, d), ref)
