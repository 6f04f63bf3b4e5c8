"""A sector plan whose extra split-K parts or residue plane do not fit the device pool is built without
them: the pool is filled but for one gap between the two sizes."""
import numpy as np
import pytest

from tamm_amd import configs

pytestmark = pytest.mark.gpu


class _Gap:
    """Leaves one free stretch of `nbytes` in the pool (and crumbs below 1 MB)."""

    def __init__(self, eng, nbytes):
        gap = eng.DeviceBuffer(nbytes)
        self.held = []
        size = 1 << 38
        while size >= 1 << 20:
            try:
                self.held.append(eng.DeviceBuffer(size))
            except eng.EngineError as e:
                assert e.code == 3  # out of pool memory
                size //= 2
        gap.free()

    def free(self):
        for b in self.held:
            b.free()


def _ladder(eng):
    wl = configs.scaled_spin(20, 40, 10, 10)
    for t in wl.tensors.values():
        t.spin = None
    return wl, configs.LADDER, eng.EXEC_SECTOR_F64, 1e-13


def _adjoint(eng):
    wl = configs.with_loss_and_grads(configs.scaled_spin(12, 60, 6, 15))
    term = next(t for t in wl.extra["adjoint_terms"] if t.name == "dV<-ladder")
    return wl, term, eng.EXEC_SPLIT_I8, 1e-9  # 35-bit operands


@pytest.mark.parametrize("case", [_ladder, _adjoint])
def test_plan_fits_without_extras(eng, case):
    wl, term, mode, tol = case(eng)
    ew = eng.EngineWorkload(wl, configs.DEFAULT_SEED)
    C = ew.tensors[term.c[0]]

    def run(c):
        C.fill(1.0)
        c.execute()
        return C.download()

    ref = run(ew.contraction(term, eng.EXEC_GROUPED_F64))
    full = ew.contraction(term, mode)
    extra = C.size * (8 * (full.schedule_info()[0] - 1) if mode == eng.EXEC_SECTOR_F64 else 1)
    need = full.workspace
    assert full.schedule_info()[0] > 4 if mode == eng.EXEC_SECTOR_F64 else full.split_info()[2] == 11
    del full
    gap = _Gap(eng, need - extra // 2)
    try:
        c = ew.contraction(term, mode)
    finally:
        gap.free()
    assert c.workspace < need - extra // 2
    got = run(c)
    assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref)
