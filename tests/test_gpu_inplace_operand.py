"""FP64 sector plans that read their first operand in place: blocks whose columns end 2, 4 or 6
past a stage of 8, row blocks that do not fill 16-row tiles, several row blocks in one tile,
split-K parts that begin inside a block, odd columns (packed instead), an operand at an address
that does not allow 16-byte loads (packed instead), a constant operand (packed once), and a
non-finite element, against the grouped path and for its reach."""
import numpy as np
import pytest

from tamm_amd import configs

pytestmark = pytest.mark.gpu
GROUPED, SECTOR = 1, 2
TOL = 1e-13  # FP64 sums of at most 1e4 products, relative Frobenius


def _workload(eng, o, v, ot, vt, spin=True):
    wl = configs.scaled_spin(o, v, ot, vt)
    if not spin:
        for t in wl.tensors.values():
            t.spin = None
    return wl, eng.EngineWorkload(wl, configs.DEFAULT_SEED)


def _run(ew, term, mode, parts=0, eng=None, **kw):
    C = ew.tensors[term.c[0]]
    C.fill(1.0)
    eng.check(eng.lib().tmx_set_parallel_split(parts))
    try:
        c = ew.contraction(term, mode)
    finally:
        eng.check(eng.lib().tmx_set_parallel_split(0))
    c.execute(**kw)
    return C.download()


# tiles of V: columns vt * vt = 196 (8 * 24 + 4), 100 (+ 4), 900 (+ 4), 324, 26 * 26 = 676, odd 225
@pytest.mark.parametrize("o,v,ot,vt", [(6, 28, 3, 14), (10, 40, 5, 10), (4, 60, 2, 30), (12, 54, 4, 18),
                                       (8, 52, 4, 26), (8, 44, 4, 12), (20, 44, 5, 22), (6, 30, 3, 15)])
@pytest.mark.parametrize("spin", [True, False])
@pytest.mark.parametrize("parts", [0, 3])
def test_matches_grouped(eng, o, v, ot, vt, spin, parts):
    wl, ew = _workload(eng, o, v, ot, vt, spin)
    for term in (configs.LADDER, configs.HOLE_HOLE):
        ref = _run(ew, term, GROUPED, eng=eng)
        got = _run(ew, term, SECTOR, parts, eng=eng)
        assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref), term.name


def test_unaligned_and_constant_operands(eng):
    wl, ew = _workload(eng, 10, 40, 5, 20)
    term = configs.LADDER
    V = ew.tensors["V"]
    ref = _run(ew, term, SECTOR, eng=eng)
    shifted = eng.DeviceBuffer(8 * V.size + 8)
    eng.check(eng.lib().tmx_memcpy(shifted.ptr + 8, V.ptr, 8 * V.size, eng.D2D, None))
    got = _run(ew, term, SECTOR, eng=eng, A=shifted.ptr + 8)
    assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)
    c = ew.contraction(term, SECTOR)
    C = ew.tensors["R"]
    for const in (False, True, True, False):
        if const != getattr(c, "_const", None):
            c.set_constant(const, False)
            c._const = const
        C.fill(1.0)
        c.execute()
        got = C.download()
        assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref), const


def test_nonfinite_element_stays_in_its_row(eng):
    """An Inf in the last column of a V row reaches that (a,b) row of R only."""
    wl, ew = _workload(eng, 6, 28, 3, 14, spin=False)
    V, term = ew.tensors["V"], configs.LADDER
    ref = _run(ew, term, SECTOR, eng=eng)
    x = V.download()
    cols = 14 * 14
    x[5 * cols - 1] = np.inf  # block (0,0,0,0): row 4, last column
    V.upload(x)
    got = _run(ew, term, SECTOR, eng=eng)
    bad = ~np.isfinite(got)
    R = ew.tensors["R"]
    nt = [len(s.offsets) - 1 for s in R.spaces]
    for key, off, size in zip(R.keys, R.offsets, R.sizes):
        b = np.unravel_index(int(key), nt)
        blk = bad[off:off + size].reshape(cols, -1)
        want = np.zeros(cols, dtype=bool)
        want[4] = b[0] == 0 and b[1] == 0
        assert (blk.all(axis=1) == want).all() and (blk.any(axis=1) == want).all()
    ok = ~bad
    assert np.linalg.norm(got[ok] - ref[ok]) <= TOL * np.linalg.norm(ref)
