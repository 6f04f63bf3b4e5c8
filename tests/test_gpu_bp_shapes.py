"""The C-tile shape that the launch model of the block-pair kernels chooses, and every shape around
the edges of its tiles, k-steps of 4 and chunks of 64 indices: all four orders of the operands, C along
either side, a non-finite row beside finite ones."""
import numpy as np
import pytest

from tamm_amd import configs

pytestmark = pytest.mark.gpu
TOL = 1e-13  # FP64 sums of at most 2.1e3 products of unit normals, relative Frobenius

# sizes of one block pair (m, n, k), and (rows, columns, shared reduction) of the shape chosen for them
KS16, KS32, KS64, LDS64, LDS16 = (16, 16, True), (32, 32, True), (64, 64, True), (64, 64, False), (16, 256, False)
CASES = [((15, 17, 5), KS16), ((130, 63, 64), KS16), ((300, 300, 70), KS16), ((4097, 15, 300), KS16),
         ((700, 700, 64), KS32), ((481, 511, 1030), KS32), ((545, 500, 700), KS32), ((800, 700, 515), KS32),
         ((1030, 1010, 1030), KS64), ((960, 1030, 1029), KS64), ((1025, 1023, 2050), KS64),
         ((1300, 1300, 600), LDS64), ((1950, 1930, 67), LDS64), ((2000, 2000, 33), LDS64),
         ((16, 240000, 66), LDS16), ((240001, 15, 35), LDS16)]


def _contraction(eng, al, bl, cl, dims):
    sp = {c: eng.Space(n, n) for c, n in dims.items()}
    t = [eng.Tensor([sp[c] for c in s]).allocate() for s in (cl, al, bl)]
    lab = {c: -(i + 1) for i, c in enumerate(dims)}
    ids = [[lab[c] for c in s] for s in (cl, al, bl)]
    return t, eng.Contraction(t[0], ids[0], 0.5, t[1], ids[1], t[2], ids[2], eng.EXEC_GROUPED_F64)


def _run(t, c, al, bl, cl, dims, assign, A=None):
    rng = np.random.default_rng(sum(dims.values()))
    x = [rng.standard_normal([dims[q] for q in s]) for s in (cl, al, bl)]
    x[1] = x[1] if A is None else A
    for ti, xi in zip(t, x):
        ti.upload(xi.ravel())
    c.set_assign(assign)
    c.execute()
    got = t[0].download().reshape(x[0].shape)
    a, b = (x[1] if al == "mk" else x[1].T), (x[2] if bl == "kn" else x[2].T)
    ref = 0.5 * (a @ b)
    return got, (ref if cl == "mn" else ref.T) + (0.0 if assign else x[0])


@pytest.mark.parametrize("size,shape", CASES, ids=lambda x: "x".join(map(str, x)))
@pytest.mark.parametrize("al,bl,cl", [("mk", "nk", "mn"), ("km", "kn", "nm"), ("mk", "kn", "nm"), ("km", "nk", "mn")])
def test_shapes(eng, size, shape, al, bl, cl):
    dims = dict(zip("mnk", size))
    t, c = _contraction(eng, al, bl, cl, dims)
    assert c.kernel_info()[:3] == shape
    got, ref = _run(t, c, al, bl, cl, dims, bool(size[2] & 1))
    assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)


@pytest.mark.parametrize("size,shape", [CASES[i] for i in (1, 5, 8, 11)], ids=lambda x: "x".join(map(str, x)))
def test_nonfinite_row_stays_in_its_row(eng, size, shape):
    dims = dict(zip("mnk", size))
    t, c = _contraction(eng, "mk", "nk", "mn", dims)
    assert c.kernel_info()[:3] == shape
    A = np.random.default_rng(1).standard_normal((dims["m"], dims["k"]))
    A[-1, -1], A[3, 0] = np.nan, np.inf
    with np.errstate(invalid="ignore"):
        got, ref = _run(t, c, "mk", "nk", "mn", dims, True, A)
    bad = np.zeros(dims["m"], dtype=bool)
    bad[[3, -1]] = True
    assert not np.isfinite(got[bad]).any()
    assert np.linalg.norm(got[~bad] - ref[~bad]) <= TOL * np.linalg.norm(ref[~bad])


# short reductions into large outputs: 64x64 tiles 24 us where 32x32 with a shared reduction take 34
@pytest.mark.parametrize("o,v,ot,vt", [(16, 40, 8, 10), (8, 40, 4, 10), (6, 40, 3, 10)])
def test_short_reductions_take_staged_tiles(eng, o, v, ot, vt):
    wl = configs.with_loss_and_grads(configs.scaled_spin(o, v, ot, vt))
    ew = eng.EngineWorkload(wl, configs.DEFAULT_SEED, allocate=False)
    term = next(t for t in wl.extra["adjoint_terms"] if t.name == "dV<-ladder")
    assert ew.contraction(term, eng.EXEC_GROUPED_F64).kernel_info()[:3] == LDS64
