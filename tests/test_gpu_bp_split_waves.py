"""The block-pair kernels whose waves share a reduction: block products around the edges of the
16x16, 32x32 and 64x64 tiles, of the 4-index k-steps and of the 64-index chunks, with operands
contiguous along K or along the rows; a batch label and a one-sided reduction; a non-finite row
beside finite ones; and spin-blocked sets of tiny ragged blocks against the FP64 sector path."""
import numpy as np
import pytest

from tamm_amd import configs

pytestmark = pytest.mark.gpu
TOL = 1e-13  # FP64 sums of at most 6.4e3 products of unit normals, relative Frobenius


def _multiply(eng, al, bl, cl, dims, is_assign, A=None):
    rng = np.random.default_rng(sum(dims.values()))
    ids = {c: -(i + 1) for i, c in enumerate(dims)}
    shape = lambda s: [dims[c] for c in s]  # noqa: E731
    A = rng.standard_normal(shape(al)) if A is None else A
    B, C = rng.standard_normal(shape(bl)), rng.standard_normal(shape(cl))
    da, db, dc = (eng.DeviceBuffer.from_array(x.ravel()) for x in (A, B, C))
    eng.block_multiply(0.5, da, shape(al), [ids[c] for c in al], db, shape(bl), [ids[c] for c in bl],
                       dc, shape(cl), [ids[c] for c in cl], is_assign=is_assign)
    got = dc.download(np.float64, C.size).reshape(C.shape)
    ref = 0.5 * np.einsum(f"{al},{bl}->{cl}", A, B, optimize=True) + (0.0 if is_assign else C)
    return got, ref


@pytest.mark.parametrize("m,n", [(1, 1), (15, 17), (16, 16), (31, 33), (33, 5), (64, 65), (130, 63)])
@pytest.mark.parametrize("k", [1, 3, 5, 63, 64, 65, 257, 1030])
@pytest.mark.parametrize("al,bl,cl", [("mk", "nk", "mn"), ("km", "kn", "nm"), ("mk", "kn", "nm"), ("km", "nk", "mn")])
def test_edges(eng, m, n, k, al, bl, cl):
    got, ref = _multiply(eng, al, bl, cl, {"m": m, "n": n, "k": k}, is_assign=bool(k & 1))
    assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)


@pytest.mark.parametrize("al,bl,cl,dims", [
    ("abcd", "cdij", "abij", dict(a=7, b=5, c=6, d=9, i=3, j=4)),       # two modes a side
    ("kbcj", "acik", "abij", dict(k=5, b=9, c=10, j=3, a=8, i=6)),      # a ring's modes
    ("abcd", "cdij", "abij", dict(a=40, b=40, c=48, d=24, i=15, j=15)),  # many tiles
    ("zmk", "zkn", "zmn", dict(z=3, m=18, k=70, n=20)),                  # batch label
    ("mkx", "kn", "mn", dict(m=17, k=9, x=11, n=33)),                    # A-only reduction
])
def test_modes(eng, al, bl, cl, dims):
    for is_assign in (False, True):
        got, ref = _multiply(eng, al, bl, cl, dims, is_assign)
        assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)


@pytest.mark.parametrize("m", [17, 33, 70])
@pytest.mark.parametrize("k", [6, 67])
def test_nonfinite_row_stays_in_its_row(eng, m, k):
    A = np.random.default_rng(m).standard_normal((m, k))
    A[m - 1, k - 1], A[3, 0] = np.nan, np.inf
    got, ref = _multiply(eng, "mk", "nk", "mn", {"m": m, "n": 21, "k": k}, True, A)
    bad = np.zeros(m, dtype=bool)
    bad[[3, m - 1]] = True
    assert not np.isfinite(got[bad]).any()
    assert np.linalg.norm(got[~bad] - ref[~bad]) <= TOL * np.linalg.norm(ref[~bad])


@pytest.mark.parametrize("o,v,ot,vt", [(4, 8, 2, 3), (6, 20, 1, 4), (10, 40, 5, 11)])
@pytest.mark.parametrize("mode", [0, 1, 4])  # per pair, grouped, AUTO
def test_sets_match_sector(eng, o, v, ot, vt, mode):
    wl = configs.with_loss_and_grads(configs.scaled_spin(o, v, ot, vt))
    ew = eng.EngineWorkload(wl, configs.DEFAULT_SEED)
    for term in wl.terms + wl.extra["adjoint_terms"]:
        C = ew.tensors[term.c[0]]
        out = []
        for md in (2, mode):  # FP64 sector first
            C.fill(1.0)
            c = ew.contraction(term, md)
            c.execute()
            out.append(C.download())
        assert np.linalg.norm(out[1] - out[0]) <= TOL * np.linalg.norm(out[0]), (term.name, mode)
