"""Block permutations in each of the cuts that a plan chooses among (whole tiles of 32x32 or 1024,
boxes of 256, 1024 and 2304 elements), at sizes where tiles, sides, runs and offset tables end, and
AddOps over many ragged blocks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILES = [((33, 31), (1, 0)), ((65, 64), (1, 0)), ((97, 49, 513), (2, 1, 0)), ((1025,), (0,)), ((3, 4, 1100), (1, 0, 2)),
         ((34, 3, 5, 33), (3, 1, 2, 0)), ((34, 3, 5, 33), (3, 0, 2, 1)), ((49, 47, 33, 32), (1, 0, 2, 3)),
         ((49, 47, 33, 32), (3, 2, 1, 0)), ((40, 9, 7, 80, 13), (0, 2, 1, 3, 4)), ((1100, 49, 47), (0, 2, 1)),
         ((17, 40000), (1, 0))]
BOXES_256 = [((60, 40, 5, 11), (1, 0, 2, 3)), ((30, 16, 15, 14), (0, 2, 1, 3)), ((300, 6, 7, 11), (0, 2, 1, 3)),
             ((1500, 10, 9), (0, 2, 1)), ((2, 3, 4, 5, 6, 7, 8, 9), (7, 6, 5, 4, 3, 2, 1, 0)),
             ((2, 3, 4, 5, 6, 7, 8, 9), (1, 0, 3, 2, 5, 4, 7, 6)), ((25, 11, 13, 40, 3), (0, 2, 1, 3, 4))]
BOXES_1024 = [((20, 30, 40, 100), (0, 2, 1, 3)), ((2, 900001), (1, 0)), ((3, 700001), (1, 0)), ((900001, 2), (1, 0))]
BOXES_2304 = [((8, 300001), (1, 0)), ((300001, 8), (1, 0)), ((49, 47, 17, 33), (1, 0, 3, 2)), ((35, 49, 33, 47), (3, 2, 1, 0)),
              ((70, 71, 16, 17), (0, 1, 3, 2)), ((6, 13, 513, 97), (2, 1, 0, 3)), ((11, 250, 7, 130), (2, 1, 0, 3)),
              ((2, 2, 2, 2, 9, 33, 35, 47), (3, 1, 2, 0, 6, 4, 5, 7)), ((33, 2, 3, 5, 7, 2, 9, 34), (7, 2, 1, 5, 4, 3, 6, 0)),
              ((100, 12, 100, 9), (0, 2, 1, 3))]


def _check(got, dst, ref, is_assign):
    if is_assign:
        assert np.array_equal(got, ref)
    else:  # one rounding of a sum (fused or not) of terms of magnitude <= ~9
        assert np.max(np.abs(got - (dst + ref))) <= 4e-15


@pytest.mark.parametrize("is_assign", [False, True])
@pytest.mark.parametrize("sdims,perm", TILES + BOXES_256 + BOXES_1024 + BOXES_2304)
def test_block_permutation(eng, sdims, perm, is_assign):
    rng = np.random.default_rng(len(sdims))
    src = rng.standard_normal(sdims)
    ddims = [sdims[p] for p in perm]
    dst = rng.standard_normal(ddims)
    sl = [-(i + 1) for i in range(len(sdims))]
    ds, dd = eng.DeviceBuffer.from_array(src.ravel()), eng.DeviceBuffer.from_array(dst.ravel())
    eng.block_assign(dd, ddims, [sl[p] for p in perm], -1.5, ds, list(sdims), sl, is_assign=is_assign)
    got = dd.download(np.float64, dst.size).reshape(ddims)
    _check(got, dst, -1.5 * np.transpose(src, perm), is_assign)


def _dense(t, packed):
    out = np.zeros([s.n for s in t.spaces])
    nt = [s.ntiles for s in t.spaces]
    for key, off, size in zip(t.keys, t.offsets, t.sizes):
        b = np.unravel_index(int(key), nt)
        sl = tuple(slice(int(s.offsets[i]), int(s.offsets[i + 1])) for s, i in zip(t.spaces, b))
        out[sl] = packed[off:off + size].reshape([x.stop - x.start for x in sl])
    return out


# V and O tiles: whole tiles (blocks of 64 and 50, of one element beside 64), boxes of 2304 and 256
@pytest.mark.parametrize("vt,ot", [([64, 50], [33, 9]), ([64, 1, 63], [32, 1]), ([20, 13, 20, 1, 19], [11, 5, 1, 11]),
                                   ([5, 3, 1, 4], [3, 2])])
@pytest.mark.parametrize("perm", ["baij", "abji", "baji", "ijab", "jiab"])
@pytest.mark.parametrize("is_assign", [False, True])
def test_ragged_addop(eng, vt, ot, perm, is_assign):
    V, O = eng.Space(sum(vt), vt), eng.Space(sum(ot), ot)
    space = dict(a=V, b=V, i=O, j=O)
    dst, src = (eng.Tensor([space[c] for c in s]).allocate() for s in ("abij", perm))
    rng = np.random.default_rng(dst.size)
    x, y = rng.standard_normal(src.size), rng.standard_normal(dst.size)
    src.upload(x), dst.upload(y)
    lab = {c: -(i + 1) for i, c in enumerate("abij")}
    eng.AddOp(dst, [lab[c] for c in "abij"], -1.5, src, [lab[c] for c in perm], is_assign).execute()
    ref = -1.5 * np.transpose(_dense(src, x), [perm.index(c) for c in "abij"])
    _check(_dense(dst, dst.download()), _dense(dst, y), ref, is_assign)
