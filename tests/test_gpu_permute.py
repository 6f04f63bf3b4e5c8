"""Block permutations at the sizes where a box of the tiling ends: sides around 32 and 48, runs
around 64 and 512, blocks of a few elements, unit modes, merged modes and up to six modes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    ((2, 3), (1, 0)), ((48, 48), (1, 0)), ((49, 47), (1, 0)), ((97, 33), (1, 0)), ((513, 5), (0, 1)),
    ((1, 7), (1, 0)), ((31, 32, 33), (2, 1, 0)), ((5, 48, 16), (1, 0, 2)), ((3, 2305), (1, 0)),
    ((48, 48, 16, 16), (1, 0, 2, 3)), ((48, 24, 16, 4), (0, 1, 3, 2)), ((48, 48, 4, 16), (1, 0, 3, 2)),
    ((7, 1, 63, 2), (3, 1, 2, 0)), ((2, 2, 2, 2, 2, 2), (5, 4, 3, 2, 1, 0)), ((3, 65, 1, 4, 5, 2), (4, 0, 5, 2, 1, 3)),
    ((700, 3, 2), (0, 2, 1)), ((), ()),
]


@pytest.mark.parametrize("is_assign", [False, True])
@pytest.mark.parametrize("sdims,perm", CASES)
def test_block_permutation(eng, sdims, perm, is_assign):
    rng = np.random.default_rng(len(sdims))
    src = rng.standard_normal(sdims)
    ddims = [sdims[p] for p in perm]
    dst = rng.standard_normal(ddims)
    sl = [-(i + 1) for i in range(len(sdims))]
    ds, dd = eng.DeviceBuffer.from_array(src.ravel()), eng.DeviceBuffer.from_array(dst.ravel())
    eng.block_assign(dd, ddims, [sl[p] for p in perm], -1.5, ds, list(sdims), sl, is_assign=is_assign)
    got = dd.download(np.float64, dst.size).reshape(ddims)
    ref = -1.5 * np.transpose(src, perm)
    if is_assign:
        assert np.array_equal(got, ref)
    else:  # one rounding of a sum (fused or not) of terms of magnitude <= ~8
        assert np.max(np.abs(got - (dst + ref))) <= 4e-15


def test_assigning_addop_zeroes_blocks_without_source(eng):
    """A dense destination over a spin-masked source: blocks the mask excludes become zero."""
    sp = eng.Space(6, 2, spin=[(0, 3, 1), (3, 6, 2)])
    src = eng.Tensor([sp] * 4, (2, 2)).allocate()
    dst = eng.Tensor([sp] * 4, None).allocate()
    src.upload(np.random.default_rng(0).standard_normal(src.size))
    dst.fill(float("nan"))
    eng.AddOp(dst, [1, 2, 3, 4], 2.0, src, [2, 1, 4, 3], is_assign=True).execute()
    got = dst.download()
    assert np.isfinite(got).all()
    assert abs(np.linalg.norm(got) - 2.0 * src.norm()) <= 1e-14 * src.norm()
    assert np.count_nonzero(got) == src.size
