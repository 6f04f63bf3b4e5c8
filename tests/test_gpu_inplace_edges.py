"""FP64 plans that read their first operand in place, asserted by the plan: K blocks that end 2, 4 and 6
columns past a stage of 8 and on one, row blocks that do not fill tiles, parts that begin inside a block,
and operands that are packed for their block count or an odd block, against numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-13  # FP64 sums of at most 1.4e3 products, relative Frobenius


def _dense(t, packed):
    out = np.zeros([s.n for s in t.spaces])
    nt = [s.ntiles for s in t.spaces]
    for key, off, size in zip(t.keys, t.offsets, t.sizes):
        b = np.unravel_index(int(key), nt)
        sl = tuple(slice(int(s.offsets[i]), int(s.offsets[i + 1])) for s, i in zip(t.spaces, b))
        out[sl] = packed[off:off + size].reshape([x.stop - x.start for x in sl])
    return out


def _product(eng, al, bl, cl, spaces, parts):
    t = {s: eng.Tensor([spaces[c] for c in s]).allocate() for s in (cl, al, bl)}
    rng = np.random.default_rng(t[al].size)
    x = {s: rng.standard_normal(q.size) for s, q in t.items()}
    for s, q in t.items():
        q.upload(x[s])
    lab = {c: -(i + 1) for i, c in enumerate(spaces)}
    eng.check(eng.lib().tmx_set_parallel_split(parts))
    try:
        c = eng.Contraction(t[cl], [lab[q] for q in cl], -0.5, t[al], [lab[q] for q in al], t[bl], [lab[q] for q in bl],
                            eng.EXEC_SECTOR_F64)
    finally:
        eng.check(eng.lib().tmx_set_parallel_split(0))
    c.execute()
    d = {s: _dense(q, x[s]) for s, q in t.items()}
    ref = d[cl] - 0.5 * np.einsum(f"{al},{bl}->{cl}", d[al], d[bl], optimize=True)
    got = _dense(t[cl], t[cl].download())
    assert np.linalg.norm(got - ref) <= TOL * np.linalg.norm(ref)
    return c.kernel_info()[3]


# columns 66 = 8*8 + 2, 68 (+ 4), 70 (+ 6), 72; two columns of their own and a long block
@pytest.mark.parametrize("kt", [[66], [70], [66, 68, 70, 72], [72, 70, 66, 2, 150], [128, 66, 1000, 70]])
@pytest.mark.parametrize("mt,nt", [([150], [40]), ([13, 100, 5, 37, 128, 1], [33, 70]), ([300, 17], [170]),
                                   ([16] * 20, [16, 64, 1])])
@pytest.mark.parametrize("parts", [0, 1, 3])
def test_columns_past_a_stage(eng, kt, mt, nt, parts):
    sp = {c: eng.Space(sum(t), t) for c, t in (("m", mt), ("n", nt), ("k", kt))}
    assert _product(eng, "mk", "kn", "mn", sp, parts)


# row-major X(i,j,k,l): K blocks of o tiles 8 x 8 and 10 x 12
@pytest.mark.parametrize("ot", [[8, 8], [10, 12, 8]])
@pytest.mark.parametrize("bl", ["klab", "abkl"])
def test_four_modes(eng, ot, bl):
    o, v = eng.Space(sum(ot), ot), eng.Space(15, [7, 8])
    assert _product(eng, "ijkl", bl, "ijab", dict(i=o, j=o, k=o, l=o, a=v, b=v), 0)


@pytest.mark.parametrize("mt,kt", [([1] * 130, [66] * 5),     # 640 block offsets in a tile of 128 rows
                                   ([100, 60], [66, 67, 70]),  # an odd block
                                   ([100, 60], [66, 20, 30])])  # 39 columns on average
def test_packed_instead(eng, mt, kt):
    sp = {c: eng.Space(sum(t), t) for c, t in (("m", mt), ("n", [90, 50]), ("k", kt))}
    assert not _product(eng, "mk", "kn", "mn", sp, 0)
