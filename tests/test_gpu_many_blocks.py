"""A sector plan whose packing pass has more than 2^24 units: an operand of 4097 x 4096 blocks of one
element, over the work items that one launch may have at a workgroup a unit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.timeout(300)
def test_more_blocks_than_work_items(eng):
    m, k, n = 4097, 4096, 3
    sm, sk, sn = eng.Space(m, 1), eng.Space(k, 1), eng.Space(n, n)
    A, B, C = (eng.Tensor(list(s)).allocate() for s in ((sm, sk), (sk, sn), (sm, sn)))
    rng = np.random.default_rng(0)
    a, b = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    A.upload(a.ravel()), B.upload(b.ravel()), C.fill(0.0)
    c = eng.Contraction(C, [-1, -3], 1.0, A, [-1, -2], B, [-2, -3], eng.EXEC_SECTOR_F64)
    c.execute()
    got, ref = C.download().reshape(m, n), a @ b
    assert np.linalg.norm(got - ref) <= 1e-13 * np.linalg.norm(ref)  # FP64 sums of 4096 products
