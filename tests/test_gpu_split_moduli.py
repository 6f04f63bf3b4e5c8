"""Moduli of split plans: a product that ten would do for takes eleven, whose residues are combined in
pairs; other counts are the smallest exact ones.  Results against the grouped path."""
import numpy as np
import pytest

from tamm_amd import configs

pytestmark = pytest.mark.gpu


# bits, moduli of the short hole-hole reductions (K <= 100): 2 bits + log2(K) + 1.05 bits needed
@pytest.mark.parametrize("bits,nmod", [(25, 8), (30, 9), (33, 11), (34, 11), (35, 11), (40, 12)])
@pytest.mark.parametrize("o,v,ot,vt", [(10, 20, 5, 10), (20, 24, 10, 7)])
def test_short_reductions(eng, bits, nmod, o, v, ot, vt):
    wl = configs.with_loss_and_grads(configs.scaled_spin(o, v, ot, vt))
    ew = eng.EngineWorkload(wl, configs.DEFAULT_SEED)
    # the hole-hole term and the ladder's adjoint: both CRT scatters (C along columns and along rows)
    for term in (configs.HOLE_HOLE, next(t for t in wl.extra["adjoint_terms"] if t.name == "dV<-ladder")):
        C = ew.tensors[term.c[0]]
        out = []
        for mode in (eng.EXEC_GROUPED_F64, eng.EXEC_SPLIT_I8):
            eng.check(eng.lib().tmx_set_split_bits(bits))
            try:
                c = ew.contraction(term, mode)
            finally:
                eng.check(eng.lib().tmx_set_split_bits(35))
            C.fill(1.0)
            c.execute()
            out.append(C.download())
        assert c.split_info() == (bits, bits, nmod)
        # 2^-bits of the row maximum (about 4 times the rms of normal data) in each factor
        assert np.linalg.norm(out[1] - out[0]) <= 8.0 * 2.0 ** (1 - bits) * np.linalg.norm(out[0])
