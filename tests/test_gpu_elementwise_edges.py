"""Reductions and the energy denominator at the sizes where their tiling ends: around a vector
pair, a workgroup, a full grid of unrolled loads; unaligned operands; denominators of tensors on
both sides of the chunk-size rule, with blocks of one element and of many chunks."""
import ctypes as C

import numpy as np
import pytest

from tamm_amd import configs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 255, 512, 513, 2047, 2049, 8 * 256 * 2048 - 1, 8 * 256 * 2048 + 3])
@pytest.mark.parametrize("shift", [0, 1])
def test_reductions(eng, n, shift):
    rng = np.random.default_rng(n)
    x, y = rng.standard_normal(n + 1), rng.standard_normal(n + 1)
    dx, dy = eng.DeviceBuffer.from_array(x), eng.DeviceBuffer.from_array(y)
    px, py = dx.ptr + 8 * shift, dy.ptr
    x, y = x[shift:shift + n], y[:n]
    r = C.c_double()
    # FP64 sums of n terms in any order: relative to the sum of magnitudes, n * 2^-53 at worst
    eng.check(eng.lib().tmx_norm(px, n, C.byref(r), None))
    assert abs(r.value - np.linalg.norm(x)) <= 1e-12 * np.linalg.norm(x)
    assert abs(eng.dot(px, py, n) - float(x @ y)) <= 1e-12 * float(np.abs(x) @ np.abs(y))
    ref = np.linalg.norm(x - y) / np.linalg.norm(y)
    assert abs(eng.rel_diff(px, py, n) - ref) <= 1e-12 * max(ref, 1.0)


@pytest.mark.parametrize("o,v,ot,vt,irrep", [(4, 8, 1, 1, False), (5, 7, 2, 3, False), (12, 24, 4, 4, True),
                                             (20, 60, 20, 60, False), (24, 70, 5, 9, False), (16, 96, 16, 48, True)])
def test_denominator(eng, o, v, ot, vt, irrep):
    ho, hv = o // 2, v // 2
    spin = lambda n, h: [(0, h, 1), (h, n, 2)]  # noqa: E731
    irr = lambda n: configs._irrep_ranges(n) if irrep else ()  # noqa: E731
    O, V = eng.Space(o, ot, spin(o, ho), irr(o)), eng.Space(v, vt, spin(v, hv), irr(v))
    t = eng.Tensor([V, V, O, O], (2, 2), irrep).allocate()
    rng = np.random.default_rng(o)
    x = rng.standard_normal(t.size)
    eo, ev = rng.uniform(-2, -0.5, o), rng.uniform(0.2, 3, v)
    t.upload(x)
    de, dv = eng.DeviceBuffer.from_array(eo), eng.DeviceBuffer.from_array(ev)
    eng.check(eng.lib().tmx_energy_denominator(t.h, t.ptr, de.ptr, dv.ptr, None))
    D = eo[None, None, :, None] + eo - ev[:, None, None, None] - ev[None, :, None, None]
    ref = np.empty_like(x)
    nt = [len(s.offsets) - 1 for s in t.spaces]
    for key, off, size in zip(t.keys, t.offsets, t.sizes):
        b = np.unravel_index(int(key), nt)
        sl = tuple(slice(int(s.offsets[i]), int(s.offsets[i + 1])) for s, i in zip(t.spaces, b))
        ref[off:off + size] = x[off:off + size] / D[sl].ravel()
    assert np.max(np.abs(t.download() - ref) / np.abs(ref)) <= 4e-16
