"""Performance cases of the block-sparse contraction engine.

What a coupled-cluster-style program has the engine do, through the public entry points of
tamm_amd.engine: sets of labeled contractions in the forward and the adjoint direction, the
doubles residual of a CC iteration as one level, permuting additions, the amplitude update
with its reductions, and the single-block kernels.  Index spaces have O occupied and V virtual
spin orbitals, from a molecule with a handful of orbitals to the largest workloads of
tamm_amd.configs; tilings are uniform, or drawn between two sizes inside every spin and C2v
irrep range, which makes ragged blocks.

A case:
  kind       terms    R = ladder + ring + hole-hole, each contraction executed on its own
             adjoint  the six adjoint contractions of those terms, into dV, dW, dX and dT
             step     the ten-term doubles residual as one level, then the energy denominator
             antisym  R(abij) = T(abij) - T(baij) - T(abji) + T(baji), four AddOps
             update   t = residual / denominator, T += t, norm of t, <residual, T>
             block    one block pair multiplied into a C block, which is then added, permuted,
                      into another block
  o, v       occupied and virtual spin orbitals
  otile, vtile      the largest tile of each space
  otile_lo, vtile_lo  the smallest one drawn; equal to the largest: uniform tiles
  tiling     seed of the drawn tile sizes
  spin       the tensors keep spin ({2,2} masks; {1,1} for one-body tensors)
  irrep      and the C2v irreps
  mode       auto (FP64) or auto_split (split precision where it pays)
"""
import numpy as np
import torch

from tamm_amd import engine

# Tensors: modes (o / v) and the scale of their normally distributed elements.
TENSORS = {
    "V": ("vvvv", 0.1), "W": ("ovvo", 0.1), "X": ("oooo", 0.1), "T": ("vvoo", 0.01),
    "L": ("vvoo", 0.01), "R": ("vvoo", 0.0), "Fv": ("vv", 0.05), "Fo": ("oo", 0.05),
    "dV": ("vvvv", 0.0), "dW": ("ovvo", 0.0), "dX": ("oooo", 0.0), "dT": ("vvoo", 0.0),
}
# C, its labels, alpha, A, its labels, B, its labels
LADDER = ("R", "abij", 1.0, "V", "abcd", "T", "cdij")
RING = ("R", "abij", 1.0, "W", "kbcj", "T", "acik")
HOLES = ("R", "abij", 1.0, "X", "klij", "T", "abkl")
FORWARD = [LADDER, RING, HOLES]
ADJOINT = [
    ("dV", "abcd", 1.0, "L", "abij", "T", "cdij"), ("dT", "cdij", 1.0, "L", "abij", "V", "abcd"),
    ("dW", "kbcj", 1.0, "L", "abij", "T", "acik"), ("dT", "acik", 1.0, "L", "abij", "W", "kbcj"),
    ("dX", "klij", 1.0, "L", "abij", "T", "abkl"), ("dT", "abkl", 1.0, "L", "abij", "X", "klij"),
]
STEP = [
    LADDER, HOLES, RING,
    ("R", "abij", -1.0, "W", "kacj", "T", "bcik"), ("R", "abij", -1.0, "W", "kbci", "T", "acjk"),
    ("R", "abij", 1.0, "W", "kaci", "T", "bcjk"),
    ("R", "abij", 1.0, "Fv", "ac", "T", "cbij"), ("R", "abij", 1.0, "Fv", "bc", "T", "acij"),
    ("R", "abij", -1.0, "Fo", "ki", "T", "abkj"), ("R", "abij", -1.0, "Fo", "kj", "T", "abik"),
]
PROGRAMS = {"terms": FORWARD, "adjoint": ADJOINT, "step": STEP}
OUTPUTS = {"terms": ["R"], "adjoint": ["dV", "dW", "dX", "dT"], "step": ["R"]}
SPACE_OF = {c: "v" for c in "abcd"} | {c: "o" for c in "ijkl"}
MODES = {"auto": engine.EXEC_AUTO, "auto_split": engine.EXEC_AUTO_SPLIT}


def _case(name, kind, o, v, otile, vtile, *, lo=None, spin=True, irrep=False, mode="auto", tiling=1):
    c = {"kind": kind, "o": o, "v": v, "otile": otile, "vtile": vtile,
         "otile_lo": lo[0] if lo else otile, "vtile_lo": lo[1] if lo else vtile,
         "spin": spin, "irrep": irrep, "mode": mode, "tiling": tiling}
    return {"name": name, **c} if name else c


def listed():
    return [
        # kernels::block_multiply and kernels::assign on one block pair, as a program that walks
        # the blocks by itself calls them
        _case("block_pair", "block", 16, 36, 16, 36, spin=False),
        # the smallest molecule: launches and their latency
        _case("terms_o4_v8", "terms", 4, 8, 2, 3),
        # many tiny ragged blocks: the residual of a small molecule with point-group symmetry
        _case("step_o12_v24", "step", 12, 24, 4, 4, lo=(1, 1), irrep=True),
        # a small dense problem without symmetry
        _case("dense_o20_v80", "terms", 20, 80, 10, 20, spin=False),
        # the ordinary iteration, in FP64 and in split precision, and its gradient
        _case("terms_o30_v180_f64", "terms", 30, 180, 16, 36),
        _case("terms_o30_v180_split", "terms", 30, 180, 16, 36, mode="auto_split"),
        _case("adjoint_o30_v180_split", "adjoint", 30, 180, 16, 36, mode="auto_split"),
        # symmetry-blocked spaces with ragged tiles
        _case("terms_o50_v320_irrep_split", "terms", 50, 320, 96, 96, lo=(24, 24), irrep=True,
              mode="auto_split"),
        # a whole doubles residual with the energy denominator
        _case("step_o60_v300_split", "step", 60, 300, 80, 80, lo=(32, 32), irrep=True,
              mode="auto_split"),
        # the largest integrals
        _case("terms_o40_v240_split", "terms", 40, 240, 16, 48, mode="auto_split"),
        # the memory-bound ends of an iteration, at the largest amplitudes
        _case("antisym_o40_v240", "antisym", 40, 240, 16, 48),
        _case("update_o40_v240", "update", 40, 240, 16, 48),
    ]


def draw(rng):
    def size(lo, hi):  # spread over the logarithm
        return int(round(lo * (hi / lo) ** rng.random()))

    kind = rng.choice(["block", "small", "terms", "terms", "adjoint", "step", "antisym", "update"])
    tiling, mode = rng.randrange(1 << 16), rng.choice(["auto", "auto_split"])
    if kind == "block":
        ot, vt = size(4, 24), size(8, 48)
        return _case(None, "block", ot, vt, ot, vt, spin=False, tiling=tiling)
    if kind == "small":
        o, v = size(4, 20), size(8, 80)
        ot, vt = size(max(2, o // 6), max(3, o // 2)), size(max(3, v // 10), max(4, v // 3))
        return _case(None, rng.choice(["terms", "step", "adjoint"]), o, v, ot, vt,
                     lo=(max(1, ot // 3), max(1, vt // 3)), spin=rng.random() < 0.8, mode=mode, tiling=tiling)
    o, v = size(16, 40), size(90, 220)
    ot, vt = size(8, 20), size(24, 60)
    if kind == "adjoint":
        v = min(v, 160)
    irrep = rng.random() < 0.4
    lo = None if rng.random() < 0.5 else (max(1, ot // 2), max(1, vt // 2))
    return _case(None, kind, o, v, ot, vt, lo=lo, irrep=irrep, mode=mode, tiling=tiling)


# --- structure, written out here so that exact() needs nothing of the engine ---------------------

def _ranges(case, n):
    """(lo, hi, spin, irrep) of the attribute ranges: two spin halves, four irreps in each."""
    if not case["spin"]:
        return [(0, n, 0, 0)]
    out, h = [], n // 2
    for spin, base, size in ((1, 0, h), (2, h, n - h)):
        counts = [(size - r + 3) // 4 if size > r else 0 for r in range(4)] if case["irrep"] else [size]
        lo = base
        for irrep, cnt in enumerate(counts):
            if cnt:
                out.append((lo, lo + cnt, spin, irrep))
                lo += cnt
    return out


def _tiles(case, which):
    """Tiles of a space: arrays of their first index, size, spin and irrep."""
    hi_t, lo_t = case[which + "tile"], case[which + "tile_lo"]
    r = np.random.RandomState(case["tiling"] * 2 + (which == "v"))
    first, size, spin, irrep = [], [], [], []
    for lo, hi, s, x in _ranges(case, case[which]):
        while lo < hi:
            t = min(hi_t if lo_t == hi_t else int(r.randint(lo_t, hi_t + 1)), hi - lo)
            first.append(lo), size.append(t), spin.append(s), irrep.append(x)
            lo += t
    return np.array(first), np.array(size), np.array(spin), np.array(irrep)


def _nonzero(case, modes, attr):
    """Mask over the tiles (or ranges) of every mode: spin of the upper half of the modes equal to
    that of the lower half, and the irreps' product the symmetric one."""
    n = len(modes)
    shape = lambda i, x: x.reshape([-1 if j == i else 1 for j in range(n)])  # noqa: E731
    ok = np.ones([len(attr[m][0]) for m in modes], dtype=bool)
    if case["spin"]:
        ok &= sum(shape(i, attr[m][0]) * (1 if i < n // 2 else -1) for i, m in enumerate(modes)) == 0
        x = 0
        for i, m in enumerate(modes):
            x = x ^ shape(i, attr[m][1])
        ok &= x == 0
    return ok


def _blocks(case, modes):
    """(offset, slices, extents) of the stored blocks in their order, and the element count."""
    tiles = {m: _tiles(case, m) for m in set(modes)}
    ok = _nonzero(case, modes, {m: t[2:] for m, t in tiles.items()})
    out, off = [], 0
    for bid in np.argwhere(ok):
        ext = [int(tiles[m][1][b]) for m, b in zip(modes, bid)]
        lo = [int(tiles[m][0][b]) for m, b in zip(modes, bid)]
        out.append((off, tuple(slice(x, x + e) for x, e in zip(lo, ext)), ext))
        off += int(np.prod(ext))
    return out, off


def _elements(case, name):
    modes = TENSORS[name][0]
    ranges = {m: _ranges(case, case[m]) for m in set(modes)}
    attr = {m: np.array([r[2:] for r in ranges[m]]).T for m in ranges}
    ok = _nonzero(case, modes, attr).astype(float)
    for m in modes:
        ok = np.tensordot(ok, np.array([r[1] - r[0] for r in ranges[m]], dtype=float), axes=(0, 0))
    return float(ok)


def _flops(case, term):
    _, cl, _, a, al, b, bl = term
    labels = sorted(set(al + bl))
    ranges = {m: _ranges(case, case[m]) for m in "ov"}
    attr = {m: np.array([r[2:] for r in ranges[m]]).T for m in "ov"}
    args = []
    for lab in (cl, al, bl):
        args += [_nonzero(case, [SPACE_OF[c] for c in lab], attr).astype(float), [labels.index(c) for c in lab]]
    for c in labels:
        args += [np.array([r[1] - r[0] for r in ranges[SPACE_OF[c]]], dtype=float), [labels.index(c)]]
    return 2.0 * float(np.einsum(*args, [], optimize=True))


def work(case):
    kind = case["kind"]
    if kind == "block":
        o, v = case["o"], case["v"]
        c = v * v * o * o
        return {"bytes": 8.0 * (v ** 4 + c + c + 2 * c), "flops": 2.0 * v ** 4 * o * o}
    amp = _elements(case, "T")
    if kind == "antisym":  # T read, R written
        return {"bytes": 8.0 * 2 * amp, "flops": 3.0 * amp}
    if kind == "update":  # residual and T read, t and T written
        return {"bytes": 8.0 * 4 * amp, "flops": 9.0 * amp}
    terms = PROGRAMS[kind]
    names = {n for t in terms for n in (t[0], t[3], t[5])}
    return {"bytes": 8.0 * sum(_elements(case, n) for n in names), "flops": sum(_flops(case, t) for t in terms)}


# --- inputs ---------------------------------------------------------------------------------------

def _gen(seed, what):
    return torch.Generator(device="cuda").manual_seed(seed * 64 + what)


def _fill(x, name, seed):
    """Elements of a tensor's stored blocks, in their order."""
    return x.normal_(0.0, TENSORS[name][1], generator=_gen(seed, list(TENSORS).index(name)))


def _energies(case, seed):
    eo = torch.rand(case["o"], generator=_gen(seed, 40), dtype=torch.float64, device="cuda") * 1.5 - 2.0
    ev = torch.rand(case["v"], generator=_gen(seed, 41), dtype=torch.float64, device="cuda") * 2.8 + 0.2
    return eo, ev


class _Memory:
    """A tensor's or buffer's device memory, for torch (which keeps the owner alive)."""

    def __init__(self, owner, n):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (int(n),), "typestr": "<f8", "data": (owner.ptr, False),
                                         "version": 3, "strides": None}


def _view(owner, n):
    return torch.as_tensor(_Memory(owner, n), device="cuda")


def _spaces(case):
    out = {}
    for w in "ov":
        r = _ranges(case, case[w])
        spin = irrep = ()
        if case["spin"]:
            spin = [(a, b, s) for a, b, s, _ in r]
            irrep = [(a, b, x) for a, b, _, x in r] if case["irrep"] else ()
        out[w] = engine.Space(case[w], [int(t) for t in _tiles(case, w)[1]], spin, irrep)
    return out


def _tensors(case, names, seed):
    """Tensors in HBM, the inputs filled, and torch's views of them."""
    sp = _spaces(case)
    ts, views = {}, {}
    for n in names:
        modes = TENSORS[n][0]
        half = len(modes) // 2
        t = engine.Tensor([sp[m] for m in modes], (half, half) if case["spin"] else None,
                          case["spin"] and case["irrep"]).allocate()
        ts[n], views[n] = t, _view(t, t.size)
        if TENSORS[n][1]:
            _fill(views[n], n, seed)
        else:
            views[n].zero_()
    return ts, views


LABEL = {c: -(i + 1) for i, c in enumerate("abcdijkl")}


def prepare(case, seed):
    engine.init(0, 0.6)
    kind = case["kind"]
    st = {"kind": kind}
    if kind == "block":
        o, v = case["o"], case["v"]
        dims = {"A": (v, v, v, v), "B": (v, v, o, o), "C": (v, v, o, o), "D": (v, v, o, o)}
        for i, (k, d) in enumerate(dims.items()):
            n = int(np.prod(d))
            st[k] = engine.DeviceBuffer(8 * n)
            st["view" + k] = _view(st[k], n)
            st["view" + k].normal_(0.0, 0.1, generator=_gen(seed, 50 + i))
        st["dims"] = dims
    elif kind in ("antisym", "update"):
        names = ["T", "R"] + (["L"] if kind == "update" else [])
        st["t"], st["views"] = _tensors(case, names, seed)
        lab = lambda s: [LABEL[c] for c in s]  # noqa: E731
        T, R = st["t"]["T"], st["t"]["R"]
        if kind == "antisym":
            st["ops"] = [engine.AddOp(R, lab("abij"), 1.0, T, lab("abij"), True)] + [
                engine.AddOp(R, lab("abij"), s, T, lab(p)) for s, p in ((-1.0, "baij"), (-1.0, "abji"), (1.0, "baji"))]
        else:
            st["ops"] = [engine.AddOp(R, lab("abij"), 1.0, st["t"]["L"], lab("abij"), True)]
            st["e"] = [engine.DeviceBuffer(8 * len(x)) for x in _energies(case, seed)]
            for b, x in zip(st["e"], _energies(case, seed)):
                _view(b, len(x)).copy_(x)
    else:
        terms = PROGRAMS[kind]
        st["t"], st["views"] = _tensors(case, dict.fromkeys(n for t in terms for n in (t[0], t[3], t[5])), seed)
        st["plans"], seen = [], set()
        for c, cl, alpha, a, al, b, bl in terms:
            p = engine.Contraction(st["t"][c], [LABEL[x] for x in cl], alpha, st["t"][a], [LABEL[x] for x in al],
                                   st["t"][b], [LABEL[x] for x in bl], MODES[case["mode"]])
            if c not in seen:  # the first term into a tensor assigns it
                p.set_assign(True)
            seen.add(c)
            st["plans"].append(p)
        if kind == "step":
            st["level"] = engine.Level(st["plans"])
            st["e"] = [engine.DeviceBuffer(8 * len(x)) for x in _energies(case, seed)]
            for b, x in zip(st["e"], _energies(case, seed)):
                _view(b, len(x)).copy_(x)
    torch.cuda.synchronize()
    return st


def _divide(st, name):
    t = st["t"][name]
    engine.check(engine.lib().tmx_energy_denominator(t.h, t.ptr, st["e"][0].ptr, st["e"][1].ptr, None))


def run(st):
    kind = st["kind"]
    if kind == "block":
        d = st["dims"]
        engine.block_multiply(0.5, st["A"], d["A"], (1, 2, 3, 4), st["B"], d["B"], (3, 4, 5, 6),
                              st["C"], d["C"], (1, 2, 5, 6), is_assign=True)
        engine.block_assign(st["D"], d["D"], (1, 2, 5, 6), -1.0, st["C"], d["C"], (2, 1, 6, 5), is_assign=False)
        return {"C": st["viewC"], "D": st["viewD"]}
    if kind == "antisym":
        for op in st["ops"]:
            op.execute()
        return {"R": st["views"]["R"]}
    if kind == "update":
        T, R, L = st["t"]["T"], st["t"]["R"], st["t"]["L"]
        st["ops"][0].execute()
        _divide(st, "R")
        T.axpy(1.0, R)
        return {"R": st["views"]["R"], "T": st["views"]["T"], "norm": R.norm(), "energy": L.dot(T)}
    if kind == "step":
        st["level"].execute()
        _divide(st, "R")
    else:
        for p in st["plans"]:
            p.execute()
    return {n: st["views"][n] for n in OUTPUTS[kind]}


# --- the same in plain torch, FP64 ----------------------------------------------------------------

def _input(case, name, seed):
    _, n = _blocks(case, TENSORS[name][0])
    return _fill(torch.empty(n, dtype=torch.float64, device="cuda"), name, seed)


def _dense(case, name, packed):
    modes = TENSORS[name][0]
    out = torch.zeros([case[m] for m in modes], dtype=torch.float64, device="cuda")
    for off, sl, ext in _blocks(case, modes)[0]:
        out[sl] = packed[off:off + int(np.prod(ext))].view(ext)
    return out


def _packed(case, name, dense):
    return torch.cat([dense[sl].reshape(-1) for _, sl, _ in _blocks(case, TENSORS[name][0])[0]])


def exact(case, seed):
    kind = case["kind"]
    if kind == "block":
        o, v = case["o"], case["v"]
        dims = {"A": (v, v, v, v), "B": (v, v, o, o), "C": (v, v, o, o), "D": (v, v, o, o)}
        x = {k: torch.empty(int(np.prod(d)), dtype=torch.float64, device="cuda")
             .normal_(0.0, 0.1, generator=_gen(seed, 50 + i)).view(d) for i, (k, d) in enumerate(dims.items())}
        c = 0.5 * torch.einsum("abcd,cdij->abij", x["A"], x["B"])
        return {"C": c.reshape(-1), "D": (x["D"] - c.permute(1, 0, 3, 2)).reshape(-1)}
    if kind == "antisym":
        t = _dense(case, "T", _input(case, "T", seed))
        t = t - t.permute(1, 0, 2, 3)
        return {"R": _packed(case, "R", t - t.permute(0, 1, 3, 2))}
    eo, ev = _energies(case, seed)
    D = lambda: (eo[:, None] + eo)[None, None] - (ev[:, None] + ev)[:, :, None, None]  # noqa: E731
    if kind == "update":
        L, T = _input(case, "L", seed), _input(case, "T", seed)
        R = L / _packed(case, "R", D())
        T = T + R
        return {"R": R, "T": T, "norm": float(R.norm()), "energy": float(torch.dot(L, T))}
    terms = PROGRAMS[kind]
    inputs = {n for t in terms for n in (t[3], t[5])}
    x = {n: _dense(case, n, _input(case, n, seed)) for n in sorted(inputs)}
    out = {}
    for c, cl, alpha, a, al, b, bl in terms:
        y = torch.einsum("%s,%s->%s" % (al, bl, cl), x[a], x[b])
        out[c] = out[c].add_(y, alpha=alpha) if c in out else y.mul_(alpha)
        del y
    x.clear()
    if kind == "step":
        out["R"] /= D()
    return {n: _packed(case, n, out.pop(n)) for n in OUTPUTS[kind]}
