// plan_bp.cpp -- label analysis, execute_bufacc pair enumeration, the fused block-pair plan,
// the contraction object and the block-level entry points.
#include <atomic>
#include <cmath>
#include <numeric>
#include <unordered_map>

#include "plan.hpp"

namespace tmx {

std::vector<int64_t> strides_of(const std::vector<int64_t>& dims) {
  std::vector<int64_t> s(dims.size(), 1);
  for (int i = (int)dims.size() - 2; i >= 0; --i) s[i] = s[i + 1] * dims[i + 1];
  return s;
}

LabelInfo analyse_labels(const LOperand& C, const LOperand& A, const LOperand& B) {
  LabelInfo li;
  auto uniq = [](const std::vector<int>& v, const char* who) {
    std::vector<int> s = v;
    std::sort(s.begin(), s.end());
    TMX_REQUIRE(std::adjacent_find(s.begin(), s.end()) == s.end(),
                std::string("a label repeats within operand ") + who);
  };
  uniq(C.labels, "C");
  uniq(A.labels, "A");
  uniq(B.labels, "B");
  auto in = [](const std::vector<int>& v, int l) { return pos_of(v, l) >= 0; };
  for (int l : C.labels) {  // multiply.hpp:238-263
    bool ia = in(A.labels, l), ib = in(B.labels, l);
    TMX_REQUIRE(ia || ib, "an output label does not occur on the right-hand side");
    if (ia && ib) li.batch.push_back(l);
    else if (ia) li.aouter.push_back(l);
    else li.bouter.push_back(l);
  }
  for (int l : A.labels) {  // :265-283
    bool ib = in(B.labels, l), ic = in(C.labels, l);
    if (ib && !ic) li.inner.push_back(l);
    else if (!ib && !ic) li.ared.push_back(l);
  }
  for (int l : B.labels)  // :285-302
    if (!in(A.labels, l) && !in(C.labels, l)) li.bred.push_back(l);
  std::vector<int> rhs = A.labels;
  rhs.insert(rhs.end(), B.labels.begin(), B.labels.end());
  std::sort(rhs.begin(), rhs.end());
  rhs.erase(std::unique(rhs.begin(), rhs.end()), rhs.end());
  for (int l : rhs)
    if (!in(C.labels, l)) li.red.push_back(l);
  // Tile sizes of each label's space; every occurrence must agree (labels of one space).
  auto add = [&](const LOperand& o) {
    for (size_t i = 0; i < o.labels.size(); ++i) {
      std::vector<int64_t> ts;
      const Space& sp = *o.t->modes[i];
      for (int64_t t = 0; t < o.ntl[i]; ++t) ts.push_back(sp.tsize(o.toff[i] + t));
      auto it = li.tile_sizes.find(o.labels[i]);
      if (it == li.tile_sizes.end()) li.tile_sizes[o.labels[i]] = ts;
      else TMX_REQUIRE(it->second == ts, "a label is used over index spaces with different tilings");
    }
  };
  add(C);
  add(A);
  add(B);
  return li;
}

std::vector<int64_t> block_dims(const LOperand& op, const std::vector<int64_t>& label_tiles) {
  std::vector<int64_t> d;
  for (size_t i = 0; i < op.labels.size(); ++i)
    d.push_back(op.t->modes[i]->tsize(op.toff[i] + label_tiles[i]));
  return d;
}

std::vector<CBlockWork> enumerate_pairs(const LOperand& C, const LOperand& A, const LOperand& B,
                                        const LabelInfo& li) {
  std::vector<CBlockWork> out;
  const size_t nc = C.labels.size(), nr = li.red.size();
  std::vector<int64_t> cext(nc), rext(nr);
  for (size_t i = 0; i < nc; ++i) cext[i] = C.ntl[i];
  for (size_t i = 0; i < nr; ++i) rext[i] = (int64_t)li.tile_sizes.at(li.red[i]).size();
  for (auto e : cext) if (e == 0) return out;
  bool red_empty = false;
  for (auto e : rext) if (e == 0) red_empty = true;
  // operand label -> source (C label index or reduction label index)
  auto src_map = [&](const LOperand& o, std::vector<int>& from_c, std::vector<int>& from_r) {
    for (int l : o.labels) {
      from_c.push_back(pos_of(C.labels, l));
      from_r.push_back(pos_of(li.red, l));
    }
  };
  std::vector<int> a_c, a_r, b_c, b_r;
  src_map(A, a_c, a_r);
  src_map(B, b_c, b_r);
  auto next = [](std::vector<int64_t>& v, const std::vector<int64_t>& e) {
    for (int i = (int)v.size() - 1; i >= 0; --i) {
      if (++v[i] < e[i]) return true;
      v[i] = 0;
    }
    return false;
  };
  std::vector<int64_t> ct(nc, 0), cb(nc), ab(A.labels.size()), bb(B.labels.size());
  do {
    for (size_t i = 0; i < nc; ++i) cb[i] = C.toff[i] + ct[i];
    if (!C.t->is_non_zero(cb.data())) continue;
    CBlockWork w;
    w.c_off = C.t->find(cb.data());
    w.ct = ct;
    if (!red_empty) {
      std::vector<int64_t> rt(nr, 0);
      do {
        for (size_t i = 0; i < ab.size(); ++i)
          ab[i] = A.toff[i] + (a_c[i] >= 0 ? ct[a_c[i]] : rt[a_r[i]]);
        if (!A.t->is_non_zero(ab.data())) continue;
        for (size_t i = 0; i < bb.size(); ++i)
          bb[i] = B.toff[i] + (b_c[i] >= 0 ? ct[b_c[i]] : rt[b_r[i]]);
        if (!B.t->is_non_zero(bb.data())) continue;
        PairRef pr;
        pr.a_off = A.t->find(ab.data());
        pr.b_off = B.t->find(bb.data());
        pr.rt = rt;
        w.pairs.push_back(std::move(pr));
      } while (next(rt, rext));
    }
    out.push_back(std::move(w));
  } while (next(ct, cext));
  return out;
}

namespace {

Radix make_radix(const std::vector<int64_t>& ext, const std::vector<int64_t>& stride) {
  Radix r;
  std::memset(&r, 0, sizeof(r));
  TMX_REQUIRE(ext.size() <= (size_t)MAXR, "too many modes in one GEMM role");
  r.n = (int)ext.size();
  for (int i = 0; i < r.n; ++i) {
    TMX_REQUIRE(ext[i] < (1ll << 31) && stride[i] < (1ll << 31), "block too large");
    r.ext[i] = (int)ext[i];
    r.stride[i] = (int)stride[i];
  }
  return r;
}

template <class T>
std::vector<int64_t> key_of(const T& v) {
  std::vector<int64_t> k(sizeof(T) / sizeof(int32_t));
  const int32_t* p = reinterpret_cast<const int32_t*>(&v);
  for (size_t i = 0; i < k.size(); ++i) k[i] = p[i];
  return k;
}

template <class T>
int intern(std::vector<T>& table, std::map<std::vector<int64_t>, int>& index, const T& v) {
  auto k = key_of(v);
  auto it = index.find(k);
  if (it != index.end()) return it->second;
  int id = (int)table.size();
  table.push_back(v);
  index[k] = id;
  return id;
}

}  // namespace

static void build_bp_plan_as(BPPlan& plan, const LOperand& C, const LOperand& A, const LOperand& B,
                             const LabelInfo& li, const std::vector<CBlockWork>& work,
                             bool per_pair_launches, double* flops_out, int64_t* npairs_out,
                             int tile) {
  const int TM = bp_tile_rows(tile), TN = bp_tile_cols(tile);
  plan.tile = tile;
  std::vector<BPTask> tasks;
  std::vector<BPPair> pairs;
  std::vector<BPCShape> cshapes;
  std::vector<BPKShape> kshapes;
  // Shapes by the tile sizes of the labels they depend on, each size as its index among the
  // label's distinct ones: C's labels for a C shape, those and the reduction's for a K shape.
  std::map<std::vector<int64_t>, int> cidx;
  std::unordered_map<std::string, int> kidx;
  auto size_ids = [&](int l) {
    const std::vector<int64_t>& sz = li.tile_sizes.at(l);
    std::vector<int64_t> distinct(sz);
    std::sort(distinct.begin(), distinct.end());
    distinct.erase(std::unique(distinct.begin(), distinct.end()), distinct.end());
    std::vector<uint16_t> id;
    for (int64_t x : sz)
      id.push_back((uint16_t)(std::lower_bound(distinct.begin(), distinct.end(), x) - distinct.begin()));
    TMX_REQUIRE(distinct.size() < 65536, "too many distinct tile sizes");
    return id;
  };
  std::vector<std::vector<uint16_t>> c_ids, r_ids;
  for (int l : C.labels) c_ids.push_back(size_ids(l));
  for (int l : li.red) r_ids.push_back(size_ids(l));
  std::vector<BPTask> pair_tasks;
  double flops = 0;
  int64_t npairs = 0;
  std::vector<std::pair<int64_t, int>> cost_task;  // for LPT ordering

  // Label -> tile index lookup for one triple.
  auto tiles_for = [&](const LOperand& o, const std::vector<int64_t>& ct,
                       const std::vector<int64_t>& rt) {
    std::vector<int64_t> t;
    for (int l : o.labels) {
      int pc = pos_of(C.labels, l);
      t.push_back(pc >= 0 ? ct[pc] : rt[pos_of(li.red, l)]);
    }
    return t;
  };
  auto dims_of = [&](const LOperand& o, const std::vector<int64_t>& tiles, const std::vector<int>& ls,
                     std::vector<int64_t>& ext, std::vector<int64_t>& str) {
    std::vector<int64_t> d = block_dims(o, tiles), s = strides_of(d);
    ext.clear();
    str.clear();
    for (int l : ls) {
      int p = pos_of(o.labels, l);
      ext.push_back(p >= 0 ? d[p] : 0);
      str.push_back(p >= 0 ? s[p] : 0);
    }
  };
  std::vector<int> kl = li.inner;  // K modes: inner, A-reduce, B-reduce
  kl.insert(kl.end(), li.ared.begin(), li.ared.end());
  kl.insert(kl.end(), li.bred.begin(), li.bred.end());
  // Digit order of each GEMM role.  The M, N and K indices are enumerations private to this
  // plan (the A/B/C radices of a role all use one order), so each role's last, fastest digit
  // is chosen as the stride-1 mode of the operand the kernel reads along it: A's last mode
  // when it is an M mode, B's when it is an N mode, and for K the stride-1 K mode of the
  // larger operand (A's on a tie).  A wave's 16 or 64 consecutive indices are then one
  // contiguous run of that operand's block; in TAMM's label order they can be a stride of
  // thousands of elements (R(a,b,i,j) += W(k,b,c,j) T(a,c,i,k): K = (k,c) puts c, of stride
  // 256 in T, where the loads along T's k expect stride 1).
  std::vector<int> mo = li.aouter, no = li.bouter;
  auto to_back = [](std::vector<int>& v, int l) {
    auto it = std::find(v.begin(), v.end(), l);
    if (it == v.end()) return false;
    v.erase(it);
    v.push_back(l);
    return true;
  };
  if (!A.labels.empty()) to_back(mo, A.labels.back());
  if (!B.labels.empty()) to_back(no, B.labels.back());
  {
    const bool ak = !A.labels.empty() && pos_of(kl, A.labels.back()) >= 0;
    const bool bk = !B.labels.empty() && pos_of(kl, B.labels.back()) >= 0;
    if (ak && (!bk || A.t->total >= B.t->total)) to_back(kl, A.labels.back());
    else if (bk) to_back(kl, B.labels.back());
  }

  std::vector<BPPair> pinfo;
  for (const CBlockWork& w : work) {
    if (w.pairs.empty()) continue;
    std::vector<int64_t> rt0(li.red.size(), 0);
    std::vector<int64_t> ctiles = tiles_for(C, w.ct, rt0);
    std::vector<int64_t> cext, cstr, nce, ncs, bte, bts;
    dims_of(C, ctiles, mo, cext, cstr);
    dims_of(C, ctiles, no, nce, ncs);
    dims_of(C, ctiles, li.batch, bte, bts);
    int64_t M = 1, N = 1, Bn = 1;
    for (auto e : cext) M *= e;
    for (auto e : nce) N *= e;
    for (auto e : bte) Bn *= e;
    BPCShape cs;
    std::memset(&cs, 0, sizeof(cs));
    cs.M = (int)M;
    cs.N = (int)N;
    cs.ncontig = !no.empty() && !C.labels.empty() && C.labels.back() == no.back() ? 1 : 0;
    cs.cm = make_radix(cext, cstr);
    cs.cn = make_radix(nce, ncs);
    int csid = intern(cshapes, cidx, cs);

    // Per pair: K shape and base offsets (batch element added below).
    pinfo.clear();
    std::string key((C.labels.size() + li.red.size()) * 2, '\0');
    auto put = [&](size_t i, uint16_t v) { std::memcpy(&key[2 * i], &v, 2); };
    for (size_t i = 0; i < C.labels.size(); ++i) put(i, c_ids[i][(size_t)w.ct[i]]);
    for (const PairRef& pr : w.pairs) {
      for (size_t i = 0; i < li.red.size(); ++i) put(C.labels.size() + i, r_ids[i][(size_t)pr.rt[i]]);
      auto it = kidx.find(key);
      if (it == kidx.end()) {
        const std::vector<int64_t> at = tiles_for(A, w.ct, pr.rt), bt = tiles_for(B, w.ct, pr.rt);
        BPKShape ks;
        std::memset(&ks, 0, sizeof(ks));
        std::vector<int64_t> e, s;
        dims_of(A, at, mo, e, s);
        ks.am = make_radix(e, s);
        dims_of(B, bt, no, e, s);
        ks.bn = make_radix(e, s);
        // K radix: extents from whichever operand holds the label, strides 0 where absent.
        std::vector<int64_t> kext, ka, kb;
        const std::vector<int64_t> ad = block_dims(A, at), as = strides_of(ad);
        const std::vector<int64_t> bd = block_dims(B, bt), bs = strides_of(bd);
        for (int l : kl) {
          int pa = pos_of(A.labels, l), pb = pos_of(B.labels, l);
          kext.push_back(pa >= 0 ? ad[pa] : bd[pb]);
          ka.push_back(pa >= 0 ? as[pa] : 0);
          kb.push_back(pb >= 0 ? bs[pb] : 0);
        }
        int64_t K = 1;
        for (auto x : kext) K *= x;
        TMX_REQUIRE(K < (1ll << 31), "reduction block too large");
        ks.K = (int)K;
        ks.ak = make_radix(kext, ka);
        ks.bk = make_radix(kext, kb);
        // Read along K when the operand's stride-1 mode is the fastest K digit (above), else
        // along its rows, whose fastest digit is then its stride-1 mode where that is an
        // outer mode.
        ks.a_kcontig = (!kl.empty() && !A.labels.empty() && A.labels.back() == kl.back()) ? 1 : 0;
        ks.b_kcontig = (!kl.empty() && !B.labels.empty() && B.labels.back() == kl.back()) ? 1 : 0;
        it = kidx.emplace(key, (int)kshapes.size()).first;
        kshapes.push_back(ks);
      }
      BPPair p;
      p.a_off = pr.a_off;
      p.b_off = pr.b_off;
      p.kshape = it->second;
      p.K = kshapes[(size_t)it->second].K;
      pinfo.push_back(p);
      flops += 2.0 * (double)M * (double)N * (double)p.K * (double)Bn;
      ++npairs;
    }
    // Batch elements: offsets of each batch index in C, A (per pair), B (per pair).
    std::vector<int64_t> bidx(li.batch.size(), 0);
    for (int64_t be = 0; be < Bn; ++be) {
      int64_t coff = w.c_off;
      {
        int64_t rem = be;
        for (int i = (int)li.batch.size() - 1; i >= 0; --i) { bidx[i] = rem % bte[i]; rem /= bte[i]; }
        for (size_t i = 0; i < li.batch.size(); ++i) coff += bidx[i] * bts[i];
      }
      int pbeg = (int)pairs.size();
      int64_t kcost = 0;
      for (size_t q = 0; q < pinfo.size(); ++q) {
        BPPair p = pinfo[q];
        if (!li.batch.empty()) {
          const std::vector<int64_t>& rt = w.pairs[q].rt;
          std::vector<int64_t> e, s;
          dims_of(A, tiles_for(A, w.ct, rt), li.batch, e, s);
          for (size_t i = 0; i < li.batch.size(); ++i) p.a_off += bidx[i] * s[i];
          dims_of(B, tiles_for(B, w.ct, rt), li.batch, e, s);
          for (size_t i = 0; i < li.batch.size(); ++i) p.b_off += bidx[i] * s[i];
        }
        pairs.push_back(p);
        kcost += p.K;
      }
      int pend = (int)pairs.size();
      for (int64_t m0 = 0; m0 < M; m0 += TM)
        for (int64_t n0 = 0; n0 < N; n0 += TN) {
          BPTask t;
          t.c_off = coff;
          t.m0 = (int)m0;
          t.n0 = (int)n0;
          t.cshape = csid;
          t.pair_begin = pbeg;
          t.pair_end = pend;
          t.pad = 0;
          cost_task.push_back({kcost, (int)tasks.size()});
          tasks.push_back(t);
        }
    }
  }
  // Tasks stay in C-block order (the tiles of a block in a row, neighbouring blocks sharing
  // operand blocks) and are cut into 8 contiguous ranges of equal reduction work, one per XCD,
  // so each XCD's L2 serves the re-reads of its own blocks' operands.
  std::vector<BPTask> ordered = tasks;
  {
    double total = 0;
    for (auto& ct : cost_task) total += (double)ct.first;
    int x = 0;
    double acc = 0;
    plan.xcd.lo[0] = 0;
    for (size_t i = 0; i < cost_task.size(); ++i) {
      acc += (double)cost_task[i].first;
      while (x < 7 && acc >= total * (x + 1) / 8.0) {
        plan.xcd.hi[x] = (int)i + 1;
        plan.xcd.lo[++x] = (int)i + 1;
      }
    }
    for (; x < 7; ) { plan.xcd.hi[x] = (int)cost_task.size(); plan.xcd.lo[++x] = (int)cost_task.size(); }
    plan.xcd.hi[7] = (int)cost_task.size();
  }
  if (per_pair_launches) {
    // One launch per block pair, in execute_bufacc order: the tiles of the C block, one pair.
    std::vector<BPTask> byblock = tasks;  // original (block-major) order
    size_t i = 0;
    while (i < byblock.size()) {
      size_t j = i;
      while (j < byblock.size() && byblock[j].pair_begin == byblock[i].pair_begin &&
             byblock[j].c_off == byblock[i].c_off)
        ++j;
      for (int p = byblock[i].pair_begin; p < byblock[i].pair_end; ++p) {
        int beg = (int)pair_tasks.size();
        for (size_t k = i; k < j; ++k) {
          BPTask t = byblock[k];
          t.pair_begin = p;
          t.pair_end = p + 1;
          pair_tasks.push_back(t);
        }
        plan.per_pair.push_back({beg, (int)pair_tasks.size()});
        plan.per_pair_first.push_back(p == byblock[i].pair_begin ? 1 : 0);
      }
      i = j;
    }
    plan.pair_tasks = upload(pair_tasks);
  }
  {
    std::vector<int64_t> zoff, zpre{0};
    for (const CBlockWork& w : work) {
      if (!w.pairs.empty()) continue;
      int64_t n = 1;
      for (int64_t d : block_dims(C, w.ct)) n *= d;
      if (n == 0) continue;
      zoff.push_back(w.c_off);
      zpre.push_back(zpre.back() + n);
    }
    plan.nzero = (int)zoff.size();
    plan.zero_elems = zpre.back();
    if (plan.nzero > 0) {
      plan.zero_off = upload(zoff);
      plan.zero_prefix = upload(zpre);
    }
  }
  plan.ntasks = (int)ordered.size();
  plan.tasks = upload(ordered);
  plan.pairs = upload(pairs);
  plan.cshapes = upload(cshapes);
  plan.kshapes = upload(kshapes);
  if (flops_out) *flops_out = flops;
  if (npairs_out) *npairs_out = npairs;
}

namespace {
// Launch model of the fused block-pair kernels, one entry per C-tile shape: the launch takes the
// longest of its padded work at the shape's full-chip rate (over whole rounds of one workgroup
// per CU) and the tasks' fixed time (tables, sums, the write) on top, its serial chains spread over
// the chip's workgroup slots, and its longest chain.  A chain is a task's fixed time and, for each of
// its block pairs, a start and a time per `unit` reduction indices.  Fitted to launches of 5 us to 5
// ms (blocks of 1 to 1600 rows, 1 to 50 pairs, K of 2 to 6400); over 324 of them the shapes taken are
// 2% above the fastest in the mean.  E.g. a 12 + 24 orbital ladder in blocks of ~6x6, 64x64 112 us, 32x32
// 28, 16x16 16; a 20 + 80 orbital dense ladder 1250 / 1472 / 2517, split 64x64 1047; a Fock
// term over blocks of 37 x 2600 with K = 37 340 / 421 / 495 / 610; the adjoint dV += L T of 25 +
// 110 orbitals (K ~ 40 a pair) 908 / 1398 / 2474 / 1354, of 16 + 40 (2 pairs of K = 64) 24 / 34 /
// 42 / 32.
struct BpShape {
  int tile, slots;
  bool swapped;
  double rate;                  // padded flops per second
  double fixed, pair, per_unit;  // us
  int unit, waves;              // the chain's pair and unit times are shared by `waves`
  double alone;                 // fixed time of a chain that waits for no other
};
constexpr BpShape kBpShapes[] = {
    {BP_TILE_64x64, 1024, false, 37.6e12, 12.5, 2.5, 1.45, 16, 1, 4.0},
    {BP_TILE_16x256, 768, false, 23.4e12, 14.0, 2.5, 1.45, 8, 1, 14.0},
    {BP_TILE_16x256, 768, true, 23.4e12, 14.0, 2.5, 1.45, 8, 1, 14.0},
    {BP_TILE_KS16, 1280, false, 14.6e12, 5.0, 0.0, 2.0, 64, 4, 5.0},
    {BP_TILE_KS32, 1024, false, 24.8e12, 8.0, 0.0, 2.5, 64, 4, 8.0},
    {BP_TILE_KS64, 512, false, 45e12, 30.0, 0.0, 9.5, 64, 4, 30.0},
};

struct BpLaunch {  // running sums of one launch
  double flops = 0, tasks = 0, chains = 0, longest = 0;
  double us(const BpShape& sh) const {
    if (tasks == 0) return 0;
    const double rounds = std::ceil(tasks / 256.0) * 256.0 / tasks;
    return std::max({flops / sh.rate * 1e6 * rounds + sh.fixed * tasks / sh.slots, chains / sh.slots, longest});
  }
};
}  // namespace

// The fastest C-tile shape by the launch model (index into kBpShapes) and its modelled time.
static int choose_bp_shape(const LOperand& C, const LOperand& A, const LOperand& B,
                           const LabelInfo& li, const std::vector<CBlockWork>& work,
                           bool per_pair_launches, double* us_out) {
  constexpr int NS = sizeof(kBpShapes) / sizeof(BpShape);
  BpLaunch all[NS];
  double total[NS] = {};
  int64_t largest = 1;  // operand block
  for (const LOperand* o : {&A, &B})
    for (int64_t sz : o->t->sizes) largest = std::max(largest, sz);
  std::vector<const std::vector<int64_t>*> red_sizes;
  for (int l : li.red) red_sizes.push_back(&li.tile_sizes.at(l));
  std::vector<int64_t> ks;
  for (const CBlockWork& w : work) {
    if (w.pairs.empty()) continue;
    const std::vector<int64_t> cd = block_dims(C, w.ct);
    double M = 1, N = 1, Bn = 1;
    for (size_t i = 0; i < C.labels.size(); ++i) {
      const int l = C.labels[i];
      if (pos_of(li.aouter, l) >= 0) M *= (double)cd[i];
      else if (pos_of(li.bouter, l) >= 0) N *= (double)cd[i];
      else Bn *= (double)cd[i];
    }
    // K of every pair, and sums over the pairs of its k-steps of 4 and units of 8, 16 and 64
    ks.clear();
    double kpad = 0, u8 = 0, u16 = 0, u64 = 0;
    for (const PairRef& pr : w.pairs) {
      int64_t k = 1;
      for (size_t i = 0; i < li.red.size(); ++i) k *= red_sizes[i]->at((size_t)pr.rt[i]);
      kpad += (double)((k + 3) / 4 * 4);
      u8 += (double)((k + 7) / 8);
      u16 += (double)((k + 15) / 16);
      u64 += (double)((k + 63) / 64);
      if (per_pair_launches) ks.push_back(k);
    }
    for (int s = 0; s < NS; ++s) {
      const BpShape& sh = kBpShapes[s];
      const double tm = bp_tile_rows(sh.tile), tn = bp_tile_cols(sh.tile);
      const double m = sh.swapped ? N : M, n = sh.swapped ? M : N;
      const double tiles = std::ceil(m / tm) * std::ceil(n / tn) * Bn;
      for (int64_t k : ks) {
        BpLaunch one;
        one.tasks = tiles;
        one.flops = 2 * tiles * tm * tn * (double)((k + 3) / 4 * 4);
        const double links = (sh.pair + sh.per_unit * (double)((k + sh.unit - 1) / sh.unit)) / sh.waves;
        one.longest = sh.alone + links;
        one.chains = tiles * (sh.fixed + links);
        total[s] += one.us(sh);
      }
      const double units = sh.unit == 8 ? u8 : sh.unit == 16 ? u16 : u64;
      const double links = (sh.pair * (double)w.pairs.size() + sh.per_unit * units) / sh.waves;
      all[s].flops += 2 * tiles * tm * tn * kpad;
      all[s].tasks += tiles;
      all[s].chains += tiles * (sh.fixed + links);
      all[s].longest = std::max(all[s].longest, sh.alone + links);
    }
  }
  int best = 0;
  double best_us = -1;
  for (int s = 0; s < NS; ++s) {
    const BpShape& sh = kBpShapes[s];
    if (sh.waves > 1 && largest > kBpKsMaxBlock) continue;
    const double us = per_pair_launches ? total[s] : all[s].us(sh);
    if (best_us < 0 || us < best_us) {
      best = s;
      best_us = us;
    }
  }
  if (us_out) *us_out = std::max(best_us, 0.0);
  return best;
}

void build_bp_plan(BPPlan& plan, const LOperand& C, const LOperand& A, const LOperand& B,
                   const LabelInfo& li, const std::vector<CBlockWork>& work,
                   bool per_pair_launches, double* flops_out, int64_t* npairs_out, int shape) {
  const int best = shape >= 0 ? shape : choose_bp_shape(C, A, B, li, work, per_pair_launches, nullptr);
  if (kBpShapes[best].swapped) {
    const LabelInfo li2 = analyse_labels(C, B, A);
    const std::vector<CBlockWork> work2 = enumerate_pairs(C, B, A, li2);
    build_bp_plan_as(plan, C, B, A, li2, work2, per_pair_launches, flops_out, npairs_out,
                     kBpShapes[best].tile);
    plan.swapped = true;
    return;
  }
  build_bp_plan_as(plan, C, A, B, li, work, per_pair_launches, flops_out, npairs_out,
                   kBpShapes[best].tile);
}

int grouped_bp_shape(const LOperand& C, const LOperand& A, const LOperand& B, const LabelInfo& li,
                     const std::vector<CBlockWork>& work, double* us) {
  return choose_bp_shape(C, A, B, li, work, false, us);
}

void launch_bp_plan(const BPPlan& bp, const BPTask* tasks, int ntasks, const BPXcd* xr,
                    const double* A, const double* B, double* C, double alpha, int is_assign,
                    hipStream_t s) {
  if (bp.swapped) std::swap(A, B);
  launch_bp_f64(tasks, ntasks, bp.pairs.as<BPPair>(), bp.cshapes.as<BPCShape>(),
                bp.kshapes.as<BPKShape>(), A, B, C, alpha, is_assign, s, xr, bp.tile);
}

}  // namespace tmx

using namespace tmx;

// ---------------------------------------------------------------------------
// Contraction object
struct tmx_contraction_s {
  int mode = TMX_EXEC_GROUPED_F64;
  double alpha = 1.0;
  LOperand C, A, B;
  double flops = 0;
  int64_t npairs = 0;
  BPPlan bp;
  SectorPlanPtr sec;
  // Inputs of the sector plan, kept so the autotuner can rebuild it with other split-K counts.
  // When C's labels list the B-outer labels before the A-outer ones, the sector plan is built
  // for C = B*A (swapped = true): a C block is then row-major over the plan's dense rows and
  // columns, which lets the split path add its results into C in one fused pass.
  LabelInfo li;
  std::vector<CBlockWork> work;
  int split_bits = 0;
  int parallel_split = 0;  // tmx_set_parallel_split at creation; 0 lets the autotuner measure split-K
  bool swapped = false;
  // tmx_contraction_set_constant: operands packed once and kept (call's A / B).
  bool const_a = false, const_b = false;
  // tmx_contraction_set_assign: C = alpha*A*B instead of C += alpha*A*B.
  bool assign = false;
  // AUTO's estimates for a product that it took off the sector path as small (0: none such): both
  // paths, and the packing of A and of B in the sector one.
  struct Small {
    double grouped_us = 0, sector_us = 0, pack_us[2] = {0, 0};
    int exec_mode = 0;
  } small;
  // Holds of live graphs that captured an execution of the contraction (GraphHold).
  std::atomic<int> graph_holds{0};
  const LOperand& sa() const { return swapped ? B : A; }
  const LOperand& sb() const { return swapped ? A : B; }
};

// Contraction and AddOp handles are owned through a registry of shared pointers: destroy drops
// the registry's reference, and a graph that captured the object holds another
// (capture_hold), so the object and its device memory live until both are gone.
template <class T>
struct HandleRegistry {
  std::mutex mu;
  std::map<const T*, std::shared_ptr<T>> live;
  T* add(std::shared_ptr<T> p) {
    std::lock_guard<std::mutex> g(mu);
    T* raw = p.get();
    live[raw] = std::move(p);
    return raw;
  }
  std::shared_ptr<T> get(const T* raw) {
    std::lock_guard<std::mutex> g(mu);
    auto it = live.find(raw);
    return it == live.end() ? nullptr : it->second;
  }
  // References beyond the registry's own (graphs holding the object).
  long held(const T* raw) {
    std::lock_guard<std::mutex> g(mu);
    auto it = live.find(raw);
    return it == live.end() ? 0 : it->second.use_count() - 1;
  }
  void drop(const T* raw) {
    std::shared_ptr<T> p;  // released outside the lock
    std::lock_guard<std::mutex> g(mu);
    auto it = live.find(raw);
    TMX_REQUIRE(it != live.end(), "unknown or already destroyed handle");
    p = std::move(it->second);
    live.erase(it);
  }
};
// Heap singletons, never destroyed (objects they still hold must not free device memory
// during static destruction).
static HandleRegistry<tmx_contraction_s>& contractions() {
  static auto* r = new HandleRegistry<tmx_contraction_s>();
  return *r;
}

// A graph's hold on a contraction, counted on the contraction, so that changes a replay must
// not see (which operands are constant, whether it assigns) are refused only while a graph
// holds it (a level's reference does not count).
struct GraphHold {
  std::shared_ptr<tmx_contraction_s> c;
  explicit GraphHold(std::shared_ptr<tmx_contraction_s> p) : c(std::move(p)) { ++c->graph_holds; }
  ~GraphHold() { --c->graph_holds; }
  GraphHold(const GraphHold&) = delete;
  GraphHold& operator=(const GraphHold&) = delete;
};
static void hold_for_graph(hipStream_t s, std::shared_ptr<tmx_contraction_s> c) {
  if (c && stream_capturing(s)) capture_hold(s, std::make_shared<GraphHold>(std::move(c)));
}

// Executes a contraction's sector plan with its operands in the plan's order.
// Executes a contraction's block-pair plan (GROUPED: one launch; BLOCKPAIR: one launch per
// block pair).  Assigning, the blocks without pairs are zeroed and each C tile is written by
// its first pair (GROUPED: its only task; BLOCKPAIR: the launch of the block's first pair).
static void run_bp(const tmx_contraction_s* c, const double* A, const double* B, double* C,
                   hipStream_t s) {
  if (c->assign)
    launch_zero_ranges(c->bp.zero_off.as<int64_t>(), c->bp.zero_prefix.as<int64_t>(), c->bp.nzero,
                       c->bp.zero_elems, C, s);
  if (c->mode == TMX_EXEC_GROUPED_F64) {
    launch_bp_plan(c->bp, c->bp.tasks.as<BPTask>(), c->bp.ntasks, &c->bp.xcd, A, B, C, c->alpha,
                   c->assign ? 1 : 0, s);
    return;
  }
  const BPTask* pt = c->bp.pair_tasks.as<BPTask>();
  for (size_t i = 0; i < c->bp.per_pair.size(); ++i) {
    const auto& r = c->bp.per_pair[i];
    launch_bp_plan(c->bp, pt + r.first, r.second - r.first, nullptr, A, B, C, c->alpha,
                   c->assign && c->bp.per_pair_first[i] ? 1 : 0, s);
  }
}

static void set_constant_flags(const tmx_contraction_s* c, SectorPlan& sp) {
  set_sector_constant(sp, c->swapped ? c->const_b : c->const_a, c->swapped ? c->const_a : c->const_b);
}

// pack_ev: optional two events around the main packing pass of the call's A operand.
static void run_sector(const tmx_contraction_s* c, SectorPlan& sp, const double* A, const double* B,
                       double* C, double alpha, hipStream_t s, hipEvent_t* ev = nullptr,
                       hipEvent_t* gemm_ev = nullptr, hipEvent_t* pack_ev = nullptr) {
  set_constant_flags(c, sp);
  set_sector_assign(sp, c->assign);
  if (c->swapped) std::swap(A, B);
  execute_sector_plan(sp, A, B, C, alpha, s, ev, gemm_ev, c->swapped ? nullptr : pack_ev,
                      c->swapped ? pack_ev : nullptr);
}

// Library-wide settings: set by the tmx_set_* calls, read when plans are built or executed,
// possibly from other threads.
static std::atomic<int> g_split_bits{35};
static std::atomic<int> g_parallel_split{0};  // 0: launch model

// Times a sector plan executing into a scratch C (average of 3 after one warm-up), in ms.
static float time_sector_plan(const tmx_contraction_s* c, SectorPlan& sp, const double* A,
                              const double* B, double* scratch, hipStream_t s, hipEvent_t e0,
                              hipEvent_t e1) {
  run_sector(c, sp, A, B, scratch, 1.0, s);
  TMX_HIP(hipEventRecord(e0, s));
  for (int r = 0; r < 3; ++r) run_sector(c, sp, A, B, scratch, 1.0, s);
  TMX_HIP(hipEventRecord(e1, s));
  TMX_HIP(hipEventSynchronize(e1));
  float ms = 0;
  TMX_HIP(hipEventElapsedTime(&ms, e0, e1));
  return ms / 3;
}

// Split-K counts by measurement: the plan is rebuilt with uniform part counts 1, 2, 3 and 4
// (pairs whose reduction is too short keep fewer), each timed end to end (packing, GEMM,
// recombination, scatter) into a scratch copy of C, and the fastest kept if it beats the launch
// model's plan by 2%; a replacement then has its tile shapes tuned.  Plans whose execution takes
// under half a millisecond are left alone.  Returns 1 when the plan was replaced.
static int autotune_split_k(tmx_contraction_s* c, const double* A, const double* B, hipStream_t s) {
  hipEvent_t e0, e1;
  TMX_HIP(hipEventCreate(&e0));
  TMX_HIP(hipEventCreate(&e1));
  struct Cleanup {
    hipEvent_t a, b;
    ~Cleanup() { (void)hipEventDestroy(a); (void)hipEventDestroy(b); }
  } cleanup{e0, e1};
  DevBuf scratch(sizeof(double) * (size_t)std::max<int64_t>(c->C.t->total, 1));
  launch_fill_bytes_zero(scratch.p, scratch.bytes, s);
  double* sc = scratch.as<double>();
  float best_ms = time_sector_plan(c, *c->sec, A, B, sc, s, e0, e1);
  if (best_ms < 0.5f) return 0;
  const bool split = c->mode == TMX_EXEC_SPLIT_I8;
  SectorPlanPtr best;
  int last_rounds = -1;
  for (int p = 1; p <= 4; ++p) {
    SectorPlanPtr cand = build_sector_plan(c->C, c->sa(), c->sb(), c->li, c->work, split, c->split_bits, p);
    int rounds = 0;
    sector_schedule_info(*cand, &rounds, nullptr, nullptr);
    if (rounds == last_rounds) continue;
    last_rounds = rounds;
    const float ms = time_sector_plan(c, *cand, A, B, sc, s, e0, e1);
    if (ms < best_ms * 0.98f) {
      best_ms = ms;
      best = std::move(cand);
    }
  }
  if (!best) return 0;
  run_sector(c, *best, A, B, sc, 1.0, s);
  autotune_sector_plan(*best, c->swapped ? B : A, s);
  c->sec = std::move(best);
  return 1;
}

static bool sector_eligible(const LabelInfo& li) {
  return li.batch.empty() && li.ared.empty() && li.bred.empty() && !li.aouter.empty() &&
         !li.bouter.empty() && !li.inner.empty();
}

// Builds the sector plan of a contraction whose label analysis and pair list are li and work;
// returns the mode it executes in.
static int build_sector(tmx_contraction_s& c, const LabelInfo& li, const std::vector<CBlockWork>& work,
                        int mode, int exec_mode) {
  std::vector<int> ab(li.aouter), ba(li.bouter);
  ab.insert(ab.end(), li.bouter.begin(), li.bouter.end());
  ba.insert(ba.end(), li.aouter.begin(), li.aouter.end());
  c.swapped = c.C.labels != ab && c.C.labels == ba;
  if (c.swapped) {
    c.li = analyse_labels(c.C, c.B, c.A);
    c.work = enumerate_pairs(c.C, c.B, c.A, c.li);
  } else {
    c.li = li;
    c.work = work;
  }
  // AUTO_SPLIT: split precision pays only where the FP64 GEMM is MFMA-bound.  A sector GEMM
  // reads (mrows + nrows) K operand elements for 2 mrows nrows K flops; below
  // kMinSplitMN (flops-weighted mrows nrows / (mrows + nrows) of the sectors, e.g. the one-O-
  // tile classes of Fo(k,i) += U(k,l,c,d) T(c,d,i,l)) both precisions stream their packed
  // operands at the same HBM rate and split packs 11 bytes per element against 8, so the
  // planner builds the plan in FP64 (before allocating anything).
  constexpr double kMinSplitMN = 32;
  c.sec = build_sector_plan(c.C, c.sa(), c.sb(), c.li, c.work, mode == TMX_EXEC_SPLIT_I8, c.split_bits,
                            c.parallel_split, exec_mode == TMX_EXEC_AUTO_SPLIT ? kMinSplitMN : 0.0);
  return mode == TMX_EXEC_SPLIT_I8 && !sector_is_split(*c.sec) ? TMX_EXEC_SECTOR_F64 : mode;
}

// A small product that AUTO put on the grouped path, once operands of it are constant: the sector
// path then packs them once, and takes the product over unless grouped is modelled 1.25 times as
// fast (ladder of 10 + 100 orbitals with constant V: 212 us grouped, 122 split; of 24 + 96 in tiles
// of 2 to 6: 587 and 206 in FP64; rings of 10 + 100 stay at 20, split 37).  For good: a level may have given the plan's product to
// other terms.  Not during a capture, whose executions stay grouped; the next call decides again.
static void reconsider_small(tmx_contraction_s& c) {
  if (c.small.grouped_us == 0 || c.sec || !(c.const_a || c.const_b)) return;
  const double us = c.small.sector_us - (c.const_a ? c.small.pack_us[0] : 0) - (c.const_b ? c.small.pack_us[1] : 0);
  if (1.25 * c.small.grouped_us < us || capture_in_progress()) return;
  const bool split = c.small.exec_mode == TMX_EXEC_AUTO_SPLIT;
  const LabelInfo li = analyse_labels(c.C, c.A, c.B);
  try {
    c.mode = build_sector(c, li, enumerate_pairs(c.C, c.A, c.B, li),
                          split ? TMX_EXEC_SPLIT_I8 : TMX_EXEC_SECTOR_F64, c.small.exec_mode);
  } catch (const Error&) {
    c.sec = nullptr;  // e.g. no memory for the packed copies: it stays grouped
  }
}

extern "C" {

int tmx_set_split_bits(int bits) {
  return guarded([&] {
    TMX_REQUIRE(bits >= 8 && bits <= 50, "split bits must be in [8, 50]");
    g_split_bits = bits;
  });
}

int tmx_set_parallel_split(int parts) {
  return guarded([&] {
    TMX_REQUIRE(parts >= 0 && parts <= 16, "parallel split must be in [0, 16]");
    g_parallel_split = parts;
  });
}

int tmx_set_scale_reuse(int on) {
  return guarded([&] {
    TMX_REQUIRE(on == 0 || on == 1, "scale reuse must be 0 or 1");
    set_scale_reuse(on != 0);
  });
}

int tmx_contraction_create(const tmx_operand* C, double alpha, const tmx_operand* A,
                           const tmx_operand* B, int exec_mode, tmx_contraction* out) {
  return guarded([&] {
    require_init();
    TMX_REQUIRE(out, "null output");
    TMX_REQUIRE(exec_mode >= 0 && exec_mode <= TMX_EXEC_AUTO_SPLIT, "unknown execution mode");
    auto c = std::make_shared<tmx_contraction_s>();
    c->alpha = alpha;
    c->C = make_loperand(C);
    c->A = make_loperand(A);
    c->B = make_loperand(B);
    TMX_REQUIRE(c->C.t.get() != c->A.t.get() && c->C.t.get() != c->B.t.get(),
                "output tensor also appears on the right-hand side (MultOp::validate)");
    LabelInfo li = analyse_labels(c->C, c->A, c->B);
    std::vector<CBlockWork> work = enumerate_pairs(c->C, c->A, c->B, li);
    int mode = exec_mode, bp_shape = -1;
    if (mode == TMX_EXEC_AUTO || mode == TMX_EXEC_AUTO_SPLIT) {
      // Average reduction length per output element: below kMinSectorK the contraction is
      // memory-bound, and the sector path's operand repacking and dense intermediate cost more
      // than the fused block-pair kernel that reads the blocks in place.
      double fl = 0, celems = 0;
      for (const CBlockWork& w : work) {
        std::vector<int64_t> cd = block_dims(c->C, w.ct);
        double mn = 1;
        for (auto d : cd) mn *= (double)d;
        celems += mn;
        for (const PairRef& pr : w.pairs) {
          double k = 1;
          for (size_t i = 0; i < li.red.size(); ++i) k *= (double)li.tile_sizes.at(li.red[i])[pr.rt[i]];
          fl += 2.0 * mn * k;
        }
      }
      const double avg_k = celems > 0 ? fl / (2.0 * celems) : 0.0;
      constexpr double kMinSectorK = 128;
      bool sector = sector_eligible(li) && avg_k >= kMinSectorK;
      // Small products: the sector path's launches, packs of blocks of a few hundred elements and
      // few-tile GEMMs over a long K cost more than the block-pair kernel.  Its time here: four
      // launches of 4.5 us (nine on the split path), packs and scatter at 3 TB/s or 6 us a block
      // over 1024 workgroups, and the GEMM at its rate or the stages of 1024 columns.  Over 528
      // products of 4 to 40 and 20 to 147 orbitals the grouped model is right in the mean (rms
      // 22%), this one 17 (split) to 45% (FP64) too high, so grouped is taken when modelled 1.6
      // times as fast (what is taken is then 2% above the faster path in the mean, at 1 and 2 times
      // 3.5 and 3), e.g. 10 + 100 orbitals: ladder 150 us grouped, 279 sector; 30 + 60: hole-hole 66
      // and 56.  On the split path 2 times: a level computes the product of a ring's four
      // permutations once there.
      // Larger products stay on the sector path (so does, from tmx_contraction_set_constant on, what
      // the sector path runs faster once it has packed a constant operand); so do streaming ones (few flops over large tensors), which the model does not cover.
      constexpr double kSmallFlops = 20e9, kSmallElems = 4e7;
      const double elems = (double)(c->A.t->total + c->B.t->total + c->C.t->total);
      if (sector && fl < kSmallFlops && elems < kSmallElems) {
        const bool split = exec_mode == TMX_EXEC_AUTO_SPLIT;
        double us = 4.5 * (split ? 9 : 4), pass_us[3];
        const LOperand* ops[3] = {&c->A, &c->B, &c->C};
        for (int i = 0; i < 3; ++i) {
          const double bytes = (double)ops[i]->t->total * (i == 2 ? (split ? 27 : 24) : (split ? 27 : 16));
          pass_us[i] = std::max(bytes / 3e6, 6.0 * (double)ops[i]->t->keys.size() / 1024.0);
          us += pass_us[i];
        }
        us += split ? std::max(fl / 120e6, avg_k / 64.0) : std::max(fl / 50e6, 0.9 * std::min(avg_k, 1024.0) / 8.0);
        double grouped_us = 0;
        bp_shape = grouped_bp_shape(c->C, c->A, c->B, li, work, &grouped_us);
        if ((split ? 2.0 : 1.6) * grouped_us < us) {
          sector = false;
          const double launches = 4.5 * (split ? 3 : 1);
          c->small = {grouped_us, us, {pass_us[0] + launches, pass_us[1] + launches}, exec_mode};
        }
      }
      mode = !sector ? TMX_EXEC_GROUPED_F64
                     : (exec_mode == TMX_EXEC_AUTO_SPLIT ? TMX_EXEC_SPLIT_I8 : TMX_EXEC_SECTOR_F64);
    }
    // One read of each setting: the plan and the fields the autotuner rebuilds it from agree.
    c->split_bits = g_split_bits.load();
    c->parallel_split = g_parallel_split.load();
    if (mode == TMX_EXEC_SECTOR_F64 || mode == TMX_EXEC_SPLIT_I8) {
      if (!sector_eligible(li))
        throw Error(TMX_ERR_UNSUPPORTED,
                    "sector execution needs aouter, bouter and inner labels and no batch or "
                    "reduce-only labels; use TMX_EXEC_GROUPED_F64");
      double fl = 0;
      int64_t np = 0;
      for (const CBlockWork& w : work) np += (int64_t)w.pairs.size();
      mode = build_sector(*c, li, work, mode, exec_mode);
      // algorithmic flops: sum over triples of 2*M*N*K
      for (const CBlockWork& w : work) {
        std::vector<int64_t> rt0(li.red.size(), 0);
        std::vector<int64_t> cd = block_dims(c->C, w.ct);
        double mn = 1;
        for (auto d : cd) mn *= (double)d;
        for (const PairRef& pr : w.pairs) {
          double k = 1;
          for (size_t i = 0; i < li.red.size(); ++i) k *= (double)li.tile_sizes.at(li.red[i])[pr.rt[i]];
          fl += 2.0 * mn * k;
        }
      }
      c->flops = fl;
      c->npairs = np;
    } else {
      build_bp_plan(c->bp, c->C, c->A, c->B, li, work, mode == TMX_EXEC_BLOCKPAIR_F64, &c->flops,
                    &c->npairs, bp_shape);
    }
    c->mode = mode;
    *out = contractions().add(std::move(c));
  });
}

int tmx_contraction_execute(tmx_contraction c, const double* A, const double* B, double* C,
                            void* stream) {
  return guarded([&] {
    TMX_REQUIRE(c, "null contraction");
    hipStream_t s = pick_stream(stream);
    TMX_REQUIRE(A && B && C, "null data pointer");
    hold_for_graph(s, contractions().get(c));
    if (c->mode == TMX_EXEC_GROUPED_F64 || c->mode == TMX_EXEC_BLOCKPAIR_F64) run_bp(c, A, B, C, s);
    else run_sector(c, *c->sec, A, B, C, c->alpha, s);
  });
}

int tmx_contraction_autotune(tmx_contraction c, const double* A, const double* B, double* C,
                             void* stream, int* changed) {
  return guarded([&] {
    TMX_REQUIRE(c, "null contraction");
    TMX_REQUIRE(A && B && C, "null data pointer");
    hipStream_t s = pick_stream(stream);
    // A graph or a level (whose terms scatter from each other's products) holds the plan.
    if (contractions().held(c) > 0)
      throw Error(TMX_ERR_STATE,
                  "the contraction is held by a captured graph or a level (its plan would be "
                  "rebuilt under them): destroy them before autotuning");
    int n = 0;
    if (c->mode == TMX_EXEC_SECTOR_F64 || c->mode == TMX_EXEC_SPLIT_I8) {
      run_sector(c, *c->sec, A, B, C, c->alpha, s);
      n = autotune_sector_plan(*c->sec, c->swapped ? B : A, s);
      if (c->parallel_split == 0) n += autotune_split_k(c, A, B, s);
    } else {
      const int rc = tmx_contraction_execute(c, A, B, C, stream);
      if (rc != TMX_OK) throw Error(rc, tmx_last_error());
    }
    TMX_HIP(hipStreamSynchronize(s));
    if (changed) *changed = n;
  });
}

// Executes once with events between the stages; ms[0] / ms[1] = packing of the call's A / B
// operand, ms[2] = GEMM, ms[3] = scatter (fused block-pair modes: their kernel as ms[2]),
// ms[4] = the longest single GEMM launch, ms[5] = the main packing pass of the call's A operand
// alone (0 when nothing was packed).
static void execute_stages(tmx_contraction c, const double* A, const double* B, double* C,
                           hipStream_t s, float ms[6]) {
  constexpr int kMaxLaunchEvents = 16, kEvents = 7 + kMaxLaunchEvents;
  hipEvent_t ev[kEvents];
  for (auto& e : ev) TMX_HIP(hipEventCreate(&e));
  struct Cleanup {
    hipEvent_t* ev;
    ~Cleanup() { for (int i = 0; i < kEvents; ++i) (void)hipEventDestroy(ev[i]); }
  } cleanup{ev};
  hipEvent_t* pack_ev = ev + 5 + kMaxLaunchEvents;
  // both recorded here first: a pass that does not run leaves them equal
  TMX_HIP(hipEventRecord(pack_ev[0], s));
  TMX_HIP(hipEventRecord(pack_ev[1], s));
  int launches = 1;
  if (c->mode == TMX_EXEC_SECTOR_F64 || c->mode == TMX_EXEC_SPLIT_I8) {
    int64_t t = 0;
    int r = 0;
    set_constant_flags(c, *c->sec);
    sector_schedule_info(*c->sec, &r, &launches, &t, c->swapped ? B : A);
    const bool per_launch = launches > 1 && launches <= kMaxLaunchEvents + 1;
    run_sector(c, *c->sec, A, B, C, c->alpha, s, ev, per_launch ? ev + 5 : nullptr, pack_ev);
    if (!per_launch) launches = 1;
  } else {
    TMX_HIP(hipEventRecord(ev[0], s));
    TMX_HIP(hipEventRecord(ev[1], s));
    TMX_HIP(hipEventRecord(ev[2], s));
    run_bp(c, A, B, C, s);
    TMX_HIP(hipEventRecord(ev[3], s));
    TMX_HIP(hipEventRecord(ev[4], s));
  }
  TMX_HIP(hipEventSynchronize(ev[4]));
  for (int i = 0; i < 4; ++i) TMX_HIP(hipEventElapsedTime(&ms[i], ev[i], ev[i + 1]));
  if (c->swapped) std::swap(ms[0], ms[1]);  // the plan packed B first
  ms[4] = ms[2];
  if (launches > 1) {  // launch i runs from event (i - 1) (ev[2] for the first) to event i
    ms[4] = 0;
    for (int i = 0; i < launches; ++i) {
      hipEvent_t a = i == 0 ? ev[2] : ev[5 + i - 1], b = i + 1 == launches ? ev[3] : ev[5 + i];
      float x = 0;
      TMX_HIP(hipEventElapsedTime(&x, a, b));
      ms[4] = std::max(ms[4], x);
    }
  }
  TMX_HIP(hipEventElapsedTime(&ms[5], pack_ev[0], pack_ev[1]));
}

int tmx_contraction_execute_timed(tmx_contraction c, const double* A, const double* B, double* C,
                                  void* stream, float* stage_ms) {
  return guarded([&] {
    TMX_REQUIRE(c && stage_ms, "null argument");
    TMX_REQUIRE(A && B && C, "null data pointer");
    float ms[6];
    execute_stages(c, A, B, C, pick_stream(stream), ms);
    stage_ms[0] = ms[0] + ms[1];
    stage_ms[1] = ms[2];
    stage_ms[2] = ms[3];
  });
}

int tmx_contraction_execute_stages(tmx_contraction c, const double* A, const double* B, double* C,
                                   void* stream, float* stage_ms) {
  return tmx_contraction_execute_stages_n(c, A, B, C, stream, stage_ms, 5);
}

int tmx_contraction_execute_stages_n(tmx_contraction c, const double* A, const double* B, double* C,
                                     void* stream, float* stage_ms, int n) {
  return guarded([&] {
    TMX_REQUIRE(c && stage_ms, "null argument");
    TMX_REQUIRE(A && B && C, "null data pointer");
    TMX_REQUIRE(n >= 1 && n <= 6, "stage count must be in [1, 6]");
    float ms[6];
    execute_stages(c, A, B, C, pick_stream(stream), ms);
    for (int i = 0; i < n; ++i) stage_ms[i] = ms[i];
  });
}

int tmx_contraction_info(tmx_contraction c, double* flops, int64_t* npairs, int64_t* ws, int* mode) {
  return guarded([&] {
    TMX_REQUIRE(c, "null contraction");
    if (flops) *flops = c->flops;
    if (npairs) *npairs = c->npairs;
    if (ws) {
      int64_t b = (int64_t)(c->bp.tasks.bytes + c->bp.pairs.bytes + c->bp.cshapes.bytes +
                            c->bp.kshapes.bytes + c->bp.pair_tasks.bytes);
      if (c->sec) b += sector_workspace_bytes(*c->sec);
      *ws = b;
    }
    if (mode) *mode = c->mode;
  });
}

int tmx_contraction_schedule_info(tmx_contraction c, int* rounds, int* launches, int64_t* tasks) {
  return guarded([&] {
    TMX_REQUIRE(c, "null contraction");
    if (!c->sec) {
      if (rounds) *rounds = 1;
      if (launches) *launches = 1;
      if (tasks) *tasks = 0;
      return;
    }
    sector_schedule_info(*c->sec, rounds, launches, tasks);
  });
}

int tmx_contraction_kernel_info(tmx_contraction c, int* tile_rows, int* tile_cols, int* shared_k, int* in_place) {
  return guarded([&] {
    TMX_REQUIRE(c, "null contraction");
    int rows = 0, cols = 0;
    bool ks = false, inp = false;
    if (c->sec) {
      sector_kernel_info(*c->sec, &rows, &cols, &inp);
    } else {
      rows = bp_tile_rows(c->bp.tile);
      cols = bp_tile_cols(c->bp.tile);
      ks = bp_tile_shares_k(c->bp.tile);
    }
    if (tile_rows) *tile_rows = rows;
    if (tile_cols) *tile_cols = cols;
    if (shared_k) *shared_k = ks ? 1 : 0;
    if (in_place) *in_place = inp ? 1 : 0;
  });
}

int tmx_contraction_split_info(tmx_contraction c, int* bits_a, int* bits_b, int* nmoduli) {
  return guarded([&] {
    TMX_REQUIRE(c, "null contraction");
    if (c->mode != TMX_EXEC_SPLIT_I8 || !c->sec) {
      if (bits_a) *bits_a = 53;
      if (bits_b) *bits_b = 53;
      if (nmoduli) *nmoduli = 0;
      return;
    }
    sector_split_info(*c->sec, bits_a, bits_b, nmoduli);
  });
}

int tmx_contraction_set_constant(tmx_contraction c, int a_constant, int b_constant) {
  return guarded([&] {
    TMX_REQUIRE(c, "null contraction");
    TMX_REQUIRE((a_constant == 0 || a_constant == 1) && (b_constant == 0 || b_constant == 1),
                "constant flags must be 0 or 1");
    if (c->graph_holds > 0)
      throw Error(TMX_ERR_STATE,
                  "the contraction is held by a captured graph: destroy the graph before changing "
                  "which operands are constant");
    c->const_a = a_constant != 0;
    c->const_b = b_constant != 0;
    reconsider_small(*c);
    if (!c->sec) return;
    set_constant_flags(c, *c->sec);
    forget_sector_packing(*c->sec);  // the next execution packs afresh
  });
}

int tmx_contraction_set_assign(tmx_contraction c, int assign) {
  return guarded([&] {
    TMX_REQUIRE(c, "null contraction");
    TMX_REQUIRE(assign == 0 || assign == 1, "assign must be 0 or 1");
    if (c->graph_holds > 0)
      throw Error(TMX_ERR_STATE,
                  "the contraction is held by a captured graph: destroy the graph before changing "
                  "whether it assigns");
    c->assign = assign != 0;
    if (c->sec) set_sector_assign(*c->sec, c->assign);  // also for a level's scatter-only terms
  });
}

// ---------------------------------------------------------------------------
// Level: contractions executed in order as one unit (a Scheduler level), where terms that
// compute the same product share it.  A term's product is the packed-operand GEMM its sector
// plan runs; two plans have the same product when they pack the same tensors with the same
// jobs and have the same sector geometry (product_key), e.g. the four permutations of a CC
// ring term, R(a,b,i,j) += W(k,b,c,j) T(a,c,i,k) and its P(ab), P(ij), P(ab)P(ij) images,
// which all pack W and T alike and differ only in where (and with which sign) the product
// lands in R.  Such a term runs only its scatter stage, from the first term's product.
struct tmx_level_s {
  std::vector<std::shared_ptr<tmx_contraction_s>> terms;
  std::vector<int> leader;  // term whose product term i reuses; i itself when it computes its own
};

static bool sector_mode(const tmx_contraction_s& c) {
  return c.mode == TMX_EXEC_SECTOR_F64 || c.mode == TMX_EXEC_SPLIT_I8;
}

int tmx_level_create(const tmx_contraction* cs, int n, tmx_level* out) {
  return guarded([&] {
    TMX_REQUIRE(out && (cs || n == 0) && n >= 0, "bad level arguments");
    auto lv = std::make_unique<tmx_level_s>();
    for (int i = 0; i < n; ++i) {
      auto c = contractions().get(cs[i]);
      TMX_REQUIRE(c, "unknown contraction in level");
      int lead = i;
      if (sector_mode(*c) && c->sec) {
        for (int j = 0; j < i; ++j) {
          const tmx_contraction_s& d = *lv->terms[j];
          if (lv->leader[j] == j && sector_mode(d) && d.mode == c->mode &&
              sector_product_key(*d.sec) == sector_product_key(*c->sec)) {
            lead = j;
            break;
          }
        }
      }
      lv->terms.push_back(std::move(c));
      lv->leader.push_back(lead);
    }
    *out = lv.release();
  });
}

int tmx_level_products(tmx_level lv, int* nproducts) {
  return guarded([&] {
    TMX_REQUIRE(lv && nproducts, "null argument");
    int k = 0;
    for (size_t i = 0; i < lv->leader.size(); ++i) k += lv->leader[i] == (int)i;
    *nproducts = k;
  });
}

int tmx_level_execute(tmx_level lv, const double* const* A, const double* const* B, double* const* C,
                      void* stream) {
  return guarded([&] {
    TMX_REQUIRE(lv && A && B && C, "null argument");
    hipStream_t s = pick_stream(stream);
    const size_t n = lv->terms.size();
    for (size_t i = 0; i < n; ++i) TMX_REQUIRE(A[i] && B[i] && C[i], "null data pointer");
    for (size_t i = 0; i < n; ++i) {
      tmx_contraction_s* c = lv->terms[i].get();
      const size_t l = (size_t)lv->leader[i];
      // Reuse only when the leader saw the same operand data and no term since the leader
      // wrote into it (a level has no such dependence, but the call is checked).
      bool reuse = l != i && A[i] == A[l] && B[i] == B[l];
      for (size_t j = l; reuse && j < i; ++j) reuse = C[j] != A[l] && C[j] != B[l];
      if (reuse) {
        if (stream_capturing(s)) {
          hold_for_graph(s, lv->terms[i]);
          hold_for_graph(s, lv->terms[l]);
        }
        execute_sector_scatter_from(*c->sec, *lv->terms[l]->sec, C[i], c->alpha, s);
      } else {
        const int rc = tmx_contraction_execute(c, A[i], B[i], C[i], stream);
        if (rc != TMX_OK) throw Error(rc, tmx_last_error());
      }
    }
  });
}

int tmx_level_destroy(tmx_level lv) {
  return guarded([&] {
    if (!lv) return;
    quiesce();
    delete lv;
  });
}

int tmx_contraction_destroy(tmx_contraction c) {
  return guarded([&] {
    if (!c) return;
    quiesce();  // the plan's workspace may still be in use by queued kernels
    contractions().drop(c);  // a graph that captured it keeps it until tmx_graph_destroy
  });
}

}  // extern "C"

// ---------------------------------------------------------------------------
// Block-level entry points.  Plans are cached per (dims, labels) signature so a call
// allocates nothing once its shape has been seen.
namespace {

struct BlockMulPlan {
  BPPlan bp;
};
struct AssignPlan {
  DevBuf tables;  // shapes, jobs, units, zero_off and zero_prefix, in one upload
  const AssignShape* shapes = nullptr;
  const AssignJob* jobs = nullptr;
  const AssignUnit* units = nullptr;
  int64_t nunits = 0;
  int box = 0;  // launch_assign's
  // Destination blocks whose source block is zero (element ranges; zero_prefix holds running
  // lengths), zeroed when the op assigns.
  const int64_t *zero_off = nullptr, *zero_prefix = nullptr;
  int nzero = 0;
  int64_t zero_elems = 0;
};
// Heap singletons, never destroyed (their device buffers must not be freed during static
// destruction, see runtime.cpp).
std::mutex& cache_mu() {
  static std::mutex* m = new std::mutex();
  return *m;
}
std::map<std::vector<int64_t>, std::unique_ptr<BlockMulPlan>>& bm_cache() {
  static auto* c = new std::map<std::vector<int64_t>, std::unique_ptr<BlockMulPlan>>();
  return *c;
}
std::map<std::vector<int64_t>, std::unique_ptr<AssignPlan>>& as_cache() {
  static auto* c = new std::map<std::vector<int64_t>, std::unique_ptr<AssignPlan>>();
  return *c;
}

// Builds a one-block "tensor" whose single block has the given dims (one tile per mode).
LOperand single_block_operand(int n, const int64_t* dims, const int* labels) {
  std::vector<std::shared_ptr<const Space>> modes;
  for (int i = 0; i < n; ++i) {
    TMX_REQUIRE(dims[i] > 0, "block dims must be positive");
    int64_t t = dims[i];
    modes.push_back(make_space(dims[i], 0, &t, 1, 0, nullptr, nullptr, nullptr, 0, nullptr, nullptr,
                               nullptr, 0, nullptr, nullptr));
  }
  LOperand o;
  o.t = make_tensor(modes, -1, 0, 0);
  for (int i = 0; i < n; ++i) {
    o.labels.push_back(labels[i]);
    o.toff.push_back(0);
    o.ntl.push_back(1);
  }
  return o;
}

}  // namespace

namespace tmx {

// Box of a block permutation: dims of the destination block and the source stride of each of its
// modes (see AssignShape).  elems = 0: whole tiles (k_assign_tile), 32 x 32 of the two contiguous
// modes or 1024 of a shared one.  Else boxes of up to `elems` elements: X starts as the
// source's contiguous mode and Y as the destination's; each side of fewer than 32 indices takes
// in the next mode of its own block's order unless that mode is already on the other side (the
// two sides together are then one contiguous piece of that block), so reads and writes come in
// runs of at least 256 bytes wherever the blocks allow it.  Z then fills the box with the
// remaining modes, the destination's fastest first; where these are too few to fill it, a cut side
// grows first.  A mode is cut into boxes of equal size.
static AssignShape make_assign_shape(const std::vector<int64_t>& dd, const std::vector<int64_t>& src_stride,
                                     int64_t elems) {
  const int64_t side = elems == kAssignElems ? 48 : elems == 1024 ? 32 : 16;
  const int64_t lds = kAssignLds * elems / 256;
  AssignShape sh;
  std::memset(&sh, 0, sizeof(sh));
  std::vector<int64_t> ext, ss;
  for (size_t i = 0; i < dd.size(); ++i) {
    TMX_REQUIRE(dd[i] < (1ll << 31), "block too large");
    if (dd[i] == 1) continue;
    if (!ext.empty() && ss.back() == src_stride[i] * dd[i] && ext.back() * dd[i] < (1ll << 31)) {
      ext.back() *= dd[i];
      ss.back() = src_stride[i];
    } else {
      ext.push_back(dd[i]);
      ss.push_back(src_stride[i]);
    }
  }
  const std::vector<int64_t> ds = strides_of(ext);
  const int n = (int)ext.size();
  TMX_REQUIRE(n <= MAXR, "too many modes in a block permutation");
  sh.n = n;
  if (n == 0) return sh;
  std::vector<int64_t> box(n, 1);
  std::vector<int> role(n, -1), X, Y, Z;  // fastest first
  // Takes mode m into a side: in full when that keeps the side at `cap` (and offsets inside the
  // box in 32 bits), else cut evenly.
  int64_t span = (1ll << 31) - 1;  // largest offset the box may still add
  auto take = [&](std::vector<int>& side, int r, int m, int64_t have, int64_t cap) {
    const int64_t stride = std::max(ss[m], ds[m]);
    const int64_t most = std::max<int64_t>(1, std::min(cap / have, 1 + span / stride));
    const int64_t cuts = (ext[m] + most - 1) / most;
    box[m] = (ext[m] + cuts - 1) / cuts;
    span -= (box[m] - 1) * stride;
    role[m] = r;
    side.push_back(m);
    return have * box[m];
  };
  std::vector<int> by_src(n);  // modes by source stride, fastest first
  std::iota(by_src.begin(), by_src.end(), 0);
  std::sort(by_src.begin(), by_src.end(), [&](int a, int b) { return ss[a] < ss[b]; });
  const bool same = by_src[0] == n - 1;
  if (elems == 0) {
    if (!same) X.push_back(by_src[0]);
    Y.push_back(n - 1);
    for (int m = n - 2; m >= 0; --m)
      if (same || m != X[0]) Z.push_back(m);
    if (same) box[n - 1] = kAssignTile * kAssignTile;
    else box[X[0]] = box[n - 1] = kAssignTile;
  } else {
    int64_t nx = 1, ny = 1, nz = 1;
    if (same) {
      const int64_t run = std::min<int64_t>(kAssignRole, elems);
      ny = take(Y, 1, n - 1, 1, run);
      for (int m = n - 2; m >= 0 && ny < 64 && box[Y.back()] == ext[Y.back()]; --m) ny = take(Y, 1, m, ny, run);
    } else {
      nx = take(X, 0, by_src[0], 1, side);
      ny = take(Y, 1, n - 1, 1, side);
      for (int k = 1; k < n && nx < std::min<int64_t>(side, 32) && box[X.back()] == ext[X.back()] && role[by_src[k]] < 0; ++k)
        nx = take(X, 0, by_src[k], nx, side);
      for (int m = n - 2; m >= 0 && ny < std::min<int64_t>(side, 32) && box[Y.back()] == ext[Y.back()] && role[m] < 0; --m)
        ny = take(Y, 1, m, ny, side);
      int64_t rest = 1;  // what Z could take
      for (int m = 0; m < n; ++m)
        if (role[m] < 0) rest = std::min(rest * ext[m], elems);
      // re-takes a side's last mode up to `cap` when it is cut
      auto grow = [&](std::vector<int>& v, int r, int64_t have, int64_t cap) {
        const int m = v.back();
        if (box[m] == ext[m] || cap < 2 * have) return have;
        have /= box[m];
        span += (box[m] - 1) * std::max(ss[m], ds[m]);
        v.pop_back();
        return take(v, r, m, have, std::min<int64_t>(cap, kAssignRole));
      };
      nx = grow(X, 0, nx, std::min(elems / (ny * rest), lds / ((ny | 1) * rest)));
      ny = grow(Y, 1, ny, std::min(elems / (nx * rest), lds / (nx * rest) - 1));
    }
    const int64_t room = std::min<int64_t>(std::min<int64_t>(elems / (nx * ny), kAssignRole),
                                           same ? kAssignRole : lds / (nx * (ny | 1)));
    for (int m = n - 1; m >= 0; --m) {
      if (role[m] >= 0) continue;
      // a side's cut mode, or Z's own, ends the run: later modes stay outside the box
      if (nz < room) nz = take(Z, 2, m, nz, room);
      else Z.push_back(m);
    }
  }
  sh.nx = (int)X.size();
  sh.ny = (int)Y.size();
  std::vector<int64_t> nt(n);
  for (int i = 0; i < n; ++i) nt[i] = (ext[i] + box[i] - 1) / box[i];
  const std::vector<int64_t> tdiv = strides_of(nt);
  int k = 0;
  for (const std::vector<int>* side : {&X, &Y, &Z})
    for (size_t i = side->size(); i-- > 0; ++k) {
      const int m = (*side)[i];
      sh.ext[k] = (int)ext[m];
      sh.box[k] = (int)box[m];
      sh.nt[k] = (int)nt[m];
      sh.tdiv[k] = (int)tdiv[m];
      sh.sstr[k] = ss[m];
      sh.dstr[k] = ds[m];
    }
  return sh;
}

// Assign plan between two operands whose labels are a permutation of each other; zeroing: lists
// the destination blocks that have no source block.
std::unique_ptr<AssignPlan> build_assign_plan(const LOperand& D, const LOperand& S, bool zeroing) {
  TMX_REQUIRE(D.labels.size() == S.labels.size(), "assign: label sets differ");
  for (int l : D.labels) TMX_REQUIRE(pos_of(S.labels, l) >= 0, "assign: labels are not a permutation");
  std::vector<AssignJob> jobs;
  std::vector<std::vector<int64_t>> geoms;  // dims and source strides of the distinct shapes
  std::vector<int64_t> uses;                // jobs of each
  std::map<std::vector<int64_t>, int> sidx;
  std::vector<int64_t> zoff, zpre{0};
  const size_t r = D.labels.size();
  std::vector<int64_t> ext(r);
  for (size_t i = 0; i < r; ++i) ext[i] = D.ntl[i];
  std::vector<int64_t> it(r, 0), db(r), sb(r);
  bool empty = false;
  for (auto e : ext) if (e == 0) empty = true;
  while (!empty) {
    for (size_t i = 0; i < r; ++i) db[i] = D.toff[i] + it[i];
    if (D.t->is_non_zero(db.data())) {
      for (size_t j = 0; j < r; ++j) sb[j] = S.toff[j] + it[pos_of(D.labels, S.labels[j])];
      int64_t doff = D.t->find(db.data());
      int64_t soff = S.t->is_non_zero(sb.data()) ? S.t->find(sb.data()) : -1;
      std::vector<int64_t> dd(r), sd(r);
      int64_t size = 1;
      for (size_t i = 0; i < r; ++i) size *= dd[i] = D.t->modes[i]->tsize(db[i]);
      for (size_t i = 0; i < r; ++i) sd[i] = S.t->modes[i]->tsize(sb[i]);
      if (soff < 0) {
        if (zeroing && size > 0) {
          zoff.push_back(doff);
          zpre.push_back(zpre.back() + size);
        }
      } else if (size > 0) {
        const std::vector<int64_t> ss = strides_of(sd);
        std::vector<int64_t> key(dd), st(r);
        for (size_t i = 0; i < r; ++i) st[i] = ss[pos_of(S.labels, D.labels[i])];
        key.insert(key.end(), st.begin(), st.end());
        const auto f = sidx.emplace(key, (int)geoms.size());
        if (f.second) {
          geoms.push_back(key);
          uses.push_back(0);
        }
        ++uses[f.first->second];
        AssignJob jb;
        jb.src_off = soff;
        jb.dst_off = doff;
        jb.shape = f.first->second;
        jb.pad = 0;
        jobs.push_back(jb);
      }
    }
    int d = (int)r - 1;
    for (; d >= 0; --d) {
      if (++it[d] < ext[d]) break;
      it[d] = 0;
    }
    if (d < 0) break;
  }
  auto shape_of_geom = [&](size_t i, int64_t elems) {
    const std::vector<int64_t>& g = geoms[i];
    return make_assign_shape({g.begin(), g.begin() + r}, {g.begin() + r, g.end()}, elems);
  };
  auto tiles_of = [](const AssignShape& sh) {
    int64_t n = 1;
    for (int i = 0; i < sh.n; ++i) n *= sh.nt[i];
    return n;
  };
  // Whole tiles or boxes, by a model of the launch fitted to blocks of 10^2 to 3e8 elements: whole
  // tiles are cheap (1.6 ns each while all fit the chip at once, then 2.8), boxes of 256, 1024 and
  // 2304 elements cost 2, 4.5 and 7.5 ns each and a longer start.  48x48x16x16 with the outer two
  // modes exchanged, in whole tiles and in boxes: 86 and 7 us; 64x64x64x64, the last two: 41 and 49;
  // 17x40000 transposed: 4.7 and 7.1.
  struct Cut { int64_t elems; double start, each; };
  int64_t elems = 0;
  double best_us = -1;
  const size_t step = (geoms.size() + 31) / 32;  // ragged blocks have thousands of shapes: 32 stand for all
  for (const Cut& c : {Cut{0, 3.0, 1.6e-3}, Cut{256, 3.5, 2e-3}, Cut{1024, 4.7, 4.5e-3}, Cut{kAssignElems, 6.3, 7.5e-3}}) {
    double n = 0, seen = 0;
    for (size_t i = 0; i < geoms.size(); i += step) {
      n += (double)tiles_of(shape_of_geom(i, c.elems)) * (double)uses[i];
      seen += (double)uses[i];
    }
    if (seen > 0) n *= (double)jobs.size() / seen;
    const double us = c.start + n * c.each + (c.elems == 0 ? std::max(0.0, n - 2048) * 1.2e-3 : 0.0);
    if (best_us >= 0 && us >= best_us) continue;
    best_us = us;
    elems = c.elems;
  }
  std::vector<AssignShape> shapes;
  for (size_t i = 0; i < geoms.size(); ++i) shapes.push_back(shape_of_geom(i, elems));
  std::vector<int64_t> tiles;
  for (const AssignShape& sh : shapes) {
    tiles.push_back(tiles_of(sh));
    TMX_REQUIRE(tiles.back() < (1ll << 31), "block too large");
  }
  std::vector<AssignUnit> units;
  size_t nunits = 0;
  for (const AssignJob& jb : jobs) nunits += (size_t)tiles[jb.shape];
  units.reserve(nunits);
  for (size_t j = 0; j < jobs.size(); ++j)
    for (int64_t t = 0; t < tiles[jobs[j].shape]; ++t) units.push_back({(int32_t)j, (int32_t)t});
  auto p = std::make_unique<AssignPlan>();
  p->nunits = (int64_t)units.size();
  p->box = (int)elems;
  p->nzero = (int)zoff.size();
  p->zero_elems = zpre.back();
  std::vector<char> bytes;
  auto put = [&](const auto& v) {  // offset of v's bytes, 8-byte aligned
    const size_t at = (bytes.size() + 7) / 8 * 8, n = v.size() * sizeof(v[0]);
    bytes.resize(at + n);
    if (n) std::memcpy(bytes.data() + at, v.data(), n);
    return at;
  };
  const size_t o_shapes = put(shapes), o_jobs = put(jobs), o_units = put(units), o_zoff = put(zoff), o_zpre = put(zpre);
  p->tables = upload(bytes);
  const char* base = p->tables.as<char>();
  p->shapes = reinterpret_cast<const AssignShape*>(base + o_shapes);
  p->jobs = reinterpret_cast<const AssignJob*>(base + o_jobs);
  p->units = reinterpret_cast<const AssignUnit*>(base + o_units);
  p->zero_off = reinterpret_cast<const int64_t*>(base + o_zoff);
  p->zero_prefix = reinterpret_cast<const int64_t*>(base + o_zpre);
  return p;
}

}  // namespace tmx

struct tmx_addop_s {
  LOperand C, A;
  double alpha = 1;
  int is_assign = 0;
  std::unique_ptr<AssignPlan> plan;
  bool whole = false;  // identical labels and layouts over whole tensors: one streaming pass
};

// C(l) (=|+=) alpha * A(l) with the same label list, both operands spanning their whole
// tensors, and the two tensors laid out identically (same blocks, same offsets): no
// permutation and no block bookkeeping, so the op is one element-wise pass over the buffer.
static bool same_layout_whole(const LOperand& C, const LOperand& A) {
  if (C.labels != A.labels || C.t->nmodes() != A.t->nmodes()) return false;
  for (int i = 0; i < C.t->nmodes(); ++i) {
    if (C.toff[i] != 0 || A.toff[i] != 0) return false;
    if (C.ntl[i] != C.t->modes[i]->ntiles() || A.ntl[i] != A.t->modes[i]->ntiles()) return false;
    if (C.t->modes[i]->ntiles() != A.t->modes[i]->ntiles()) return false;
    for (int64_t k = 0; k < C.t->modes[i]->ntiles(); ++k)
      if (C.t->modes[i]->tsize(k) != A.t->modes[i]->tsize(k)) return false;
  }
  return C.t->total == A.t->total && C.t->keys == A.t->keys && C.t->offs == A.t->offs;
}

extern "C" {

int tmx_block_multiply(double alpha, const double* A, int andim, const int64_t* adims,
                       const int* alabels, const double* B, int bndim, const int64_t* bdims,
                       const int* blabels, double* C, int cndim, const int64_t* cdims,
                       const int* clabels, int is_assign, void* stream) {
  return guarded([&] {
    hipStream_t s = pick_stream(stream);
    TMX_REQUIRE(A && B && C, "null block pointer");
    TMX_REQUIRE(andim >= 0 && bndim >= 0 && cndim >= 0, "negative rank");
    std::vector<int64_t> key{andim, bndim, cndim};
    for (int i = 0; i < andim; ++i) { key.push_back(adims[i]); key.push_back(alabels[i]); }
    for (int i = 0; i < bndim; ++i) { key.push_back(bdims[i]); key.push_back(blabels[i]); }
    for (int i = 0; i < cndim; ++i) { key.push_back(cdims[i]); key.push_back(clabels[i]); }
    BlockMulPlan* plan;
    {
      std::lock_guard<std::mutex> g(cache_mu());
      auto& g_bm_cache = bm_cache();
      auto it = g_bm_cache.find(key);
      if (it == g_bm_cache.end()) {
        LOperand Co = single_block_operand(cndim, cdims, clabels);
        LOperand Ao = single_block_operand(andim, adims, alabels);
        LOperand Bo = single_block_operand(bndim, bdims, blabels);
        LabelInfo li = analyse_labels(Co, Ao, Bo);
        std::vector<CBlockWork> work = enumerate_pairs(Co, Ao, Bo, li);
        auto p = std::make_unique<BlockMulPlan>();
        build_bp_plan(p->bp, Co, Ao, Bo, li, work, false, nullptr, nullptr);
        it = g_bm_cache.emplace(key, std::move(p)).first;
      }
      plan = it->second.get();
    }
    launch_bp_plan(plan->bp, plan->bp.tasks.as<BPTask>(), plan->bp.ntasks, &plan->bp.xcd, A, B, C,
                   alpha, is_assign, s);
  });
}

int tmx_block_assign(double* dst, int ndim, const int64_t* ddims, const int* dlabels, double scale,
                     const double* src, const int64_t* sdims, const int* slabels, int is_assign,
                     void* stream) {
  return guarded([&] {
    hipStream_t s = pick_stream(stream);
    TMX_REQUIRE(dst && src, "null block pointer");
    std::vector<int64_t> key{ndim};
    for (int i = 0; i < ndim; ++i) { key.push_back(ddims[i]); key.push_back(dlabels[i]); }
    for (int i = 0; i < ndim; ++i) { key.push_back(sdims[i]); key.push_back(slabels[i]); }
    AssignPlan* plan;
    {
      std::lock_guard<std::mutex> g(cache_mu());
      auto& g_as_cache = as_cache();
      auto it = g_as_cache.find(key);
      if (it == g_as_cache.end()) {
        LOperand D = single_block_operand(ndim, ddims, dlabels);
        LOperand S = single_block_operand(ndim, sdims, slabels);
        for (int i = 0; i < ndim; ++i) {
          int p = pos_of(S.labels, D.labels[i]);
          TMX_REQUIRE(p >= 0 && sdims[p] == ddims[i], "assign: dims do not match the permutation");
        }
        it = g_as_cache.emplace(key, build_assign_plan(D, S, false)).first;
      }
      plan = it->second.get();
    }
    launch_assign(plan->jobs, plan->units, plan->nunits, plan->box, plan->shapes, src, dst, scale, is_assign, s);
  });
}

static HandleRegistry<tmx_addop_s>& addops() {
  static auto* r = new HandleRegistry<tmx_addop_s>();
  return *r;
}

int tmx_addop_create(const tmx_operand* C, double alpha, const tmx_operand* A, int is_assign,
                     tmx_addop* out) {
  return guarded([&] {
    require_init();
    auto op = std::make_shared<tmx_addop_s>();
    op->C = make_loperand(C);
    op->A = make_loperand(A);
    op->alpha = alpha;
    op->is_assign = is_assign;
    LabelInfo li = analyse_labels(op->C, op->A, op->A);  // validates tilings of shared labels
    (void)li;
    op->whole = same_layout_whole(op->C, op->A);
    if (!op->whole) op->plan = build_assign_plan(op->C, op->A, is_assign != 0);
    *out = addops().add(std::move(op));
  });
}

int tmx_addop_execute(tmx_addop op, const double* A, double* C, void* stream) {
  return guarded([&] {
    TMX_REQUIRE(op && A && C, "null argument");
    hipStream_t s = pick_stream(stream);
    if (stream_capturing(s)) capture_hold(s, addops().get(op));
    if (op->whole) {
      if (op->is_assign) launch_scale_copy(op->C.t->total, op->alpha, A, C, s);
      else launch_axpy(op->C.t->total, op->alpha, A, C, s);
      return;
    }
    const AssignPlan& p = *op->plan;
    launch_zero_ranges(p.zero_off, p.zero_prefix, p.nzero, p.zero_elems, C, s);
    launch_assign(p.jobs, p.units, p.nunits, p.box, p.shapes, A, C, op->alpha, op->is_assign, s);
  });
}

int tmx_addop_destroy(tmx_addop op) {
  return guarded([&] {
    if (!op) return;
    quiesce();
    addops().drop(op);
  });
}

}  // extern "C"
