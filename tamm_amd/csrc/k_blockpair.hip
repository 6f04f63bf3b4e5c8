// k_blockpair.hip -- fused block-pair FP64 contraction and LDS-tiled block assign (gfx950).
//
// k_bp_f64 replaces TAMM's per-pair transpose -> dgemm -> transpose sequence
// (src/tamm/kernels/multiply.hpp:159-210 + gpu_blas.cpp:43-85): the permutation of A and B
// into GEMM order is folded into the global->LDS load (per-pair offset tables in LDS), the
// product runs on v_mfma_f64_16x16x4f64, and the epilogue accumulates straight into the C
// block in its own mode order.  One workgroup owns one C tile and loops over every
// reduction pair of that C block, so C is read and written once per tile and needs no
// atomics (TAMM zeroes, accumulates and copies a C staging buffer per block instead,
// multop.hpp:690-839).
//
// k_assign replaces kernels::assign / librett (assign.hpp:466-485, multiply.hpp:108-157):
// dst(dl) (+)= scale * src(sl) for a label permutation, in boxes of up to 2304 elements that
// pass through LDS so both the source read (along the source's contiguous mode) and the
// destination write (along the destination's contiguous mode) are coalesced.
#include "tmx_device.hpp"
#include "tmx_kernels.hpp"

namespace tmx {

typedef double d4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Fused block-pair FP64 GEMM.  256 threads = 4 waves in a WM x (4/WM) grid over a TM x TN C
// tile; each wave owns (TM/WM) x (TN*WM/4) = FM x FN MFMA 16x16 tiles; BK k per LDS stage,
// double buffered (global -> registers -> LDS).  Tile shapes: 64x64 (2x2 waves of 32x32, BK 16)
// for general blocks; 16x256 (1x4 waves of 16x64, BK 8) for blocks with few rows, such as
// one-body terms R(a,b,i,j) += F(k,i) T(a,b,k,j) whose row extent is one O tile, where a
// 64-row tile would be mostly padding (the plan puts the small side on the rows).
//
// LDS layout: As[m][k] and Bs[n][k] with an odd row stride (BK + 1 doubles).  The MFMA reads of
// a 16x4 fragment (lane l -> row l%16, k l/16) and both global->LDS write patterns (k-fastest
// or row-fastest) then spread over the banks.
constexpr int BP_KC = 512;

// 64x64: four workgroups per CU (128 VGPRs, 40 KB of LDS; 7-9% faster than three, which 136
// registers gave); 16x256: three (45 KB of LDS).
template <int TM, int TN, int WM, int BK>
__global__ __launch_bounds__(256, TM == 64 ? 4 : 3) void k_bp_f64(const BPTask* __restrict__ tasks, int ntasks,
                                                const BPPair* __restrict__ pairs,
                                                const BPCShape* __restrict__ cshapes,
                                                const BPKShape* __restrict__ kshapes,
                                                const double* __restrict__ A,
                                                const double* __restrict__ B,
                                                double* __restrict__ C, double alpha,
                                                int is_assign, BPXcd xr) {
  constexpr int WN = 4 / WM;
  constexpr int WTM = TM / WM, WTN = TN / WN;  // wave tile
  constexpr int FM = WTM / 16, FN = WTN / 16;  // MFMA tiles per wave
  constexpr int LD = BK + 1;
  constexpr int NA = (TM * BK + 255) / 256, NB = (TN * BK + 255) / 256;  // loads per thread
  static_assert(WM * WN == 4 && FM >= 1 && FN >= 1 && WTM % 16 == 0 && WTN % 16 == 0, "wave grid");
  static_assert(BK % 4 == 0 && BP_KC % BK == 0, "k stage");
  __shared__ double As[2][TM * LD];
  __shared__ double Bs[2][TN * LD];
  __shared__ int offAm[TM], offBn[TN], offCm[TM], offCn[TN];
  __shared__ int offAk[BP_KC], offBk[BP_KC];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave % WM, wn = wave / WM;

  const int xcd = blockIdx.x & 7, per_xcd = gridDim.x >> 3;
  for (int task_id = xr.lo[xcd] + (blockIdx.x >> 3); task_id < xr.hi[xcd]; task_id += per_xcd) {
    const BPTask tk = tasks[task_id];
    const BPCShape& cs = cshapes[tk.cshape];
    const int M = cs.M, N = cs.N;

    d4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};

    for (int p = tk.pair_begin; p < tk.pair_end; ++p) {
      const BPPair pr = pairs[p];
      const BPKShape& ks = kshapes[pr.kshape];
      const int K = ks.K;
      const double* Ablk = A + pr.a_off;
      const double* Bblk = B + pr.b_off;
      __syncthreads();  // previous users of the offset tables are done
      for (int t = tid; t < TM + TN; t += 256) {
        if (t < TM) {
          int m = tk.m0 + t;
          offAm[t] = m < M ? radix_off(ks.am, m) : -1;
        } else {
          int c = t - TM;
          int n = tk.n0 + c;
          offBn[c] = n < N ? radix_off(ks.bn, n) : -1;
        }
      }
      for (int kc = 0; kc < K; kc += BP_KC) {
        const int klen = min(BP_KC, K - kc);
        __syncthreads();
        for (int t = tid; t < BP_KC; t += 256) {
          int k = kc + t;
          bool ok = t < klen;
          offAk[t] = ok ? radix_off(ks.ak, k) : -1;
          offBk[t] = ok ? radix_off(ks.bk, k) : -1;
        }
        __syncthreads();
        const int nsteps = (klen + BK - 1) / BK;

        // Element q = tid + 256 e of a stage tile (rows x BK): along k when the operand is read
        // along K (its stride-1 mode is the fastest K digit), else along rows.
        double ra[NA], rb[NB];
        auto coord = [&](int q, int rows, bool kcontig, int& r, int& k) {
          if (kcontig) { k = q % BK; r = q / BK; }
          else { r = q % rows; k = q / rows; }
        };
        // No load is conditional: places past the block read its first element and their values
        // are replaced by 0 when they go to LDS.
        uint32_t ina = 0, inb = 0;
        auto load_stage = [&](int step) {
          const int kb = step * BK;
          ina = inb = 0;
#pragma unroll
          for (int e = 0; e < NA; ++e) {
            const int q = min(tid + 256 * e, TM * BK - 1);
            int r, k;
            coord(q, TM, ks.a_kcontig, r, k);
            const int om = offAm[r], ok = offAk[kb + k];
            const bool in = (om | ok) >= 0;
            ra[e] = Ablk[in ? om + ok : 0];
            ina |= in ? 1u << e : 0u;
          }
#pragma unroll
          for (int e = 0; e < NB; ++e) {
            const int q = min(tid + 256 * e, TN * BK - 1);
            int r, k;
            coord(q, TN, ks.b_kcontig, r, k);
            const int on = offBn[r], ok = offBk[kb + k];
            const bool in = (on | ok) >= 0;
            rb[e] = Bblk[in ? on + ok : 0];
            inb |= in ? 1u << e : 0u;
          }
        };
        auto store_stage = [&](int buf) {
#pragma unroll
          for (int e = 0; e < NA; ++e) {
            const int q = tid + 256 * e;
            int r, k;
            coord(q, TM, ks.a_kcontig, r, k);
            if (q < TM * BK) As[buf][r * LD + k] = ina >> e & 1 ? ra[e] : 0.0;
          }
#pragma unroll
          for (int e = 0; e < NB; ++e) {
            const int q = tid + 256 * e;
            int r, k;
            coord(q, TN, ks.b_kcontig, r, k);
            if (q < TN * BK) Bs[buf][r * LD + k] = inb >> e & 1 ? rb[e] : 0.0;
          }
        };

        load_stage(0);
        store_stage(0);
        __syncthreads();
        for (int s = 0; s < nsteps; ++s) {
          const int buf = s & 1;
          if (s + 1 < nsteps) load_stage(s + 1);
#pragma unroll
          for (int kk = 0; kk < BK / 4; ++kk) {
            const int kq = 4 * kk + (lane >> 4);
            double a[FM], b[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) a[i] = As[buf][(WTM * wm + 16 * i + (lane & 15)) * LD + kq];
#pragma unroll
            for (int j = 0; j < FN; ++j) b[j] = Bs[buf][(WTN * wn + 16 * j + (lane & 15)) * LD + kq];
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
              for (int j = 0; j < FN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
          }
          if (s + 1 < nsteps) store_stage(buf ^ 1);
          __syncthreads();
        }
      }
    }

    // Epilogue: C(clabels) (=|+=) alpha * acc, straight into the block's own mode order.
    __syncthreads();
    for (int t = tid; t < TM + TN; t += 256) {
      if (t < TM) {
        int m = tk.m0 + t;
        offCm[t] = m < M ? radix_off(cs.cm, m) : -1;
      } else {
        int c = t - TM;
        int n = tk.n0 + c;
        offCn[c] = n < N ? radix_off(cs.cn, n) : -1;
      }
    }
    __syncthreads();
    // v_mfma_f64_16x16x4f64 result: register e of lane l holds row 4e + l/16, col l%16.  All old
    // values are loaded before any is stored (places past the block read its first element);
    // one by one each load waited for the store before it: one-body terms over 3e7 elements 341, 321,
    // 243 and 230 -> 306, 283, 227 and 230 us.
    double* Cblk = C + tk.c_off;
    const auto place = [&](int i, int j, int e) {  // -1: past the block
      const int om = offCm[WTM * wm + 16 * i + 4 * e + (lane >> 4)], on = offCn[WTN * wn + 16 * j + (lane & 15)];
      return (om | on) >= 0 ? om + on : -1;
    };
    double old[FM][FN][4];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) old[i][j][e] = is_assign ? 0.0 : Cblk[max(place(i, j, e), 0)];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int o = place(i, j, e);
          const double v = alpha * acc[i][j][e];
          if (o >= 0) Cblk[o] = is_assign ? v : old[i][j][e] + v;
        }
  }
}

// ---------------------------------------------------------------------------
// Fused block-pair FP64 GEMM, the reduction split over the waves of a workgroup: for small
// blocks, whose cost in k_bp_f64 is a chain of barriers and table loads per pair, and for
// products with too few C tiles to fill the chip.  The NW waves of a workgroup share one
// (16 FM) x (16 FN) C tile; the reduction is a stream of chunks of up to 64 indices of one block
// pair, dealt round-robin to the waves.  A wave needs no barrier for a chunk: its 64 lanes put
// the chunk's K offsets into the wave's own LDS row, and operands go straight from the TAMM
// blocks into MFMA registers (lane l: row l%16, k l/16), the next G k-steps loading while G
// multiply.  At the end the waves' partial tiles are summed through LDS, in wave order, and
// written along C's contiguous direction.
// Bound by the loads: a K-contiguous operand's load touches 16 rows x 32 B, about 43 cycles of a
// CU's address pipe averaged over both operands, so larger tiles (fewer loads per MFMA) run
// faster where there are enough of them: 16x16 / 32x32 / 64x64 at 14.6 / 29.7 / 45 TFLOP/s of
// padded work on a dense 20 + 80 orbital ladder (k_bp_f64 37.6).  16-byte loads of two k per
// lane, eight or sixteen waves per tile and deeper prefetch measured the same or slower.
// 12 + 24 orbitals in blocks of ~6x6: ladder 112 -> 18 us, Fock terms 15-23 -> 6; one pair of
// 36x36x36x36 and 36x36x16x16 blocks: 119 -> 55 us.
constexpr int BP_KCH = 64;

// G: k-steps (of 4) per group of loads.
template <int FM, int FN, int NW, int G, int OCC>
__global__ __launch_bounds__(64 * NW, OCC) void k_bp_ks(const BPTask* __restrict__ tasks, int ntasks,
                                                        const BPPair* __restrict__ pairs,
                                                        const BPCShape* __restrict__ cshapes,
                                                        const BPKShape* __restrict__ kshapes,
                                                        const double* __restrict__ A,
                                                        const double* __restrict__ B,
                                                        double* __restrict__ C, double alpha,
                                                        int is_assign, BPXcd xr) {
  constexpr int TM = 16 * FM, TN = 16 * FN, LD = TN + 1;
  constexpr int NP = NW * TM * LD * 8 <= 36 * 1024 ? NW : 1;  // partial tiles in LDS
  __shared__ double part[NP][TM * LD];
  __shared__ uint32_t offK[NW][2][2][BP_KCH];  // byte offsets of a chunk's K indices in A and B
  __shared__ int offCm[TM], offCn[TN];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lk = lane >> 4;
  const int xcd = blockIdx.x & 7, per_xcd = gridDim.x >> 3;
  for (int task_id = xr.lo[xcd] + (blockIdx.x >> 3); task_id < xr.hi[xcd]; task_id += per_xcd) {
    const BPTask tk = tasks[task_id];
    const BPCShape& cs = cshapes[tk.cshape];
    const int M = cs.M, N = cs.N;
    for (int t = tid; t < TM + TN; t += 64 * NW) {
      if (t < TM) offCm[t] = tk.m0 + t < M ? radix_off(cs.cm, tk.m0 + t) : -1;
      else offCn[t - TM] = tk.n0 + t - TM < N ? radix_off(cs.cn, tk.n0 + t - TM) : -1;
    }
    d4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
    int turn = wave;  // chunks until this wave's next one
    for (int p = tk.pair_begin; p < tk.pair_end; ++p) {
      const BPPair pr = pairs[p];
      const int K = pr.K, nch = (K + BP_KCH - 1) / BP_KCH;
      if (turn >= nch) {
        turn -= nch;
        continue;
      }
      const BPKShape& ks = kshapes[pr.kshape];
      const char* Ab = reinterpret_cast<const char*>(A + pr.a_off);
      const char* Bb = reinterpret_cast<const char*>(B + pr.b_off);
      // rows beyond the block repeat its last one: their products land in C rows never written
      uint32_t ra[FM], rb[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) ra[i] = 8u * (uint32_t)radix_off(ks.am, min(tk.m0 + 16 * i + l16, M - 1));
#pragma unroll
      for (int j = 0; j < FN; ++j) rb[j] = 8u * (uint32_t)radix_off(ks.bn, min(tk.n0 + 16 * j + l16, N - 1));
      int tb = 0, klen = 0, g = 0;  // offset table in use, its chunk's length, group in the chunk
      auto open_chunk = [&](int t) {
        klen = min(BP_KCH, K - turn * BP_KCH);
        const int kk = turn * BP_KCH + min(lane, klen - 1);
        offK[wave][t][0][lane] = 8u * (uint32_t)radix_off(ks.ak, kk);
        offK[wave][t][1][lane] = 8u * (uint32_t)radix_off(ks.bk, kk);
        tb = t;
        g = 0;
        __builtin_amdgcn_wave_barrier();
      };
      double a[2][G][FM], b[2][G][FN];
      auto load = [&](double (&av)[G][FM], double (&bv)[G][FN]) {
#pragma unroll
        for (int s = 0; s < G; ++s) {
          const int k = 4 * (G * g + s) + lk;
          const uint32_t oa = offK[wave][tb][0][k], ob = offK[wave][tb][1][k];
#pragma unroll
          for (int i = 0; i < FM; ++i) av[s][i] = *reinterpret_cast<const double*>(Ab + (ra[i] + oa));
#pragma unroll
          for (int j = 0; j < FN; ++j) bv[s][j] = *reinterpret_cast<const double*>(Bb + (rb[j] + ob));
        }
      };
      // multiplies group gg of a chunk of length len
      auto mul = [&](double (&av)[G][FM], double (&bv)[G][FN], int gg, int len) {
#pragma unroll
        for (int s = 0; s < G; ++s) {
          const int k0 = 4 * (G * gg + s);
          if (k0 >= len) break;
          if (k0 + 4 > len) {  // beyond the chunk: zeros on both sides
            const bool in = k0 + lk < len;
#pragma unroll
            for (int i = 0; i < FM; ++i) av[s][i] = in ? av[s][i] : 0.0;
#pragma unroll
            for (int j = 0; j < FN; ++j) bv[s][j] = in ? bv[s][j] : 0.0;
          }
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[s][i], bv[s][j], acc[i][j], 0, 0, 0);
        }
      };
      // Steps to the next group of this wave's chunks of the pair and starts its loads; then the
      // group before it is multiplied.
      auto step = [&](double (&na)[G][FM], double (&nb)[G][FN], double (&ca)[G][FM], double (&cb)[G][FN]) {
        const int cg = g, clen = klen;
        bool more = true;
        if ((g + 1) * 4 * G < klen) {
          ++g;
        } else {
          turn += NW;
          more = turn < nch;
          if (more) open_chunk(tb ^ 1);
        }
        if (more) load(na, nb);
        mul(ca, cb, cg, clen);
        return more;
      };
      open_chunk(0);
      load(a[0], b[0]);
      while (step(a[1], b[1], a[0], b[0]) && step(a[0], b[0], a[1], b[1])) {
      }
      turn -= nch;
    }
    // partial tiles -> LDS; v_mfma_f64_16x16x4f64 result: register e of lane l holds row
    // 4e + l/16, col l%16
    auto put = [&](double* pw, bool add) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            double* q = pw + (16 * i + 4 * e + lk) * LD + 16 * j + l16;
            *q = add ? *q + acc[i][j][e] : acc[i][j][e];
          }
    };
    if constexpr (NP == NW) {
      put(part[wave], false);
    } else {
      for (int w = 0; w + 1 < NW; ++w) {
        if (wave == w) put(part[0], w > 0);
        __syncthreads();
      }
      if (wave == NW - 1) put(part[0], true);
    }
    __syncthreads();
    double* Cblk = C + tk.c_off;
    constexpr int PER = TM * TN / (64 * NW), STEP = PER < 4 ? PER : 4;
    static_assert(PER * 64 * NW == TM * TN && PER % STEP == 0, "tile not a whole number of passes");
    for (int k0 = 0; k0 < PER; k0 += STEP) {
      double old[STEP];
      int off[STEP], at[STEP];
#pragma unroll
      for (int k = 0; k < STEP; ++k) {
        const int e = tid + 64 * NW * (k0 + k);
        const int row = cs.ncontig ? e / TN : e % TM, col = cs.ncontig ? e % TN : e / TM;
        const int om = offCm[row], on = offCn[col];
        off[k] = om >= 0 && on >= 0 ? om + on : -1;
        at[k] = row * LD + col;
        old[k] = !is_assign && off[k] >= 0 ? Cblk[off[k]] : 0.0;
      }
#pragma unroll
      for (int k = 0; k < STEP; ++k) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < NP; ++w) v += part[w][at[k]];
        if (off[k] >= 0) Cblk[off[k]] = is_assign ? alpha * v : old[k] + alpha * v;
      }
    }
    __syncthreads();  // the next tile rewrites the partials and offsets
  }
}

bool bp_tile_shares_k(int tile) { return tile == BP_TILE_KS16 || tile == BP_TILE_KS32 || tile == BP_TILE_KS64; }
int bp_tile_rows(int tile) {
  return tile == BP_TILE_16x256 || tile == BP_TILE_KS16 ? 16 : tile == BP_TILE_KS32 ? 32 : 64;
}
int bp_tile_cols(int tile) {
  return tile == BP_TILE_16x256 ? 256 : tile == BP_TILE_KS16 ? 16 : tile == BP_TILE_KS32 ? 32 : 64;
}

void launch_bp_f64(const BPTask* tasks, int ntasks, const BPPair* pairs, const BPCShape* cshapes,
                   const BPKShape* kshapes, const double* A, const double* B, double* C,
                   double alpha, int is_assign, hipStream_t s, const BPXcd* xr, int tile) {
  if (ntasks <= 0) return;
  BPXcd r;
  if (xr) {
    r = *xr;
  } else {
    for (int x = 0; x < 8; ++x) {
      r.lo[x] = (int)((int64_t)ntasks * x / 8);
      r.hi[x] = (int)((int64_t)ntasks * (x + 1) / 8);
    }
  }
  int longest = 1;
  for (int x = 0; x < 8; ++x) {
    TMX_REQUIRE(0 <= r.lo[x] && r.lo[x] <= r.hi[x] && r.hi[x] <= ntasks, "bad XCD task ranges");
    longest = std::max(longest, r.hi[x] - r.lo[x]);
  }
  const int grid = 8 * std::min(longest, 65535);
#define TMX_BP_LAUNCH(KERNEL_, THREADS_)                                                              \
  hipLaunchKernelGGL(KERNEL_, dim3(grid), dim3(THREADS_), 0, s, tasks, ntasks, pairs, cshapes, kshapes, \
                     A, B, C, alpha, is_assign, r)
  if (tile == BP_TILE_16x256) TMX_BP_LAUNCH((k_bp_f64<16, 256, 1, 8>), 256);
  else if (tile == BP_TILE_KS16) TMX_BP_LAUNCH((k_bp_ks<1, 1, 4, 8, 4>), 256);
  else if (tile == BP_TILE_KS32) TMX_BP_LAUNCH((k_bp_ks<2, 2, 4, 4, 4>), 256);
  else if (tile == BP_TILE_KS64) TMX_BP_LAUNCH((k_bp_ks<4, 4, 4, 2, 2>), 256);
  else TMX_BP_LAUNCH((k_bp_f64<64, 64, 2, 16>), 256);
#undef TMX_BP_LAUNCH
  TMX_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Block assign / transpose-accumulate: HBM-bound (16 B per element, 24 when accumulating).
//
// A workgroup iteration of k_assign takes one box of a (dst block, src block) pair (AssignShape; blocks
// that fill whole tiles take k_assign_tile below).  The
// offsets of the box's X, Y and Z indices go to LDS tables once; elements are read with X
// fastest, then Y, then Z (the source's contiguous mode along the lanes), pass through an LDS
// tile and are written with Y fastest, then X, then Z.  Without X modes both orders are the same
// and the tile is skipped.  Each thread has its PER source loads and, accumulating, its PER
// destination loads in flight together: 1, 4 or 9 for boxes of 256, 1024 or 2304 elements.  Boxes
// span as many modes as it takes to hold that many: in whole tiles or runs of the contiguous mode,
// amplitude blocks of 48x48x16x16 gave each workgroup 256 or 16 elements: over 3.5e7 elements, R(a,b,i,j) -=
// T(b,a,i,j) went from 9.49 to 0.17 ms (5.0 TB/s) and R(a,b,i,j) -= T(a,b,j,i) from 0.93 to 0.17.
struct AssignTable {
  int s, d;
};
__device__ __forceinline__ uint32_t div_magic(uint32_t d) { return d > 1 ? 0xffffffffu / d + 1 : 0; }
// e / d for e, d <= 4096 and m = div_magic(d).
__device__ __forceinline__ uint32_t div_by(uint32_t e, uint32_t d, uint32_t m) {
  return d > 1 ? __umulhi(e, m) : e;
}

template <int PER>
__global__ __launch_bounds__(256) void k_assign(const AssignJob* __restrict__ jobs,
                                                const AssignUnit* __restrict__ units, int64_t nunits,
                                                const AssignShape* __restrict__ shapes,
                                                const double* __restrict__ src,
                                                double* __restrict__ dst, double scale,
                                                int is_assign) {
  __shared__ double tile[kAssignLds * PER];
  __shared__ AssignTable tab[kAssignTable];
  __shared__ int act[MAXR];
  __shared__ int64_t first_s[MAXR], first_d[MAXR];
  const int tid = threadIdx.x;
  for (int64_t u = blockIdx.x; u < nunits; u += gridDim.x) {
    const AssignUnit un = units[u];
    const AssignJob jb = jobs[un.job];
    const AssignShape& sh = shapes[jb.shape];
    // the box's start and its extents (short at the end of a mode), a lane per mode
    const int n_modes = sh.n, by = sh.nx, bz = sh.nx + sh.ny;
    if (tid < MAXR) {
      int a = 1, start = 0;
      if (tid < n_modes) {
        const uint32_t q = (uint32_t)un.tile / (uint32_t)sh.tdiv[tid], nt = (uint32_t)sh.nt[tid];
        start = (int)(q % nt) * sh.box[tid];
        a = min(sh.box[tid], sh.ext[tid] - start);
      }
      act[tid] = a;
      first_s[tid] = tid < n_modes ? start * sh.sstr[tid] : 0;
      first_d[tid] = tid < n_modes ? start * sh.dstr[tid] : 0;
    }
    __syncthreads();
    int64_t sb = jb.src_off, db = jb.dst_off;
    int X = 1, Y = 1, Z = 1;
#pragma unroll
    for (int k = 0; k < MAXR; ++k) {
      sb += first_s[k];
      db += first_d[k];
      X *= k < by ? act[k] : 1;
      Y *= k >= by && k < bz ? act[k] : 1;
      Z *= k >= bz ? act[k] : 1;
    }
    // offsets of index i of the role with modes [b, e)
    auto entry = [&](int b, int e, int i) {
      AssignTable t{0, 0};
      for (int k = e - 1; k >= b; --k) {
        int dig = i;
        if (k > b) {  // the slowest mode's digit is what is left
          const uint32_t q = (uint32_t)i / (uint32_t)act[k];
          dig = i - (int)q * act[k];
          i = (int)q;
        }
        t.s += dig * (int)sh.sstr[k];
        t.d += dig * (int)sh.dstr[k];
      }
      return t;
    };
    const int XY = X * Y, n = XY * Z;
    AssignTable *tx = tab, *ty = tx + X, *tz = ty + Y;
    for (int i = tid; i < X; i += 256) tx[i] = entry(0, by, i);
    for (int i = tid; i < Y; i += 256) ty[i] = entry(by, bz, i);
    for (int i = tid; i < Z; i += 256) tz[i] = entry(bz, n_modes, i);
    const uint32_t mx = div_magic(X), my = div_magic(Y), mxy = div_magic(XY);
    __syncthreads();
    const double* sp = src + sb;
    double* dp = dst + db;
    double v[PER], old[PER];
    int dof[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = tid + 256 * k;
      v[k] = 0.0;
      if (e < n) {
        const int z = div_by(e, XY, mxy), r = e - z * XY, y = div_by(r, X, mx), x = r - y * X;
        v[k] = sp[tx[x].s + ty[y].s + tz[z].s];
      }
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = tid + 256 * k;
      old[k] = 0.0;
      dof[k] = 0;
      if (e < n) {
        const int z = div_by(e, XY, mxy), r = e - z * XY, x = div_by(r, Y, my), y = r - x * Y;
        dof[k] = tx[x].d + ty[y].d + tz[z].d;
        if (!is_assign) old[k] = dp[dof[k]];
      }
    }
    if (X > 1) {
      const int ld = Y | 1;
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int e = tid + 256 * k;
        if (e < n) {
          const int z = div_by(e, XY, mxy), r = e - z * XY, y = div_by(r, X, mx), x = r - y * X;
          tile[(z * X + x) * ld + y] = v[k];
        }
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int e = tid + 256 * k;
        if (e < n) {
          const int q = div_by(e, Y, my);  // z * X + x
          v[k] = tile[q * ld + (e - q * Y)];
        }
      }
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = tid + 256 * k;
      if (e < n) {
        const double t = scale * v[k];
        dp[dof[k]] = is_assign ? t : old[k] + t;
      }
    }
    __syncthreads();  // the next box rewrites the tables and the tile
  }
}

// Whole tiles (make_assign_shape without `elems`): 32 x 32 of the source's and the destination's
// contiguous modes through LDS, or 1024 elements of a shared contiguous mode.  No tables and hardly
// any index arithmetic, so blocks that fill such tiles, and small ones, run faster than in boxes
// (the rule is at build_assign_plan): 64x64x64x64 with the last two modes exchanged 41 against 49 us
// (6.5 TB/s), 3e7 contiguous elements 88 against 191, 17x40000 transposed 4.7 against 7.1.  The
// order of the tiles: with X first instead of Y, 94x92x60x161 to modes (3,1,2,0) 417 against 373 us.
__global__ __launch_bounds__(256) void k_assign_tile(const AssignJob* __restrict__ jobs,
                                                     const AssignUnit* __restrict__ units, int64_t nunits,
                                                     const AssignShape* __restrict__ shapes,
                                                     const double* __restrict__ src,
                                                     double* __restrict__ dst, double scale,
                                                     int is_assign) {
  __shared__ double tile[kAssignTile][kAssignTile + 1];
  const int tid = threadIdx.x, lx = tid & 31, ly = tid >> 5;  // 32 x 8
  for (int64_t u = blockIdx.x; u < nunits; u += gridDim.x) {
    const AssignUnit un = units[u];
    const AssignJob jb = jobs[un.job];
    const AssignShape& sh = shapes[jb.shape];
    int64_t sb = jb.src_off, db = jb.dst_off;
    int left[2] = {1, 1};  // elements of the first two listed modes from the tile's start on
    uint32_t t = (uint32_t)un.tile;
    for (int i = 0; i < sh.n; ++i) {  // tiles along Y first, then X, then the rest, fastest first
      const int k = i <= sh.nx ? sh.nx - i : sh.n + sh.nx - i;
      const uint32_t q = i + 1 < sh.n ? t / (uint32_t)sh.nt[k] : 0;
      const int start = (int)(t - q * (uint32_t)sh.nt[k]) * sh.box[k];
      t = q;
      sb += start * sh.sstr[k];
      db += start * sh.dstr[k];
      if (k < 2) left[k] = sh.ext[k] - start;
    }
    const double* sp = src + sb;
    double* dp = dst + db;
    if (sh.nx == 0) {
      for (int e = tid; e < min(kAssignTile * kAssignTile, left[0]); e += 256) {
        const double r = scale * sp[e];
        dp[e] = is_assign ? r : dp[e] + r;
      }
      continue;
    }
    const int64_t ys = sh.sstr[1], xd = sh.dstr[0];  // the other stride of X and of Y is 1
    double v[4], old[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int y = ly + 8 * k;
      v[k] = lx < left[0] && y < left[1] ? sp[lx + y * ys] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int x = ly + 8 * k;
      old[k] = !is_assign && x < left[0] && lx < left[1] ? dp[lx + x * xd] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) tile[ly + 8 * k][lx] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int x = ly + 8 * k;
      const double r = scale * tile[lx][x];
      if (x < left[0] && lx < left[1]) dp[lx + x * xd] = is_assign ? r : old[k] + r;
    }
    __syncthreads();  // the next tile is written
  }
}

void launch_assign(const AssignJob* jobs, const AssignUnit* units, int64_t nunits, int box,
                   const AssignShape* shapes, const double* src, double* dst, double scale,
                   int is_assign, hipStream_t s) {
  if (nunits <= 0) return;
  const int grid = (int)std::min<int64_t>(nunits, 65536);
  const auto kernel = box == 0 ? &k_assign_tile : box == 256 ? &k_assign<1> : box == 1024 ? &k_assign<4> : &k_assign<9>;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, s, jobs, units, nunits, shapes, src, dst, scale, is_assign);
  TMX_HIP(hipGetLastError());
}

}  // namespace tmx
