// k_elementwise.hip -- fills, scaling, reductions, synthetic inputs, energy denominator.
//
// These cover TAMM's SetOp (C() = v), scale/axpy updates, norm (tamm_utils.hpp:1197-1254:
// sqrt of the sum of squares over stored blocks) and the element-wise update of a doubles
// residual by orbital-energy denominators.  All are HBM-bound streaming kernels with
// 16-byte accesses and a grid sized to a few waves per CU.
#include "tmx_kernels.hpp"
#include "tmx_rng.h"

namespace tmx {

namespace {
inline int grid_for(int64_t n, int per_block) {
  int64_t g = (n + per_block - 1) / per_block;
  return (int)std::max<int64_t>(1, std::min<int64_t>(g, 8192));
}
}  // namespace

__global__ __launch_bounds__(256) void k_fill(double* __restrict__ p, int64_t n, double v) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = v;
}
__global__ __launch_bounds__(256) void k_zero_bytes(uint8_t* __restrict__ p, size_t n) {
  for (size_t i = blockIdx.x * 256ull + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = 0;
}
__global__ __launch_bounds__(256) void k_zero_u4(uint4* __restrict__ p, size_t n) {
  for (size_t i = blockIdx.x * 256ull + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
    p[i] = make_uint4(0, 0, 0, 0);
}
__global__ __launch_bounds__(256) void k_scale(double* __restrict__ p, int64_t n, double a) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] *= a;
}
__global__ __launch_bounds__(256) void k_axpy(int64_t n, double a, const double* __restrict__ x,
                                              double* __restrict__ y) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    y[i] += a * x[i];
}

void launch_fill(double* p, int64_t n, double v, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill, dim3(grid_for(n, 256 * 4)), dim3(256), 0, s, p, n, v);
  TMX_HIP(hipGetLastError());
}
// Zeroes the element ranges [off[i], off[i] + prefix[i+1] - prefix[i]) of C (prefix: running
// sums of the range lengths, prefix[0] = 0, prefix[n] = total): the blocks of an assigning
// contraction that no block pair writes.
__global__ __launch_bounds__(256) void k_zero_ranges(const int64_t* __restrict__ off,
                                                     const int64_t* __restrict__ prefix, int n,
                                                     double* __restrict__ C) {
  const int64_t total = prefix[n];
  for (int64_t e = blockIdx.x * 256ll + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (prefix[mid] <= e) lo = mid;
      else hi = mid - 1;
    }
    C[off[lo] + (e - prefix[lo])] = 0.0;
  }
}
void launch_zero_ranges(const int64_t* off, const int64_t* prefix, int n, int64_t total, double* C,
                        hipStream_t s) {
  if (n <= 0 || total <= 0) return;
  hipLaunchKernelGGL(k_zero_ranges, dim3(grid_for(total, 256 * 4)), dim3(256), 0, s, off, prefix, n, C);
  TMX_HIP(hipGetLastError());
}
void launch_fill_bytes_zero(void* p, size_t bytes, hipStream_t s) {
  if (bytes == 0) return;
  uintptr_t a = reinterpret_cast<uintptr_t>(p);
  if (a % 16 == 0 && bytes % 16 == 0) {
    hipLaunchKernelGGL(k_zero_u4, dim3(grid_for((int64_t)(bytes / 16), 1024)), dim3(256), 0, s,
                       static_cast<uint4*>(p), bytes / 16);
  } else {
    hipLaunchKernelGGL(k_zero_bytes, dim3(grid_for((int64_t)bytes, 1024)), dim3(256), 0, s,
                       static_cast<uint8_t*>(p), bytes);
  }
  TMX_HIP(hipGetLastError());
}
void launch_scale(double* p, int64_t n, double a, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_scale, dim3(grid_for(n, 1024)), dim3(256), 0, s, p, n, a);
  TMX_HIP(hipGetLastError());
}
void launch_axpy(int64_t n, double a, const double* x, double* y, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_axpy, dim3(grid_for(n, 1024)), dim3(256), 0, s, n, a, x, y);
  TMX_HIP(hipGetLastError());
}

// y = a * x (an assigning AddOp over whole tensors: one read and one write per element).
__global__ __launch_bounds__(256) void k_scale_copy(int64_t n, double a, const double* __restrict__ x,
                                                    double* __restrict__ y) {
  for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    y[i] = a * x[i];
}

void launch_scale_copy(int64_t n, double a, const double* x, double* y, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_scale_copy, dim3(grid_for(n, 1024)), dim3(256), 0, s, n, a, x, y);
  TMX_HIP(hipGetLastError());
}

// ---- reductions: per-block partial sums in FP64, summed by one workgroup on the device ----
// HBM-bound (8 or 16 B per element).  Each thread has eight nontemporal 8-byte loads per operand
// in flight (a workgroup's are one contiguous piece) and eight independent sums.  Read alone,
// 3.5e7 elements take 42 us (6.5 TB/s) this way, 46 with ordinary 8- or 16-byte loads in any
// order; the operands are not read again soon, so they need not displace the caches.  Right after
// an update that leaves the caches full of its writes the norm went from 66 to 40 us.
constexpr int kReduceUnroll = 8;
template <int OP>
__device__ __forceinline__ double reduce_term(double a, double b) {
  if (OP == 0) return a * a;
  if (OP == 1) return a * b;
  const double d = a - b;
  return d * d;
}
// Sum over a workgroup of 256 threads, valid in thread 0.
__device__ __forceinline__ double block_sum(double s) {
  __shared__ double sh[4];
  for (int w = 32; w > 0; w >>= 1) s += __shfl_down(s, w);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

template <int OP>
__global__ __launch_bounds__(256) void k_reduce(const double* __restrict__ x,
                                                const double* __restrict__ y, int64_t n,
                                                double* __restrict__ partial) {
  constexpr int U = kReduceUnroll, PIECE = 256 * U;
  double s[U] = {};
  const int64_t whole = n / PIECE * PIECE;
  for (int64_t i = (int64_t)blockIdx.x * PIECE + threadIdx.x; i < whole; i += (int64_t)gridDim.x * PIECE) {
    double a[U], b[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      a[k] = __builtin_nontemporal_load(x + i + 256 * k);
      b[k] = OP == 0 ? a[k] : __builtin_nontemporal_load(y + i + 256 * k);
    }
#pragma unroll
    for (int k = 0; k < U; ++k) s[k] += reduce_term<OP>(a[k], b[k]);
  }
  for (int64_t i = whole + (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    s[0] += reduce_term<OP>(x[i], OP == 0 ? x[i] : y[i]);
#pragma unroll
  for (int w = U / 2; w > 0; w >>= 1)
#pragma unroll
    for (int k = 0; k < w; ++k) s[k] += s[k + w];
  const double r = block_sum(s[0]);
  if (threadIdx.x == 0) partial[blockIdx.x] = r;
}

// Sums the partials with one workgroup into *out (device or pinned host memory), in an order
// that depends on their count alone.
__global__ __launch_bounds__(256) void k_reduce_finish(const double* __restrict__ partial, int g,
                                                       double* __restrict__ out) {
  double s = 0.0;
  for (int i = threadIdx.x; i < g; i += 256) s += partial[i];
  s = block_sum(s);
  if (threadIdx.x == 0) *out = s;
}

constexpr int kMaxPartials = 2048;
static int reduce_grid(int64_t n) { return std::min(grid_for(n, 256 * kReduceUnroll), kMaxPartials); }

// Partial sums into `partial` (reduce_grid(n) doubles), their sum into *out.
template <int OP>
static void launch_reduce(const double* x, const double* y, int64_t n, double* partial, double* out,
                          hipStream_t s) {
  const int g = reduce_grid(n);
  hipLaunchKernelGGL(k_reduce<OP>, dim3(g), dim3(256), 0, s, x, y, n, partial);
  hipLaunchKernelGGL(k_reduce_finish, dim3(1), dim3(256), 0, s, partial, g, out);
  TMX_HIP(hipGetLastError());
}

template <int OP>
static double reduce(const double* x, const double* y, int64_t n, hipStream_t s) {
  if (n <= 0) return 0.0;
  DevBuf part(sizeof(double) * (reduce_grid(n) + 1));
  // The finished sum lands in pinned host memory; without a free slot it is copied from the
  // buffer's last element.
  ResultSlot slot;
  double* out = slot.dev ? slot.dev : part.as<double>() + reduce_grid(n);
  launch_reduce<OP>(x, y, n, part.as<double>(), out, s);
  double r = 0.0;
  if (!slot.dev) TMX_HIP(hipMemcpyAsync(&r, out, sizeof(double), hipMemcpyDeviceToHost, s));
  TMX_HIP(hipStreamSynchronize(s));  // `part` and the slot are given back only after this
  return slot.dev ? *const_cast<volatile double*>(slot.host) : r;
}
// ---- norm without allocation (tmx_norm_noalloc) ----
// The partial sums of k_reduce (at most kMaxPartials workgroups) and the finished sum go
// to a file-scope device array instead of pool memory.  Each GPU holds its own copy of the
// array until the process ends; its address on a device comes from hipGetSymbolAddress, taken
// once per device by noalloc_setup (called from tmx_init with that device current).  Calls
// that overlap on one GPU share the array and race.
__device__ __align__(256) double scratch[kMaxPartials + 1];  // partials, then the sum
constexpr int kMaxDevices = 64;
static double* g_scratch_ptr[kMaxDevices] = {};

void noalloc_setup(int device) {
  TMX_REQUIRE(device >= 0 && device < kMaxDevices, "device index beyond the scratch table");
  if (g_scratch_ptr[device]) return;
  void* p = nullptr;
  TMX_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  g_scratch_ptr[device] = static_cast<double*>(p);
}

double reduce_sumsq_noalloc(const double* x, int64_t n, hipStream_t s, int device) {
  TMX_REQUIRE(device >= 0 && device < kMaxDevices && g_scratch_ptr[device],
              "no-allocation scratch not set up on this device (tmx_init)");
  if (n <= 0) return 0.0;
  double* sc = g_scratch_ptr[device];
  launch_reduce<0>(x, nullptr, n, sc, sc + kMaxPartials, s);
  double r = 0.0;
  TMX_HIP(hipMemcpyAsync(&r, sc + kMaxPartials, sizeof(double), hipMemcpyDeviceToHost, s));
  TMX_HIP(hipStreamSynchronize(s));
  return r;
}

double reduce_sumsq(const double* x, int64_t n, hipStream_t s) { return reduce<0>(x, nullptr, n, s); }
double reduce_dot(const double* x, const double* y, int64_t n, hipStream_t s) { return reduce<1>(x, y, n, s); }
double reduce_diffsq(const double* x, const double* y, int64_t n, hipStream_t s) { return reduce<2>(x, y, n, s); }

// ---- synthetic inputs: one workgroup per block, elements in block (row-major) order ----
struct GenDims {
  int nmodes;
  int64_t n[MAXR];
};

__global__ __launch_bounds__(256) void k_fill_normal(const GenBlock* __restrict__ blocks,
                                                     int64_t nblocks, GenDims gd,
                                                     double* __restrict__ data, uint64_t seed,
                                                     uint64_t tensor_id, double scale,
                                                     int symmetrize) {
  for (int64_t b = blockIdx.y * (int64_t)gridDim.x + blockIdx.x; b < nblocks;
       b += (int64_t)gridDim.x * gridDim.y) {
    const GenBlock gb = blocks[b];
    int64_t size = 1;
    for (int d = 0; d < gd.nmodes; ++d) size *= gb.ext[d];
    for (int64_t e = threadIdx.x; e < size; e += 256) {
      int64_t rem = e;
      int64_t idx[MAXR];
      for (int d = gd.nmodes - 1; d >= 0; --d) {
        idx[d] = gb.lo[d] + rem % gb.ext[d];
        rem /= gb.ext[d];
      }
      int64_t g = 0;
      for (int d = 0; d < gd.nmodes; ++d) g = g * gd.n[d] + idx[d];
      double z = tmx_rng_normal(seed, tensor_id, (uint64_t)g);
      if (symmetrize && gd.nmodes == 4) {
        int64_t g2 = ((idx[1] * gd.n[0] + idx[0]) * gd.n[3] + idx[3]) * gd.n[2] + idx[2];
        double z2 = tmx_rng_normal(seed, tensor_id, (uint64_t)g2);
        z = 0.5 * (z + z2);
      }
      data[gb.off + e] = scale * z;
    }
  }
}

void launch_fill_normal(const GenBlock* blocks, int64_t nblocks, int nmodes, const int64_t* mode_n,
                        int64_t /*max_block*/, double* data, uint64_t seed, uint64_t tensor_id,
                        double scale, int symmetrize, hipStream_t s) {
  if (nblocks <= 0) return;
  GenDims gd;
  std::memset(&gd, 0, sizeof(gd));
  gd.nmodes = nmodes;
  for (int i = 0; i < nmodes; ++i) gd.n[i] = mode_n[i];
  int gx = (int)std::min<int64_t>(nblocks, 65535);
  int gy = (int)std::min<int64_t>((nblocks + gx - 1) / gx, 64);
  hipLaunchKernelGGL(k_fill_normal, dim3(gx, gy), dim3(256), 0, s, blocks, nblocks, gd, data, seed,
                     tensor_id, scale, symmetrize);
  TMX_HIP(hipGetLastError());
}

// R(a,b,i,j) /= (e_i + e_j - e_a - e_b); blocks of a (V,V,O,O) tensor, lo = global indices.
// HBM-bound (16 B per element).  A workgroup takes a chunk of 256 E consecutive elements of the
// tensor, wherever the block boundaries fall: `first` lists the block each chunk starts in, so
// the chunk's blocks are known before any search, their starts go to LDS, and a thread finds the
// block of its E consecutive elements there, takes the first one's digits apart once and steps
// them.  E = 4 (two 16-byte loads); tensors too small to give every CU such a chunk take E = 1.
// With chunks of 4096 elements, blocks stepped through one by one and three integer divisions
// per element, 6.6e3 elements in blocks of ~20 took 130 us and 3.5e7 elements 173 us (3.2 TB/s);
// now 4.1 and 107 us (5.2 TB/s).
template <int E>
__global__ __launch_bounds__(256) void k_denominator(const GenBlock* __restrict__ blocks,
                                                     const int32_t* __restrict__ first,
                                                     int64_t nchunks, int64_t total,
                                                     double* __restrict__ data,
                                                     const double* __restrict__ eo,
                                                     const double* __restrict__ ev, int aligned) {
  constexpr int CHUNK = 256 * E;
  __shared__ int start[CHUNK + 2];  // block starts relative to the chunk (0 for its first block)
  const int tid = threadIdx.x;
  for (int64_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
    const int64_t c0 = c * CHUNK;
    const int n = (int)min((int64_t)CHUNK, total - c0);
    const int b0 = first[c], nb = first[c + 1] - b0 + 1;
    int e = tid * E;
    double* p = data + c0 + e;
    double v[E];
    if (E > 1 && aligned && e + E <= n) {
#pragma unroll
      for (int k = 0; k < E; k += 2) {
        const double2 t = *reinterpret_cast<const double2*>(p + k);
        v[k] = t.x;
        v[k + (E > 1)] = t.y;
      }
    } else {
#pragma unroll
      for (int k = 0; k < E; ++k) v[k] = e + k < n ? p[k] : 0.0;
    }
    for (int i = tid; i <= nb; i += 256)
      start[i] = i == 0 ? 0 : i == nb ? CHUNK : (int)min(blocks[b0 + i].off - c0, (int64_t)CHUNK);
    __syncthreads();
    if (e < n) {
      int lo = 0, hi = nb - 1;  // the last block starting at or before e
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (start[mid] <= e) lo = mid;
        else hi = mid - 1;
      }
      const GenBlock* gb = blocks + b0 + lo;
      uint32_t n1 = gb->ext[1], n2 = gb->ext[2], n3 = gb->ext[3];
      // a block holds fewer than 2^31 elements: its indices come apart in 32-bit arithmetic
      const uint32_t r = (uint32_t)(c0 + e - gb->off);
      const uint32_t q3 = r / n3, q2 = q3 / n2;
      uint32_t j = r - q3 * n3, i = q3 - q2 * n2, a = q2 / n1, b = q2 - a * n1;
      const double *pj = eo + gb->lo[3], *pi = eo + gb->lo[2], *pb = ev + gb->lo[1], *pa = ev + gb->lo[0];
      double ei = pi[i], ea = pa[a], eb = pb[b];
      double q[E];
#pragma unroll
      for (int k = 0; k < E; ++k) {
        q[k] = 0.0;
        if (e >= n) continue;
        q[k] = v[k] / (ei + pj[j] - ea - eb);
        ++e;
        if (k + 1 < E && (++j == n3 || e >= start[lo + 1])) {
          j = 0;
          if (e >= n) continue;
          if (e >= start[lo + 1]) {  // blocks hold at least one element: the next one starts here
            ++lo;
            ++gb;
            n1 = gb->ext[1], n2 = gb->ext[2], n3 = gb->ext[3];
            pj = eo + gb->lo[3], pi = eo + gb->lo[2], pb = ev + gb->lo[1], pa = ev + gb->lo[0];
            i = a = b = 0;
          } else if (++i == n2) {
            i = 0;
            if (++b == n1) {
              b = 0;
              ++a;
            }
          }
          ei = pi[i];
          ea = pa[a];
          eb = pb[b];
        }
      }
      e = tid * E;
      if (E > 1 && aligned && e + E <= n) {
#pragma unroll
        for (int k = 0; k < E; k += 2) *reinterpret_cast<double2*>(p + k) = make_double2(q[k], q[k + (E > 1)]);
      } else {
#pragma unroll
        for (int k = 0; k < E; ++k)
          if (e + k < n) p[k] = q[k];
      }
    }
    __syncthreads();  // the next chunk rewrites the starts
  }
}

int denominator_chunk(int64_t total) { return total >= 1024 * 1024 ? 1024 : 256; }

void launch_denominator(const GenBlock* blocks, const int32_t* first, int64_t total, double* data,
                        const double* e_occ, const double* e_vir, hipStream_t s) {
  if (total <= 0) return;
  const int chunk = denominator_chunk(total);
  const int64_t nchunks = (total + chunk - 1) / chunk;
  const int g = (int)std::min<int64_t>(nchunks, 65536);
  const int aligned = reinterpret_cast<uintptr_t>(data) % 16 == 0;
  if (chunk == 1024)
    hipLaunchKernelGGL(k_denominator<4>, dim3(g), dim3(256), 0, s, blocks, first, nchunks, total, data,
                       e_occ, e_vir, aligned);
  else
    hipLaunchKernelGGL(k_denominator<1>, dim3(g), dim3(256), 0, s, blocks, first, nchunks, total, data,
                       e_occ, e_vir, aligned);
  TMX_HIP(hipGetLastError());
}

}  // namespace tmx
