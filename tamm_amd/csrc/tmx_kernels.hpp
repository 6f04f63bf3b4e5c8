// tmx_kernels.hpp -- kernel descriptors and launcher declarations.
#pragma once

#include "tmx_internal.hpp"

namespace tmx {

// Block assign (permutation) descriptors.  Unit modes are dropped and modes that are neighbours
// in both blocks merged; a tile is a box of box[k] indices of every mode.  The modes have three
// roles and are listed by role, X's nx first, then Y's ny, then Z's, each slowest first: X holds
// the source's contiguous mode, Y the destination's, Z the rest.  When both blocks share their
// contiguous mode X is empty.  Offsets inside a box fit 32 bits.
struct AssignShape {
  int32_t n, nx, ny;
  int32_t ext[MAXR], box[MAXR], nt[MAXR];  // extent, box extent and boxes of each mode
  int32_t tdiv[MAXR];              // boxes: tile / tdiv % nt is the mode's box (destination order)
  int64_t sstr[MAXR], dstr[MAXR];  // source and destination strides
};
struct AssignJob {
  int64_t src_off, dst_off;
  int32_t shape, pad;
};
struct AssignUnit {
  int32_t job, tile;
};
// Boxes hold 256, 1024 or 2304 elements.  kAssignLds: LDS doubles of a staged box (X * Z rows of
// Y | 1) for each 256 of them; kAssignTable: entries of the X, Y and Z offset tables together, where
// no role has more than kAssignRole indices.  kAssignTile: side of a whole tile, whose square is its
// elements.
constexpr int kAssignElems = 2304, kAssignLds = 288, kAssignTable = 520, kAssignRole = 480, kAssignTile = 32;

// xr: XCD task ranges (null: the tasks split into 8 equal contiguous ranges).
// C-tile shapes of the fused block-pair kernels (rows x columns of one task): 64x64 and 16x256 of
// k_bp_f64 (operands staged in LDS), 16x16, 32x32 and 64x64 of k_bp_ks (the reduction split over
// a workgroup's waves; blocks of at most kBpKsMaxBlock elements).
enum { BP_TILE_64x64 = 0, BP_TILE_16x256 = 1, BP_TILE_KS16 = 2, BP_TILE_KS32 = 3, BP_TILE_KS64 = 4 };
constexpr int64_t kBpKsMaxBlock = int64_t(1) << 29;  // byte offsets inside a block in 32 bits
int bp_tile_rows(int tile);
int bp_tile_cols(int tile);
bool bp_tile_shares_k(int tile);  // of k_bp_ks
void launch_bp_f64(const BPTask* tasks, int ntasks, const BPPair* pairs, const BPCShape* cshapes,
                   const BPKShape* kshapes, const double* A, const double* B, double* C,
                   double alpha, int is_assign, hipStream_t s, const BPXcd* xr = nullptr,
                   int tile = BP_TILE_64x64);
// box: elements of a unit's box (256, 1024 or kAssignElems), or 0 for whole tiles.
void launch_assign(const AssignJob* jobs, const AssignUnit* units, int64_t nunits, int box,
                   const AssignShape* shapes, const double* src, double* dst, double scale,
                   int is_assign, hipStream_t s);

// Element-wise kernels (k_elementwise.hip)
void launch_fill(double* p, int64_t n, double v, hipStream_t s);
void launch_fill_bytes_zero(void* p, size_t bytes, hipStream_t s);
// Zeroes n element ranges of C: range i starts at off[i] and has prefix[i+1] - prefix[i]
// elements (device arrays; total = prefix[n]).
void launch_zero_ranges(const int64_t* off, const int64_t* prefix, int n, int64_t total, double* C,
                        hipStream_t s);
void launch_scale(double* p, int64_t n, double a, hipStream_t s);
void launch_axpy(int64_t n, double a, const double* x, double* y, hipStream_t s);
void launch_scale_copy(int64_t n, double a, const double* x, double* y, hipStream_t s);
// Partial sums of squares / products / squared differences -> host result (synchronous).
double reduce_sumsq(const double* x, int64_t n, hipStream_t s);
double reduce_dot(const double* x, const double* y, int64_t n, hipStream_t s);
double reduce_diffsq(const double* x, const double* y, int64_t n, hipStream_t s);
// reduce_sumsq with its partial sums in a file-scope device array (no allocation); the
// array's address on `device` is taken by noalloc_setup, which tmx_init calls.
void noalloc_setup(int device);
double reduce_sumsq_noalloc(const double* x, int64_t n, hipStream_t s, int device);

struct GenBlock {  // one block of a generated tensor
  int64_t off;
  int32_t lo[MAXR];   // global index of the block's first element per mode
  int32_t ext[MAXR];  // block extent per mode
};
void launch_fill_normal(const GenBlock* blocks, int64_t nblocks, int nmodes, const int64_t* mode_n,
                        int64_t max_block, double* data, uint64_t seed, uint64_t tensor_id,
                        double scale, int symmetrize, hipStream_t s);
// first: for each chunk of denominator_chunk(total) elements the block it starts in, and one
// more entry, the last block.
int denominator_chunk(int64_t total);
void launch_denominator(const GenBlock* blocks, const int32_t* first, int64_t total, double* data,
                        const double* e_occ, const double* e_vir, hipStream_t s);

}  // namespace tmx
