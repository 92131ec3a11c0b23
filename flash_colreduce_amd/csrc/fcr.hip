// libfcr: column reduction of softmax attention for MI355X (gfx950, CDNA4).
//
// Two sweeps, both built on v_mfma_f32_16x16x32_{f16,bf16} (fp32 operands as two fp16 parts each) with
// the product taken as S^T = K * Q^T (keys are MFMA rows, queries are MFMA columns).  In a 16x16
// accumulator a lane owns ONE query (lane & 15) and 4 keys (row 4*(lane/16) + r for register r), so
//   - everything that is per query row (softmax reference exponent, running sum, lse) is one
//     scalar per lane and needs no cross-lane traffic inside the sweep;
//   - everything that is per key column accumulates in the lane's registers over the whole
//     sweep and is reduced across the 16 query lanes once, at the end.
// The sweeps are bound by the vector instruction port (an MFMA keeps it for about 10 cycles, the fma,
// exp2 and add of the 64 scores it produces for 16 more) and, on random operands, by the package power
// limit.  The 16x16x32 shape is used because the 32x32x16 one, which would halve the MFMAs' share of the
// port, draws more power on random operands and ends up slower there.
//
//   row_lse_kernel    a workgroup keeps 256 query rows in registers (64 per wave; 128 and 32 for
//                     few or ragged M and for rows longer than 256 bytes) and streams key tiles through
//                     LDS; writes lse2[bh, i] = log2 sum_j 2^(s_ij).
//   col_reduce_kernel a workgroup keeps 256 key rows in registers and streams query tiles (and
//                     their lse2) through LDS; writes out[bh, j] = sum_i or max_i 2^(s_ij-lse2_i).
//   row_lse_f32_kernel, col_reduce_f32_kernel   the same for fp32 operands, whose rows are split on the way to LDS.
//   both_sweeps_kernel  both in one launch: column sweeps start where row sweeps leave a CU and wait for the lse they need.
//   col_small_kernel  the same result for at most 128 query rows against many keys: queries resident
//                     in every wave, keys streamed (HBM bound).
//   col_fused_kernel  both sweeps in one for at most 128 query rows against many 16-bit keys: the scores of
//                     1024 keys stay in registers while the workgroups that share a (batch, head) pair
//                     exchange their row sums through tagged 64-bit slots, so the keys are read once.
//   few_keys_kernel   both sweeps in one for pairs whose 16-bit keys fit the registers of a workgroup (up to 512).
//   topk_mask_kernel  keep-mask of the k largest columns of every row of the result (one workgroup per
//                     row; topk_spread_* kernels share a long row between workgroups).
// where s_ij = scale * log2(e) * <q_i, k_j>.  The column kernels store the result type of the caller's choice
// and divide the means as they store (store_column).  The streamed operand goes from global memory straight
// into a swizzled ring of LDS stages (buffer loads with the LDS as destination).  Nothing of size M*N
// is written anywhere and nothing in global memory is updated by read-modify-write atomics: one workgroup
// owns its output rows / columns (col_fused_kernel hands its partial row values to its team with atomic
// 64-bit stores and loads, value and round number in one word; both_sweeps_kernel its lse, word by word, to column sweeps).
//
// Replaces the Triton kernel of the reference (flash_colreduce/flash.py:11-274).

#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <stdio.h>

#include <atomic>
#include <mutex>
#include <type_traits>

#include "f32_tiles.h"
#include "fcr.h"

// The file can be compiled whole, or in parts that are linked together (the build script does that to
// use several cores): part 0 holds the C ABI and the small kernels, parts 1-4 the sweeps of one element
// type each (fp16, bf16, fp32 rows up to 512 bytes, longer fp32 rows), parts 5 and 6 the sweeps over fp16 and
// bf16 rows of more than 512 bytes, parts 7 and 8 the single sweep for fp16 and bf16, parts 9 and 10 few_keys_kernel for them,
// parts 11 and 12 both_sweeps_kernel, part 13 few_keys_f32_kernel.
#ifndef FCR_PART
#define FCR_PART -1
#endif
#define FCR_HAS(part) (FCR_PART == -1 || FCR_PART == (part))

namespace fcr_detail {
struct Params {
  const char* q;
  const char* k;
  float* lse;        // [BH, M]
  float* part;       // [splits, BH, M] partial lse of key ranges when splits > 1
  int splits;        // key ranges per row tile in the row kernel (1 = whole sweep in one workgroup)
  void* out;         // [BH, N]: column sums or means (or the only result)
  void* out2;        // [BH, N]: column maxima when one sweep produces both
  int64_t q_sb, q_sh, q_sr;  // strides in BYTES: batch, head, row
  int64_t k_sb, k_sh, k_sr;
  int H, M, N;
  int dgran;         // D / 8: valid 16-byte granules per row
  int c;             // max(N - M, 0): the causal right-alignment offset
  float scale2;      // scale * log2(e)
  float split_most;  // fp32 operands: see SplitRing::limit
  int tiles;         // resident tiles per (b,h)
  int bh_count;      // B * H
  int group;         // (b,h) pairs whose workgroups are launched together (see map_block)
  int fill;          // with the mask: workgroups that give every CU one (see map_group), 0 = plain order
  int stream_once;   // col_small_kernel: load the keys non-temporally
  int total;         // tiles * B * H workgroups
  // How the column kernels write a finished column (see store_column)
  int out_fmt;       // element type of out and out2: FCR_DTYPE_F32, FCR_DTYPE_F16 or FCR_DTYPE_BF16
  int mean_from;     // < 0: out holds the sums.  Else out holds means: columns below mean_from are
  float inv_m;       //   multiplied by inv_m = 1/M, column j from there on is divided by N - j
  // col_fused_kernel: teams of `splits` workgroups, team t takes (b,h) = t, t + teams, ..
  int teams;
  unsigned* sync;    // error word; zero at launch, like the slots at `part`.  both_sweeps_kernel: null if the workspace has no room for it;
                     // row_lse_kernel clears it for the calls that take two launches instead
  int spin_limit;    // polls of the counter after which a wait gives up
  // both_sweeps_kernel: `tiles`, `group`, `fill` and `total` are of the row sweeps
  int col_tiles, col_group;
  int row_blocks, col_blocks;
  int run_chunks;    // col_fused_kernel: chunks of keys a workgroup takes of a pair
  int parts;         // few_keys_f32_kernel: ranges of a pair's queries whose columns are added up apart
};
// which: 0 = row statistics, 1 = column sweep, 2 = column sweep for few queries, 3 = both sweeps in one for few
// queries, mode + 4 for more than 64 of them (2 and 3: 16-bit types only)
void sweeps_f16(int which, const Params& p, int ksteps, bool causal, int mode, hipStream_t s);
void sweeps_bf16(int which, const Params& p, int ksteps, bool causal, int mode, hipStream_t s);
void sweeps_f32(int which, const Params& p, int ksteps, bool causal, int mode, hipStream_t s);
void sweeps_f32_long_rows(int which, const Params& p, int ksteps, bool causal, int mode, hipStream_t s);
void sweeps_f16_single(const Params& p, int ksteps, bool causal, int mode, hipStream_t s);    // col_fused_kernel
void sweeps_bf16_single(const Params& p, int ksteps, bool causal, int mode, hipStream_t s);
void sweeps_f16_few_keys(const Params& p, int ksteps, bool causal, int mode, int form, hipStream_t s);   // few_keys_kernel
void sweeps_bf16_few_keys(const Params& p, int ksteps, bool causal, int mode, int form, hipStream_t s);
void sweeps_f32_few_keys(const Params& p, int ksteps, bool causal, int mode, int form, hipStream_t s);    // few_keys_f32_kernel
void sweeps_f16_both(const Params& p, int ksteps, bool causal, int mode, hipStream_t s);   // both_sweeps_kernel
void sweeps_bf16_both(const Params& p, int ksteps, bool causal, int mode, hipStream_t s);
void sweeps_f16_long_rows(int which, const Params& p, int ksteps, bool causal, int mode, hipStream_t s);
void sweeps_bf16_long_rows(int which, const Params& p, int ksteps, bool causal, int mode, hipStream_t s);
extern thread_local bool fused_refused;   // set by a launcher of col_fused_kernel that did not launch
}  // namespace fcr_detail

namespace {
using fcr_detail::Params;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
// k-steps are 64 bytes of a row: 32 16-bit elements of D, or 16 floats.  A wave keeps resident rows in groups of 16 (one MFMA operand each);
// two 32-row blocks (four groups) while their fragments fit the register file next to the
// accumulators (D <= 128: 4 k-steps), one block for larger D.  A workgroup keeps 4 * 32 * blocks rows.
__host__ __device__ constexpr int blocks_per_wave(int ksteps) { return ksteps <= 4 ? 2 : 1; }
// Compute units of the current device, asked once per device.  The tile, split and group choices below
// are stated in workgroups per CU (these kernels run two per CU).  256, an MI355X in its default
// partition mode, when no device can be asked (argument checks on a host without a GPU).
inline int chip_cus() {
  static int cached[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    (void)hipGetLastError();
    return 256;
  }
  int n = __atomic_load_n(&cached[dev], __ATOMIC_RELAXED);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) {
      (void)hipGetLastError();
      n = 256;
    }
    __atomic_store_n(&cached[dev], n, __ATOMIC_RELAXED);
  }
  return n;
}
// The row kernel has both forms for D <= 128 and the host picks per problem.  Waves whose rows are all
// padding do no arithmetic, so a launch costs (rows in waves with at least one query) x (cost per
// row); one block per wave costs about 3 % per k-step more per row (every streamed fragment feeds
// half as many MFMAs) but rounds M up to 32 instead of 64 rows per wave: it wins for M <= 128 and
// for a few ragged M above that.
inline int64_t rows_swept(int M, int nb) {
  const int trows = kWaves * 32 * nb;
  const int rem = M % trows;
  const int waves = rem ? (rem + 31) / 32 : 0;   // blocks of the last tile that hold queries
  return (int64_t)(M / trows) * trows + (waves < kWaves ? waves : kWaves) * 32 * nb;
}
// One block also wins when two would give between one and two workgroups per CU (with fewer than
// one the keys of a tile are split over workgroups instead, see row_splits; that case does not depend
// on `causal`, so the size of the lse buffer does not either).  With the mask exactly two per CU is
// still too coarse: the chip then waits for the workgroup with the longest sweep.  Against at most
// 1024 keys one block wins below one workgroup per CU as well: twice the workgroups beat splitting
// sweeps of 16 chunks (32 heads of 1024 x 1024: 16.5 -> 14 us, 16 heads of 512 x 512: 13 -> 8.6 us).
inline int row_blocks_per_wave(int ksteps, int M, int N, int64_t bh, bool causal) {
  if (ksteps > 4) return 1;
  if (rows_swept(M, 1) * (100 + 3 * ksteps) < rows_swept(M, 2) * 100) return 1;
  const int64_t wgs2 = bh * ((M + kWaves * 64 - 1) / (kWaves * 64));
  const int cus = chip_cus();
  if (wgs2 < cus && N <= 1024) return 1;
  return (wgs2 >= cus && wgs2 < 2 * cus + (causal ? 1 : 0)) ? 1 : 2;
}
// fp32 operands of D >= 32 are multiplied as two fp16 parts by kernels of their own, shorter ones on the fp32 instructions by the
// kernels of the 16-bit types (per call, against the staging through registers that those kernels do: 8 heads of 1024 x 1024 x 16
// 21 us against 33, 32 of 4096 x 4096 x 16 376 against 601, 2 x 16 of 2048 x 2048 x 28 causal 89 against 94).
inline bool in_parts(int dtype, int D) { return dtype == FCR_DTYPE_F32 && D >= 32; }
// Those on the fp32 instructions that give at most one workgroup of 128 rows on every other CU take tiles of 64 rows, one 16-row
// group per wave (NB = 0): such a launch lasts as long as one workgroup, and half the resident rows halve its matrix instructions.
// So do those of at most 64 rows.  A row sweep of 16 chunks or more is split over the idle CUs (row_splits) and keeps its tile if
// it has more rows than that.
inline bool half_tiles(int dtype, int D, int64_t rows, int64_t bh) {
  return dtype == FCR_DTYPE_F32 && !in_parts(dtype, D) && (rows <= 64 || 2 * bh * ((rows + 127) / 128) <= chip_cus());
}
inline bool row_half_tiles(int dtype, int D, int M, int N, int64_t bh) { return (M <= 64 || N <= 15 * 64) && half_tiles(dtype, D, M, bh); }
using fcr_tiles::F32Tile;
inline F32Tile f32_col_tile(int ksteps, bool both, int M, int N, int64_t bh, bool causal) {
  return fcr_tiles::f32_col_tile(ksteps, both, M, N, bh, causal, chip_cus());
}
inline F32Tile f32_row_tile(int M, int N, int64_t bh, bool causal) { return fcr_tiles::f32_row_tile(M, N, bh, causal, chip_cus()); }
inline int f32_ksteps(int ksteps) { return (ksteps + 1) / 2; }   // k-steps of 32 d from k-steps of 64 bytes
inline int elem_bytes(int dtype) { return dtype == FCR_DTYPE_F32 ? 4 : 2; }
inline int ksteps_of(int dtype, int D) { return (D * elem_bytes(dtype) + 63) / 64; }
inline int row_tile_rows(int dtype, int D, int M, int N, int64_t bh, bool causal) {
  if (in_parts(dtype, D)) return f32_row_tile(M, N, bh, causal).rows();
  if (row_half_tiles(dtype, D, M, N, bh)) return kWaves * 16;
  return kWaves * 32 * row_blocks_per_wave(ksteps_of(dtype, D), M, N, bh, causal);
}
constexpr int kMaxKSteps = 8;                 // rows of up to 512 bytes: two workgroups per CU
constexpr int kMaxKStepsF32 = 16;             // rows of up to 1 KiB (fp32: D <= 256, 16-bit elements: D <= 512), one workgroup per CU
constexpr int kChunk = 64;                    // streamed rows per LDS stage (two 32-row sub-steps)
using fcr_tiles::kMaxWorkgroups;
constexpr float kNegInf = -__builtin_inff();
constexpr float kPosInf = __builtin_inff();


// D[16 keys][16 queries] += A[16 keys][32 d] * B[32 d][16 queries].  Lane l supplies, for A and for
// B alike, the 8 consecutive d-elements [8*(l/16), +8) of row / column l & 15, and receives
// D[4*(l/16) + r][l & 15] in register r.
template <int DT>
__device__ __forceinline__ f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (DT == FCR_DTYPE_F16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                  0, 0, 0);
  } else if constexpr (DT == FCR_DTYPE_BF16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                   c, 0, 0, 0);
  } else {
    // fp32 operands: the same 16 bytes per lane are four floats, d = 4*(l/16) + e of a 16-float k-step.
    // v_mfma_f32_16x16x4_f32 number e contracts over the four lane groups' element e, so the four of
    // them cover the 16 floats once (the order of the terms of a dot product is free).
    const f32x4 af = __builtin_bit_cast(f32x4, a), bf = __builtin_bit_cast(f32x4, b);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(af[0], bf[0], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(af[1], bf[1], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(af[2], bf[2], c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(af[3], bf[3], c, 0, 0, 0);
    return c;
  }
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }

// Work order.  The (b,h) pairs are taken in groups of `group`; inside a group workgroup w takes
// (b,h) = first + w % g and the tile of rank w / g, tiles ranked by the length of their sweep,
// longest first: with more workgroups than the chip holds at once, the short ones fill in behind
// the long ones and the causal triangle finishes level.  A group is sized to about what the chip
// holds at once, so all tiles of a (b,h) run at the same time and its streamed operand comes from
// HBM once.  Workgroups are dealt to the 8 XCDs round-robin by v, so with group a multiple of 8
// every (b,h) stays on XCD (b,h) % 8 and that operand is shared through the XCD's L2.
//
// A causal launch of a few workgroups per CU, two at a time: in plain longest-first order the second workgroup of a
// CU is as many places behind the first as the chip has CUs, so the CU with the longest sweep also gets the longest of
// the second helping.  That helping is dealt backwards instead (p.fill; eight places at a time, which keeps the XCDs), so the
// two sweeps of every CU add up to about the same length; what is left follows in plain order.  Host: fill_places.
__device__ __forceinline__ void map_group(const Params& p, int v, int per_bh, int& bh, int& r) {
  const int second = v - p.fill, dealt = (min(2 * p.fill, p.total) - p.fill) & ~7;
  if (p.fill > 0 && second >= 0 && second < dealt) v = p.fill + (dealt - 8 - (second & ~7)) + (second & 7);
  const int per = p.group * per_bh;
  const int chunk = v / per;
  const int first = chunk * p.group;
  const int g = min(p.group, p.bh_count - first);
  const int w = v - chunk * per;
  r = w / g;
  bh = first + (w - r * g);
}

__device__ __forceinline__ void map_block(const Params& p, int v, bool longest_is_last_tile, int& bh, int& tile) {
  int rank;
  map_group(p, v, p.tiles, bh, rank);
  tile = longest_is_last_tile ? p.tiles - 1 - rank : rank;
}

// Row kernel with the keys of a tile split over several workgroups (few query rows, many keys):
// inside a group the order is (b,h), then the tile, then the key range: the tiles that stream the
// same keys start next to each other on the same XCD and share them through its L2.
__device__ __forceinline__ void map_block_split(const Params& p, int v, bool longest_is_last_tile, int& bh, int& tile,
                                                int& split) {
  int r;
  map_group(p, v, p.tiles * p.splits, bh, r);
  const int back = r / p.tiles;   // the last key range first: with the mask it holds the diagonal, the slow part
  const int rank = r - back * p.tiles;
  split = p.splits - 1 - back;
  tile = longest_is_last_tile ? p.tiles - 1 - rank : rank;
}

// First rows of the wave's resident 16-row groups.  With two blocks per wave a workgroup's 256
// resident rows are eight 32-row blocks and wave w keeps blocks w and 7-w: on a causal diagonal
// block b has b+1 (rows) or 8-b (columns) visible sub-tiles out of 8, so every wave gets 9 of the 36
// and the four waves reach each barrier together.  With one block per wave, wave w keeps block w
// of four.
// With NB = 0 a wave keeps one group, w of four.
__host__ __device__ constexpr int wave_group_count(int nb) { return nb ? 2 * nb : 1; }
template <int NB>
__device__ __forceinline__ void wave_groups(int tile, int wave, int (&rows)[wave_group_count(NB)]) {
  const int t0 = tile * (kWaves * 16 * wave_group_count(NB));
  if constexpr (NB == 0) rows[0] = t0 + 16 * wave;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    // blocks w, 7-w (, 8+w, 15-w): even positions count up, odd ones count down inside a run of eight
    const int blk = (NB == 1) ? wave : 8 * (i / 2) + ((i & 1) ? 7 - wave : wave);
    rows[2 * i] = t0 + 32 * blk;
    rows[2 * i + 1] = t0 + 32 * blk + 16;
  }
}

// Raw buffer view of rows [row0, nrows) of a row-major operand.  Loads through it return zero
// past the last row instead of faulting, so ragged tails need neither branches nor clamps.
// Offsets inside the view are 32 bit; the host checks that 64 rows fit.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_view(const char* base, int64_t row_bytes, int row0,
                                                            int nrows) {
  int64_t bytes = (int64_t)(nrows - row0) * row_bytes;
  bytes = bytes < 0 ? 0 : (bytes > 0xfffffff0ll ? 0xfffffff0ll : bytes);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base) + (int64_t)row0 * row_bytes, 0,
                                           (int)(uint32_t)bytes, 0x00020000);
}

// AUX is the cache policy of the load: 0 = default, kLoadOnce = non-temporal, for bytes that no
// workgroup of the launch will ask for again.
constexpr int kLoadOnce = 2;
template <int AUX = 0>
__device__ __forceinline__ u32x4 view_load16(__amdgpu_buffer_rsrc_t v, uint32_t byte_off) {
  return __builtin_amdgcn_raw_buffer_load_b128(v, (int)byte_off, 0, AUX);
}

// The operand a wave keeps for the whole sweep: NG groups of 16 rows starting at rows[g], as MFMA
// fragments.  Lane l holds, for k-step ks, the 8 elements [32*ks + 8*(l/16), +8) of row l & 15.
template <int KS, int NG>
__device__ __forceinline__ void load_resident(u32x4 (&f)[NG][KS], const char* base, int64_t row_bytes,
                                              const int (&rows)[NG], int nrows, int dgran, int lane) {
  const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const __amdgpu_buffer_rsrc_t view = rows_view(base, row_bytes, rows[g], nrows);
    const uint32_t roff = (uint32_t)(lane & 15) * (uint32_t)row_bytes;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int gi = ks * 4 + (lane >> 4);
      const u32x4 v = view_load16(view, roff + (uint32_t)min(gi, dgran - 1) * 16u);
      f[g][ks] = (gi < dgran) ? v : zero;  // zero padding of D up to the k-step
    }
  }
}

// Global -> LDS staging of the streamed operand, kChunk rows at a time, without passing through
// registers: buffer loads with the LDS as destination write 16 bytes per lane, 1 KiB per wave and
// instruction, to consecutive LDS addresses, while every lane chooses which 16 bytes of global memory it
// fetches.  A ring of stages is filled several chunks ahead of its use, so a load has one or two whole
// chunk periods to arrive and no wave ever waits for memory in the sweep.
//
// LDS layout of a stage: kChunk rows of kPitch bytes, no padding.  The 16-byte granule c of row r sits
// at granule position c ^ swz(r) of its row: a 16-byte fragment read is served in passes of lanes
// {0-7, 16-23}, {8-15, 24-31}, .. (eight consecutive rows at two neighbouring granule columns), and the
// swizzle sends those sixteen granules to sixteen different 16-byte slots modulo 256 bytes, i.e. to all
// 64 banks once.  Granule columns at or past D/8 (the zero padding up to the MFMA k-step, and up to the
// pitch) are fetched from an offset past the end of the buffer view, which yields zeros; so do rows
// past the end of the operand.  Behind the rows a stage has room for 64 floats (the column kernel's lse).
constexpr uint32_t kPastEnd = 0xfffffff0u;   // never inside a view: rows_view keeps sizes below it

// Stages of the ring in the two big sweeps: four while two workgroups of them fit a CU's 160 KiB (loads
// then have two to three chunk periods to arrive), two for the 32 KiB stages of D > 128.
__host__ __device__ constexpr int ring_stages(int ksteps) { return ksteps <= 4 ? 4 : 2; }

template <int AUX>
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t view, uint32_t byte_off, char* lds_wave_base) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(view, (__attribute__((address_space(3))) void*)lds_wave_base, 16,
                                           (int)byte_off, 0, 0, AUX);
}
constexpr int kFromMemory = 16;   // sc1: past the caches of the workgroup's die, as atomic loads at device scope are done
template <int AUX = 0>
__device__ __forceinline__ void dma4(__amdgpu_buffer_rsrc_t view, uint32_t byte_off, char* lds_wave_base) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(view, (__attribute__((address_space(3))) void*)lds_wave_base, 4,
                                           (int)byte_off, 0, 0, AUX);
}

// Waits until at most N of this wave's loads are outstanding and all its LDS reads have returned, then
// meets the other waves.  After it, what every wave loaded before its N newest loads is visible to
// all, and no wave is still reading what it read before the barrier, so those stages may be refilled.
// The empty asm statements keep the compiler from moving LDS accesses across the barrier (there is no
// fence, which would wait for every outstanding load).
// The value a float has after a round trip through the result's element type (round to nearest even,
// overflow to infinity, NaN kept), as the float16_t / bfloat16 casts of torch do it.
__device__ __forceinline__ float round_trip(int fmt, float v) {
  if (fmt == FCR_DTYPE_F16) return (float)(_Float16)v;
  if (fmt == FCR_DTYPE_BF16) {
    uint32_t b = __builtin_bit_cast(uint32_t, v);
    b = (v != v) ? 0x7fc00000u : ((b + 0x7fffu + ((b >> 16) & 1u)) & 0xffff0000u);
    return __builtin_bit_cast(float, b);
  }
  return v;
}

// Writes column `key` of row `bh` of a [BH, N] result whose elements have type p.out_fmt.  The
// reference casts its fp32 accumulation to the result type first (flash.py:308) and divides the means
// afterwards, in that type (flash.py:377-384): columns left of the causal offset by the Python scalar
// M, which torch turns into a multiplication by the fp32 reciprocal, the others by a tensor of counts
// that torch converts to the result type before the fp32 division.  The same steps, in the same order.
__device__ __forceinline__ void store_column(const Params& p, void* base, bool is_sum, int bh, int key, float v) {
  const int fmt = p.out_fmt;
  if (is_sum && p.mean_from >= 0) {
    v = round_trip(fmt, v);
    v = (key < p.mean_from) ? v * p.inv_m : v / round_trip(fmt, (float)(p.N - key));
  }
  const int64_t at = (int64_t)bh * p.N + key;
  if (fmt == FCR_DTYPE_F32) {
    static_cast<float*>(base)[at] = v;
  } else if (fmt == FCR_DTYPE_F16) {
    static_cast<_Float16*>(base)[at] = (_Float16)v;
  } else {
    static_cast<uint16_t*>(base)[at] = (uint16_t)(__builtin_bit_cast(uint32_t, round_trip(FCR_DTYPE_BF16, v)) >> 16);
  }
}

template <int N>
__device__ __forceinline__ void ring_sync() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (0 << 8));  // vmcnt(N) lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int CTRL>
__device__ __forceinline__ float dpp_row(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// All LDS accesses of this wave done, then the workgroup's barrier.  Loads and stores to memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((15) | (3 << 14) | (7 << 4) | (0 << 8));   // vmcnt(63) expcnt(7) lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// clamp(x, 0, kChunk) on the scalar unit (written out because the compiler turns min(max()) into a
// three-operand median that only the vector unit has, which would make everything derived from it,
// here a buffer descriptor, a per-lane value)
template <int CR = kChunk>
__device__ __forceinline__ int rows_in_chunk(int rows_left) {
  int live;
  asm("s_max_i32 %0, %1, 0\n\ts_min_i32 %0, %0, %2" : "=s"(live) : "s"(rows_left), "n"(CR) : "scc");
  return live;
}

// LW: the waves that issue the loads (their index is what init() takes as wave_id); CR: rows of a chunk
template <int KS, int NS = ring_stages(KS), int LW = kWaves, int CR = kChunk>
struct Ring {
  static constexpr int kN = NS;
  static constexpr int kPitch = KS <= 1 ? 64 : KS == 2 ? 128 : KS <= 4 ? 256 : KS <= 8 ? 512 : 1024;   // LDS row pitch
  static constexpr int kRowsPerLoad = 1024 / kPitch;                 // rows one wave-wide load covers
  static constexpr int kPer = CR / (LW * kRowsPerLoad);              // loads per loading wave and chunk
  static_assert(kPer * LW * kRowsPerLoad == CR, "whole loads");
  static constexpr int kRows = CR * kPitch;                          // bytes of rows in a stage
  static constexpr int kStage = kRows + CR * 4;                      // rows + a float for each
  static constexpr int kBytes = kN * kStage;
  static constexpr int kSwz = kPitch < 256 ? kPitch : 256;
  static __host__ __device__ constexpr int swz(int row) { return 2 * ((row * kSwz / 256) & (kSwz / 32 - 1)); }

  uint32_t voff[kPer];   // source byte offset inside a chunk of the granule this lane fetches, per load
  uint32_t ko[KS];       // LDS byte offset inside a 16-row group of this lane's fragment, per k-step
  int wave;              // wave-uniform

  __device__ __forceinline__ void init(int64_t row_bytes, int dgran, int lane, int wave_id) {
    wave = wave_id;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int byte = (wave * kPer + i) * 1024 + lane * 16;   // where the lane's 16 bytes land in the stage
      const int row = byte / kPitch;
      const int c = ((byte % kPitch) / 16) ^ swz(row);         // the granule that belongs there
      voff[i] = (c < dgran) ? (uint32_t)row * (uint32_t)row_bytes + (uint32_t)c * 16u : kPastEnd;
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int r = lane & 15, c = 4 * ks + (lane >> 4);
      ko[ks] = (uint32_t)(r * kPitch + ((c ^ swz(r)) * 16));
    }
  }
  // Chunks are fetched in order, so where the next one comes from is kept as a running address and a
  // count of the rows left (scalar registers, a handful of scalar instructions per chunk): rows
  // [row0, nrows) of the operand at `base` are what may be fetched, the rest arrives as zeros
  // without touching memory.
  const char* next_ptr;
  int rows_left;
  uint32_t row_bytes32;
  __device__ __forceinline__ void start(const char* base, int64_t row_bytes, int row0, int nrows) {
    next_ptr = base + (int64_t)row0 * row_bytes;
    rows_left = nrows - row0;
    row_bytes32 = (uint32_t)row_bytes;
  }
  // The next CR rows into `stage`.
  template <int AUX = 0>
  __device__ __forceinline__ void issue_next(char* stage) {
    const int live = rows_in_chunk<CR>(rows_left);   // the view covers this chunk's rows only
    const __amdgpu_buffer_rsrc_t view = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(next_ptr), 0, (int)((uint32_t)live * row_bytes32), 0x00020000);
#pragma unroll
    for (int i = 0; i < kPer; ++i) dma16<AUX>(view, voff[i], stage + (wave * kPer + i) * 1024);
    next_ptr += (int64_t)CR * row_bytes32;
    rows_left -= CR;
  }
  // CR rows from `ptr` on into `stage`, of which the first `rows` (clamped to [0, CR]) exist;
  // for sweeps that do not walk one operand front to back.
  template <int AUX = 0>
  __device__ __forceinline__ void issue_at(char* stage, const char* ptr, int rows) {
    const int live = rows_in_chunk<CR>(rows);
    const __amdgpu_buffer_rsrc_t view = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(ptr), 0, (int)((uint32_t)live * row_bytes32), 0x00020000);
#pragma unroll
    for (int i = 0; i < kPer; ++i) dma16<AUX>(view, voff[i], stage + (wave * kPer + i) * 1024);
  }
  // Fragment of the 16-row group sg of sub-step `sub` (32 rows) for k-step ks.
  __device__ __forceinline__ u32x4 frag(const char* stage, int sub, int sg, int ks) const {
    return *reinterpret_cast<const u32x4*>(stage + (sub * 32 + sg * 16) * kPitch + ko[ks]);
  }
};

// One sub-step of a sweep: 32 streamed rows (two groups of 16, fragments f) against the wave's NG
// resident groups: 2*NG independent 16x16 accumulator chains n[g][sg].  S^T = K * Q^T, so keys are
// the A operand.  A streamed fragment stays put for NG consecutive MFMAs.  When REFILL, each fragment
// register is reloaded for the sub-step after this one as soon as its MFMAs are issued, a whole
// sub-step ahead of its use.
template <int DT, int KS, int NG, bool RESIDENT_IS_KEYS, bool REFILL, class RingT>
__device__ __forceinline__ void mma_groups(f32x4 (&n)[NG][2], u32x4 (&f)[2][KS], const u32x4 (&res)[NG][KS],
                                           const RingT& rg, const char* next_lds, int next_sub) {
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    n[g][0] = zero;
    n[g][1] = zero;
  }
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
    for (int sg = 0; sg < 2; ++sg) {
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        if (RESIDENT_IS_KEYS) n[g][sg] = mma<DT>(res[g][ks], f[sg][ks], n[g][sg]);
        else n[g][sg] = mma<DT>(f[sg][ks], res[g][ks], n[g][sg]);
      }
      if (REFILL) f[sg][ks] = rg.frag(next_lds, next_sub, sg, ks);
      // MFMAs and LDS reads keep this order (the refill stays a sub-step ahead of its use instead of
      // sinking to just before it); vector, transcendental and scalar instructions may move across.
      __builtin_amdgcn_sched_barrier(0x2 | 0x4 | 0x400);
    }
  }
}

// Ring protocol.  advance(t) = ring_sync, then the load of the next chunk, t + kN - 1, into the stage
// chunk t - 1 lived in.  A loop calls it once per chunk, in order, before it first touches chunk t; loads are issued
// in chunk order, kPer (+1 with an lse row) per wave and chunk, so at that point "all but the newest
// kN - 2 chunks' loads have arrived" is exactly "chunk t has arrived".  Before the first advance the
// loads of the first kN - 1 chunks of the sweep have been issued.
//
// Branch-free sweep over chunks [ta, tb) of the streamed operand, none of which needs a mask.
// Steady state, per chunk t (two sub-steps s0, s1), one barrier:
//     advance(t+1)       chunk t+1 visible; nobody reads chunk t any more, its stage is being refilled
//     MFMA(s1 of t)   || VALU of s0 of t   || fragments <- s0 of t+1
//     MFMA(s0 of t+1) || VALU of s1 of t   || fragments <- s1 of t+1
// Every LDS read is issued a sub-step before its use.
// aux_of(t, stage, sub) reads what the consumer needs per sub-step besides the scores (the column
// kernel: lse of the lane's queries); it travels with the fragments so that it too is read before
// the barrier that lets the stage be refilled.
template <int DT, int KS, int NG, bool RESIDENT_IS_KEYS, class Aux, class RingT, class AdvF, class StageF,
          class AuxF, class ConsumeF>
__device__ __forceinline__ void pipelined_sweep(int ta, int tb, const u32x4 (&res)[NG][KS], const RingT& rg,
                                                AdvF&& advance, StageF&& stage_of, AuxF&& aux_of,
                                                ConsumeF&& consume) {
  if (ta >= tb) return;
  u32x4 f[2][KS];
  f32x4 pa[NG][2], pb[NG][2];  // scores of the sub-step being consumed / being produced, swapping roles
  Aux af, ap, an;
  advance(ta);
  {
    const char* lds = stage_of(ta);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      f[0][ks] = rg.frag(lds, 0, 0, ks);
      f[1][ks] = rg.frag(lds, 0, 1, ks);
    }
    ap = aux_of(ta, lds, 0);
    mma_groups<DT, KS, NG, RESIDENT_IS_KEYS, true>(pa, f, res, rg, lds, 1);
    af = aux_of(ta, lds, 1);
  }
  for (int t = ta; t + 1 < tb; ++t) {
    advance(t + 1);
    const char* nxt = stage_of(t + 1);
    an = af;
    mma_groups<DT, KS, NG, RESIDENT_IS_KEYS, true>(pb, f, res, rg, nxt, 0);
    af = aux_of(t + 1, nxt, 0);
    consume(pa, ap);
    ap = af;
    mma_groups<DT, KS, NG, RESIDENT_IS_KEYS, true>(pa, f, res, rg, nxt, 1);
    af = aux_of(t + 1, nxt, 1);
    consume(pb, an);
  }
  mma_groups<DT, KS, NG, RESIDENT_IS_KEYS, false>(pb, f, res, rg, nullptr, 0);
  consume(pa, ap);
  consume(pb, af);
}

// ---------------------------------------------------------------------------------------------
// Row statistics.  Per lane and resident 16-query group the state is (mref, l) with
//   sum over the keys seen so far of 2^(s) = l * 2^mref.
// mref is a reference exponent, not the running maximum: the common path (lse_fast) adds
// 2^(s - mref) without looking for a maximum.  The sum is renormalised (lse_renorm) only when it
// leaves [1, 2^64) -- the first visible keys of a row, or a jump of the scores by more than 64
// binades -- and then exactly as the classic online softmax would (new reference = old +
// max(tile max, 0)).  Invariant after the first visible key: 1 <= l < 2^64, hence
// mref <= lse < mref + 64, so terms that underflow are below 2^-126 of the total and overflow is
// caught by the range check.
// a[sg][r] is the score of the lane's query against key 16*sg + 4*(lane/16) + r of the sub-step;
// with MASK, keys whose offset 16*sg + r exceeds lim (already reduced by 4*(lane/16)) are hidden.
template <bool MASK, int SG>
__device__ __forceinline__ float lse_fast(const f32x4 (&a)[SG], float scale2, float mref, float l, int lim) {
  const float nm = -mref;
  float ln = l;  // one add per score and nothing else: the groups of a wave give the adder its parallelism
#pragma unroll
  for (int sg = 0; sg < SG; ++sg)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float x = fmaf(a[sg][r], scale2, nm);
      if (MASK) x = (16 * sg + r <= lim) ? x : kNegInf;
      ln += fast_exp2(x);
    }
  return ln;
}

__device__ __forceinline__ bool lse_in_range(float l) { return (l >= 1.0f) && (l < 1.8446744e19f); }

template <bool MASK, int SG>
__device__ __forceinline__ void lse_renorm(const f32x4 (&a)[SG], float scale2, float& mref, float& l, int lim) {
  const float nm = -mref;
  float t[4 * SG];
#pragma unroll
  for (int sg = 0; sg < SG; ++sg)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float x = fmaf(a[sg][r], scale2, nm);
      if (MASK) x = (16 * sg + r <= lim) ? x : kNegInf;
      t[sg * 4 + r] = x;
    }
  float tmax = t[0];
#pragma unroll
  for (int i = 1; i < 4 * SG; ++i) tmax = fmaxf(tmax, t[i]);
  // Nothing seen yet: the tile maximum becomes the reference (it may be far below zero, so the
  // empty sum must not be scaled: 0 * 2^(+big) is not a number).  Otherwise only ever move up.
  const bool empty = (l == 0.f);
  const float delta = empty ? ((tmax > kNegInf) ? tmax : 0.f) : fmaxf(tmax, 0.f);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4 * SG; ++i) s += fast_exp2(t[i] - delta);
  l = empty ? s : l * fast_exp2(-delta) + s;
  mref += delta;
}

template <bool MASK, int SG>
__device__ __forceinline__ void lse_update(const f32x4 (&a)[SG], float scale2, float& mref, float& l, int lim) {
  const float ln = lse_fast<MASK>(a, scale2, mref, l, lim);
  if (__builtin_amdgcn_ballot_w64(!lse_in_range(ln)) == 0) l = ln;
  else lse_renorm<MASK>(a, scale2, mref, l, lim);
}

// All groups of a fully visible sub-step; one rarely taken branch at the very end so that the
// arithmetic above it can be scheduled against the MFMAs of the next sub-step.
template <int NG, int SG>
__device__ __forceinline__ void lse_update_groups(const f32x4 (&a)[NG][SG], const float (&scale2)[NG], float (&mref)[NG],
                                                  float (&l)[NG]) {
  float ln[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) ln[g] = lse_fast<false>(a[g], scale2[g], mref[g], l[g], 0);
  // one range check for all groups, on the smallest and the largest sum (NaN scores stay NaN on
  // either path, so they need no test of their own)
  float lo = ln[0], hi = ln[0];
#pragma unroll
  for (int g = 1; g < NG; ++g) {
    lo = fminf(lo, ln[g]);
    hi = fmaxf(hi, ln[g]);
  }
  const bool ok = (lo >= 1.0f) && (hi < 1.8446744e19f);
  if (__builtin_amdgcn_ballot_w64(!ok) == 0) {
#pragma unroll
    for (int g = 0; g < NG; ++g) l[g] = ln[g];
  } else {
#pragma unroll
    for (int g = 0; g < NG; ++g) {   // group by group: the bits of a row do not depend on what else the wave holds
      if (__builtin_amdgcn_ballot_w64(!lse_in_range(ln[g])) == 0) l[g] = ln[g];
      else lse_renorm<false>(a[g], scale2[g], mref[g], l[g], 0);
    }
  }
}

// log2(2^a + 2^b); a NaN in either (a row with a NaN or +inf score) stays a NaN: fmaxf / fminf alone
// would drop it.
__device__ __forceinline__ float lse_merge(float a, float b) {
  const float hi = fmaxf(a, b), lo = fminf(a, b);
  if (a != a || b != b) return a + b;
  if (hi == kNegInf) return kNegInf;
  return hi + fast_log2(1.0f + fast_exp2(lo - hi));
}

struct NoAux {};

// STREAM_ONCE: the launch has one row tile per (b,h), so every key is read by exactly one workgroup,
// and so many keys that none of them survives in a cache until the column kernel: they are loaded
// non-temporally (7.0 instead of 6.2 TB/s on 34 GB of keys).  With several row tiles, or few keys, the
// default policy is the faster one.
// TELL: column sweeps of the same launch wait for the values (both_sweeps_kernel).
template <int DT, int KS, bool CAUSAL, int NB, bool STREAM_ONCE, bool TELL>
__device__ __forceinline__ void row_sweep(const Params& p, char* smem, int tid, int bh, int tile, int split) {
  using Rg = Ring<KS>;
  constexpr int NG = wave_group_count(NB);
  constexpr int kTileRows = kWaves * 16 * NG;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, keeps the row views scalar
  const int b = bh / p.H, h = bh - b * p.H;
  const char* qb = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
  const char* kb = p.k + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh;

  int q0[NG];  // first query of each of this wave's groups
  wave_groups<NB>(tile, wave, q0);

  // Keys [0, kend) matter to this workgroup.  Chunks [0, t_int) are seen in full by every one of
  // its queries and lie inside [0, N): they take the branch-free pipelined sweep.  The rest (the
  // causal diagonal, the ragged tail) take the general loop.
  // With splits > 1 this workgroup only sweeps chunks [c_begin, c_end) of that range and writes a
  // partial lse; lse_combine_kernel merges the partials.
  const int kend = CAUSAL ? min(p.N, tile * kTileRows + kTileRows + p.c) : p.N;
  const int per_split = ((p.N + kChunk - 1) / kChunk + p.splits - 1) / p.splits;
  const int c_begin = split * per_split;
  const int nchunks = min((kend + kChunk - 1) / kChunk, c_begin + per_split);
  const int t_int = min(nchunks, CAUSAL ? min((tile * kTileRows + p.c + 1) / kChunk, p.N / kChunk) : p.N / kChunk);
  const int keys_end = min(p.N, nchunks * kChunk);   // nothing is fetched from here on

  float mref[NG], l[NG], scale2[NG];
  int last[NG];  // last key a lane's query may see, minus the lane's row offset in a group
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    mref[g] = 0.f;
    l[g] = 0.f;
    scale2[g] = p.scale2;
    const int i = q0[g] + (lane & 15);
    last[g] = (CAUSAL ? min(p.N - 1, i + p.c) : p.N - 1) - 4 * (lane >> 4);
  }

  Rg rg;
  rg.init(p.k_sr, p.dgran, lane, wave);
  auto stage_of = [&](int t) { return smem + ((uint32_t)t % Rg::kN) * Rg::kStage; };
  rg.start(kb, p.k_sr, c_begin * kChunk, keys_end);
  auto issue = [&](int t) { rg.template issue_next<(STREAM_ONCE ? kLoadOnce : 0)>(stage_of(t)); };
  auto advance = [&](int t) {
    ring_sync<(Rg::kN - 2) * Rg::kPer>();
    issue(t + Rg::kN - 1);
  };
  // The first chunks of the streamed operand are requested before the resident one, so that all of
  // them are in flight together.
#pragma unroll
  for (int i = 0; i < Rg::kN - 1; ++i) issue(c_begin + i);

  // A wave whose rows all lie past M (a ragged last tile, fewer than 128 queries) only helps staging.
  if (q0[0] >= p.M) {
    for (int t = c_begin; t < nchunks; ++t) advance(t);
    ring_sync<0>();
    return;
  }
  u32x4 qf[NG][KS];
  load_resident<KS, NG>(qf, qb, p.q_sr, q0, p.M, p.dgran, lane);

  pipelined_sweep<DT, KS, NG, false, NoAux>(
      c_begin, t_int, qf, rg, advance, stage_of, [](int, const char*, int) { return NoAux{}; },
      [&](const f32x4(&a)[NG][2], NoAux) { lse_update_groups(a, scale2, mref, l); });

  for (int t = max(t_int, c_begin); t < nchunks; ++t) {
    advance(t);
    const char* lds = stage_of(t);
#pragma unroll
    for (int sub = 0; sub < kChunk / 32; ++sub) {
      const int key0 = t * kChunk + sub * 32;
      if (key0 >= p.N) continue;
      // the sub-step's fragments once, for all groups that see it
      u32x4 kf[2][KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        kf[0][ks] = rg.frag(lds, sub, 0, ks);
        kf[1][ks] = rg.frag(lds, sub, 1, ks);
      }
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const int qg = q0[g];
        if (CAUSAL && key0 > qg + 15 + p.c) continue;  // no query of the group sees this sub-tile
        f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          acc[0] = mma<DT>(kf[0][ks], qf[g][ks], acc[0]);
          acc[1] = mma<DT>(kf[1][ks], qf[g][ks], acc[1]);
        }
        const bool need_mask = (key0 + 32 > p.N) || (CAUSAL && key0 + 31 > qg + p.c);
        if (need_mask) lse_update<true>(acc, p.scale2, mref[g], l[g], last[g] - key0);
        else lse_update<false>(acc, p.scale2, mref[g], l[g], 0);
      }
    }
  }
  ring_sync<0>();   // the loads past the last chunk write their zeros before the LDS is given back

#pragma unroll
  for (int g = 0; g < NG; ++g) {
    float v = (l[g] == 0.f) ? kNegInf : mref[g] + fast_log2(l[g]);   // l is positive, zero (no key seen) or NaN
    v = lse_merge(v, __shfl_xor(v, 16));  // the four lane groups hold different keys of the same query
    v = lse_merge(v, __shfl_xor(v, 32));
    const int i = q0[g] + lane;
    float* dst = (p.splits > 1) ? p.part + (int64_t)split * p.bh_count * p.M : p.lse;
    if (lane < 16 && i < p.M) {
      if (TELL) __hip_atomic_store(reinterpret_cast<uint32_t*>(dst) + (int64_t)bh * p.M + i, v != v ? 0x7fc00000u : __builtin_bit_cast(uint32_t, v),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else dst[(int64_t)bh * p.M + i] = v;
    }
  }
}

template <int DT, int KS, bool CAUSAL, int NB, bool STREAM_ONCE>
__global__ __launch_bounds__(kThreads, (KS > 8 ? 1 : 2)) void row_lse_kernel(const Params p) {
  __shared__ __attribute__((aligned(1024))) char smem[Ring<KS>::kBytes];
  if (p.sync != nullptr && blockIdx.x == 0 && threadIdx.x == 0) p.sync[0] = 0u;
  int bh, tile, split;
  map_block_split(p, (int)blockIdx.x, CAUSAL, bh, tile, split);
  row_sweep<DT, KS, CAUSAL, NB, STREAM_ONCE, false>(p, smem, (int)threadIdx.x, bh, tile, split);
}

// lse[r] = log2 sum_s 2^part[s][r] over the key ranges of a split row sweep.  One thread per row; the
// partials are fetched eight at a time (independent loads: a round trip to memory per batch, not per
// value) and folded into a running (maximum, sum); a NaN partial makes the result NaN.
__global__ __launch_bounds__(256) void lse_combine_kernel(const float* __restrict__ part, float* __restrict__ lse,
                                                          int64_t rows, int splits) {
  const int64_t r = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (r >= rows) return;
  float m = kNegInf, acc = 0.f;
  bool nan = false;   // fmaxf drops a NaN partial
  for (int s0 = 0; s0 < splits; s0 += 8) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (s0 + i < splits) ? part[(int64_t)(s0 + i) * rows + r] : kNegInf;
    float bm = v[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) bm = fmaxf(bm, v[i]);
#pragma unroll
    for (int i = 0; i < 8; ++i) nan = nan || (v[i] != v[i]);
    const float nm = fmaxf(m, bm);
    if (nm > kNegInf) {
      acc *= fast_exp2(m - nm);   // m = -inf: acc is 0 and stays 0
#pragma unroll
      for (int i = 0; i < 8; ++i) acc += fast_exp2(v[i] - nm);
      m = nm;
    }
  }
  lse[r] = nan ? __builtin_nanf("") : ((m > kNegInf) ? m + fast_log2(acc) : kNegInf);
}

// ---------------------------------------------------------------------------------------------
// What a column sweep produces.
constexpr int kModeSum = 0, kModeMax = 1, kModeBoth = 2;

// a[sg][r] is the score of key 4*(lane/16) + r of a resident group against the lane's query in
// streamed group sg, whose lse is lse2[sg].  x = s*scale2 - lse is the base-2 log of the probability.
// Sums add 2^x; maxima track x itself and exponentiate once at the end of the sweep (2^x is monotone),
// so a max-only sweep has no exp.  With MASK, register r of group sg is hidden when r > lim + 16*sg.
template <bool MASK, int MODE, int SG>
__device__ __forceinline__ void col_update(const f32x4 (&a)[SG], const float (&scale2)[SG], const float (&lse2)[SG], f32x4& csum,
                                           f32x4& cmax, int lim) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float x[SG];
#pragma unroll
    for (int sg = 0; sg < SG; ++sg) {
      x[sg] = fmaf(a[sg][r], scale2[sg], -lse2[sg]);
      if (MASK) x[sg] = (r <= lim + 16 * sg) ? x[sg] : kNegInf;
      if (MODE != kModeMax) csum[r] += fast_exp2(x[sg]);
    }
    if (MODE != kModeSum) {   // two groups in one v_max3_f32 (32 heads of 32768, sums and maxima: 7556 -> 7406 us per call)
      if constexpr (SG == 2) cmax[r] = fmaxf(fmaxf(cmax[r], x[0]), x[1]);
      else cmax[r] = fmaxf(cmax[r], x[0]);
    }
  }
}

// End of a column sweep: reduces the wave's NG groups over the 16 query lanes (a transpose through LDS, one output key per
// lane and pass; a pass writes out four groups) and stores the columns.  Nobody uses the LDS any more.
// nans: NaN in their place.
template <int MODE, int NG>
__device__ __forceinline__ void col_store(const Params& p, char* smem, int bh, const int (&k0)[NG], const f32x4 (&csum)[NG],
                                          const f32x4 (&cmax)[NG], int lane, int wave, bool nans = false) {
  float* red = reinterpret_cast<float*>(smem) + wave * (NG * 4 * 64);
  const int w = lane & 15;                 // key inside its group
  if (MODE != kModeMax) {
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[(g * 4 + r) * 64 + lane] = csum[g][r];
    __syncthreads();
#pragma unroll
    for (int g4 = 0; g4 < NG; g4 += 4) {
      const int grp = g4 + (lane >> 4);      // which of the wave's groups this lane writes out
      if (grp < NG) {                        // lanes 32.. idle when a wave keeps two groups
        const float* src = red + (grp * 4 + (w & 3)) * 64 + (w >> 2) * 16;
        float v = 0.f;
#pragma unroll
        for (int j = 0; j < 16; ++j) v += src[(j + lane) & 15];
        const int key = k0[grp] + w;
        if (key < p.N) store_column(p, p.out, true, bh, key, nans ? __builtin_nanf("") : v);
      }
    }
  }
  if (MODE != kModeSum) {
    if (MODE == kModeBoth) __syncthreads();
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[(g * 4 + r) * 64 + lane] = cmax[g][r];
    __syncthreads();
#pragma unroll
    for (int g4 = 0; g4 < NG; g4 += 4) {
      const int grp = g4 + (lane >> 4);
      if (grp < NG) {
        const float* src = red + (grp * 4 + (w & 3)) * 64 + (w >> 2) * 16;
        float v = kNegInf;
#pragma unroll
        for (int j = 0; j < 16; ++j) v = fmaxf(v, src[(j + lane) & 15]);
        const int key = k0[grp] + w;
        if (key < p.N) store_column(p, (MODE == kModeBoth) ? p.out2 : p.out, false, bh, key, nans ? __builtin_nanf("") : fast_exp2(v));
      }
    }
  }
}

struct LsePair {
  float v[2];
};

// Blocks per wave the host asks for.  Strictly between one and two workgroups of 256 keys per CU
// leave CUs unevenly loaded, and with the mask one or two per CU are too coarse as well (the chip
// waits for the longest sweep): those launches use 128-key tiles.
// Sums and maxima together gain by two blocks too, but less the shorter the rows (16-bit, per call, one block against two: 32 heads of
// 32768 x 128 causal 7987 us, 7406; of 4096 x 128 268, 253; of 4096 x 64 182, 176), and lose in rows of one k-step (256 heads of
// 2351 x 32 394, 400; 160 of 987 x 32 53, 57) and, of two, where two blocks leave a part of a second round (160 of 1024 x 64,
// 2.5 workgroups of 256 keys per CU, 72, 77; 44 of 4096 x 64, 2.75, 266, 264) or no more than one per CU (11 of 4096 x 64 97.5, 99.5).
inline int col_tile_blocks(int ksteps, int mode, int N, int64_t bh, bool causal) {
  const int nb = blocks_per_wave(ksteps);
  if (nb != 2) return nb;
  const int64_t wgs2 = bh * ((N + kWaves * 64 - 1) / (kWaves * 64)), wgs1 = bh * ((N + kWaves * 32 - 1) / (kWaves * 32));
  const int cus = chip_cus();
  if (mode == kModeBoth && ksteps == 1) return 1;
  if (mode == kModeBoth && ksteps == 2 && !causal && (wgs2 <= cus || (wgs2 > 2 * cus && 8 * wgs2 < 22 * cus))) return 1;
  // two-block tiles only when they still give two workgroups per CU; with fewer, CUs idle or run a single
  // workgroup (32 heads of 1024 x 1024: the call takes 37 us with 128 two-block tiles, 32 us with 256 one-block tiles)
  // (without the mask one workgroup on most CUs does better with two blocks, 16 heads of 4096 x 4096 76 -> 66 us, unless the
  // 128-key tiles are no more than the CUs either: 252 of them, 12 heads of 2661 x 2661 x 128, 60.5 us, 132 two-block ones 72.5)
  if (causal) return wgs2 <= 2 * cus ? 1 : 2;
  if (wgs2 <= cus) return wgs1 > cus ? 2 : 1;
  return wgs2 < 2 * cus ? 1 : 2;
}

// FOLLOW: row sweeps of the same launch may not have stored the lse of the streamed rows yet (both_sweeps_kernel).
constexpr uint32_t kNotYet = 0xffffffffu;   // an lse that is still to come: no row sweep stores this NaN,
constexpr uint32_t kBegun = 0xfffffffeu;    // nor this one, which stands at the first row of a tile that a running workgroup has in hand
__device__ __forceinline__ bool still_to_come(uint32_t lse) { return lse >= kBegun; }
constexpr int kLseSlots = 8;                // of 64 rows each
template <int KS, int NB, bool FOLLOW>
__host__ __device__ constexpr int col_sweep_bytes() {
  const int red = kWaves * wave_group_count(NB) * 4 * 64 * 4;      // end-of-sweep transpose buffer
  const int ring = Ring<KS>::kBytes + (FOLLOW ? kLseSlots * kChunk * 4 : 0);
  return ring > red ? ring : red;
}
template <int DT, int KS, bool CAUSAL, int MODE, int NB, bool FOLLOW>
__device__ __forceinline__ void col_sweep(const Params& p, char* smem, int bh, int tile) {
  using Rg = Ring<KS>;
  static_assert(!FOLLOW || Rg::kN + 1 <= kLseSlots, "a slot for every chunk whose lse is read or on its way");
  constexpr int NG = wave_group_count(NB);
  constexpr int kTileRows = kWaves * 16 * NG;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform, keeps the row views scalar
  const int b = bh / p.H, h = bh - b * p.H;
  const char* qb = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
  const char* kb = p.k + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh;
  const float* lse = p.lse + (int64_t)bh * p.M;
  const float scale2[2] = {p.scale2, p.scale2};

  int k0[NG];  // first key of each of this wave's groups
  wave_groups<NB>(tile, wave, k0);

  f32x4 csum[NG], cmax[NG];  // the set a MODE does not use is never touched and costs no registers
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    csum[g] = (f32x4){0.f, 0.f, 0.f, 0.f};
    cmax[g] = (f32x4){kNegInf, kNegInf, kNegInf, kNegInf};
  }

  // Query chunks [t0, nchunks) can see keys of this tile.  Chunks [t_int, nfull) are whole chunks whose
  // queries all see every key of the tile: they take the branch-free pipelined sweep (keys past N are
  // computed and never stored, so they need no mask).  The chunks on the causal diagonal before them
  // and a ragged last chunk (rows past M read as zeros, their lse too) take the general loop.
  const int nchunks = (p.M + kChunk - 1) / kChunk;
  const int t0 = CAUSAL ? max(0, tile * kTileRows - p.c) / kChunk : 0;
  const int nfull = max(t0, p.M / kChunk);
  const int t_int = CAUSAL ? min(nfull, max(t0, (tile * kTileRows + kTileRows - 1 - p.c + kChunk - 1) / kChunk)) : 0;
  // lim = i + c - key0(group) - 4*(lane/16), with i the lane's query in group 0 of the current sub-tile
  const int lim_lane = (lane & 15) + p.c - 4 * (lane >> 4);

  // A stage is kChunk query rows plus their lse.
  Rg rg;
  rg.init(p.q_sr, p.dgran, lane, wave);
  auto stage_of = [&](int t) { return smem + ((uint32_t)t % Rg::kN) * Rg::kStage; };
  rg.start(qb, p.q_sr, t0 * kChunk, p.M);
  const float* lse_next = lse + t0 * kChunk;   // walks along with the ring's cursor
  int lse_left = p.M - t0 * kChunk;            // (FOLLOW: the lse is ahead of the rows)
  auto lse_slot = [&](int t) { return smem + Rg::kBytes + (t & (kLseSlots - 1)) * (kChunk * 4); };   // (FOLLOW)
  auto issue_lse = [&](char* to, int live) {
    const __amdgpu_buffer_rsrc_t view = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(lse_next), 0, live * 4, 0x00020000);
    dma4<(FOLLOW ? kFromMemory : 0)>(view, (uint32_t)lane * 4u, to);   // every wave writes the same 64 values: no branch
    lse_next += kChunk;
    lse_left -= kChunk;
  };
  // FOLLOW: the lse is requested a chunk ahead of its rows, into slots of its own, so that a wave can look at it a chunk before its use
  // (`word`: of the chunk that comes next, the lane's row).
  uint32_t word = 0;
  bool given_up = false;
  auto issue = [&](int t) {
    char* stage = stage_of(t);
    const int live = rows_in_chunk(FOLLOW ? lse_left : rg.rows_left);
    rg.issue_next(stage);
    issue_lse(FOLLOW ? lse_slot(t + 1) : stage + Rg::kRows, live);
  };
  auto wait_for = [&](int t) {   // every wave by itself: the slot then holds the same values whoever wrote last
    const int i = t * kChunk + lane;
    const uint32_t* at = reinterpret_cast<const uint32_t*>(lse) + (i < p.M ? i : p.M - 1);
    int polls = 0;
    uint32_t x = kNotYet;
    for (;;) {
      x = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (__builtin_amdgcn_ballot_w64(still_to_come(x)) == 0) break;
      if (given_up || ++polls > p.spin_limit) {
        given_up = true;
        break;
      }
      __builtin_amdgcn_s_sleep(8);
    }
    if (!still_to_come(x)) reinterpret_cast<uint32_t*>(lse_slot(t))[lane] = x;   // (a wave that gave up leaves what another has got)
  };
  auto advance = [&](int t) {
    ring_sync<(Rg::kN - 2) * (Rg::kPer + 1)>();
    if constexpr (FOLLOW) {
      if (t == t0) word = reinterpret_cast<const uint32_t*>(lse_slot(t))[lane];
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(still_to_come(word)) != 0, 0)) wait_for(t);
      word = reinterpret_cast<const uint32_t*>(lse_slot(t + 1))[lane];
    }
    issue(t + Rg::kN - 1);
  };
  auto aux_of = [&](int t, const char* lds, int sub) {
    const float* v = reinterpret_cast<const float*>(FOLLOW ? lse_slot(t) : lds + Rg::kRows) + sub * 32 + (lane & 15);
    return LsePair{{v[0], v[16]}};
  };
  if (FOLLOW) issue_lse(lse_slot(t0), rows_in_chunk(lse_left));
  // The first chunks of the streamed operand are requested before the resident one, so that all of
  // them are in flight together.
#pragma unroll
  for (int i = 0; i < Rg::kN - 1; ++i) issue(t0 + i);
  u32x4 kf[NG][KS];
  load_resident<KS, NG>(kf, kb, p.k_sr, k0, p.N, p.dgran, lane);

  auto general_chunk = [&](int t, auto ragged_tag) {
    constexpr bool RAGGED = decltype(ragged_tag)::value;   // rows past M are among the chunk's
    advance(t);
    const char* lds = stage_of(t);
#pragma unroll
    for (int sub = 0; sub < kChunk / 32; ++sub) {
      const int qs = t * kChunk + sub * 32;  // first query of the sub-tile
      if (RAGGED && qs >= p.M) continue;
      LsePair lq = aux_of(t, lds, sub);
      // +inf for rows past M: they contribute 2^-inf = 0
      if (RAGGED && qs + (lane & 15) >= p.M) lq.v[0] = kPosInf;
      if (RAGGED && qs + 16 + (lane & 15) >= p.M) lq.v[1] = kPosInf;
      // the sub-step's fragments once, for all groups that see it
      u32x4 qfrag[2][KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        qfrag[0][ks] = rg.frag(lds, sub, 0, ks);
        qfrag[1][ks] = rg.frag(lds, sub, 1, ks);
      }
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const int kg = k0[g];
        if (kg >= p.N) continue;
        if (CAUSAL && kg > qs + 31 + p.c) continue;  // no query of the sub-tile sees this group
        f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          acc[0] = mma<DT>(kf[g][ks], qfrag[0][ks], acc[0]);
          acc[1] = mma<DT>(kf[g][ks], qfrag[1][ks], acc[1]);
        }
        if (RAGGED && qs + 32 > p.M) {   // rows of padding, zeros, may have met a non-finite key
          if (qs + (lane & 15) >= p.M) acc[0] = (f32x4){0.f, 0.f, 0.f, 0.f};
          if (qs + 16 + (lane & 15) >= p.M) acc[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
        }
        const bool need_mask = CAUSAL && (kg + 15 > qs + p.c);
        if (need_mask) col_update<true, MODE>(acc, scale2, lq.v, csum[g], cmax[g], lim_lane + qs - kg);
        else col_update<false, MODE>(acc, scale2, lq.v, csum[g], cmax[g], 0);
      }
    }
  };

  for (int t = t0; t < t_int; ++t) general_chunk(t, std::false_type());

  pipelined_sweep<DT, KS, NG, true, LsePair>(
      t_int, nfull, kf, rg, advance, stage_of, aux_of,
      [&](const f32x4(&a)[NG][2], const LsePair& lq) {
        // the lse values are first touched here, a sub-step after their LDS read was issued
#pragma unroll
        for (int g = 0; g < NG; ++g) col_update<false, MODE>(a[g], scale2, lq.v, csum[g], cmax[g], 0);
      });

  for (int t = nfull; t < nchunks; ++t) general_chunk(t, std::true_type());

  ring_sync<0>();   // every load has landed (those past the last chunk write zeros): the LDS can be reused
  if (FOLLOW && given_up && p.sync != nullptr) p.sync[0] = 1u;
  col_store<MODE, NG>(p, smem, bh, k0, csum, cmax, lane, wave, given_up);
}

template <int DT, int KS, bool CAUSAL, int MODE, int NB>
__global__ __launch_bounds__(kThreads, ((NB > 2 || KS > 8) ? 1 : 2)) void col_reduce_kernel(const Params p) {
  __shared__ __attribute__((aligned(1024))) char smem[col_sweep_bytes<KS, NB, false>()];
  int bh, tile;
  map_block(p, (int)blockIdx.x, false, bh, tile);
  col_sweep<DT, KS, CAUSAL, MODE, NB, false>(p, smem, bh, tile);
}

// Both sweeps in one launch: workgroups [0, p.total) take row tiles as row_lse_kernel does, those from the next multiple of eight on
// (which keeps the XCDs) column tiles as col_reduce_kernel.  The row statistics start as kNotYet (fill_words_kernel), a row sweep stores its rows' values with
// device scope, and a column sweep takes a chunk of queries once their values are there: every word says so by itself, so there is
// no order between words and there are no fences.  A column sweep first looks whether every row tile that it needs has begun: the workgroup whose place
// it is marks the tile's first row with kBegun when it starts.  If one has not (another die is behind, other kernels hold its CUs), the workgroup gives it
// kPatience polls, then takes the tile in hand itself, marks it and sweeps it (the place's own workgroup will store the same bits once more).  So a
// column sweep waits only for row tiles that a running workgroup has in hand, and those wait for nobody: every wait ends, whatever the order in which
// workgroups start and whatever else holds CUs meanwhile, be it kernels that wait for each other, and no launch has to be kept apart from another.
// The bound on a wait (p.spin_limit polls, then the columns become NaN and p.sync[0] is set) is for a host that lowers it.
// Mark and look (a round trip to memory per column tile, beside another workgroup's sweep) cost 0.8 % in the geometric mean of 2900 shapes, up to 1.3 % of calls of
// several rounds.  The row sweep stands here twice: in one loop for both kinds of places it cost another 0.4 %.  Started in the reverse order, columns first, the launch gives the same bits in 1.2 to 2.3 times the time.  (Tickets
// for all tiles instead, rows first, cost 4.9 %, up to half of a short call: 64 to 128 atomics on a line before the first load of a
// workgroup, and workgroups that share a CU no longer get a long tile and a short one.)
// A captured graph gets the two launches, whose bits it has always had.
// What it is for: a launch that waits for its longest or last sweeps keeps CUs idle at its end, and here only the second one does.  With
// the mask, the first column tile needs only the rows of the first row tile at first, which end early, and follows the row sweeps chunk
// by chunk.  A column sweep looks at a chunk's values a chunk ahead, one LDS read and one branch per chunk, within 1 % of a sweep of its
// own (32 heads of 8192 x 8192 x 128 467 -> 472 us, where nothing is gained).  When a CU holds two workgroups the older one runs at nearly its
// full speed and the younger one on what is left (1.15 us and 3.3 per chunk of 64 rows against 1.05 alone), so the order of
// dispatch decides what ends together: see map_group, and both_plan for what was measured.
constexpr int kPatience = 32;   // polls, a microsecond or so each
template <int DT, int KS, bool CAUSAL, int MODE, int NBR, int NBC>
__global__ __launch_bounds__(kThreads, 2) void both_sweeps_kernel(const Params p) {
  constexpr int kCols = col_sweep_bytes<KS, NBC, true>();
  __shared__ __attribute__((aligned(1024))) char smem[kCols > Ring<KS>::kBytes ? kCols : Ring<KS>::kBytes];
  constexpr int kRowTile = kWaves * 16 * wave_group_count(NBR), kColTile = kWaves * 16 * wave_group_count(NBC);
  const int v = (int)blockIdx.x, rows = (p.total + 7) & ~7, tid = (int)threadIdx.x;
  auto words_of = [&](int bh) {
    uint32_t* words = reinterpret_cast<uint32_t*>(p.lse) + (int64_t)bh * p.M;
    asm volatile("" : "+v"(words));   // (opaque: per-lane arithmetic on it is not to draw that of the sweeps into vector registers)
    return words;
  };
  auto mark = [&](uint32_t* word) {   // whether the tile was not marked before
    uint32_t none = kNotYet;
    return __hip_atomic_compare_exchange_strong(word, &none, kBegun, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  if (v < rows) {   // a row tile's place
    if (v >= p.total) return;
    int bh, tile, split;
    map_block_split(p, v, CAUSAL, bh, tile, split);
    int place = tile;
    asm volatile("" : "+v"(place));   // (as words_of)
    uint32_t* const words = words_of(bh);
    if (tid == 0) mark(words + place * kRowTile);   // (the answer is not waited for)
    row_sweep<DT, KS, CAUSAL, NBR, false, true>(p, smem, tid, bh, tile, split);
    return;
  }
  Params c = p;
  c.tiles = p.col_tiles;
  c.group = p.col_group;
  c.fill = 0;
  int bh, tile;
  map_block(c, v - rows, false, bh, tile);
  {
    const int last = (p.M - 1) / kRowTile;
    int next = CAUSAL ? max(0, tile * kColTile - p.c) / kChunk * kChunk / kRowTile : 0;   // the first row tile that it needs
    asm volatile("" : "+v"(next));
    int patience = min(p.spin_limit, kPatience);
    uint32_t* const words = words_of(bh);
    for (;;) {
      if (tid < 64) {   // a row tile of the pair that nobody has begun
        while (next <= last) {
          const uint32_t x = __hip_atomic_load(words + min(next + tid, last) * kRowTile, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          const uint64_t missing = __builtin_amdgcn_ballot_w64(x == kNotYet);
          if (missing == 0) {
            next += 64;
            continue;
          }
          next += __builtin_ctzll(missing);
          if (patience > 0) {
            --patience;
            __builtin_amdgcn_s_sleep(8);
          } else if (__builtin_amdgcn_ballot_w64(tid == 0 && mark(words + next * kRowTile)) != 0) {
            break;
          }
        }
        if (tid == 0) *reinterpret_cast<int*>(smem) = next <= last ? next : -1;
      }
      lds_barrier();
      const int row = __builtin_amdgcn_readfirstlane(*reinterpret_cast<const int*>(smem));
      lds_barrier();
      if (row < 0) break;
      // (opaque: what the sweep derives from these is not to be kept in registers around the loop, and a split of 0 that the compiler knows
      // would put its chunk numbers into vector registers)
      const __attribute__((address_space(4))) Params* at = (const __attribute__((address_space(4))) Params*)__builtin_amdgcn_kernarg_segment_ptr();
      int thread = tid, split = 0;
      asm volatile("" : "+s"(at), "+v"(thread), "+s"(split));
      row_sweep<DT, KS, CAUSAL, NBR, false, true>(*(const Params*)at, smem, thread, bh, row, split);
    }
  }
  col_sweep<DT, KS, CAUSAL, MODE, NBC, true>(c, smem, bh, tile);
}

// ---------------------------------------------------------------------------------------------
// Both sweeps in one for a pair whose keys all fit the registers of one workgroup: every wave keeps 16 * NG keys (groups w, w + NW,
// w + 2 NW, .., which levels the mask), the queries stream through the ring 16 * SQ at a time, and a workgroup that sees a query
// sees all of its keys, so a score is formed once and its row's sum is a matter of the workgroup.  Per chunk and behind one barrier:
// the waves' sums of the rows of the chunk before are added up, and what was kept of its scores, times the reciprocal, goes
// to the columns; the chunk's own scores become 2^score (maxima keep the score itself), each wave's sum per row goes to LDS.
// Sums are of 2^score itself.  One outside [1, 2^100), which a NaN, an infinity, a row without a visible key and scores far from
// zero all end in, is not used: the workgroup forms that chunk again, and the rest of its chunks once, row maximum first (`exact`; every
// wave reads the same sums and so comes to the same conclusion).  Where every score is that far off, the two kernels -> this one, fp16
// sums: 512 pairs of 512 x 512 x 128 81 -> 79 us, with the mask 77 -> 77, of 256 x 256 x 64 21 -> 18 and 18.4 -> 20.1 (the worst), 8 pairs of 8192 x
// 512 x 128 88 -> 38; with every chunk formed both ways they took 145, 145, 31, 31 and 44.
// A 2^score below 2^-126 is 0, which is a probability below 2^-126 if the row's sum is 1 or more.  So sums below 1 are good only in chunks
// whose first row sees less than 64 keys, where they are common, and there a wave that finds such a 2^score makes its sum a NaN.
// The accumulators of hidden keys, those past N and those behind the mask, start at -inf.
// The queries of a pair are dealt chunk by chunk to p.splits workgroups, which leave fp32 columns behind each other for
// merge_columns_kernel (p.out, p.out2: [splits, BH, N]); one workgroup per pair stores the final form.
// Bound by the vector port, then by the chain through one barrier per chunk (32 queries against 512 keys of 128: 2560 cycles of
// port work on two waves per SIMD, 2810 taken; of 64: 1960, 2350), and where a CU gets one workgroup by reading its keys first (6000 of
// 28000 cycles for 512 keys of 64).  Scores formed and exponentiated once take 30 port cycles per 64 of D = 128 where the two sweeps
// take 52.  Per call, two kernels -> this one, fp16 sums: 512 pairs of 512 x 512 x 128 79.5 -> 53.5 us, of 256 x 256 34.7 -> 19.4, of
// 100 x 100 18.5 -> 7.6; 128 pairs of 512 x 512 x 64 18.9 -> 15.0, 2 pairs 14.1 -> 8.3; 8 pairs of 8192 x 512 x 128 86 -> 19.
// More than 512 keys of 64 were built with eight groups per wave and sixteen queries per chunk, and with 64 queries per chunk: both
// keep registers in memory in some forms and gave up to 1.3 times on 1024 keys without a mask, nothing or less with one.
__device__ __forceinline__ void swap_halves(float& a, float& b) {   // upper half of a with the lower half of b
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ void swap_rows(float& a, float& b) {     // odd rows of 16 lanes of a with the even rows of b
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
// Sums (maxima) over the four rows of lanes.  One value: in every lane.  Two: the first in the lower half, the second in the upper.
template <bool MAX>
__device__ __forceinline__ float lane_rows_reduce(const float (&v)[1]) {
  float a = v[0], b = v[0];
  swap_halves(a, b);
  a = MAX ? fmaxf(a, b) : a + b;
  b = a;
  swap_rows(a, b);
  return MAX ? fmaxf(a, b) : a + b;
}
template <bool MAX>
__device__ __forceinline__ float lane_rows_reduce(const float (&v)[2]) {
  float a = v[0], b = v[1];
  swap_halves(a, b);
  a = MAX ? fmaxf(a, b) : a + b;
  b = a;
  swap_rows(a, b);
  return MAX ? fmaxf(a, b) : a + b;
}

// Sum (maximum) of each of 16 values over the 16 lanes of a row: lane l of a row ends up with value l, v[l / 4][l % 4].
template <bool MAX>
__device__ __forceinline__ float lanes16_scatter(const f32x4 (&v)[4], int lane) {
  auto join = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
  float x[8], y[4], z[2];
#pragma unroll
  for (int j = 0; j < 8; ++j) {   // lanes 8.. keep the upper half of the values, of the mirrored lanes as well
    const float lo = v[j >> 2][j & 3], hi = v[2 + (j >> 2)][j & 3];
    x[j] = join((lane & 8) ? hi : lo, dpp_row<0x140>((lane & 8) ? lo : hi));
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) y[j] = join((lane & 4) ? x[j + 4] : x[j], dpp_row<0x141>((lane & 4) ? x[j] : x[j + 4]));
#pragma unroll
  for (int j = 0; j < 2; ++j) z[j] = join((lane & 2) ? y[j + 2] : y[j], dpp_row<0x4E>((lane & 2) ? y[j] : y[j + 2]));
  return join((lane & 1) ? z[1] : z[0], dpp_row<0xB1>((lane & 1) ? z[0] : z[1]));
}

// Sum (maximum) of each of 8 values over the four rows of lanes: row rho of lanes ends up with values 2 rho and 2 rho + 1 in v[0], v[1].
template <bool MAX>
__device__ __forceinline__ void lane_rows_scatter(float (&v)[8]) {
  float y[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float a = v[j], b = v[j + 4];
    swap_halves(a, b);
    y[j] = MAX ? fmaxf(a, b) : a + b;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    float a = y[j], b = y[j + 2];
    swap_rows(a, b);
    v[j] = MAX ? fmaxf(a, b) : a + b;
  }
}
// log2 of a row sum, the exponent apart: rounded once at the size of the result.
__device__ __forceinline__ float log2_of_sum(float l) { return (float)__builtin_amdgcn_frexp_expf(l) + fast_log2(__builtin_amdgcn_frexp_mantf(l)); }

// 16-row groups of keys per wave where there are more than 128 keys: what leaves room for a chunk's scores beside their fragments.
constexpr int few_keys_groups(int ks) { return ks > 4 ? 2 : 4; }
constexpr int few_keys_queries(int ks) { return ks > 4 ? 1 : 2; }   // streamed 16-row groups per chunk

template <int DT, int KS, bool CAUSAL, int MODE, int NG, int NW>
__global__ __launch_bounds__(64 * NW, 2) void few_keys_kernel(const Params p) {
  constexpr int SQ = few_keys_queries(KS), CR = 16 * SQ;
  static_assert(!CAUSAL || 16 * NW > CR + 14, "a chunk's diagonal meets one group of a wave");
  constexpr int kLoads = CR * Ring<KS>::kPitch / 1024;
  constexpr int LW = kLoads < NW ? kLoads : NW;
  constexpr int NS = 8;
  using Rg = Ring<KS, NS, LW, CR>;
  constexpr int kSums = CR * NW;
  __shared__ __attribute__((aligned(1024))) char smem[Rg::kBytes + 4 * kSums * 4];
  float* const sums = reinterpret_cast<float*>(smem + Rg::kBytes);   // two sets by parity of the chunk, [query][wave]
  float* const redo = sums + 2 * kSums;                              // maxima and sums of a chunk that is done again
  // grid: heads, batch, splits
  const int split = (int)blockIdx.z, S = p.splits, bh = (int)blockIdx.y * p.H + (int)blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const char* qb = p.q + (int64_t)blockIdx.y * p.q_sb + (int64_t)blockIdx.x * p.q_sh;
  const char* kb = p.k + (int64_t)blockIdx.y * p.k_sb + (int64_t)blockIdx.x * p.k_sh;

  int k0[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) k0[g] = 16 * (wave + NW * g);
  // of this workgroup: split, split + S, ..  (uniform, which a division hides from the compiler)
  const int chunks = S == 1 ? (p.M + CR - 1) / CR : __builtin_amdgcn_readfirstlane(((p.M + CR - 1) / CR - split + S - 1) / S);
  Rg rg;
  rg.init(p.q_sr, p.dgran, lane, wave);
  rg.start(qb, p.q_sr, split * CR, p.M);
  auto stage_of = [&](int i) { return smem + ((uint32_t)i % NS) * Rg::kStage; };
  auto first_row = [&](int i) { return (split + i * S) * CR; };
  const int64_t step = (int64_t)(S - 1) * CR * p.q_sr;
  auto issue = [&](int i) __attribute__((always_inline)) {   // in order: the cursor walks over the workgroup's chunks
    if (wave >= LW) return;
    rg.issue_next(stage_of(i));
    rg.next_ptr += step;
    rg.rows_left -= (S - 1) * CR;
  };
  // The stage of the chunk before the current one is not refilled yet: it may be done again.
#pragma unroll
  for (int i = 0; i < NS - 2; ++i) issue(i);
  // The keys through one view (the host checks that the workgroup's rows end below 2 GiB; granules past D come from past that).
  u32x4 kf[NG][KS];
  {
    const __amdgpu_buffer_rsrc_t view = rows_view(kb, p.k_sr, 0, p.N);
    uint32_t off[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int gi = ks * 4 + (lane >> 4);
      off[ks] = gi < p.dgran ? (uint32_t)(16 * wave + (lane & 15)) * (uint32_t)p.k_sr + (uint32_t)gi * 16u : 0x80000000u;
    }
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kf[g][ks] = view_load16(view, off[ks] + (uint32_t)(16 * NW * g) * (uint32_t)p.k_sr);
  }

  const int live_all = max(0, min(NG, (p.N - 16 * wave + 16 * NW - 1) / (16 * NW)));   // groups with keys
  const float hidden = p.scale2 < 0.f ? kPosInf : kNegInf;   // (times a scale of 0: a NaN, and the chunk is done again)
  f32x4 csum[NG], cmax[NG];   // the set a MODE does not use is never touched and costs no registers
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    csum[g] = (f32x4){0.f, 0.f, 0.f, 0.f};
    cmax[g] = (f32x4){kNegInf, kNegInf, kNegInf, kNegInf};
  }

  // groups that some query of a chunk sees; only the last of them can need a mask (they are 16 * NW keys apart)
  auto live_groups = [&](int q0) __attribute__((always_inline)) {
    if (!CAUSAL) return live_all;
    const int last = q0 + CR - 1 + p.c - 16 * wave;
    return last < 0 ? 0 : min(live_all, last / (16 * NW) + 1);
  };
  // first chunk from which on every query sees every key of the wave, and all of its groups are whole
  int i_full = 1 << 30;
  if (k0[NG - 1] + 16 <= p.N) {
    const int row = CAUSAL ? max(0, k0[NG - 1] + 15 - p.c) : 0;   // first row that sees the wave's last key
    i_full = CAUSAL ? __builtin_amdgcn_readfirstlane(max(0, ((row + CR - 1) / CR - split + S - 1) / S)) : 0;
  }
  // a wave's sums (maxima) per row, reduced over its lanes
  auto write_reduced = [&](float* set, float x) __attribute__((always_inline)) {
    if constexpr (SQ == 1) {
      if (lane < 16) set[lane * NW + wave] = x;
    } else {
      if ((lane & 16) == 0) set[((lane >> 5) * 16 + (lane & 15)) * NW + wave] = x;
    }
  };
  auto read_partials = [&](const float* set, float (&w)[SQ][NW]) __attribute__((always_inline)) {
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq)
#pragma unroll
      for (int i = 0; i < NW; i += 4) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(set + (16 * sq + (lane & 15)) * NW + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[sq][i + e] = x[e];
      }
  };
  auto add_up = [&](const float (&w)[SQ][NW], float (&l)[SQ]) __attribute__((always_inline)) {
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) {
      l[sq] = (w[sq][0] + w[sq][1]) + (w[sq][2] + w[sq][3]);
#pragma unroll
      for (int v = 4; v < NW; v += 4) l[sq] += (w[sq][v] + w[sq][v + 1]) + (w[sq][v + 2] + w[sq][v + 3]);
    }
  };

  u32x4 f[SQ][KS];   // fragments of the chunk that comes next
  auto read_fragments = [&](int i) __attribute__((always_inline)) {
    const char* stage = stage_of(i);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int sq = 0; sq < SQ; ++sq) f[sq][ks] = rg.frag(stage, 0, sq, ks);
  };
  // 2^score of a group, into the row sums; s is what adding it up needs of it
  auto exponents = [&](const f32x4(&t)[SQ], f32x4(&s)[SQ], float (&part)[SQ]) __attribute__((always_inline)) {
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = t[sq][r] * p.scale2, e = fast_exp2(x);
        part[sq] += e;
        s[sq][r] = MODE == kModeSum ? e : x;
      }
  };

  auto store_lse = [&](int q0, const float (&lse)[SQ]) __attribute__((always_inline)) {
    float v = lse[0];
#pragma unroll
    for (int sq = 1; sq < SQ; ++sq) v = lane >> 4 == sq ? lse[sq] : v;
    if (lane < CR && q0 + lane < p.M) p.lse[(int64_t)bh * p.M + q0 + lane] = v;
  };
  // Chunk i for rows whose sums of 2^score are unusable: every wave takes its own maximum of a row first, and behind one barrier the
  // waves' sums are brought to a common one.  Scaling a product and taking a maximum or the lse off rounds once, as in the two
  // kernels.  Keys come with the sign of the scale, up = |scale|.
  const float up = fabsf(p.scale2);
  auto exact = [&](int i, auto masked_tag, auto barrier) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;   // some key is hidden from some row: of the last live group, or all from rows past M
    const int q0 = first_row(i), live = MASKED ? live_groups(q0) : NG;
    const bool tail = q0 + CR > p.M;
    int lane_again = lane;   // opaque: what follows from it is not to be kept in registers from chunk to chunk
    asm volatile("" : "+v"(lane_again));
    // body(g, sq, seen) for every group in use; seen(r) is a question only in groups that are hidden in part, and there if it has to be
    auto groups = [&](bool ask, auto body) __attribute__((always_inline)) {
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        if (g >= live) continue;
        if (!MASKED || !ask || (g + 1 < live && !tail)) {
#pragma unroll
          for (int sq = 0; sq < SQ; ++sq) body(g, sq, [](int) { return true; });
        } else {
#pragma unroll
          for (int sq = 0; sq < SQ; ++sq) {
            const int key = k0[g] + 4 * (lane_again >> 4), q = q0 + 16 * sq + (lane_again & 15);
            const int lim = q >= p.M ? -1 : CAUSAL ? min(p.N - 1 - key, q + p.c - key) : p.N - 1 - key;
            body(g, sq, [lim](int r) { return r <= lim; });
          }
        }
      }
    };
    read_fragments(i);
    f32x4 x[NG][SQ];   // products, hidden ones -inf; later (sums) 2^score relative to the wave's maximum
    float most[SQ], part[SQ], factor[SQ], lse[SQ];
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) most[sq] = kNegInf, part[sq] = 0.f;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      if (g >= live) continue;
#pragma unroll
      for (int sq = 0; sq < SQ; ++sq) x[g][sq] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int sq = 0; sq < SQ; ++sq) x[g][sq] = mma<DT>(kf[g][ks], f[sq][ks], x[g][sq]);
    }
    groups(true, [&](int g, int sq, auto seen) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        x[g][sq][r] = seen(r) ? x[g][sq][r] : kNegInf;
        most[sq] = fmaxf(most[sq], x[g][sq][r]);
      }
    });
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) {   // the largest score; -inf if the row sees none of the wave's keys
      const float m[1] = {most[sq] == kNegInf ? kNegInf : most[sq] * up};
      most[sq] = lane_rows_reduce<true>(m);
    }
    groups(up == 0.f, [&](int g, int sq, auto seen) __attribute__((always_inline)) {   // (-inf times 0 is a NaN)
      const float ref = most[sq] == kNegInf ? 0.f : most[sq];
#pragma unroll
      for (int r = 0; r < 4; ++r) {   // (+inf - inf is a NaN, as the row kernel's lse then is)
        const float e = seen(r) ? fast_exp2(fmaf(x[g][sq][r], up, -ref)) : 0.f;
        part[sq] += e;
        if (MODE == kModeSum) x[g][sq][r] = e;
      }
    });
    float* const set_m = redo + (i & 1) * kSums;
    float* const set_l = sums + (i & 1) * kSums;
    write_reduced(set_m, SQ == 1 || lane < 32 ? most[0] : most[SQ - 1]);
    write_reduced(set_l, lane_rows_reduce<false>(part));
    barrier();
    // Each row of lanes takes its share of the waves.
    constexpr int PW = NW / 4;
    bool odd = up == 0.f;
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) {
      const int at = (16 * sq + (lane & 15)) * NW + PW * (lane >> 4);
      float wm[PW], wl[PW], m[1], l[1] = {0.f};
#pragma unroll
      for (int v = 0; v < PW; ++v) wm[v] = set_m[at + v], wl[v] = set_l[at + v];
      m[0] = wm[0];
#pragma unroll
      for (int v = 1; v < PW; ++v) m[0] = fmaxf(m[0], wm[v]);
      m[0] = lane_rows_reduce<true>(m);
      const float ref = m[0] == kNegInf ? 0.f : m[0];
#pragma unroll
      for (int v = 0; v < PW; ++v) l[0] = fmaf(wl[v], fast_exp2(wm[v] - ref), l[0]);   // (a wave without a key: 0 times 0)
      l[0] = lane_rows_reduce<false>(l);
      lse[sq] = l[0] == 0.f ? kNegInf : ref + fast_log2(l[0]);
      factor[sq] = (most[sq] == kNegInf ? 0.f : fast_exp2(most[sq] - ref)) * __builtin_amdgcn_rcpf(l[0]);
    }
    if (wave == 0) store_lse(q0, lse);
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) {
      if (MASKED && q0 + 16 * sq + (lane & 15) >= p.M) factor[sq] = 0.f, lse[sq] = kPosInf;
      odd = odd || !(MODE == kModeSum ? factor[sq] < kPosInf : lse[sq] > kNegInf);   // a NaN, or a row whose scores are all -inf
    }
    groups(__builtin_amdgcn_ballot_w64(odd) != 0, [&](int g, int sq, auto seen) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (MODE == kModeSum) {
          csum[g][r] = seen(r) ? fmaf(x[g][sq][r], factor[sq], csum[g][r]) : csum[g][r];
        } else {
          const float y = seen(r) ? fmaf(x[g][sq][r], up, -lse[sq]) : kNegInf;
          if (MODE == kModeBoth) csum[g][r] += fast_exp2(y);
          cmax[g][r] = fmaxf(cmax[g][r], y);
        }
      }
    });
  };

  f32x4 s[NG][SQ];   // of the chunk whose columns are added up next: 2^score, or (maxima) the scaled score
  float fact[SQ];    // per row of that chunk: the reciprocal of its sum, or its lse; such that rows past M add nothing
  auto add_group = [&](int g) __attribute__((always_inline)) {
    if constexpr (MODE == kModeSum) {
#pragma unroll
      for (int sq = 0; sq < SQ; ++sq)
#pragma unroll
        for (int r = 0; r < 4; ++r) csum[g][r] = fmaf(s[g][sq][r], fact[sq], csum[g][r]);
    } else {
      float one[SQ];
#pragma unroll
      for (int sq = 0; sq < SQ; ++sq) one[sq] = 1.f;
      col_update<false, MODE>(s[g], one, fact, csum[g], cmax[g], 0);
    }
  };
  constexpr int GP = SQ == 1 ? 2 : 1, NBT = NG / GP;   // groups side by side: two independent chains of matrix instructions
  f32x4 t[2][GP][SQ];
  auto scores = [&](int bt, auto init) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < GP; ++e) init(k0[bt * GP + e], t[bt & 1][e]);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int e = 0; e < GP; ++e)
#pragma unroll
        for (int sq = 0; sq < SQ; ++sq) t[bt & 1][e][sq] = mma<DT>(kf[bt * GP + e][ks], f[sq][ks], t[bt & 1][e][sq]);
  };
  auto visible = [](int, f32x4(&c)[SQ]) __attribute__((always_inline)) {
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) c[sq] = (f32x4){0.f, 0.f, 0.f, 0.f};
  };
  auto arrive = [&](int i) __attribute__((always_inline)) {
    ring_sync<(NS - 4) * Rg::kPer>();   // chunk i + 1 is there, the sums of chunk i - 1 are
    issue(i + NS - 2);
  };
  // some row of chunk i sees less than 64 keys
  auto few_seen = [&](int i) __attribute__((always_inline)) { return (CAUSAL ? min(p.N, first_row(i) + p.c + 1) : p.N) < 64; };
  // The wave's sums of chunk i to LDS.  (A minimum per score, of numbers that are not negative, in the first chunk behind the mask: 0.1 to 0.15 us
  // of a call.  In every chunk it cost 2-4 %.)
  auto write_sums = [&](int i, int live, const float (&v)[SQ]) __attribute__((always_inline)) {
    float x = lane_rows_reduce<false>(v);
    if (MODE == kModeSum && __builtin_expect(few_seen(i) && live > 0 && __builtin_amdgcn_ballot_w64(x < 1.f) != 0, 0)) {
      uint32_t smallest = 0x3f800000u;
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        if (g >= live) continue;
        const int key = k0[g] + 4 * (lane >> 4);
#pragma unroll
        for (int sq = 0; sq < SQ; ++sq) {
          int lim = p.N - 1 - key;
          if (CAUSAL) lim = min(lim, first_row(i) + 16 * sq + (lane & 15) + p.c - key);
#pragma unroll
          for (int r = 0; r < 4; ++r) smallest = min(smallest, r <= lim ? __builtin_bit_cast(uint32_t, s[g][sq][r]) : 0x3f800000u);
        }
      }
      if (__builtin_amdgcn_ballot_w64(smallest < 0x00800000u) != 0) x = __builtin_nanf("");
    }
    write_reduced(sums + (i & 1) * kSums, x);
  };
  // What the rows of chunk i contribute with, into `fact`; whether a row's sum is unusable (the same in every wave).  all_seen: no row sees
  // less than 64 keys.
  auto row_facts = [&](int i, float (&l)[SQ], bool all_seen = false) __attribute__((always_inline)) {
    const int q0 = first_row(i);
    float w[SQ][NW];
    read_partials(sums + (i & 1) * kSums, w);
    add_up(w, l);
    bool good = true;
    const float least = MODE != kModeSum || (!all_seen && few_seen(i)) ? 9.5367432e-7f : 1.f;   // (maxima take a logarithm off the score)
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) {
      good = good && l[sq] >= least && l[sq] < 1.2676506e30f;
      const bool row = q0 + 16 * sq + (lane & 15) < p.M;
      if (MODE == kModeSum) fact[sq] = row ? __builtin_amdgcn_rcpf(l[sq]) : 0.f;
      else fact[sq] = row ? log2_of_sum(l[sq]) : kPosInf;
    }
    return __builtin_amdgcn_ballot_w64(!good) != 0;
  };
  auto lse_of = [&](int i, const float (&l)[SQ]) __attribute__((always_inline)) {
    if (wave != 0) return;
    float lse[SQ];
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) lse[sq] = log2_of_sum(l[sq]);
    store_lse(first_row(i), lse);
  };
  int batches = 0;   // of GP groups, in use in the chunk whose columns are added up next
  auto add_batches = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int bt = 0; bt < NBT; ++bt)
      if (bt < batches) {
#pragma unroll
        for (int e = 0; e < GP; ++e) add_group(bt * GP + e);
      }
  };

  // Chunk i: its scores and their exponents, and, unless it is the first of a run, the columns of the chunk before between the two.
  // Returns without the exponents if a row of that one is unusable (the same in every wave).
  // A chunk that some key of the wave is hidden from, or the one behind them (whose predecessor's groups are not all in use):
  auto some_hidden = [&](int i) __attribute__((always_inline)) {
    arrive(i);
    if (__builtin_expect(i == 0, 0)) read_fragments(0);
    const int q0 = first_row(i), live = live_groups(q0), in_use = (live + GP - 1) / GP;
    int lane_again = lane;
    asm volatile("" : "+v"(lane_again));
    // the last batch holds what is hidden: the diagonal, keys past N, a group that nobody sees
    auto masked = [&](int key0, f32x4(&c)[SQ]) __attribute__((always_inline)) {
      const int key = key0 + 4 * (lane_again >> 4);
      int lim = p.N - 1 - key;
#pragma unroll
      for (int sq = 0; sq < SQ; ++sq) {
        if (CAUSAL) lim = min(p.N - 1 - key, q0 + 16 * sq + (lane_again & 15) + p.c - key);
#pragma unroll
        for (int r = 0; r < 4; ++r) c[sq][r] = r <= lim ? 0.f : hidden;
      }
    };
    auto batch = [&](int bt) __attribute__((always_inline)) {
      if (bt + 1 < in_use) scores(bt, visible);
      else if (bt < in_use) scores(bt, masked);
    };
    batch(0);
    if (NBT > 1) batch(1);
    if (__builtin_expect(i > 0, 1)) {
      float l[SQ];
      if (__builtin_expect(row_facts(i - 1, l), 0)) return false;
      add_batches();
      lse_of(i - 1, l);
    }
    float part[SQ];
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) part[sq] = 0.f;
#pragma unroll
    for (int bt = 0; bt < NBT; ++bt) {
      if (bt < in_use) {
#pragma unroll
        for (int e = 0; e < GP; ++e) exponents(t[bt & 1][e], s[bt * GP + e], part);
      }
      if (bt + 2 < NBT) batch(bt + 2);
    }
    read_fragments(i + 1);
    write_sums(i, live, part);
    batches = in_use;
    return true;
  };
  // The others, without branches but for such rows: the columns of chunk i - 1 are added up, and the exponents of each group of chunk i
  // taken, under the matrix instructions of the groups behind it.
  auto all_visible = [&](int i) __attribute__((always_inline)) {
    arrive(i);
    if (__builtin_expect(i == 0, 0)) read_fragments(0);
    scores(0, visible);
    if (NBT > 1) scores(1, visible);
    if (__builtin_expect(i > 0, 1)) {
      float l[SQ];
      if (__builtin_expect(row_facts(i - 1, l, !CAUSAL), 0)) return false;
#pragma unroll
      for (int g = 0; g < NG; ++g) add_group(g);
      lse_of(i - 1, l);
    }
    float part[SQ];
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) part[sq] = 0.f;
#pragma unroll
    for (int bt = 0; bt < NBT; ++bt) {
#pragma unroll
      for (int e = 0; e < GP; ++e) exponents(t[bt & 1][e], s[bt * GP + e], part);
      if (bt + 2 < NBT) scores(bt + 2, visible);
      if (bt + 3 == NBT || (NBT < 3 && bt == 0)) read_fragments(i + 1);
    }
    write_reduced(sums + (i & 1) * kSums, lane_rows_reduce<false>(part));   // (a wave's last key is past the 64th: no few_seen chunk)
    return true;
  };

  constexpr int kCalm = 2;
  // Columns: a reduce-scatter over the 16 query lanes, 16 values (four groups) at a time; lane l ends up with group (l & 15) / 4,
  // key 4 * (l / 16) + (l & 3) of it.
  auto store_columns = [&]() __attribute__((always_inline)) {
    Params mine = p;
    if (S > 1) {
      const int64_t at = (int64_t)split * p.bh_count * p.N * 4;
      mine.out = static_cast<char*>(p.out) + at;
      mine.out2 = static_cast<char*>(p.out2) + at;
    }
    const int r = lane & 3;
#pragma unroll
    for (int g4 = 0; g4 < NG; g4 += 4) {
      const int grp = g4 + ((lane & 15) >> 2);
      const int key = 16 * (wave + NW * grp) + 4 * (lane >> 4) + r;
      f32x4 c4[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) c4[g] = g4 + g < NG ? csum[(g4 + g) % NG] : (f32x4){0.f, 0.f, 0.f, 0.f};
      const float sum = MODE != kModeMax ? lanes16_scatter<false>(c4, lane) : 0.f;
#pragma unroll
      for (int g = 0; g < 4; ++g) c4[g] = g4 + g < NG ? cmax[(g4 + g) % NG] : (f32x4){0.f, 0.f, 0.f, 0.f};
      const float most = MODE != kModeSum ? lanes16_scatter<true>(c4, lane) : 0.f;
      if (grp < NG && key < p.N) {
        if (MODE != kModeMax) store_column(mine, mine.out, true, bh, key, sum);
        if (MODE != kModeSum) store_column(mine, MODE == kModeBoth ? mine.out2 : mine.out, false, bh, key, fast_exp2(most));
      }
    }
  };

  int i = 0;
  bool usable = true;
#pragma unroll 1
  for (; i < chunks && i_full > 0 && i <= i_full; ++i) {
    usable = some_hidden(i);
    if (__builtin_expect(!usable, 0)) break;
  }
  if (__builtin_expect(usable, 1)) {
#pragma unroll 1
    for (; i < chunks; ++i) {
      usable = all_visible(i);
      if (__builtin_expect(!usable, 0)) break;
      batches = NBT;
    }
  }
  if (__builtin_expect(usable, 1)) {
    ring_sync<0>();   // (and the loads past the last chunk have written their zeros)
    float l[SQ];
    usable = !row_facts(chunks - 1, l);
    if (__builtin_expect(usable, 1)) {
      add_batches();
      lse_of(chunks - 1, l);
      store_columns();
      return;
    }
  }
  // Chunk i - 1 has such a row.  It and all that follow are done the other way at once, formed once, behind one barrier each, the one that
  // the next chunk is there after.  (Back to the usual way after a few chunks without one was built; the loops above then keep
  // less in registers and lose 2-6 %.)
  lds_barrier();   // (everybody has read the plain sums, whose place is used again)
  if (p.scale2 < 0.f) {
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) kf[g][ks] ^= (u32x4){0x80008000u, 0x80008000u, 0x80008000u, 0x80008000u};
  }
  int at = i - 1;
  auto next_is_there = [&]() __attribute__((always_inline)) {
    if (at < i && i < chunks) lds_barrier();   // chunk i has been waited for
    else if (at + 1 < chunks) arrive(at + 1);
    else ring_sync<0>();
  };
#pragma unroll 1
  do {
    if (at < i_full || first_row(at) + CR > p.M) exact(at, std::true_type(), next_is_there);
    else exact(at, std::false_type(), next_is_there);
  } while (++at < chunks);
  store_columns();
}

// out = the sums or maxima of p.splits columns that lie BH * N apart at p.part (both: maxima p.splits * BH * N behind the sums).
template <int MODE>
__global__ __launch_bounds__(256) void merge_columns_kernel(const Params p) {
  const int64_t n = (int64_t)p.bh_count * p.N, at = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (at >= n) return;
  const int bh = (int)(at / p.N), key = (int)(at - (int64_t)bh * p.N);
  const float* src = p.part + at;
  if (MODE != kModeMax) {
    float v = 0.f;
#pragma unroll 8
    for (int s = 0; s < p.splits; ++s) v += src[s * n];
    store_column(p, p.out, true, bh, key, v);
  }
  if (MODE != kModeSum) {
    if (MODE == kModeBoth) src += p.splits * n;
    float v = 0.f;   // (maxima of probabilities)
#pragma unroll 8
    for (int s = 0; s < p.splits; ++s) v = fmaxf(v, src[s * n]);
    store_column(p, MODE == kModeBoth ? p.out2 : p.out, false, bh, key, v);
  }
}

// ---------------------------------------------------------------------------------------------
// fp32 operands.  Each row is scaled by a power of two that puts its largest element at 2^14..2^15 and every element x is split
// into two fp16 numbers, h = fp16(x) and l = fp16(x - h): x to 2^-23 (one element in four loses its last bit), and elements smaller
// than 2^-16 of the row's largest to 2^-39 of that one (see SplitRing::set_limit).  A product is h h' + h l' + l h', each
// exact in fp32 and added up by v_mfma_f32_16x16x32_f16: 48 matrix cycles per 16 x 16 x 32 block where
// v_mfma_f32_16x16x4_f32 takes 256.  What is left out, l l', is up to 2^-22 of it, so a product may be off by 2^-21 in all; the
// rounding of the running sum, 24 times at D = 256 where the fp32 instructions round 64 times, is the larger part in sums
// of more than about a dozen terms of like size.  Error of the scores against sums in 64 bits, relative 2-norm over N(0,1) rows (and over
// rows whose elements spread by e^(3 N(0,1))): D = 32 8.8e-8 (8.6e-8), 64 1.1e-7 (1.1e-7), 128 1.4e-7 (1.4e-7), 256
// 1.9e-7 (1.6e-7); the fp32 instructions, which round the running sum after every term: 1.0e-7 (1.2e-7), 1.5e-7
// (1.5e-7), 2.0e-7 (1.9e-7), 2.9e-7 (2.5e-7).  Results over the shapes and key distributions of the timed cases (geometric mean of 40
// calls, sums and maxima; in brackets the fp32 instructions): N(0,1) 3.19e-7 and 4.3e-7 (3.21e-7, 5.7e-7), keys with an offset
// 3.04e-7, 4.6e-7 (3.07e-7, 6.1e-7), with sinks 5.5e-7, 1.40e-6 (5.6e-7, 1.42e-6).  Where few terms make a score the fp32 instructions are the more
// exact: one product per score 8.3e-8 against 2.5e-8 (largest 4.8e-7, 6e-8), scores of 60 from two products each sums 2.6e-6
// against 2.3e-7.  Giving those back was measured and costs more than it gives: l l' as a fourth product, 5 to 21 % of the time, one
// product 7e-8, scores of 60 unchanged; three bf16 parts and six products, exact operands, 2.6e-8 and 2.2e-7, 1.35 to 1.85 times the time.
// Rows shorter than 32 have few terms to round (D = 16 8.4e-8 against 7.4e-8) and do
// not come here (in_parts).  A row with an infinity or a
// NaN has no scale; chunks and resident rows that hold one are multiplied on the fp32 instructions, from memory (exact_scores).
//
// Streamed rows are split once per workgroup on their way to LDS: global -> registers (a chunk ahead) -> two planes of a
// stage, each laid out like a stage of Ring.  A workgroup is NW waves of NG 16-row groups (F32Tile).  What bounds the long
// sweeps is the vector port (per 32 x 128 streamed floats and wave: the split 70 instructions in workgroups of 128 rows, 35 in
// those of 256, scale, fma, exp2 and add of 16 scores per lane 64, 48 matrix instructions of about 10 port cycles), then package power;
// short ones the latency of a chunk.  32 heads of 1024 x 1024 x 128: 137 -> 64 us per call, 4096 x 4096 x 128 2250 -> 730.
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

struct Planes {   // h and l of eight values of a row
  u32x4 p[2];
};

__device__ __forceinline__ float maximum3(float a, float b, float c) {   // a NaN wins
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c);
}
__device__ __forceinline__ uint32_t largest8(const f32x4& a, const f32x4& b) {   // bits of the largest magnitude
  float m = maximum3(fabsf(a[0]), fabsf(a[1]), fabsf(a[2]));
  m = maximum3(m, fabsf(a[3]), fabsf(b[0]));
  m = maximum3(m, fabsf(b[1]), fabsf(b[2]));
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_maximum(m, fabsf(b[3])));
}
// The power of two that a row's elements are multiplied by and the one that undoes it, from the bits of the row's largest
// magnitude (2^126 at most: rows below 2^-112 are not brought all the way up).
__device__ __forceinline__ void row_scale(uint32_t largest, float& up, float& down) {
  const uint32_t e = max(largest & 0x7f800000u, 15u << 23);
  up = __builtin_bit_cast(float, (268u << 23) - e);
  down = __builtin_bit_cast(float, e - (14u << 23));
}
// Infinities, NaNs, and rows from 2^104 on: a sum of up to 256 products of two scaled rows reaches 2^38 and is first multiplied by
// what undoes the scale of the key, 2^(E - 14) for a row whose largest element is at 2^E, whatever the query is.
constexpr uint32_t kNoScale = 231u << 23;
__device__ __forceinline__ bool has_no_scale(uint32_t largest) { return largest >= kNoScale; }

__device__ __forceinline__ Planes split8(const f32x4& a, const f32x4& b, float up) {
  Planes s;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x2 x = (i < 2) ? (f32x2){a[2 * i], a[2 * i + 1]} : (f32x2){b[2 * i - 4], b[2 * i - 3]};
    const f16x2 h = __builtin_convertvector((f32x2){x[0] * up, x[1] * up}, f16x2);
    const f32x2 rest = {fmaf(x[0], up, -(float)h[0]), fmaf(x[1], up, -(float)h[1])};
    s.p[0][i] = __builtin_bit_cast(uint32_t, h);
    s.p[1][i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(rest, f16x2));
  }
  return s;
}

// Largest value over aligned groups of LANES lanes (4, 8, 16 or 32); every lane of a group ends up with it.
template <int CTRL>
__device__ __forceinline__ uint32_t max_dpp(uint32_t v) {
  return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true));
}
template <int LANES>
__device__ __forceinline__ uint32_t lanes_max(uint32_t v) {
  v = max_dpp<0xB1>(v);                        // quad_perm [1,0,3,2]
  v = max_dpp<0x4E>(v);                        // quad_perm [2,3,0,1]
  if (LANES >= 8) v = max_dpp<0x141>(v);       // row_half_mirror
  if (LANES >= 16) v = max_dpp<0x140>(v);      // row_mirror
  if (LANES >= 32) {
    // odd rows of 16 lanes of the one register change places with even rows of the other (written out: the compiler
    // takes the two results of __builtin_amdgcn_permlane16_swap for one)
    uint32_t w = v;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(v), "+v"(w));
    v = max(v, w);
  }
  return v;
}

// Rows of D <= 128 are streamed 32 at a time, D <= 64 64, longer ones 16: two stages take at most 32 KiB.
constexpr int f32_chunk(int ks, int nw) { return (ks <= 2 ? 64 : ks <= 4 ? 32 : 16) * (nw / 4); }
constexpr int f32_groups(int ks) { return ks <= 4 ? 2 : 1; }   // streamed 16-row groups per sub-step

// KS: k-steps of 32 d; CR: rows of a chunk.
template <int KS, int NW, int CR = f32_chunk(KS, NW)>
struct SplitRing {
  static constexpr int kNumThreads = 64 * NW;
  static constexpr int kChunkRows = CR;
  static constexpr int kPitch = Ring<KS>::kPitch;            // bytes of a row in one plane
  static constexpr int kRowGranules = kPitch / 16;           // of eight values: threads that share a row
  static constexpr int kPlane = kChunkRows * kPitch;
  static constexpr int kStage = 2 * kPlane;
  static constexpr int kRowFloats = 2 * kChunkRows;          // two floats per row of a stage: its scale, and what the caller adds
  // two stages, their row floats, a word for each (see `bad`) and two for each wave (see `set_limit`)
  static constexpr int kBytes = 2 * kStage + 2 * kRowFloats * 4 + 16 + 8 * NW;
  static constexpr int kGranules = kChunkRows * kRowGranules;
  static constexpr bool kAll = kGranules >= kNumThreads;                // every thread stages; else the first kGranules of them, whole waves
  static constexpr int kPer = kAll ? kGranules / kNumThreads : 1;        // granules per staging thread
  static_assert(kAll ? kPer * kNumThreads == kGranules : kGranules % 64 == 0, "whole granules per thread, whole waves");

  char* smem;
  uint32_t src[kPer];     // source byte offset inside a chunk of a granule
  bool half[kPer];        // its second 16 bytes lie past D
  uint32_t dst[kPer];     // where its parts go in each plane
  uint32_t frag0;         // the lane's fragment of k-step 0 inside a 16-row group; k-step ks: ^ (ks * 64)
  f32x4 raw[kPer][2];     // the chunk in flight
  const char* next_ptr;
  int rows_left, row_bytes;
  uint32_t limit;         // bits of the magnitude from which on a streamed row is not multiplied as two parts

  __device__ __forceinline__ void init(char* lds, const char* base, int64_t row_bytes64, int row0, int nrows, int dgran,
                                       int tid) {
    smem = lds;
    const int lane = tid & 63;
    row_bytes = (int)row_bytes64;
    next_ptr = base + (int64_t)row0 * row_bytes64;
    rows_left = nrows - row0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int idx = i * kNumThreads + tid, row = idx / kRowGranules, c = idx % kRowGranules;
      src[i] = (2 * c < dgran) ? (uint32_t)row * (uint32_t)row_bytes + (uint32_t)c * 32u : kPastEnd;
      half[i] = 2 * c + 1 >= dgran;
      dst[i] = (uint32_t)(row * kPitch + ((c ^ Ring<KS>::swz(row)) * 16));
    }
    // (the swizzle is an exclusive or over granule numbers, and so is adding 4 * ks to a number below 4)
    frag0 = (uint32_t)((lane & 15) * kPitch + (((lane >> 4) ^ Ring<KS>::swz(lane & 15)) * 16));
    if (tid < 2) bad()[tid] = -1;
  }
  // bad()[s]: the last chunk staged in stage s that holds a row without a scale, or one that is too large for the resident rows
  __device__ __forceinline__ int* bad() const { return reinterpret_cast<int*>(smem + 2 * kStage + 2 * kRowFloats * 4); }
  __device__ __forceinline__ char* stage_of(int t) const { return smem + (t & 1) * kStage; }
  __device__ __forceinline__ float* scale_of(int t) const { return reinterpret_cast<float*>(smem + 2 * kStage) + (t & 1) * kRowFloats; }
  __device__ __forceinline__ float* extra_of(int t) const { return scale_of(t) + kChunkRows; }

  // The next chunk on its way to the registers; rows past the end arrive as zeros.
  template <int AUX = 0>
  __device__ __forceinline__ void fetch(bool staging = true) {   // staging: of the waves that stage (see kAll)
    const int live = __builtin_amdgcn_readfirstlane(staging ? min(max(rows_left, 0), kChunkRows) : 0);
    const __amdgpu_buffer_rsrc_t view =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(next_ptr), 0, (int)((uint32_t)live * (uint32_t)row_bytes), 0x00020000);
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      raw[i][0] = __builtin_bit_cast(f32x4, view_load16<AUX>(view, src[i]));
      raw[i][1] = __builtin_bit_cast(f32x4, view_load16<AUX>(view, half[i] ? kPastEnd : src[i] + 16u));
    }
    next_ptr += (int64_t)kChunkRows * row_bytes;
    rows_left -= kChunkRows;
  }
  // The chunk in the registers, number t, to its stage: granule by granule, or whole.
  __device__ __forceinline__ void put_granule(int i, int t, int tid, uint32_t& largest) {
    const uint32_t m = lanes_max<kRowGranules>(largest8(raw[i][0], raw[i][1]));
    largest = max(largest, m);
    float up, down;
    row_scale(m, up, down);
    const Planes s = split8(raw[i][0], raw[i][1], up);
    scale_of(t)[(i * kNumThreads + tid) / kRowGranules] = down;   // (by every thread of the row)
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) *reinterpret_cast<u32x4*>(stage_of(t) + t2 * kPlane + dst[i]) = s.p[t2];
  }
  // What an element loses that is small beside the largest of its row, up to 2^-39 of that one, is lost in a score times the
  // largest element of the other row.  Where no channel is large in both rows the score does not grow with that product, so the
  // product has a limit: Params::split_most = 2^17 / (scale2 sqrt(D)) puts the error, as a sum of D such terms of
  // either sign, at 2^-22 in the exponent of 2, what the fp32 instructions lose on N(0,1) rows of D = 128 (2.0e-7 of a score
  // of about one).  Rows of the default scale get there with elements of 300 in both; keys and queries of
  // N(0,1) are at 2^5, keys times eight at 2^8.
  __device__ __forceinline__ void publish(int wave, uint32_t res_largest, uint32_t first_largest) {   // first_largest: of the wave's part of the first chunk
    bad()[4 + wave] = has_no_scale(res_largest) ? 0 : (int)res_largest;   // (such a wave multiplies on the fp32 instructions anyway)
    bad()[4 + NW + wave] = (int)first_largest;
  }
  // Behind a barrier after publish(); returns whether the first chunk holds a row that `bad` is to tell of.
  __device__ __forceinline__ bool set_limit(float split_most) {
    uint32_t x = 0, first = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      x = max(x, (uint32_t)bad()[4 + w]);
      first = max(first, (uint32_t)bad()[4 + NW + w]);
    }
    const float y = split_most * __builtin_amdgcn_rcpf(__builtin_bit_cast(float, x));   // (x = 0: infinity)
    limit = __builtin_amdgcn_readfirstlane(min(__builtin_bit_cast(uint32_t, y), kNoScale));   // (a NaN has larger bits)
    return (uint32_t)__builtin_amdgcn_readfirstlane(first) >= limit;
  }
  __device__ __forceinline__ void note(int t, uint32_t largest) {
    if (largest >= limit) bad()[t & 1] = t;
  }
  __device__ __forceinline__ void put(int t, int tid) {
    uint32_t largest = 0;
#pragma unroll
    for (int i = 0; i < kPer; ++i) put_granule(i, t, tid, largest);
    note(t, largest);
  }
  __device__ __forceinline__ bool is_bad(int t) const {
    return __builtin_amdgcn_readfirstlane(bad()[t & 1]) == t;
  }
  // Fragment of 16-row group `group`, k-step ks, plane t2.
  __device__ __forceinline__ u32x4 frag(const char* stage, int group, int ks, int t2) const {
    return *reinterpret_cast<const u32x4*>(smem + (((uint32_t)(stage - smem) + frag0) ^ (uint32_t)(ks * 64)) +
                                           group * 16 * kPitch + t2 * kPlane);
  }
};

// The wave's resident rows as planes; down[g] undoes the scale of group g's row lane & 15.  Returns the bits of their largest
// magnitude.
template <int KS, int NG>
__device__ __forceinline__ uint32_t load_resident_split(Planes (&f)[KS][NG], float (&down)[NG], const char* base, int64_t row_bytes,
                                                    const int (&rows)[NG], int nrows, int dgran, int lane) {
  uint32_t worst = 0;
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const __amdgpu_buffer_rsrc_t view = rows_view(base, row_bytes, rows[g], nrows);
    const uint32_t roff = (uint32_t)(lane & 15) * (uint32_t)row_bytes;
    f32x4 x[KS][2];
    uint32_t m = 0;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int gi = 2 * (ks * 4 + (lane >> 4));   // 16-byte granule of the row
      x[ks][0] = __builtin_bit_cast(f32x4, view_load16(view, gi < dgran ? roff + gi * 16u : kPastEnd));
      x[ks][1] = __builtin_bit_cast(f32x4, view_load16(view, gi + 1 < dgran ? roff + gi * 16u + 16u : kPastEnd));
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) m = max(m, largest8(x[ks][0], x[ks][1]));
    m = max(m, (uint32_t)__shfl_xor((int)m, 16));
    m = max(m, (uint32_t)__shfl_xor((int)m, 32));
    worst = max(worst, m);
    float up;
    row_scale(m, up, down[g]);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) f[ks][g] = split8(x[ks][0], x[ks][1], up);
  }
  return __builtin_amdgcn_readfirstlane(lanes_max<16>(worst));   // (the four rows of lanes hold the same)
}

// The same scores from the operands in memory, on the fp32 instructions.
template <bool RESIDENT_IS_KEYS, int NG, int SG>
__device__ __forceinline__ void exact_scores(f32x4 (&acc)[NG][SG], const char* res, int64_t res_bytes, const int (&r0)[NG],
                                             int res_rows, const char* str, int64_t str_bytes, int s0, int str_rows,
                                             int dgran, int lane) {
  const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll 1
  for (int k0 = 0; k0 < dgran; k0 += 4) {
    const int gi = k0 + (lane >> 4);
    const uint32_t col = (uint32_t)min(gi, dgran - 1) * 16u;
    u32x4 r[NG], t[SG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const u32x4 v = view_load16(rows_view(res, res_bytes, r0[g], res_rows), (uint32_t)(lane & 15) * (uint32_t)res_bytes + col);
      r[g] = gi < dgran ? v : zero;
    }
#pragma unroll
    for (int sg = 0; sg < SG; ++sg) {
      const u32x4 v = view_load16(rows_view(str, str_bytes, s0 + 16 * sg, str_rows),
                                  (uint32_t)(lane & 15) * (uint32_t)str_bytes + col);
      t[sg] = gi < dgran ? v : zero;
    }
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int sg = 0; sg < SG; ++sg)
        acc[g][sg] = RESIDENT_IS_KEYS ? mma<FCR_DTYPE_F32>(r[g], t[sg], acc[g][sg]) : mma<FCR_DTYPE_F32>(t[sg], r[g], acc[g][sg]);
  }
}

// Scaled scores of sub-step `sub` (16 * SG streamed rows) of a staged chunk against the wave's resident rows; keys are the A
// operand.  Fragments are read a k-step ahead of their matrix instructions, those of the first by the
// caller; `between(ks)` runs behind the matrix instructions of k-step ks.
// Matrix instructions and memory accesses keep this order, vector instructions may move across.
template <int SG>
struct Fragments {
  u32x4 f[2][SG];   // per plane and group
};
template <int SG, int KS, int NW, int CR>
__device__ __forceinline__ Fragments<SG> read_fragments(const SplitRing<KS, NW, CR>& rg, const char* stage, int sub, int ks) {
  Fragments<SG> x;
#pragma unroll
  for (int t2 = 1; t2 >= 0; --t2)
#pragma unroll
    for (int sg = 0; sg < SG; ++sg) x.f[t2][sg] = rg.frag(stage, sub * SG + sg, ks, t2);
  return x;
}
template <bool RESIDENT_IS_KEYS, int KS, int NG, int SG, int NW, int CR, class BetweenF>
__device__ __forceinline__ void split_scores(f32x4 (&acc)[NG][SG], const Planes (&res)[KS][NG], const SplitRing<KS, NW, CR>& rg,
                                             const char* stage, int sub, const Fragments<SG>& first, BetweenF&& between) {
  // products by plane: streamed l with h, h with l, h with h
  constexpr int kProducts = 3;
  constexpr int str_of[kProducts] = {1, 0, 0}, res_of[kProducts] = {0, 1, 0};
  constexpr int kType = FCR_DTYPE_F16;
  Fragments<SG> f[2];
  f[0] = first;
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int sg = 0; sg < SG; ++sg) acc[g][sg] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    if (ks + 1 < KS) f[(ks + 1) & 1] = read_fragments<SG>(rg, stage, sub, ks + 1);
    __builtin_amdgcn_sched_barrier(0x2 | 0x4 | 0x400);
#pragma unroll
    for (int t = 0; t < kProducts; ++t)
#pragma unroll
      for (int sg = 0; sg < SG; ++sg)
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          const u32x4 r = res[ks][g].p[res_of[t]], s = f[ks & 1].f[str_of[t]][sg];
          acc[g][sg] = RESIDENT_IS_KEYS ? mma<kType>(r, s, acc[g][sg]) : mma<kType>(s, r, acc[g][sg]);
        }
    between(ks);
    __builtin_amdgcn_sched_barrier(0x2 | 0x4 | 0x400);
  }
}

// A sweep over chunks [t0, t1), the first of them fetched by the caller, whose scaled scores go to `consume` a sub-step at a time,
// in order; those of [ta, tb) need no mask.
// Per chunk one barrier, behind which it is staged and the other stage is free.  Under the matrix instructions of an
// unmasked chunk run the split of the next one (fetched a chunk ago) and `consume` for the sub-step before, whose scores are kept for
// it.  aux_of(t, sub) is what consume needs besides the scores, extra(t) what travels with a chunk; general(t, exact) does
// a chunk that needs a mask or, `exact`, has a row without a scale.
template <bool RESIDENT_IS_KEYS, int AUX, class Aux, int KS, int NG, int NW, class ExtraF, class AuxF, class ConsumeF,
          class GeneralF>
__device__ __forceinline__ void split_sweep(int t0, int ta, int tb, int t1, const Planes (&res)[KS][NG],
                                            SplitRing<KS, NW>& rg, int tid, bool idle, uint32_t res_largest, float split_most, ExtraF&& extra,
                                            AuxF&& aux_of, ConsumeF&& consume, GeneralF&& general) {
  using Rg = SplitRing<KS, NW>;
  constexpr int SG = f32_groups(KS), SUBS = Rg::kChunkRows / (16 * SG), STEPS = SUBS * KS, PER = Rg::kPer;
  if (t0 >= t1) return;
  const bool res_bad = has_no_scale(res_largest);
  uint32_t first_largest = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) rg.put_granule(i, t0, tid, first_largest);
  extra(t0);
  rg.template fetch<AUX>();
  first_largest = lanes_max<16>(first_largest);
  uint32_t wave_largest = 0;
#pragma unroll
  for (int l = 0; l < 64; l += 16) wave_largest = max(wave_largest, (uint32_t)__builtin_amdgcn_readlane((int)first_largest, l));
  rg.publish(tid >> 6, res_largest, wave_largest);   // (the resident rows may still be on their way up to here)
  ring_sync<63>();   // the first chunk is staged
  const bool first_bad = rg.set_limit(split_most);
  f32x4 kept[NG][SG];   // the scores not yet consumed
  Aux kept_aux;
  auto chunk = [&](int t, const Fragments<SG>& first, auto first_tag) {
    constexpr bool FIRST = decltype(first_tag)::value;
    const char* stage = rg.stage_of(t);
    uint32_t largest = 0;
    Fragments<SG> next = first;
#pragma unroll
    for (int sub = 0; sub < SUBS; ++sub) {
      f32x4 acc[NG][SG];
      const Aux aux = aux_of(t, sub);
      split_scores<RESIDENT_IS_KEYS>(acc, res, rg, stage, sub, next, [&](int ks) {
        const int step = sub * KS + ks;
#pragma unroll
        for (int i = 0; i < PER; ++i)
          if (step == max(0, (i + 1) * STEPS / (PER + 1) - 1)) rg.put_granule(i, t + 1, tid, largest);
        if (step == STEPS - 1) {
          extra(t + 1);
          rg.template fetch<AUX>();
        }
        if (ks == KS - 1 && sub + 1 < SUBS) next = read_fragments<SG>(rg, stage, sub + 1, 0);
      });
      if (!FIRST || sub > 0) consume(kept, kept_aux);
#pragma unroll
      for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int sg = 0; sg < SG; ++sg) kept[g][sg] = acc[g][sg];
      kept_aux = aux;
    }
    rg.note(t + 1, largest);
  };
  bool entered = true;
  for (int t = t0; t < t1;) {
    if (!entered) ring_sync<63>();   // waits for LDS accesses only: the fetch stays in flight
    entered = false;
    Fragments<SG> first = read_fragments<SG>(rg, rg.stage_of(t), 0, 0);   // (in flight while the word is looked at)
    const bool exact = res_bad || (t == t0 ? first_bad : rg.is_bad(t));
    if (idle || exact || t < ta || t >= tb) {
      rg.put(t + 1, tid);
      extra(t + 1);
      rg.template fetch<AUX>();
      if (!idle) general(t, exact);
      ++t;
      continue;
    }
    chunk(t, first, std::true_type());
    for (++t; t < tb; ++t) {
      ring_sync<63>();
      first = read_fragments<SG>(rg, rg.stage_of(t), 0, 0);
      entered = rg.is_bad(t);
      if (entered) break;
      chunk(t, first, std::false_type());
    }
    consume(kept, kept_aux);
  }
}

// See row_lse_kernel: the same work order, key ranges, row state and result for fp32 operands.
template <int KS, bool CAUSAL, int NG, bool STREAM_ONCE, int NW>
__global__ __launch_bounds__(64 * NW, 2) void row_lse_f32_kernel(const Params p) {
  using Rg = SplitRing<KS, NW>;
  constexpr int SG = f32_groups(KS), kRows = Rg::kChunkRows, kTileRows = NW * 16 * NG;
  __shared__ __attribute__((aligned(1024))) char smem[Rg::kBytes];
  int bh, tile, split;
  map_block_split(p, (int)blockIdx.x, CAUSAL, bh, tile, split);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = bh / p.H, h = bh - b * p.H;
  const char* qb = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
  const char* kb = p.k + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh;

  const int kend = CAUSAL ? min(p.N, tile * kTileRows + kTileRows + p.c) : p.N;
  const int per_split = ((p.N + kRows - 1) / kRows + p.splits - 1) / p.splits;
  const int c_begin = split * per_split;
  const int nchunks = min((kend + kRows - 1) / kRows, c_begin + per_split);
  const int keys_end = min(p.N, nchunks * kRows);
  // chunks that every query of the workgroup sees in full
  const int t_int = min(nchunks, CAUSAL ? min((tile * kTileRows + p.c + 1) / kRows, p.N / kRows) : p.N / kRows);

  int q0[NG], last[NG];
  float mref[NG], l[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    q0[g] = tile * kTileRows + wave * 16 * NG + 16 * g;
    mref[g] = 0.f;
    l[g] = 0.f;
    const int i = q0[g] + (lane & 15);
    last[g] = (CAUSAL ? min(p.N - 1, i + p.c) : p.N - 1) - 4 * (lane >> 4);
  }
  Rg rg;
  rg.init(smem, kb, p.k_sr, c_begin * kRows, keys_end, p.dgran, tid);
  rg.template fetch<(STREAM_ONCE ? kLoadOnce : 0)>();   // in flight together with the resident rows
  Planes qf[KS][NG];
  float qs2[NG];   // scale2 times what undoes the scale of the lane's query
  const uint32_t q_largest = load_resident_split<KS, NG>(qf, qs2, qb, p.q_sr, q0, p.M, p.dgran, lane);
#pragma unroll
  for (int g = 0; g < NG; ++g) qs2[g] *= p.scale2;
  const bool idle = q0[0] >= p.M;   // a wave whose rows all lie past M only helps staging

  struct KeyScales {
    f32x4 v[SG];   // of the lane's four keys per group
  };
  auto scales_at = [&](int t, int sub) {
    KeyScales s;
#pragma unroll
    for (int sg = 0; sg < SG; ++sg)
      s.v[sg] = *reinterpret_cast<const f32x4*>(rg.scale_of(t) + (sub * SG + sg) * 16 + 4 * (lane >> 4));
    return s;
  };
  auto rescale = [&](f32x4(&a)[NG][SG], const KeyScales& s) {
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int sg = 0; sg < SG; ++sg) a[g][sg] *= s.v[sg];
  };
  auto general = [&](int t, bool exact) {
    const char* stage = rg.stage_of(t);
#pragma unroll
    for (int sub = 0; sub < kRows / (16 * SG); ++sub) {
      const int key0 = t * kRows + sub * 16 * SG;
      if (key0 >= p.N || (CAUSAL && key0 > q0[NG - 1] + 15 + p.c)) continue;   // nobody sees these keys
      f32x4 acc[NG][SG] = {};
      if (!exact) {
        split_scores<false>(acc, qf, rg, stage, sub, read_fragments<SG>(rg, stage, sub, 0), [](int) {});
        rescale(acc, scales_at(t, sub));
      } else {
        exact_scores<false>(acc, qb, p.q_sr, q0, p.M, kb, p.k_sr, key0, p.N, p.dgran, lane);
      }
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const float s2 = exact ? p.scale2 : qs2[g];
        const bool need_mask = (key0 + 16 * SG > p.N) || (CAUSAL && key0 + 16 * SG - 1 > q0[g] + p.c);
        if (need_mask) lse_update<true>(acc[g], s2, mref[g], l[g], last[g] - key0);
        else lse_update<false>(acc[g], s2, mref[g], l[g], 0);
      }
    }
  };
  split_sweep<false, (STREAM_ONCE ? kLoadOnce : 0), KeyScales>(
      c_begin, c_begin, t_int, nchunks, qf, rg, tid, idle, q_largest, p.split_most, [](int) {}, scales_at,
      [&](f32x4(&a)[NG][SG], const KeyScales& s) {
        rescale(a, s);
        lse_update_groups(a, qs2, mref, l);
      },
      general);

#pragma unroll
  for (int g = 0; g < NG; ++g) {
    float v = (l[g] == 0.f) ? kNegInf : mref[g] + fast_log2(l[g]);
    v = lse_merge(v, __shfl_xor(v, 16));
    v = lse_merge(v, __shfl_xor(v, 32));
    const int i = q0[g] + lane;
    float* out = (p.splits > 1) ? p.part + (int64_t)split * p.bh_count * p.M : p.lse;
    if (lane < 16 && i < p.M) out[(int64_t)bh * p.M + i] = v;
  }
}

// See col_reduce_kernel.
template <int KS, bool CAUSAL, int MODE, int NG, int NW>
__global__ __launch_bounds__(64 * NW, 2) void col_reduce_f32_kernel(const Params p) {
  using Rg = SplitRing<KS, NW>;
  constexpr int SG = f32_groups(KS), kRows = Rg::kChunkRows, kTileRows = NW * 16 * NG;
  constexpr int kRed = NW * NG * 4 * 64 * 4;
  __shared__ __attribute__((aligned(1024))) char smem[Rg::kBytes > kRed ? Rg::kBytes : kRed];
  int bh, tile;
  map_block(p, (int)blockIdx.x, false, bh, tile);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = bh / p.H, h = bh - b * p.H;
  const char* qb = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
  const char* kb = p.k + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh;
  const float* lse = p.lse + (int64_t)bh * p.M;

  int k0[NG];
  f32x4 csum[NG], cmax[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    k0[g] = tile * kTileRows + wave * 16 * NG + 16 * g;
    csum[g] = (f32x4){0.f, 0.f, 0.f, 0.f};
    cmax[g] = (f32x4){kNegInf, kNegInf, kNegInf, kNegInf};
  }
  const int t0 = CAUSAL ? max(0, tile * kTileRows - p.c) / kRows : 0;
  const int nchunks = (p.M + kRows - 1) / kRows;
  // chunks from t_int on: their queries all see every key of the tile (rows past M add 2^-inf)
  const int t_int = CAUSAL ? max(t0, (tile * kTileRows + kTileRows - 1 - p.c + kRows - 1) / kRows) : t0;
  const int lim_lane = (lane & 15) + p.c - 4 * (lane >> 4);

  Rg rg;
  rg.init(smem, qb, p.q_sr, t0 * kRows, p.M, p.dgran, tid);
  // the lse of a chunk's queries (+inf past M: they contribute 2^-inf) travels with its rows
  float lse_raw = 0.f;
  auto lse_fetch = [&](int t) {
    const int i = t * kRows + tid;
    if (tid < kRows) lse_raw = (i < p.M) ? lse[i] : kPosInf;
  };
  rg.fetch();   // in flight together with the resident rows
  lse_fetch(t0);
  Planes kf[KS][NG];
  f32x4 ks4[NG];   // what undoes the scale of the lane's four keys per group
  uint32_t k_largest;
  {
    float down[NG];
    k_largest = load_resident_split<KS, NG>(kf, down, kb, p.k_sr, k0, p.N, p.dgran, lane);
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) ks4[g][r] = __shfl(down[g], 4 * (lane >> 4) + r);
  }
  const bool idle = k0[0] >= p.N;

  auto extra = [&](int t) {
    if (tid < kRows) rg.extra_of(t)[tid] = lse_raw;
    lse_fetch(t + 1);
  };
  struct QueryFacts {
    float lse[SG], s2[SG];   // of the lane's query per group: lse, scale2 times what undoes its scale
  };
  auto facts_at = [&](int t, int sub) {
    QueryFacts q;
#pragma unroll
    for (int sg = 0; sg < SG; ++sg) {
      const int at = (sub * SG + sg) * 16 + (lane & 15);
      q.lse[sg] = rg.extra_of(t)[at];
      q.s2[sg] = rg.scale_of(t)[at] * p.scale2;
    }
    return q;
  };
  auto general = [&](int t, bool exact) {
    const char* stage = rg.stage_of(t);
#pragma unroll
    for (int sub = 0; sub < kRows / (16 * SG); ++sub) {
      const int qs = t * kRows + sub * 16 * SG;
      if (qs >= p.M || (CAUSAL && k0[0] > qs + 16 * SG - 1 + p.c)) continue;   // none of these queries sees a key of the wave
      QueryFacts q = facts_at(t, sub);
      f32x4 acc[NG][SG] = {};
      if (!exact) {
        split_scores<true>(acc, kf, rg, stage, sub, read_fragments<SG>(rg, stage, sub, 0), [](int) {});
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
          for (int sg = 0; sg < SG; ++sg) acc[g][sg] *= ks4[g];
      } else {
        exact_scores<true>(acc, kb, p.k_sr, k0, p.N, qb, p.q_sr, qs, p.M, p.dgran, lane);
#pragma unroll
        for (int sg = 0; sg < SG; ++sg) q.s2[sg] = p.scale2;
#pragma unroll
        for (int g = 0; g < NG; ++g)   // a row of padding may have met a non-finite key
#pragma unroll
          for (int sg = 0; sg < SG; ++sg)
            if (qs + 16 * sg + (lane & 15) >= p.M) acc[g][sg] = (f32x4){0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const bool need_mask = CAUSAL && (k0[g] + 15 > qs + p.c);
        if (need_mask) col_update<true, MODE>(acc[g], q.s2, q.lse, csum[g], cmax[g], lim_lane + qs - k0[g]);
        else col_update<false, MODE>(acc[g], q.s2, q.lse, csum[g], cmax[g], 0);
      }
    }
  };
  split_sweep<true, 0, QueryFacts>(
      t0, t_int, nchunks, nchunks, kf, rg, tid, idle, k_largest, p.split_most, extra, facts_at,
      [&](f32x4(&a)[NG][SG], const QueryFacts& q) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
#pragma unroll
          for (int sg = 0; sg < SG; ++sg) a[g][sg] *= ks4[g];
          col_update<false, MODE>(a[g], q.s2, q.lse, csum[g], cmax[g], 0);
        }
      },
      general);
  ring_sync<63>();
  col_store<MODE, NG>(p, smem, bh, k0, csum, cmax, lane, wave);
}

// ---------------------------------------------------------------------------------------------
// few_keys_kernel for fp32 operands: the same work order, groups of keys, splits and columns, and the parts, limits and exact chunks of
// the fp32 sweeps.  A row's maximum comes first in every chunk: every wave takes its own, its 2^score and their sum are relative to that, and
// behind the barrier of the next chunk the waves' (maximum, sum) are merged, so no scores need another form.  Forming a score
// is three matrix instructions per k-step and the split of its row, which the maximum adds little to.  At most 256 keys: two groups per
// wave are what the registers hold in parts beside a chunk's scores (four groups of D <= 64 and 16 queries per chunk were built: 256 pairs of 512 x
// 512 x 64 77 -> 63 us, with the mask 60 -> 67, and some forms kept registers in memory; of what is kept the forms for D > 224, at most 128 keys, maxima
// and both keep 2 to 7, 12 to 20 bytes per lane, at 0.61 of the two kernels' time all the same).  Bound by the chain of a chunk, barrier, merge,
// products, maximum, exponents, sum, on two waves per SIMD: 4700 cycles per chunk of 32 queries against 256 keys of 128, of which 1540 are
// matrix and 3000 port cycles.  Per call, two kernels -> this one: see few_keys_f32_plan.

template <int KS, bool CAUSAL, int MODE, int NG, int NW>
__global__ __launch_bounds__(64 * NW, 2) void few_keys_f32_kernel(const Params p) {
  constexpr int SQ = f32_groups(KS), CR = 16 * SQ;
  using Rg = SplitRing<KS, NW, CR>;
  constexpr int kSums = CR * NW;
  constexpr int kSetsAt = (Rg::kBytes + 15) & ~15;
  __shared__ __attribute__((aligned(1024))) char smem[kSetsAt + 4 * kSums * 4];
  float* const sets = reinterpret_cast<float*>(smem + kSetsAt);   // by parity of the chunk: maxima, then sums, [query][wave]
  const int split = (int)blockIdx.z, S = p.splits, bh = (int)blockIdx.y * p.H + (int)blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const char* qb = p.q + (int64_t)blockIdx.y * p.q_sb + (int64_t)blockIdx.x * p.q_sh;
  const char* kb = p.k + (int64_t)blockIdx.y * p.k_sb + (int64_t)blockIdx.x * p.k_sh;
  const bool staging = Rg::kAll || wave * 64 < Rg::kGranules;
  // The chunks of a pair are dealt in p.parts ranges of L, the last one shorter perhaps, and a workgroup takes ranges split, split + S, ..
  const int all = (p.M + CR - 1) / CR, L = __builtin_amdgcn_readfirstlane((all + p.parts - 1) / p.parts);
  const int ranges = __builtin_amdgcn_readfirstlane((p.parts - split + S - 1) / S);
  const int chunks = min(ranges * L, all - (split + (ranges - 1) * S) * L + (ranges - 1) * L);   // of this workgroup

  Rg rg;
  rg.init(smem, qb, p.q_sr, split * L * CR, p.M, p.dgran, tid);
  int fetched = 0;   // of a range
  auto fetch = [&]() __attribute__((always_inline)) {   // in order: the cursor walks over the workgroup's chunks
    rg.fetch(staging);
    if (++fetched == L) {
      fetched = 0;
      rg.next_ptr += (int64_t)(S - 1) * L * CR * p.q_sr;
      rg.rows_left -= (S - 1) * L * CR;
    }
  };
  uint32_t largest = 0;
  auto put = [&](int i) __attribute__((always_inline)) {
    if (!staging) return;
#pragma unroll
    for (int j = 0; j < Rg::kPer; ++j) rg.put_granule(j, i, tid, largest);
  };
  fetch();   // in flight together with the keys
  int k0[NG];
  f32x4 csum[NG], cmax[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    k0[g] = 16 * (wave + NW * g);
    csum[g] = (f32x4){0.f, 0.f, 0.f, 0.f};
    cmax[g] = (f32x4){kNegInf, kNegInf, kNegInf, kNegInf};
  }
  Planes kf[KS][NG];
  f32x4 ks4[NG];   // what undoes the scale of the lane's four keys per group, with the sign of the scale
  const float sign = p.scale2 < 0.f ? -1.f : 1.f, up = fabsf(p.scale2);
  uint32_t k_largest;
  {
    float down[NG];
    k_largest = load_resident_split<KS, NG>(kf, down, kb, p.k_sr, k0, p.N, p.dgran, lane);
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) ks4[g][r] = sign * __shfl(down[g], 4 * (lane >> 4) + r);
  }
  const bool res_bad = has_no_scale(k_largest);

  const int live_all = max(0, min(NG, (p.N - 16 * wave + 16 * NW - 1) / (16 * NW)));   // groups with keys
  auto live_groups = [&](int q0) __attribute__((always_inline)) {   // those that some query of a chunk sees
    if (!CAUSAL) return live_all;
    const int last = q0 + CR - 1 + p.c - 16 * wave;
    return last < 0 ? 0 : min(live_all, last / (16 * NW) + 1);
  };
  // first row from which on every query sees every key of the wave, and all of its groups are whole
  const int full_row = k0[NG - 1] + 16 > p.N ? 0x7fffffff : CAUSAL ? max(0, k0[NG - 1] + 15 - p.c) : 0;

  // Of the chunk whose columns are added up next: its products (sums: 2^score relative to the wave's maximum), the maximum per row, what
  // its queries' products are scaled by, and whether some key is hidden from some row of it (or a row is padding).
  f32x4 x[NG][SQ];
  float most[SQ], s2[SQ];
  bool some_hidden = false, no_scale = false;   // no_scale: some s2 is 0, which makes a NaN of a hidden product (-inf)
  int live = 0, kept_row = 0;
  // body(g, sq, seen) for every group in use; seen(r) is a question only in groups that are hidden in part, and there if it has to be
  auto groups = [&](auto masked_tag, bool ask, int lane_again, auto body) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      if (MASKED && g >= live) continue;
      if (!MASKED || !ask || (g + 1 < live && kept_row + CR <= p.M)) {
#pragma unroll
        for (int sq = 0; sq < SQ; ++sq) body(g, sq, [](int) { return true; });
      } else {
#pragma unroll
        for (int sq = 0; sq < SQ; ++sq) {
          const int key = k0[g] + 4 * (lane_again >> 4), q = kept_row + 16 * sq + (lane_again & 15);
          const int lim = q >= p.M ? -1 : CAUSAL ? min(p.N - 1 - key, q + p.c - key) : p.N - 1 - key;
          body(g, sq, [lim](int r) { return r <= lim; });
        }
      }
    }
  };
  // The (maximum, sum) that the waves left of the rows of chunk i: each row of lanes takes its share of the waves.
  constexpr int PW = NW / 4;
  float wm[SQ][PW], wl[SQ][PW];
  auto read_partials = [&](int i) __attribute__((always_inline)) {
    const float* const set = sets + (i & 1) * 2 * kSums;
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq)
#pragma unroll
      for (int v = 0; v < PW; ++v) {
        const int at = (16 * sq + (lane & 15)) * NW + PW * (lane >> 4) + v;
        wm[sq][v] = set[at];
        wl[sq][v] = set[kSums + at];
      }
  };
  // Columns of the kept chunk, whose partials have been read.
  auto columns = [&](auto masked_tag) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    int lane_again = lane;   // opaque: what follows from it is not to be kept in registers from chunk to chunk
    asm volatile("" : "+v"(lane_again));
    float factor[SQ], lse[SQ];
    bool odd = no_scale;
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) {
      float m[1] = {wm[sq][0]}, l[1] = {0.f};
#pragma unroll
      for (int v = 1; v < PW; ++v) m[0] = fmaxf(m[0], wm[sq][v]);
      m[0] = lane_rows_reduce<true>(m);
      const float ref = m[0] == kNegInf ? 0.f : m[0];
#pragma unroll
      for (int v = 0; v < PW; ++v) l[0] = fmaf(wl[sq][v], fast_exp2(wm[sq][v] - ref), l[0]);   // (a wave without a key: 0 times 0)
      l[0] = lane_rows_reduce<false>(l);
      lse[sq] = l[0] == 0.f ? kNegInf : ref + fast_log2(l[0]);
      factor[sq] = (most[sq] == kNegInf ? 0.f : fast_exp2(most[sq] - ref)) * __builtin_amdgcn_rcpf(l[0]);
    }
    if (wave == 0) {
      float v = lse[0];
#pragma unroll
      for (int sq = 1; sq < SQ; ++sq) v = lane_again >> 4 == sq ? lse[sq] : v;
      if (lane_again < CR && kept_row + lane_again < p.M) p.lse[(int64_t)bh * p.M + kept_row + lane_again] = v;
    }
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) {
      if (MASKED && kept_row + 16 * sq + (lane_again & 15) >= p.M) factor[sq] = 0.f, lse[sq] = kPosInf;
      odd = odd || !(MODE == kModeSum ? factor[sq] < kPosInf : lse[sq] > kNegInf);   // a NaN, or a row whose scores are all -inf
    }
    groups(masked_tag, MASKED && __builtin_amdgcn_ballot_w64(odd) != 0, lane_again, [&](int g, int sq, auto seen) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (MODE == kModeSum) {
          csum[g][r] = seen(r) ? fmaf(x[g][sq][r], factor[sq], csum[g][r]) : csum[g][r];
        } else {
          const float y = seen(r) ? fmaf(x[g][sq][r], s2[sq], -lse[sq]) : kNegInf;
          if (MODE == kModeBoth) csum[g][r] += fast_exp2(y);
          cmax[g][r] = fmaxf(cmax[g][r], y);
        }
      }
    });
  };
  // The products of chunk i, whose groups in use are `live`, become the kept ones.
  auto exponents = [&](int i, f32x4(&acc)[NG][SQ], bool exact, auto masked_tag) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    int lane_again = lane;
    asm volatile("" : "+v"(lane_again));
    float part[SQ];
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) {
      s2[sq] = MASKED && exact ? up : up * rg.scale_of(i)[16 * sq + (lane_again & 15)];
      most[sq] = kNegInf;
      part[sq] = 0.f;
    }
    if (MASKED) no_scale = __builtin_amdgcn_ballot_w64(s2[0] == 0.f || s2[SQ - 1] == 0.f) != 0;   // (a scale of 0, or rows so small, padding too)
    groups(masked_tag, MASKED, lane_again, [&](int g, int sq, auto seen) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float y = acc[g][sq][r] * (MASKED && exact ? sign : ks4[g][r]);
        x[g][sq][r] = seen(r) ? y : kNegInf;
        most[sq] = fmaxf(most[sq], x[g][sq][r]);
      }
    });
#pragma unroll
    for (int sq = 0; sq < SQ; ++sq) {   // the largest score; -inf if the row sees none of the wave's keys
      const float m[1] = {most[sq] == kNegInf ? kNegInf : most[sq] * s2[sq]};
      most[sq] = lane_rows_reduce<true>(m);
    }
    groups(masked_tag, MASKED && no_scale, lane_again, [&](int g, int sq, auto seen) __attribute__((always_inline)) {
      const float ref = most[sq] == kNegInf ? 0.f : most[sq];
#pragma unroll
      for (int r = 0; r < 4; ++r) {   // (+inf - inf is a NaN, as the row kernel's lse then is)
        const float e = seen(r) ? fast_exp2(fmaf(x[g][sq][r], s2[sq], -ref)) : 0.f;
        part[sq] += e;
        if (MODE == kModeSum) x[g][sq][r] = e;
      }
    });
    float* const set_m = sets + (i & 1) * 2 * kSums;
    auto write_reduced = [&](float* set, float v) __attribute__((always_inline)) {
      if constexpr (SQ == 1) {
        if (lane_again < 16) set[lane_again * NW + wave] = v;
      } else {
        if ((lane_again & 16) == 0) set[((lane_again >> 5) * 16 + (lane_again & 15)) * NW + wave] = v;
      }
    };
    write_reduced(set_m, SQ == 1 || lane_again < 32 ? most[0] : most[SQ - 1]);
    write_reduced(set_m + kSums, lane_rows_reduce<false>(part));
  };

  put(0);
  fetch();
  {
    const uint32_t first = lanes_max<16>(largest);
    uint32_t wave_largest = 0;
#pragma unroll
    for (int l = 0; l < 64; l += 16) wave_largest = max(wave_largest, (uint32_t)__builtin_amdgcn_readlane((int)first, l));
    rg.publish(wave, k_largest, wave_largest);
  }
  ring_sync<63>();   // the first chunk is staged (waits for LDS accesses only: the fetch stays in flight)
  const bool first_bad = rg.set_limit(p.split_most);
  // the products of the first G groups, the keys in parts
  auto products = [&](f32x4(&acc)[NG][SQ], const char* stage, auto groups_tag, auto between) __attribute__((always_inline)) {
    constexpr int G = decltype(groups_tag)::value;
    if constexpr (G == NG) {
      split_scores<true>(acc, kf, rg, stage, 0, read_fragments<SQ>(rg, stage, 0, 0), between);
    } else {
      Planes keys[KS][G];
      f32x4 part[G][SQ];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int g = 0; g < G; ++g) keys[ks][g] = kf[ks][g];
      split_scores<true>(part, keys, rg, stage, 0, read_fragments<SQ>(rg, stage, 0, 0), between);
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int sq = 0; sq < SQ; ++sq) acc[g][sq] = part[g][sq];
    }
  };
  // The columns of a range: a reduce-scatter over the 16 query lanes; lane l ends up with key 4 * (l / 16) + (l & 3) of group (l & 15) / 4.
  const int col_grp = (lane & 15) >> 2, col_key = 16 * (wave + NW * col_grp) + 4 * (lane >> 4) + (lane & 3);
  const bool col_mine = col_grp < NG && col_key < p.N;
  float sum = 0.f, peak = 0.f;   // S == 1: of the ranges so far, added up in the order of merge_columns_kernel
  auto end_range = [&](int range) __attribute__((always_inline)) {
    f32x4 c4[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) c4[g] = g < NG ? csum[g % NG] : (f32x4){0.f, 0.f, 0.f, 0.f};
    const float s = MODE != kModeMax ? lanes16_scatter<false>(c4, lane) : 0.f;
#pragma unroll
    for (int g = 0; g < 4; ++g) c4[g] = g < NG ? cmax[g % NG] : (f32x4){0.f, 0.f, 0.f, 0.f};
    const float m = MODE != kModeSum ? fast_exp2(lanes16_scatter<true>(c4, lane)) : 0.f;
    if (S == 1) {
      sum += s;
      peak = fmaxf(peak, m);
    } else if (col_mine) {
      const int64_t at = ((int64_t)range * p.bh_count + bh) * p.N + col_key;
      if (MODE != kModeMax) static_cast<float*>(p.out)[at] = s;
      if (MODE != kModeSum) static_cast<float*>(MODE == kModeBoth ? p.out2 : p.out)[at] = m;
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      csum[g] = (f32x4){0.f, 0.f, 0.f, 0.f};
      cmax[g] = (f32x4){kNegInf, kNegInf, kNegInf, kNegInf};
    }
  };
  auto finish_chunk = [&](int i) __attribute__((always_inline)) {
    read_partials(i);
    if (some_hidden) columns(std::true_type());
    else columns(std::false_type());
  };
  // Chunk i: the columns of the chunk before, its own products, their exponents.
  int range = split, in_range = 0, q0 = split * L * CR;
#pragma unroll 1
  for (int i = 0; i < chunks; ++i) {
    if (i > 0) ring_sync<63>();
    const bool exact = res_bad || (i == 0 ? first_bad : rg.is_bad(i));
    const char* stage = rg.stage_of(i);
    f32x4 acc[NG][SQ];
    largest = 0;
    if (i > 0) {
      finish_chunk(i - 1);
      if (in_range == 0) end_range(range - S);
    }
    if (exact || q0 < full_row || q0 + CR > p.M) {
      const int in_use = live_groups(q0);
      put(i + 1);
      fetch();
      if (exact) {
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
          for (int sq = 0; sq < SQ; ++sq) acc[g][sq] = (f32x4){0.f, 0.f, 0.f, 0.f};
        exact_scores<true>(acc, kb, p.k_sr, k0, p.N, qb, p.q_sr, q0, p.M, p.dgran, lane);
      } else if (in_use > NG / 2) {
        products(acc, stage, std::integral_constant<int, NG>(), [](int) {});
      } else if (in_use > 0) {
        products(acc, stage, std::integral_constant<int, NG / 2>(), [](int) {});
      }
      live = in_use;
      kept_row = q0;
      some_hidden = true;
      exponents(i, acc, exact, std::true_type());
    } else {
      products(acc, stage, std::integral_constant<int, NG>(), [&](int ks) {
        if (ks == 0) {
          put(i + 1);
          fetch();
        }
      });
      live = NG;
      kept_row = q0;
      some_hidden = false;
      exponents(i, acc, false, std::false_type());
    }
    rg.note(i + 1, largest);
    q0 += CR;
    if (++in_range == L) {
      in_range = 0;
      range += S;
      q0 += (S - 1) * L * CR;
    }
  }
  ring_sync<63>();
  finish_chunk(chunks - 1);
  end_range(in_range == 0 ? range - S : range);
  if (S == 1 && col_mine) {
    if (MODE != kModeMax) store_column(p, p.out, true, bh, col_key, sum);
    if (MODE != kModeSum) store_column(p, MODE == kModeBoth ? p.out2 : p.out, false, bh, col_key, peak);
  }
}

// ---------------------------------------------------------------------------------------------
// Column sweep for at most 128 query rows against many keys, where the sweep is bound by reading K.
// The roles are swapped: every wave keeps ALL queries resident (NG = 4 or 8 groups of 16) and the keys
// stream through LDS in chunks of 64, fully coalesced and two chunks ahead.  Wave w takes keys
// [16w, 16w+16) of each chunk with S = Q * K^T, so a lane holds one key (lane & 15) against the
// queries 16g + 4*(lane/16) + r: the column reduction is an in-register sum over g and r plus two
// cross-lane steps, and each wave stores its 16 finished columns.  Workgroup v sweeps key chunks
// [split*per, split*per + per) of one (b,h), p.splits ranges per (b,h).  Every key is read by exactly
// one workgroup; p.stream_once makes those loads non-temporal (set when K is too large to stay cached).
// The general kernel reads the same keys as MFMA fragments, 64 bytes per row and instruction, and
// reaches 4.9 TB/s where this one reaches 6 (measured on 34 GB of keys).
constexpr int kSmallRows = 128;

template <int DT, int KS, bool CAUSAL, int MODE, int NG>
__global__ __launch_bounds__(kThreads, (NG <= 4 ? 3 : 2)) void col_small_kernel(const Params p) {
  using Rg = Ring<KS, 3>;   // three workgroups share a CU: 3 x 3 stages of 16 KiB
  // Finished columns wait in obuf and go to memory kFlush chunks at a time, 1 KiB per store instruction:
  // up to 10 % faster than a 64-byte store per wave and chunk.  (What the columns cost beyond that does
  // not depend on how they are stored: 134 MB of them beside 8.6 GB of keys take 15 % of the sweep, which
  // runs at the row kernel's rate with the stores disabled.)  The ring and obuf are ONE LDS object:
  // with two, the compiler orders every read of the ring after all loads in flight.
  constexpr int kFlush = (MODE == kModeBoth) ? 8 : 16;   // 4 KiB of LDS either way
  constexpr int kObufBytes = (MODE == kModeBoth ? 2 : 1) * kFlush * kChunk * 4;
  __shared__ __attribute__((aligned(1024))) char smem[Rg::kBytes + kObufBytes];
  float* const obuf = reinterpret_cast<float*>(smem + Rg::kBytes);
  int bh, split;
  map_group(p, (int)blockIdx.x, p.splits, bh, split);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = bh / p.H, h = bh - b * p.H;
  const char* qb = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
  const char* kb = p.k + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh;
  const float* lse = p.lse + (int64_t)bh * p.M;

  const int nchunks = (p.N + kChunk - 1) / kChunk;
  const int per = (nchunks + p.splits - 1) / p.splits;
  const int c0 = split * per, c1 = min(nchunks, c0 + per);
  if (c0 >= c1) return;  // the whole workgroup
  const int keys_end = min(p.N, c1 * kChunk);   // nothing is fetched from here on

  // The ring keeps two chunks of keys in flight per workgroup.
  Rg rg;
  rg.init(p.k_sr, p.dgran, lane, wave);
  const bool once = p.stream_once != 0;
  auto stage_of = [&](int t) { return smem + ((uint32_t)t % Rg::kN) * Rg::kStage; };
  rg.start(kb, p.k_sr, c0 * kChunk, keys_end);
  auto issue = [&](int t) {
    if (once) rg.template issue_next<kLoadOnce>(stage_of(t));
    else rg.template issue_next<0>(stage_of(t));
  };
#pragma unroll
  for (int i = 0; i < Rg::kN - 1; ++i) issue(c0 + i);

  // -lse of the lane's queries; -inf hides the rows past M
  const int qrow = 4 * (lane >> 4);
  float nlse[NG][4];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * g + qrow + r;
      const float v = lse[min(i, p.M - 1)];
      nlse[g][r] = (i < p.M) ? -v : kNegInf;
    }
  }
  // Rows past M are copies of the last one, which are as finite as that one is against every key (zeros against an infinite key
  // would make its columns NaN).
  u32x4 qf[NG][KS];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int first = min(16 * g, (p.M - 1) & ~15);   // of the sixteen rows that are read
    const __amdgpu_buffer_rsrc_t view = rows_view(qb, p.q_sr, first, p.M);
    const uint32_t roff = (uint32_t)min(lane & 15, p.M - 1 - first) * (uint32_t)p.q_sr;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int gi = ks * 4 + (lane >> 4);
      const u32x4 v = view_load16(view, roff + (uint32_t)min(gi, p.dgran - 1) * 16u);
      qf[g][ks] = gi < p.dgran ? v : (u32x4){0u, 0u, 0u, 0u};
    }
  }

  void* const out_max = (MODE == kModeBoth) ? p.out2 : p.out;
  float* obuf_max = obuf + (MODE == kModeBoth ? kFlush * kChunk : 0);
  // Columns of chunks [ta, ta + kFlush) from obuf to memory, up to the end of this workgroup's range;
  // all waves have passed a barrier since they wrote them.
  auto flush = [&](int ta) {
    const int key0 = ta * kChunk, nkeys = keys_end - key0;
#pragma unroll
    for (int r = 0; r < kFlush * kChunk / kThreads; ++r) {
      const int i = tid + r * kThreads;
      if (i < nkeys) {
        if (MODE != kModeMax) store_column(p, p.out, true, bh, key0 + i, obuf[i]);
        if (MODE != kModeSum) store_column(p, out_max, false, bh, key0 + i, obuf_max[i]);
      }
    }
  };
  for (int t = c0; t < c1; ++t) {
    ring_sync<(Rg::kN - 2) * Rg::kPer>();   // chunk t visible, the stage of chunk t - 1 is free
    issue(t + Rg::kN - 1);
    if (t > c0 && (t - c0) % kFlush == 0) {
      flush(t - kFlush);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();   // obuf is free again before anyone writes chunk t's columns
      asm volatile("" ::: "memory");
    }
    const char* lds = stage_of(t);
    const int key = t * kChunk + 16 * wave + (lane & 15);
    // query i sees the key iff key <= i + c; chunks that end at or before key c need no mask
    const bool need_mask = CAUSAL && (t * kChunk + kChunk - 1 > p.c);
    const int first = key - p.c - qrow;  // register (g, r) is visible iff 16g + r >= first
    float vsum = 0.f, vmax = kNegInf;
    // four query groups at a time, so that at most four accumulators are live
#pragma unroll
    for (int gb = 0; gb < NG; gb += 4) {
      f32x4 acc[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) acc[g] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const u32x4 kfrag = rg.frag(lds, wave >> 1, wave & 1, ks);
#pragma unroll
        for (int g = 0; g < 4; ++g) acc[g] = mma<DT>(qf[gb + g][ks], kfrag, acc[g]);
      }
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int r2 = 0; r2 < 4; ++r2) {
          float x = fmaf(acc[g][r2], p.scale2, nlse[gb + g][r2]);
          // (rows past M are copies of others, which an infinite key that only later rows see makes a NaN)
          if (need_mask) x = (16 * (gb + g) + r2 >= first && 16 * (gb + g) + r2 < p.M - qrow) ? x : kNegInf;
          if (MODE != kModeSum) vmax = fmaxf(vmax, x);
          if (MODE != kModeMax) vsum += fast_exp2(x);
        }
    }
    // the four lane groups hold different queries of the same key
    const int slot = ((t - c0) % kFlush) * kChunk + 16 * wave + lane;
    if (MODE != kModeMax) {
      vsum += __shfl_xor(vsum, 16);
      vsum += __shfl_xor(vsum, 32);
      if (lane < 16) obuf[slot] = vsum;
    }
    if (MODE != kModeSum) {
      vmax = fmaxf(vmax, __shfl_xor(vmax, 16));
      vmax = fmaxf(vmax, __shfl_xor(vmax, 32));
      if (lane < 16) obuf_max[slot] = fast_exp2(vmax);
    }
  }
  ring_sync<0>();   // the loads past the last chunk write their zeros before the LDS is given back
  flush(c0 + (c1 - c0 - 1) / kFlush * kFlush);
}


// ---------------------------------------------------------------------------------------------
// Both sweeps in one for at most 128 query rows against many keys: the keys are read from memory ONCE.
// A team of p.splits workgroups shares a (b,h) pair; workgroup s of the team owns 16 chunks of 64 keys (8
// with more than 64 queries); a wave takes 16 keys of a chunk against 64 queries (as in col_small_kernel).
// Per pair a workgroup
//   1. streams its keys through the LDS ring and computes their scores, which STAY IN REGISTERS (16 per
//      lane and step): for column sums as 2^score, otherwise (maxima) as the scaled scores themselves;
//   2. sums 2^score per row over its own keys and publishes the 32, 64 or 128 sums.  A sum outside [2^-60, 2^100)
//      (scores far from zero, a row that sees none of these keys, a NaN) is not trusted: the scores are then
//      reduced the exact way, row maximum first -- from the registers if they hold scores, else after a second sweep
//      over the same keys that keeps the scores -- and the log2 of the sum is published;
//   3. reads what the other workgroups of its team have published for this pair and adds it up (every workgroup of the
//      team does this for itself; a log2 among the values turns the addition into a merge);
//   4. turns what it kept into probabilities (2^score times the reciprocal of the sum: one multiply-add per score),
//      reduces them down the rows and leaves its columns in LDS, from where they go to memory under the next sweep.
// The grid is teams * splits workgroups and never more than the CUs hold at once (one of eight waves, two of four), so every workgroup of a team is
// running when its partners wait for it; team t takes pairs t, t + teams, t + 2 teams, ..  The first keys
// of the next pair stream into the ring while a workgroup does steps 2-4, and the next pair's queries are
// staged in LDS a whole sweep ahead.  A wait is bounded: after p.spin_limit polls the workgroup gives up,
// sets the error word, stores NaN columns for that pair and goes on, so every workgroup reaches its end
// whatever happens to the others.
// Between workgroups: a partial value travels together with the number of its round as ONE 64-bit word,
// written and read with device-scope relaxed atomics (performed where every workgroup of the device
// sees them), so a word that shows the round shows the value; there is no counter, no fence and nobody
// waits for a store to complete.  The slots start at zero (a small kernel in front clears them), rounds
// count from 1, and the slots alternate between two sets by the parity of the round: a workgroup can be at
// most one round ahead of the slowest of its team.  The barriers between the steps wait for LDS only, so
// the keys in flight stay in flight.
// Registers are the limit (128 for the scores, 64 for the queries during step 1): what depends on the
// thread is derived again after step 1 from opaque copies instead of being kept across it.
// chunks of 64 keys per workgroup and pair: 16 for up to 64 queries, 8 for up to 128; 32 when a wave holds two
// groups of sixteen queries (nq) instead of four
__host__ __device__ constexpr int fused_chunks(int qh, int nq = 4) { return qh == 1 ? 16 * (4 / nq) : 8; }
constexpr int kFusedSteps = 8;
constexpr unsigned kIsLog = 0x80000000u;   // of a slot's round number: the value is a log2

// Sum or maximum over each row of 16 lanes; every lane of the row ends up with the result.
template <bool MAX>
__device__ __forceinline__ float row16_reduce(float v) {
  float o = dpp_row<0xB1>(v);    // quad_perm [1,0,3,2]
  v = MAX ? fmaxf(v, o) : v + o;
  o = dpp_row<0x4E>(v);          // quad_perm [2,3,0,1]
  v = MAX ? fmaxf(v, o) : v + o;
  o = dpp_row<0x141>(v);         // row_half_mirror
  v = MAX ? fmaxf(v, o) : v + o;
  o = dpp_row<0x140>(v);         // row_mirror
  v = MAX ? fmaxf(v, o) : v + o;
  return v;
}

// n words from w on get `value`, and the word at `zero`, if there is one, 0: in front of both_sweeps_kernel.
__global__ __launch_bounds__(256) void fill_words_kernel(unsigned* __restrict__ w, int64_t n, unsigned value, unsigned* __restrict__ zero) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + (int)threadIdx.x) * 4;
  if ((reinterpret_cast<uintptr_t>(w) & 15) == 0 && i + 4 <= n) {
    *reinterpret_cast<u32x4*>(w + i) = (u32x4){value, value, value, value};
  } else {
    for (int64_t j = i; j < n && j < i + 4; ++j) w[j] = value;
  }
  if (i == 0 && zero != nullptr) *zero = 0u;
}

// n words from w on, and the word at `one`.  (A workspace of one of the calls without a size may start at any multiple of 8 bytes.)  A launch of its own in front of every single sweep: 16 bytes per
// thread, and of a launch of one round one of the two sets of slots (32 pairs of 128 x 4096 x 128 17.8 -> 17.4 us per call).
__global__ __launch_bounds__(256) void zero_words_kernel(unsigned* __restrict__ w, int n, unsigned* __restrict__ one) {
  const int i = ((int)blockIdx.x * 256 + (int)threadIdx.x) * 4;
  if ((reinterpret_cast<uintptr_t>(w) & 15) == 0 && i + 4 <= n) {
    *reinterpret_cast<u32x4*>(w + i) = (u32x4){0u, 0u, 0u, 0u};
  } else {
    for (int j = i; j < n && j < i + 4; ++j) w[j] = 0u;
  }
  if (i == 0) *one = 0u;
}

// Eight waves, one workgroup per CU, or four, two per CU; eight steps per workgroup and pair (sixteen with two query groups).  Up to 64 queries (QH = 1, KH = 2):
// a step is two chunks of 64 keys, waves 0-3 take (and load) the first, waves 4-7 the second.  Up to 128
// queries (QH = 2, KH = 1): a step is one chunk, waves 4-7 hold queries 64-127, waves 0-3 load.
// NQ: groups of sixteen queries a wave holds (4; 2 for at most 32 queries: the registers then hold the scores of
// twice as many keys per pair, and the time between two sweeps is spread over that many.  One group and four
// times the keys was built as well and was slower than two: 1568 against 1499 us on 64 x 32 pairs of 16384 keys).
// SKIP: chunks past a workgroup's last key (spread_keys deals them evenly, so these are its last ones) are left out instead of being computed
// and hidden score by score.  When the team's last workgroup held all of them, it waited for that one: 6 x 40 pairs of 111 x 7284 x 128 206 -> 165 us per call, 5 x 24 of 89 x 3776 x 64 51 -> 43,
// 7 x 24 of 100 x 15756 x 128 249 -> 237 (bf16, sums).
// NW: waves.  Four (a step is one chunk, and a pair's keys are shared by twice the workgroups) leave room for two
// workgroups on a CU, of different teams or key ranges: one streams while the other exchanges its row sums.  For at most 32 queries
// (NQ = 2): 512 pairs of 32 x 16384 x 128 411 -> 369 us, 347 with the shorter exchange below.  With 64 they
// lose, 397 -> 412: every workgroup reads a word per row of every other one of its team, 0.27 GB beside 2.1 GB of keys.
// The time between two sweeps, 64 queries and 1024 keys, in cycles: row sums 3000 -> 2600, the team's values 2300 -> 1800, their
// merge 2200 -> 1900 (sums instead of logarithms), columns 3600 -> 1100 (no question per step), their way to memory 1500 -> 0.
template <int DT, int KS, bool CAUSAL, int MODE, int QH, int NQ, bool SKIP, int NW>
__global__ __launch_bounds__(64 * NW, 2) void col_fused_kernel(const Params p) {
  static_assert(NQ == 4 || (QH == 1 && NQ == 2), "fewer query groups only with one query half");
  static_assert(NW == 8 || (NW == 4 && NQ == 2), "four waves hold two query groups");
  constexpr int KG = kFusedSteps * (4 / NQ);     // steps per pair
  constexpr int KH = NW == 4 ? 1 : 3 - QH;       // chunks per step
  // ring stages (chunks): 130 KiB or 98 KiB for 256-byte rows, 49 with four waves
  constexpr int NS = NW == 4 ? (KS <= 2 ? 6 : 3) : (QH == 1) ? 8 : 6;
  using Rg = Ring<KS, NS>;                       // four loads of 1 KiB per loading wave and chunk for 256-byte rows
  constexpr int kQBytes = QH * Rg::kRows;        // the queries of a pair, staged like a chunk of keys per 64 rows
  constexpr int kNumThreads = 64 * NW;
  constexpr int kRowsWg = 16 * NQ * QH;          // query rows a workgroup holds
  constexpr int kBatchKeys = kFusedSteps * KH * kChunk;   // finished columns leave eight steps at a time
  constexpr int kBatches = KG / kFusedSteps;
  constexpr int kRes = (MODE == kModeBoth) ? 2 : 1;
  constexpr int kObufFloats = QH * kRes * kBatchKeys;
  constexpr int kRedFloats = NW * 64;
  // waves per row that share the merge of the team's partial values (half of them when two results are
  // buffered for 1024 keys: the LDS is full)
  constexpr int kMergeWaves = (NW / QH) / ((kRes == 2 && QH == 1 && NW == 8) ? 2 : 1);
  constexpr int kBatch = 4 * QH * (8 / NW);                 // slots a lane fetches together: one round trip for teams of up to 32
  constexpr int kMrgFloats = kMergeWaves * kRowsWg * 2;
  // Column sums: the row sums are taken as the scores come, while the sweep waits for memory, or, where the registers do not reach for that (five in
  // memory for 65 to 128 queries that skip nothing, many more for two query groups), after it.  65 to 128 queries that skip: 0.97 of the time.
  constexpr bool kSumsInSweep = NQ == 4 && (QH == 1 || SKIP);
  constexpr int kAhead = NS / KH - 1;            // steps in flight in front of the one being computed
  constexpr int kInFlight = (NS / KH - 2) * Rg::kPer;   // loads a loading wave may have outstanding when a step starts
  // (one LDS object: see col_small_kernel)
  // one LDS object: ring | queries | finished columns | per-wave row partials | merge | per-row values | flags
  __shared__ __attribute__((aligned(1024))) char smem[Rg::kBytes + kQBytes + (kObufFloats + kRedFloats + kMrgFloats + kRowsWg + 4) * 4];
  char* const qlds = smem + Rg::kBytes;
  float* const obuf = reinterpret_cast<float*>(smem + Rg::kBytes + kQBytes);
  float* const red = obuf + kObufFloats;
  float* const mrg = red + kRedFloats;
  float* const rowv = mrg + kMrgFloats;
  int* const flag = reinterpret_cast<int*>(rowv + kRowsWg);

  const int tid0 = threadIdx.x, lane0 = tid0 & 63;   // (the loop over the pairs has its own copies, see there)
  const int wave = __builtin_amdgcn_readfirstlane(tid0 >> 6);
  const int qh = (QH == 2) ? (wave >> 2) : 0;    // which 64 queries
  const int kh = (KH == 2) ? (wave >> 2) : 0;    // which chunk of a step
  const int wq = wave & 3;                       // which 16 keys of the chunk
  const bool loader = (KH == 2) || (wave < 4);   // (four waves: all)
  const int S = p.splits, T = p.teams;
  const int team = (int)blockIdx.x / S, split = (int)blockIdx.x - team * S;
  const int c0 = split * p.run_chunks;           // first chunk of this workgroup's keys
  const int key0 = c0 * kChunk;
  const int keys_end = min(p.N, key0 + p.run_chunks * kChunk);
  const int rounds = (p.bh_count - team + T - 1) / T;
  const int qrow0 = 4 * (lane0 >> 4);
  int spin_limit = p.spin_limit;
  // flag[0]: a row of this workgroup has a sum that must be redone; flag[1]: the team was met.  Each is
  // written and read on different sides of a barrier.
  if (tid0 == 0) flag[0] = 0;

  Rg rg;
  rg.init(p.k_sr, p.dgran, lane0, 0);   // (for the fragment offsets; the loads are issued below)
  const bool once = p.stream_once != 0;
  auto stage_of = [&](int c) { return smem + ((uint32_t)c % NS) * Rg::kStage; };
  // The loaders walk the workgroup's stream of chunks with a running address: KG * KH chunks of one pair,
  // then the same range of keys of the next pair of the team.  Chunk number c goes to stage c % NS.
  const int64_t chunk_bytes = (int64_t)kChunk * p.k_sr;
  const char* run_ptr = nullptr;
  int run_rows = 0, run_chunk = 0;
  auto run_to_pair = [&](int bh) {               // the cursor to the start of this workgroup's keys of pair bh
    const int bhc = min(bh, p.bh_count - 1);
    const int b = bhc / p.H, h = bhc - b * p.H;
    run_ptr = p.k + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh + (int64_t)key0 * p.k_sr;
    run_rows = (bh < p.bh_count) ? keys_end - key0 : 0;   // past the last pair: zeros, nothing is fetched
  };
  // Where a lane's 16 bytes of each load come from (see Ring::init).  The swizzle repeats every eight rows,
  // so the kPer loads of a wave have at most kPat different patterns and the rest follow by adding rows.
  constexpr int kPat = (Rg::kRowsPerLoad >= 8) ? 1 : 8 / Rg::kRowsPerLoad;
  const int lw = wave & 3;                         // which of the loading waves
  uint32_t src_off[kPat];
  bool src_ok[kPat];
#pragma unroll
  for (int e = 0; e < kPat; ++e) {
    const int byte = (lw * Rg::kPer + e) * 1024 + lane0 * 16;
    const int row = byte / Rg::kPitch;
    const int c = ((byte % Rg::kPitch) / 16) ^ Rg::swz(row);
    src_ok[e] = c < p.dgran;
    src_off[e] = (uint32_t)row * (uint32_t)p.k_sr + (uint32_t)c * 16u;
  }
  const uint32_t pat_bytes = (uint32_t)(kPat * Rg::kRowsPerLoad) * (uint32_t)p.k_sr;
  auto issue_step = [&]() {   // the wave's chunk of the next step
    char* stage = stage_of(run_chunk + kh);
    const char* src = run_ptr + (KH == 2 && kh ? chunk_bytes : 0);
    const int live = rows_in_chunk(run_rows - kh * kChunk);
    run_chunk += KH;        // (every wave keeps the cursor, only the loading ones issue)
    run_ptr += KH * chunk_bytes;
    run_rows -= KH * kChunk;
    if (!loader) return;
    const __amdgpu_buffer_rsrc_t view = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char*>(src), 0, (int)((uint32_t)live * (uint32_t)p.k_sr), 0x00020000);
    uint32_t so[kPat];   // opaque copies: the kPer offsets are made per call, not kept in registers between calls
#pragma unroll
    for (int e = 0; e < kPat; ++e) {
      so[e] = src_off[e];
      asm volatile("" : "+v"(so[e]));
    }
    if (once) {
#pragma unroll
      for (int i = 0; i < Rg::kPer; ++i) {
        const uint32_t off = src_ok[i % kPat] ? so[i % kPat] + (uint32_t)(i / kPat) * pat_bytes : kPastEnd;
        dma16<kLoadOnce>(view, off, stage + (lw * Rg::kPer + i) * 1024);
      }
    } else {
#pragma unroll
      for (int i = 0; i < Rg::kPer; ++i) {
        const uint32_t off = src_ok[i % kPat] ? so[i % kPat] + (uint32_t)(i / kPat) * pat_bytes : kPastEnd;
        dma16<0>(view, off, stage + (lw * Rg::kPer + i) * 1024);
      }
    }
  };
  int cons_chunk = 0;       // number of the next chunk to be computed (its stage: cons_chunk % NS)

  u32x4 qf[NQ][KS];
  // The queries of a pair go from memory to LDS like a chunk of keys (64 rows per stage-like tile, same
  // swizzle), long before they are needed, and from there into the registers when the pair's sweep starts:
  // no wave ever waits for them, and they take no registers between two sweeps.  Waves 0-3 load.
  auto stage_queries = [&](int bh) {
    if (wave >= 4) return;
    const int b = bh / p.H, h = bh - b * p.H;
    const char* qb = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh;
#pragma unroll
    for (int t = 0; t < QH; ++t) {
      const int live = rows_in_chunk(p.M - 64 * t);
      const __amdgpu_buffer_rsrc_t view = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<char*>(qb + (int64_t)(64 * t) * p.q_sr), 0, (int)((uint32_t)live * (uint32_t)p.q_sr), 0x00020000);
#pragma unroll
      for (int i = 0; i < Rg::kPer; ++i) {
        const int byte = (lw * Rg::kPer + i) * 1024 + lane0 * 16;
        const int row = byte / Rg::kPitch;
        const int c = ((byte % Rg::kPitch) / 16) ^ Rg::swz(row);
        const uint32_t off = (c < p.dgran) ? (uint32_t)row * (uint32_t)p.q_sr + (uint32_t)c * 16u : kPastEnd;
        dma16<0>(view, off, qlds + t * Rg::kRows + (lw * Rg::kPer + i) * 1024);
      }
    }
  };
  auto read_queries = [&]() {
#pragma unroll
    for (int g = 0; g < NQ; ++g)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) qf[g][ks] = rg.frag(qlds + qh * Rg::kRows, g >> 1, g & 1, ks);
  };
  // the first pair's queries, then the first steps of its keys: the loads return in this order, so the
  // wait in front of the first step covers the queries
  stage_queries(team);
  run_to_pair(team);
#pragma unroll
  for (int i = 0; i < kAhead; ++i) issue_step();

  // Register (g, r) of a lane is query 64*qh + 16g + qrow + r against the lane's key.  It takes part iff
  // the query exists and may see the key: 16g + r in [first, mlim).
  const int mlim0 = p.M - 64 * qh - qrow0;
  const bool ragged_rows = p.M < 16 * NQ * (qh + 1);
  constexpr int kRowWaves = NW / QH;   // row tid (tid < kRowsWg) is held by all waves, or by 0-3 / 4-7 for rows below / from 64

  // Columns of batch bt of pair bh from their buffer to memory (all waves have passed a barrier since they wrote them).
  bool waiting = false, met = true;   // the last batch of the pair before is still in the buffer; its team was met
  auto store_columns = [&](int bh, int bt, bool met) __attribute__((always_inline)) {
    void* const out_max = (MODE == kModeBoth) ? p.out2 : p.out;
    const float poison = __builtin_nanf("");
    const int bkey0 = key0 + bt * kBatchKeys;
    int tid_here = threadIdx.x;
    asm volatile("" : "+v"(tid_here));
#pragma unroll
    for (int r = 0; r < kBatchKeys / kNumThreads; ++r) {
      const int i = tid_here + r * kNumThreads;
      if (bkey0 + i < keys_end) {
        if (MODE != kModeMax) {
          float v = obuf[i];
          if (QH == 2) v += obuf[kRes * kBatchKeys + i];
          store_column(p, p.out, true, bh, bkey0 + i, met ? v : poison);
        }
        if (MODE != kModeSum) {
          const float* om = obuf + (MODE == kModeBoth ? kBatchKeys : 0);
          float v = om[i];
          if (QH == 2) v = fmaxf(v, om[kRes * kBatchKeys + i]);
          store_column(p, out_max, false, bh, bkey0 + i, met ? v : poison);
        }
      }
    }
  };

  for (int it = 0; it < rounds; ++it) {
    const int bh = team + it * T;
    // What the registers keep per score: for column sums 2^score (step 4 is then one multiply-add per score),
    // otherwise, or when a row's sum of 2^score is unusable, the score itself.  In the second case of a sum
    // the scores are gone by the time it shows, and the keys of the pair are streamed once more.
    f32x4 sc[KG][NQ];
    f32x4 rs[NQ];   // per row (register) and key (lane): sum of 2^score over the steps
    bool odd_padding = false;   // row tid does not exist and has met a non-finite key
    float my_lse = kNegInf;   // of row tid over this workgroup's keys, for tid < kRowsWg (where the plain sums are not usable)
    // A partial value and the number of its round travel as ONE 64-bit word, so a word that carries this round's number carries this
    // round's value: nobody waits for a store to complete and there is no counter.  The slots start at zero (round
    // numbers start at 1).  The value is the row's sum of 2^score, or, with the top bit set, its log2.
    unsigned long long* const slots =
        reinterpret_cast<unsigned long long*>(p.part) + ((int64_t)((it & 1) * T + team) * S) * kRowsWg;
    const unsigned round_no = (unsigned)it + 1u;
    // A row is published once, whatever becomes of the others: the team adds up the same values.
    bool published = false;
    auto publish = [&](int row, unsigned kind, float v) __attribute__((always_inline)) {
      if (published) return;
      published = true;
      __hip_atomic_store(slots + (int64_t)split * kRowsWg + row,
                         ((unsigned long long)(round_no | kind) << 32) | __builtin_bit_cast(unsigned, v), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    };
    // Steps 1 and the first half of 2, in two forms (KEEP: the registers end up holding the scores).  Returns
    // whether some row's sum of 2^score is unusable.
    auto sweep = [&](auto keep_tag) -> bool {
    constexpr bool KEEP = decltype(keep_tag)::value;
    if (KEEP) {
#pragma unroll
      for (int g = 0; g < NQ; ++g) rs[g] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    {
    const int tid = tid0, lane = lane0, qrow = qrow0, mlim = mlim0;
    // 1. scores of this workgroup's keys, scaled, hidden ones at -inf
    // (what the mask needs is derived afresh from an opaque copy of c0 here and in step 4: kept across the
    // steps, or hoisted out of the loop over the pairs, it would cost registers that the scores need)
    int c0a = c0;
    asm volatile("" : "+s"(c0a));
#pragma unroll
    for (int j = 0; j < KG; ++j) {
      ring_sync<kInFlight>();   // the chunks of this step are visible, the stages of the step before are free
      if (j + kAhead == KG) run_to_pair(bh + T);   // the steps from here on belong to the next pair
      issue_step();
      if (j == 0) read_queries();   // (staged at least a whole sweep ago; the barrier above has published them)
      if (j == 1 && it + 1 < rounds) stage_queries(bh + T);   // every wave has read this pair's by now
      if (j == 1 && waiting) {   // the columns of the pair before, under the loads of this one (the barriers above have published them)
        store_columns(bh - T, kBatches - 1, met);
        waiting = false;
      }
      const char* lds = stage_of(cons_chunk + j * KH + kh);
      if (SKIP && (c0a + j * KH + kh) * kChunk >= keys_end) {
        const float none = KEEP ? kNegInf : 0.f;
#pragma unroll
        for (int g = 0; g < NQ; ++g) {
          sc[j][g] = (f32x4){none, none, none, none};
          if (kSumsInSweep && !KEEP && j == 1) rs[g] = sc[0][g];
        }
        continue;
      }
#pragma unroll
      for (int g = 0; g < NQ; ++g) sc[j][g] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const u32x4 kfrag = rg.frag(lds, wq >> 1, wq & 1, ks);
#pragma unroll
        for (int g = 0; g < NQ; ++g) sc[j][g] = mma<DT>(qf[g][ks], kfrag, sc[j][g]);
      }
      const int kbase = (c0a + j * KH + kh) * kChunk;
      const int key = kbase + 16 * wq + (lane & 15);
      // Rows past M are rows of zeros: their scores are 0 and their 2^score is 1, which nothing downstream uses
      // (step 4 multiplies by 0 or adds -inf), so they are not hidden.  Only a key with a non-finite element makes them
      // NaN; the row threads below look for that, and step 4 then hides them (of plain sums after a second sweep).
      const bool need_mask = kbase + kChunk > p.N || (CAUSAL && kbase + kChunk - 1 > p.c + 64 * qh);
      if (need_mask) {
        int first = CAUSAL ? key - p.c - 64 * qh - qrow : -(1 << 30);
        if (key >= p.N) first = 1 << 30;
#pragma unroll
        for (int g = 0; g < NQ; ++g)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int o = 16 * g + r;
            sc[j][g][r] = (o >= first && o < mlim) ? sc[j][g][r] * p.scale2 : kNegInf;
          }
      } else {
#pragma unroll
        for (int g = 0; g < NQ; ++g) sc[j][g] *= p.scale2;
      }
      if (KEEP) {
#pragma unroll
        for (int g = 0; g < NQ; ++g)
#pragma unroll
          for (int r = 0; r < 4; ++r) rs[g][r] += fast_exp2(sc[j][g][r]);
      } else {
#pragma unroll
        for (int g = 0; g < NQ; ++g)
#pragma unroll
          for (int r = 0; r < 4; ++r) sc[j][g][r] = fast_exp2(sc[j][g][r]);
        if (kSumsInSweep && j > 0) {
#pragma unroll
          for (int g = 0; g < NQ; ++g) rs[g] = (j == 1) ? sc[0][g] + sc[1][g] : rs[g] + sc[j][g];
        }
      }
    }
    cons_chunk += KG * KH;
    }
    if (!KEEP && !kSumsInSweep) {
#pragma unroll
      for (int g = 0; g < NQ; ++g) {
        rs[g] = sc[0][g];
#pragma unroll
        for (int j = 1; j < KG; ++j) rs[g] += sc[j][g];
      }
    }
    // From here on, everything that depends on the thread is derived afresh from an opaque copy of its
    // number: values kept for these steps across step 1 would take registers from the scores (and come
    // back from scratch memory, a round trip each).
    int tid_again = threadIdx.x;
    asm volatile("" : "+v"(tid_again));
    const int tid = tid_again, lane = tid & 63, qrow = 4 * (lane >> 4);
    const float* const red_row = red + (QH == 2 ? (tid >> 6) * (kWaves * 64) : 0) + (tid & 63);

    // 2. log-sum-exp of every row over this workgroup's keys.  The sums of 2^x were taken as the scores
    // came; they are good unless a sum left fp32's comfortable range (or a row saw no key at all), and then
    // the scores, still in registers, are reduced again the exact way: row maximum first.
    {
      f32x4 all[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) all[g] = g < NQ ? rs[g % NQ] : (f32x4){0.f, 0.f, 0.f, 0.f};
      const float v = lanes16_scatter<false>(all, lane);   // row 16 * ((lane & 15) / 4) + qrow + (lane & 3)
      const int g = (lane & 15) >> 2;
      if (g < NQ) red[wave * 64 + 16 * g + qrow + (lane & 3)] = v;
    }
    lds_barrier();
    if (tid < kRowsWg) {
      float l = 0.f;
#pragma unroll
      for (int w = 0; w < kRowWaves; ++w) l += red_row[64 * w];
      // 2^-60 <= l < 2^100: terms flushed to zero are far below the sum's last bit, and 2^score times 2^-lse
      // (the lse of all keys is at least this one) neither overflows nor loses anything above 2^-26
      // A row that the mask lets see none of this workgroup's keys adds nothing, and that is its sum: no reason to sweep them again.  The last
      // workgroup of a team, with fewer keys than there are queries, made all of it wait for that: 7400 shapes of 33 to 128 queries 0.93 of the
      // time in the geometric mean, one in ten below 0.68, 0.48 at best (maxima and both, reduced again from registers: 0.97, 0.74).
      const bool none = CAUSAL && tid + p.c < key0;
      const bool good = none || ((l >= 8.6736174e-19f) && (l < 1.2676506e30f));
      if (!good && tid < p.M) flag[0] = 1;   // (written by whoever finds a bad row; thread 0 resets it below)
      odd_padding = tid >= p.M && !(l < kPosInf);   // a row of zeros met a non-finite key
      if (!KEEP && odd_padding) flag[0] = 1;
      if (tid == 0) flag[1] = 1;
      if (good || tid >= p.M) publish(tid, 0u, none ? 0.f : good ? l : 1.f);   // (rows that do not exist: anything finite)
    }
    lds_barrier();
    return flag[0] != 0;   // uniform over the workgroup
    };   // sweep
    bool keep_scores = (MODE != kModeSum);
    bool bad_sum;
    if (MODE == kModeSum) {
      bad_sum = sweep(std::false_type());
      if (bad_sum) {
        // once more through the keys of this pair: the loads in flight (for the next pair) land and are
        // dropped, the loader goes back to this pair's first chunk and the ring starts afresh
        ring_sync<0>();
        if (tid0 == 0) flag[0] = 0;
        stage_queries(bh);   // (the sweep above has already replaced them by the next pair's)
        run_to_pair(bh);
        cons_chunk = run_chunk;
#pragma unroll
        for (int i = 0; i < kAhead; ++i) issue_step();
        keep_scores = true;
        bad_sum = sweep(std::true_type());
      }
    } else {
      bad_sum = sweep(std::true_type());
    }
    int tid_once_more = threadIdx.x;
    asm volatile("" : "+v"(tid_once_more));
    const int tid = tid_once_more, lane = tid & 63, qrow = 4 * (lane >> 4);
    const int mlim = p.M - 64 * qh - qrow;
    const float* const red_row = red + (QH == 2 ? (tid >> 6) * (kWaves * 64) : 0) + (tid & 63);
    if (bad_sum) {
      f32x4 rm[NQ];
#pragma unroll
      for (int g = 0; g < NQ; ++g) {
        rm[g] = sc[0][g];
#pragma unroll
        for (int j = 1; j < KG; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) rm[g][r] = fmaxf(rm[g][r], sc[j][g][r]);
#pragma unroll
        for (int r = 0; r < 4; ++r) rm[g][r] = row16_reduce<true>(rm[g][r]);
        if ((lane & 15) == 0) *reinterpret_cast<f32x4*>(red + wave * 64 + 16 * g + qrow) = rm[g];
      }
      lds_barrier();
      float my_max = kNegInf;
      if (tid < kRowsWg) {
#pragma unroll
        for (int w = 0; w < kRowWaves; ++w) my_max = fmaxf(my_max, red_row[64 * w]);
        rowv[tid] = (my_max == kNegInf) ? 0.f : my_max;   // no visible key: any finite reference
      }
      lds_barrier();
#pragma unroll
      for (int g = 0; g < NQ; ++g) {
        const f32x4 ref = *reinterpret_cast<const f32x4*>(rowv + 64 * qh + 16 * g + qrow);
        rs[g] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < KG; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) rs[g][r] += fast_exp2(sc[j][g][r] - ref[r]);
#pragma unroll
        for (int r = 0; r < 4; ++r) rs[g][r] = row16_reduce<false>(rs[g][r]);
        if ((lane & 15) == 0) *reinterpret_cast<f32x4*>(red + wave * 64 + 16 * g + qrow) = rs[g];
      }
      lds_barrier();
      if (tid < kRowsWg) {
        float l = 0.f;
#pragma unroll
        for (int w = 0; w < kRowWaves; ++w) l += red_row[64 * w];
        // a +inf score makes inf - inf above, a NaN score stays: both give a NaN here, as the row kernel does
        my_lse = (my_max == kNegInf) ? kNegInf : my_max + fast_log2(l);
      }
    }
    // 3. meet the team.
    if (bad_sum && tid < kRowsWg) publish(tid, kIsLog, my_lse);
    // All waves share the team's slots: lane = row, the waves of a row take every kMergeWaves-th slot, poll
    // until it carries this round, and fold the values into (max, sum).  (The keys a wave has in flight
    // for the next pair return before these loads do; they were requested during the last steps above.)
    // Plain sums are added up; where one is a log2 all are taken as such, as (max, sum) pairs.
    if (wave / QH < kMergeWaves) {
      const int rgroup = wave % QH, sub = wave / QH;
      const bool row_here = 64 * rgroup + lane < kRowsWg;   // (fewer than 64 rows per workgroup with NQ < 4)
      const unsigned long long* mine = slots + 64 * rgroup + lane;
      float m = 0.f, acc = 0.f;
      bool nan = false, ok = true;
      int polls = 0;
      for (int s0 = sub; s0 < S; s0 += kMergeWaves * kBatch) {
        unsigned long long w[kBatch];
        for (;;) {
          bool all = true;
#pragma unroll
          for (int i = 0; i < kBatch; ++i) {
            const int sidx = s0 + i * kMergeWaves;
            w[i] = (sidx < S && row_here) ? __hip_atomic_load(mine + (int64_t)sidx * kRowsWg, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                              : ((unsigned long long)round_no << 32);   // a sum of 0
          }
#pragma unroll
          for (int i = 0; i < kBatch; ++i) all = all && (((unsigned)(w[i] >> 32) & ~kIsLog) == round_no);
          if (all) break;
          if (++polls > spin_limit) {
            ok = false;
            break;
          }
          __builtin_amdgcn_s_sleep(8);
        }
        if (!ok) break;
        float v[kBatch];
#pragma unroll
        for (int i = 0; i < kBatch; ++i) v[i] = __builtin_bit_cast(float, (unsigned)w[i]);
        bool logs = false;
#pragma unroll
        for (int i = 0; i < kBatch; ++i) logs = logs || (int)(w[i] >> 32) < 0;
        if (__builtin_amdgcn_ballot_w64(logs || m != 0.f) == 0) {
#pragma unroll
          for (int i = 0; i < kBatch; ++i) acc += v[i];
          continue;
        }
#pragma unroll
        for (int i = 0; i < kBatch; ++i)
          if ((int)(w[i] >> 32) >= 0) v[i] = fast_log2(v[i]);   // (0: -inf, adds nothing)
        float bm = v[0];
#pragma unroll
        for (int i = 1; i < kBatch; ++i) bm = fmaxf(bm, v[i]);
#pragma unroll
        for (int i = 0; i < kBatch; ++i) nan = nan || (v[i] != v[i]);
        if (acc == 0.f) m = kNegInf;   // nothing yet
        const float nm = fmaxf(m, bm);
        if (nm > kNegInf) {
          acc *= fast_exp2(m - nm);   // m = -inf: acc is 0 and stays 0
#pragma unroll
          for (int i = 0; i < kBatch; ++i) acc += fast_exp2(v[i] - nm);
          m = nm;
        }
      }
      if (!ok) {
        __hip_atomic_store(p.sync, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        flag[1] = 0;
      }
      // a NaN partial (fmaxf drops it) makes the row's lse NaN
      if (row_here) {
        mrg[(sub * kRowsWg + 64 * rgroup + lane) * 2] = nan ? __builtin_nanf("") : m;
        mrg[(sub * kRowsWg + 64 * rgroup + lane) * 2 + 1] = acc;
      }
    }
    lds_barrier();
    if (tid < kRowsWg) {
      float mv[kMergeWaves], av[kMergeWaves];
#pragma unroll
      for (int w = 0; w < kMergeWaves; ++w) {
        const float2 ma = *reinterpret_cast<const float2*>(mrg + (w * kRowsWg + tid) * 2);
        mv[w] = ma.x;
        av[w] = ma.y;
      }
      bool plain = true;
#pragma unroll
      for (int w = 0; w < kMergeWaves; ++w) plain = plain && mv[w] == 0.f;
      float lse, factor;
      if (__builtin_amdgcn_ballot_w64(!plain) == 0) {
        float sum = av[0];
#pragma unroll
        for (int w = 1; w < kMergeWaves; ++w) sum += av[w];
        lse = log2_of_sum(sum);
        factor = __builtin_amdgcn_rcpf(sum);
      } else {
        float m = kNegInf;
        bool nan = false;
#pragma unroll
        for (int w = 0; w < kMergeWaves; ++w) {
          nan = nan || (mv[w] != mv[w]);
          m = fmaxf(m, av[w] == 0.f ? kNegInf : mv[w]);   // (a wave without a slot has nothing to say)
        }
        const float ref = (m > kNegInf) ? m : 0.f;
        float acc = 0.f;
#pragma unroll
        for (int w = 0; w < kMergeWaves; ++w) acc += av[w] == 0.f ? 0.f : av[w] * fast_exp2(mv[w] - ref);
        lse = nan ? __builtin_nanf("") : ((m > kNegInf) ? m + fast_log2(acc) : kNegInf);
        factor = lse != kNegInf ? fast_exp2(-lse) : 0.f;
      }
      // what step 4 adds to a score, or multiplies 2^score by (nothing for rows that do not exist)
      // (a NaN lse stays a NaN factor: the row's visible columns become NaN, as in the other kernels)
      if (keep_scores) rowv[tid] = tid < p.M ? -lse : odd_padding ? __builtin_nanf("") : kNegInf;
      else rowv[tid] = tid < p.M ? factor : 0.f;
      if (split == 0 && tid < p.M) p.lse[(int64_t)bh * p.M + tid] = lse;   // (not meaningful if the team was not met)
    }
    lds_barrier();
    met = flag[1] != 0;
    if (tid == 0) flag[0] = 0;
    if (!met) spin_limit = min(spin_limit, 64);   // the call has failed: later waits of this workgroup are short
    // 4. probabilities, reduced down the rows
    f32x4 nl[NQ];
#pragma unroll
    for (int g = 0; g < NQ; ++g) nl[g] = *reinterpret_cast<const f32x4*>(rowv + 64 * qh + 16 * g + qrow);
    // What is hidden is 0 (sums) or -inf in the registers and stays so beside rows whose value is below infinity: no masks, then.
    bool odd = false;
#pragma unroll
    for (int g = 0; g < NQ; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) odd = odd || !(nl[g][r] < kPosInf);
    const bool plain_rows = __builtin_amdgcn_ballot_w64(odd) == 0;
    float* const osum = obuf + qh * (kRes * kBatchKeys);
    float* const omax = osum + (MODE == kModeBoth ? kBatchKeys : 0);
    int c0b = c0;
    asm volatile("" : "+s"(c0b));
    auto columns = [&](auto batch_tag) __attribute__((always_inline)) {   // eight steps at a time through the column buffer
    constexpr int bt = decltype(batch_tag)::value;
    float vs[kFusedSteps], vm[kFusedSteps];   // per step: the lane's key, reduced over the lane's queries
    // The usual cases, without a question per step.  (Per call, step by step and so, in the geometric mean of 13500 shapes: maxima of up to 64 queries 0.76, of
    // up to 128 0.81, both 0.82 and 0.86, sums, which asked wherever the mask cut a workgroup's keys, 0.93 and 0.95: 512 pairs of 64 x 16384 x 128
    // fp16 399 -> 384 us, 32 of 128 x 4096 17.7 -> 16.9.  Part of it is that sweeps that keep scores hide no rows of padding any more.)
    if (MODE != kModeSum && plain_rows) {
#pragma unroll
      for (int jj = 0; jj < kFusedSteps; ++jj) {
        f32x4 part = {0.f, 0.f, 0.f, 0.f};
        float vmax = kNegInf;
#pragma unroll
        for (int g = 0; g < NQ; ++g) {
          const f32x4 x = sc[bt * kFusedSteps + jj][g] + nl[g];
          vmax = fmaxf(fmaxf(vmax, x[0]), x[1]);
          vmax = fmaxf(fmaxf(vmax, x[2]), x[3]);
          if (MODE == kModeBoth) {
#pragma unroll
            for (int r = 0; r < 4; ++r) part[r] += fast_exp2(x[r]);
          }
        }
        vs[jj] = (part[0] + part[1]) + (part[2] + part[3]);
        vm[jj] = vmax;
      }
    } else if (MODE == kModeSum && !keep_scores && plain_rows) {   // 3000 -> 1100 cycles on 1024 keys and 64 queries
#pragma unroll
      for (int jj = 0; jj < kFusedSteps; ++jj) {
        f32x4 part = sc[bt * kFusedSteps + jj][0] * nl[0];
#pragma unroll
        for (int g = 1; g < NQ; ++g)
#pragma unroll
          for (int r = 0; r < 4; ++r) part[r] = fmaf(sc[bt * kFusedSteps + jj][g][r], nl[g][r], part[r]);
        vs[jj] = (part[0] + part[1]) + (part[2] + part[3]);
      }
    } else {
#pragma unroll
    for (int jj = 0; jj < kFusedSteps; ++jj) {
      const int j = bt * kFusedSteps + jj;
      const int kbase = (c0b + j * KH + kh) * kChunk;
      const int key = kbase + 16 * wq + (lane & 15);
      const bool need_mask = (keep_scores && ragged_rows) || kbase + kChunk > p.N || (CAUSAL && kbase + kChunk - 1 > p.c + 64 * qh);
      f32x4 part = {0.f, 0.f, 0.f, 0.f};   // four independent chains
      float vmax = kNegInf;
      if (MODE == kModeSum && !keep_scores) {   // the registers hold 2^score, nl holds 2^-lse
        if (need_mask) {
          int first = CAUSAL ? key - p.c - 64 * qh - qrow : -(1 << 30);
          if (key >= p.N) first = 1 << 30;
#pragma unroll
          for (int g = 0; g < NQ; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int o = 16 * g + r;
              part[r] += (o >= first && o < mlim) ? sc[j][g][r] * nl[g][r] : 0.f;
            }
        } else {
#pragma unroll
          for (int g = 0; g < NQ; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[r] = fmaf(sc[j][g][r], nl[g][r], part[r]);
        }
      } else if (need_mask) {   // hidden entries stay hidden from a row whose lse is not a number
        int first = CAUSAL ? key - p.c - 64 * qh - qrow : -(1 << 30);
        if (key >= p.N) first = 1 << 30;
#pragma unroll
        for (int g = 0; g < NQ; ++g)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int o = 16 * g + r;
            const float x = (o >= first && o < mlim) ? sc[j][g][r] + nl[g][r] : kNegInf;
            if (MODE != kModeSum) vmax = fmaxf(vmax, x);
            if (MODE != kModeMax) part[r] += fast_exp2(x);
          }
      } else {
#pragma unroll
        for (int g = 0; g < NQ; ++g)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float x = sc[j][g][r] + nl[g][r];
            if (MODE != kModeSum) vmax = fmaxf(vmax, x);
            if (MODE != kModeMax) part[r] += fast_exp2(x);
          }
      }
      vs[jj] = (part[0] + part[1]) + (part[2] + part[3]);
      vm[jj] = vmax;
    }
    }
    // the four rows of lanes hold different queries of the same key: a reduce-scatter, after which row rho of lanes has
    // steps 2 rho and 2 rho + 1
    const int at = ((lane >> 4) * 2 * KH + kh) * kChunk + 16 * wq + (lane & 15);
    if (MODE != kModeMax) {
      lane_rows_scatter<false>(vs);
      osum[at] = vs[0];
      osum[at + KH * kChunk] = vs[1];
    }
    if (MODE != kModeSum) {
      lane_rows_scatter<true>(vm);
      omax[at] = fast_exp2(vm[0]);
      omax[at + KH * kChunk] = fast_exp2(vm[1]);
    }
    if (bt + 1 < kBatches) {   // the next batch writes the buffer again
      lds_barrier();
      store_columns(bh, bt, met);
      lds_barrier();
    }
    };
    columns(std::integral_constant<int, 0>());
    if constexpr (kBatches == 2) columns(std::integral_constant<int, 1>());
    waiting = true;
    // the next writers of obuf, red, rowv and flag are behind the ring barriers of the next pair
  }
  ring_sync<0>();   // the loads past the last chunk write their zeros before the LDS is given back
  if (waiting) store_columns(team + (rounds - 1) * T, kBatches - 1, met);
}

// ---------------------------------------------------------------------------------------------
// One query (a decoded token): every score is used by one row only, so there is nothing for a tile to share and
// the call is the reading of the keys.  Workgroups stream disjoint ranges of keys from memory straight into
// registers, LPR lanes per key row and 16 bytes per lane and load, multiply on the vector unit in fp32, and
// leave the raw products (4 bytes per key, against a row of 16 to 1024) and one (maximum, sum) of 2^score in
// scratch; a second launch merges those pairs and stores the columns.  No workgroup waits for another, and a key
// meets no matrix instruction with fifteen rows of padding.
// Bound by HBM: eight loads of 1 KiB are in flight per wave and eight waves per SIMD (64 registers, hence the launch
// bound); the 26 vector instructions per load take a fifth of its time.  256 pairs of 9001 keys of 128 bf16: 146 us
// with the single sweep -> 102 us, 5.8 TB/s of keys (a large copy on the same card: 5.2; 112 us with loads that
// are not marked non-temporal); what the single sweep does not take gains more: 80 x 30011 x 256 bf16 448 -> 220,
// 64 x 16384 x 192 fp32 696 -> 127, 256 x 4096 x 64 fp32 207 -> 46, and at the small end 8 x 1024 x 128 14.4 -> 10,
// 512 x 128 x 128 11.2 -> 9.5, 2 x 64 x 64 10.3 -> 9.6.
constexpr int kOneLoads = 8;
constexpr int kOneCols = 4;   // columns per thread of the second launch

// (m, l) stands for l * 2^m, the sum of 2^score over the keys seen so far; m is their maximum, -inf before the
// first one.  A NaN or +inf score makes l a NaN, for good.
__device__ __forceinline__ void one_query_merge(float& m, float& l, float m2, float l2) {
  const float mx = fmaxf(m, m2);
  const float ref = (mx == kNegInf) ? 0.f : mx;
  l = l * fast_exp2(m - ref) + l2 * fast_exp2(m2 - ref);
  m = mx;
}
__device__ __forceinline__ void one_query_merge_wave(float& m, float& l) {
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const float m2 = __shfl_xor(m, d), l2 = __shfl_xor(l, d);
    one_query_merge(m, l, m2, l2);
  }
}

// Sum over each aligned group of LPR lanes, in all of its lanes.
template <int LPR>
__device__ __forceinline__ float group_sum(float v) {
  if constexpr (LPR >= 2) v += dpp_row<0xB1>(v);     // quad_perm [1,0,3,2]
  if constexpr (LPR >= 4) v += dpp_row<0x4E>(v);     // quad_perm [2,3,0,1]
  if constexpr (LPR >= 8) v += dpp_row<0x141>(v);    // row_half_mirror
  if constexpr (LPR >= 16) v += dpp_row<0x140>(v);   // row_mirror
  if constexpr (LPR >= 32) v += __shfl_xor(v, 16);
  if constexpr (LPR >= 64) v += __shfl_xor(v, 32);
  return v;
}

// one_query_merge over each aligned group of LPR lanes: the maximum first, then every sum is scaled once and the scaled ones
// are added pairwise.
template <int LPR>
__device__ __forceinline__ void one_query_join(float& m, float& l) {
  float mx = m;
#pragma unroll
  for (int d = 1; d < LPR; d <<= 1) mx = fmaxf(mx, __shfl_xor(mx, d));
  l = group_sum<LPR>(l * fast_exp2(m - ((mx == kNegInf) ? 0.f : mx)));
  m = mx;
}

// The elements of a 16-byte granule as floats.
template <int DT>
__device__ __forceinline__ void granule_floats(u32x4 v, float (&f)[DT == FCR_DTYPE_F32 ? 4 : 8]) {
  if constexpr (DT == FCR_DTYPE_F32) {
    const f32x4 x = __builtin_bit_cast(f32x4, v);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = x[e];
  } else if constexpr (DT == FCR_DTYPE_F16) {
    const f16x8 x = __builtin_bit_cast(f16x8, v);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = (float)x[e];
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[2 * e] = __builtin_bit_cast(float, v[e] << 16);
      f[2 * e + 1] = __builtin_bit_cast(float, v[e] & 0xffff0000u);
    }
  }
}

// A workgroup takes keys [split * rows_wg, + rows_wg) of one pair, all ranges of a pair in a row, or with p.group > 1
// the same range of all p.group = B batch entries of a head in a row.  scores: [BH, pitch].  ONCE: no other pair reads
// these keys (both: see launch_one_query).
template <int DT, int LPR, bool ONCE>
__global__ __launch_bounds__(256, 8) void one_query_scores_kernel(const Params p, float* __restrict__ scores,
                                                               int64_t pitch, int rows_wg) {
  constexpr int E = DT == FCR_DTYPE_F32 ? 4 : 8;
  constexpr int kRows = 64 / LPR;                               // key rows per load
  constexpr int kSel = kOneLoads > LPR ? kOneLoads / LPR : 1;   // finished scores per lane and step
  constexpr int kStep = kOneLoads * kRows;                      // key rows per wave and step
  __shared__ float wave_m[4], wave_l[4];
  const int lane = threadIdx.x & 63, g = lane & (LPR - 1), r0 = lane / LPR;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int turn = (int)blockIdx.x / p.group, member = (int)blockIdx.x - turn * p.group;
  const int pair = turn / p.splits, split = turn - pair * p.splits;
  const int bh = p.group > 1 ? member * p.H + pair : pair;
  const int b = bh / p.H, h = bh - b * p.H;
  const char* kb = p.k + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh + (int64_t)g * 16;
  const char* qb = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)g * 16;
  const bool live = g < p.dgran;   // the lanes past the end of a row neither load nor count
  const u32x4 zero = {0u, 0u, 0u, 0u};
  float qf[E];
  granule_floats<DT>(live ? *reinterpret_cast<const u32x4*>(qb) : zero, qf);
  const int first = split * rows_wg, end = min(p.N, first + rows_wg);
  float* out = scores + (int64_t)bh * pitch;
  float m = kNegInf, l = 0.f;
  for (int row = first + wave * kStep; row < end; row += 4 * kStep) {
    u32x4 v[kOneLoads];
#pragma unroll
    for (int u = 0; u < kOneLoads; ++u) {
      const u32x4* src = reinterpret_cast<const u32x4*>(kb + (int64_t)min(row + u * kRows + r0, p.N - 1) * p.k_sr);
      v[u] = zero;
      if (live) {
        if constexpr (ONCE) v[u] = __builtin_nontemporal_load(src);
        else v[u] = *src;
      }
    }
    float done[kSel];
#pragma unroll
    for (int i = 0; i < kSel; ++i) done[i] = 0.f;
#pragma unroll
    for (int u = 0; u < kOneLoads; ++u) {
      float f[E], s = 0.f;
      granule_floats<DT>(v[u], f);
#pragma unroll
      for (int e = 0; e < E; ++e) s = fmaf(f[e], qf[e], s);
      s = group_sum<LPR>(s);
      if (g == (u & (LPR - 1))) done[u / LPR] = s;   // lane g of a group keeps load g's row (and every LPR-th after it)
    }
#pragma unroll
    for (int i = 0; i < kSel; ++i) {
      const int r = row + (i * LPR + g) * kRows + r0;
      if (i * LPR + g < kOneLoads && r < end) {
        out[r] = done[i];
        one_query_merge(m, l, done[i] * p.scale2, 1.f);
      }
    }
  }
  one_query_merge_wave(m, l);
  if (lane == 0) {
    wave_m[wave] = m;
    wave_l[wave] = l;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < 4; ++w) one_query_merge(m, l, wave_m[w], wave_l[w]);
    float* part = p.part + 2 * ((int64_t)bh * p.splits + split);
    part[0] = m;
    part[1] = l;
  }
}

// p.tiles workgroups of 256 * kOneCols columns per pair; also the row statistic and the status word (p.sync, if any).
template <int MODE>
__global__ __launch_bounds__(256) void one_query_columns_kernel(const Params p, const float* __restrict__ scores,
                                                                int64_t pitch) {
  __shared__ float wave_m[4], wave_l[4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int bh = (int)blockIdx.x / p.tiles, tile = (int)blockIdx.x - bh * p.tiles;
  const int col0 = tile * 256 * kOneCols + tid;
  const float* src = scores + (int64_t)bh * pitch;
  float a[kOneCols];
#pragma unroll
  for (int i = 0; i < kOneCols; ++i) a[i] = src[min(col0 + 256 * i, p.N - 1)];
  float m = kNegInf, l = 0.f;
  const float* part = p.part + 2 * (int64_t)bh * p.splits;
  // Few pairs have many ranges each; the four waves then take a quarter of them instead of all: 2 x 262144 x 128 bf16
  // 33.4 -> 26.7 us per call (single sweep 31.8), 1 x 10^6 x 128 79 -> 52.
  const bool many = p.splits > 64;
  for (int s = many ? tid : lane; s < p.splits; s += many ? 256 : 64) one_query_merge(m, l, part[2 * s], part[2 * s + 1]);
  one_query_merge_wave(m, l);
  if (many) {
    if (lane == 0) {
      wave_m[tid >> 6] = m;
      wave_l[tid >> 6] = l;
    }
    __syncthreads();
    m = wave_m[0];
    l = wave_l[0];
#pragma unroll
    for (int w = 1; w < 4; ++w) one_query_merge(m, l, wave_m[w], wave_l[w]);
  }
  if (tile == 0 && tid == 0) p.lse[bh] = m + fast_log2(l);
  if (blockIdx.x == 0 && tid == 0 && p.sync) *p.sync = 0u;
  const float ref = (m == kNegInf) ? 0.f : m, inv = 1.0f / l;   // no score above -inf: 0 * inf, NaN sums
#pragma unroll
  for (int i = 0; i < kOneCols; ++i) {
    const int key = col0 + 256 * i;
    const float v = fast_exp2(fmaf(a[i], p.scale2, -ref)) * inv;
    if (key < p.N) {
      if (MODE != kModeMax) store_column(p, p.out, true, bh, key, v);
      if (MODE != kModeSum) store_column(p, MODE == kModeBoth ? p.out2 : p.out, false, bh, key, fmaxf(v, 0.f));   // drops a NaN
    }
  }
}

// The whole of it in one launch, a workgroup per pair, whose raw products wait in LDS (one_query_alone has where and why).  A CU
// alone has 16 waves with eight to sixteen loads of 1 KiB in flight and reads about 70 bytes per ns; with a workgroup on every CU the
// memory is the limit again.
constexpr int kOnePairThreads = 1024;
constexpr int kOnePairKeys = 8192;   // 32 KiB of products

template <int DT, int LPR>
__global__ __launch_bounds__(kOnePairThreads) void one_query_pair_kernel(const Params p, int mode) {
  constexpr int E = DT == FCR_DTYPE_F32 ? 4 : 8;
  constexpr int kRows = 64 / LPR;                               // key rows per load
  constexpr int kSel = kOneLoads > LPR ? kOneLoads / LPR : 1;   // finished scores per lane and step
  constexpr int kStep = kOneLoads * kRows;                      // key rows per wave and step
  constexpr int kW = kOnePairThreads / 64;
  __shared__ float scores[kOnePairKeys];
  __shared__ float wave_m[kW], wave_l[kW];
  const int tid = threadIdx.x, lane = tid & 63, g = lane & (LPR - 1), r0 = lane / LPR;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bh = (int)blockIdx.x, b = bh / p.H, h = bh - b * p.H;
  const char* kb = p.k + (int64_t)b * p.k_sb + (int64_t)h * p.k_sh + (int64_t)g * 16;
  const char* qb = p.q + (int64_t)b * p.q_sb + (int64_t)h * p.q_sh + (int64_t)g * 16;
  const bool live = g < p.dgran;   // the lanes past the end of a row neither load nor count
  const u32x4 zero = {0u, 0u, 0u, 0u};
  float qf[E];
  granule_floats<DT>(live ? *reinterpret_cast<const u32x4*>(qb) : zero, qf);
  float m = kNegInf, l = 0.f;
  auto load = [&](u32x4(&v)[kOneLoads], int row) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kOneLoads; ++u) {
      v[u] = zero;
      if (live) v[u] = *reinterpret_cast<const u32x4*>(kb + (int64_t)min(row + u * kRows + r0, p.N - 1) * p.k_sr);
    }
  };
  auto take = [&](const u32x4(&v)[kOneLoads], int row) __attribute__((always_inline)) {
    float done[kSel];
#pragma unroll
    for (int i = 0; i < kSel; ++i) done[i] = 0.f;
#pragma unroll
    for (int u = 0; u < kOneLoads; ++u) {
      float f[E], s = 0.f;
      granule_floats<DT>(v[u], f);
#pragma unroll
      for (int e = 0; e < E; ++e) s = fmaf(f[e], qf[e], s);
      s = group_sum<LPR>(s);
      if (g == (u & (LPR - 1))) done[u / LPR] = s;   // lane g of a group keeps load g's row (and every LPR-th after it)
    }
#pragma unroll
    for (int i = 0; i < kSel; ++i) {
      const int r = row + (i * LPR + g) * kRows + r0;
      if (i * LPR + g < kOneLoads && r < p.N) {
        scores[r] = done[i];
        one_query_merge(m, l, done[i] * p.scale2, 1.f);
      }
    }
  };
  // a step ahead: the next keys are on their way while these are multiplied
  constexpr int kPass = kW * kStep;
  u32x4 va[kOneLoads], vb[kOneLoads];
  int row = wave * kStep;
  if (row < p.N) load(va, row);
  for (; row < p.N; row += 2 * kPass) {
    if (row + kPass < p.N) load(vb, row + kPass);
    take(va, row);
    if (row + kPass >= p.N) break;
    if (row + 2 * kPass < p.N) load(va, row + 2 * kPass);
    take(vb, row + kPass);
  }
  // Merging the waves one after the other rescales and rounds the sum fifteen times.
  one_query_join<64>(m, l);
  if (lane == 0) {
    wave_m[wave] = m;
    wave_l[wave] = l;
  }
  __syncthreads();
  m = wave_m[lane & (kW - 1)];
  l = wave_l[lane & (kW - 1)];
  one_query_join<kW>(m, l);
  if (tid == 0) p.lse[bh] = m + fast_log2(l);
  if (bh == 0 && tid == 0 && p.sync) *p.sync = 0u;
  const float ref = (m == kNegInf) ? 0.f : m, inv = 1.0f / l;   // as one_query_columns_kernel
  for (int key = tid; key < p.N; key += kOnePairThreads) {
    const float v = fast_exp2(fmaf(scores[key], p.scale2, -ref)) * inv;
    if (mode != kModeMax) store_column(p, p.out, true, bh, key, v);
    if (mode != kModeSum) store_column(p, mode == kModeBoth ? p.out2 : p.out, false, bh, key, fmaxf(v, 0.f));   // drops a NaN
  }
}

// ---------------------------------------------------------------------------------------------
// fp32 operands packed by the caller.  x = hi + lo with hi = fp16(x), lo = fp16(x - hi) carries 22 bits of x.  Packing
// queries as [hi | hi | lo] and keys as [hi | lo | hi] along d makes the fp16 kernels compute
// q_hi.k_hi + q_hi.k_lo + q_lo.k_hi, the product to about 2^-22 (the lo.lo term is dropped), with fp32
// accumulation.  With terms == 1 only [hi] is written (both operands rounded to fp16).
// dst rows are terms * dpad halves, each segment zero padded from D to dpad.
__global__ __launch_bounds__(256) void pack_f32_kernel(const float* __restrict__ src, _Float16* __restrict__ dst,
                                                       int64_t rows, int D, int dpad, int terms, int is_key) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= rows * dpad) return;
  const int64_t row = idx / dpad;
  const int d = (int)(idx - row * dpad);
  const float x = (d < D) ? src[row * D + d] : 0.f;
  const _Float16 hi = (_Float16)x;
  _Float16* out = dst + row * (int64_t)(terms * dpad) + d;
  out[0] = hi;
  if (terms == 3) {
    const _Float16 lo = (_Float16)(x - (float)hi);
    out[dpad] = is_key ? lo : hi;
    out[2 * dpad] = is_key ? hi : lo;
  }
}

// ---------------------------------------------------------------------------------------------
// Keep-mask of the k largest scores of every row (what a pruning caller does with the reduced
// columns).  Floats are mapped to integers of the same order and the key T of the k-th largest element is
// found from the top down; keys equal to T are kept from the lowest column up until k are kept.
//
// Rows that fit the registers of one workgroup (topk_mask_kernel): the row is read once, 16 bytes per lane and
// load, and its keys stay in registers.  T is found by narrowing: the keys between the smallest and the
// largest one are counted in 2 * T equal bins in LDS, the bin that holds the k-th largest one becomes the
// range of the next count, and as soon as a bin holds few enough keys they are gathered and ranked against
// each other.  A count takes 11 bits of the range (9 in the smaller workgroup), so at most three (four) are
// needed, and one or two are for scores that are spread at all.  The search bit by bit that stood
// here before took 34 passes of one barrier each and read the rows with every lane on a line of its own; this
// one is bound by the vector instructions over the keys and the latency of eight or so barriers.  Kernel time, 32 rows:
// 1024 columns fp32 11.9 -> 4.2 us, 8192 fp32 14.7 -> 5.8, fp16 18.6 -> 6.1, 32768 fp32 31.2 -> 14.3, fp16 44.3 -> 14.5;
// with nine columns in ten equal 15.5 -> 7.7 (8192 fp32) and 31.8 -> 20.9 (32768 fp32).
// Longer rows without scratch (topk_mask_long_kernel) are re-read from memory in every pass, so T is found
// eight bits at a time from a 256-bin histogram in LDS; a wave whose keys all fall into one bin (the usual
// case for the top digits) adds its count with one atomic.
__device__ __forceinline__ uint32_t order_key(float x) {
  uint32_t b = __builtin_bit_cast(uint32_t, x);
  if (b == 0x80000000u) b = 0u;  // -0 and +0 are one value
  if ((b & 0x7fffffffu) > 0x7f800000u) return 0xffffffffu;  // a NaN of either sign: one value above +inf (torch.topk's order)
  return b ^ ((uint32_t)((int32_t)b >> 31) | 0x80000000u);  // monotone in x for all non-NaN floats
}

// Score rows come as fp32, fp16 or bf16 (what the column kernels store); keys are taken from the widened
// value, which is exact, so order and ties are those of the stored values.
template <typename ET> __device__ __forceinline__ float widen(ET x) { return (float)x; }
template <> __device__ __forceinline__ float widen<uint16_t>(uint16_t x) {   // bf16 bits
  return __builtin_bit_cast(float, (uint32_t)x << 16);
}
__device__ __forceinline__ float key_value(uint32_t key) {
  return __builtin_bit_cast(float, (key & 0x80000000u) ? (key ^ 0x80000000u) : ~key);
}

constexpr int kTopkThreads = 1024;
constexpr int kTopk16Columns = 64 * kTopkThreads;   // of a 16-bit row that one workgroup selects from in one launch

// Sum of v over the 64 lanes, as a wave-uniform value: butterflies inside rows of 16 lanes, then the row
// totals are passed on to the rows behind and lane 63 holds the total.
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, true);    // quad_perm [1,0,3,2]
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, true);    // quad_perm [2,3,0,1]
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true);   // row_half_mirror
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, true);   // row_mirror: every lane has its row's sum
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// Largest v over the 64 lanes, as a wave-uniform value.
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xf, 0xf, true));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xf, 0xf, true));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xf, 0xf, true));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xf, 0xf, true));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false));
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// Inclusive prefix sums over the 64 lanes.
__device__ __forceinline__ uint32_t wave_scan(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);   // row_shr 1, 2, 4, 8
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true);
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15 into rows 1 and 3
  v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31 into rows 2 and 3
  return v;
}

// Exclusive rank of this thread's first tie among the ties of the row, by column, given that thread t
// owns a contiguous run of columns and has `mine` ties.
__device__ __forceinline__ uint32_t ties_before(uint32_t mine, uint32_t* wave_eq, int lane, int wave) {
  const uint32_t incl = wave_scan(mine);
  if (lane == 63) wave_eq[wave] = incl;
  __syncthreads();
  uint32_t before = incl - mine;
  for (int w = 0; w < wave; ++w) before += wave_eq[w];
  return before;
}

// A row of at most T * VPT columns in the registers of one workgroup: thread t holds W consecutive columns
// from (j * T + t) * W on, for j < VPT / W, so loads (16 bytes per lane) and stores (W bytes) are dense.
template <int T, int VPT>
__global__ __launch_bounds__(T) void topk_mask_kernel(const float* __restrict__ scores, uint8_t* __restrict__ mask,
                                                      float* __restrict__ threshold, int N, int k) {
  constexpr int kW = T / 64;
  constexpr int W = 4;
  constexpr int J = VPT / W;
  constexpr int kBins = 2 * T, kBinBits = __builtin_ctz(kBins);
  // Keys that are ranked against each other, one per thread.  Ranking takes time with the square of their number, one more
  // count with VPT; rows of which one value fills the bin need no more than its minimum and maximum.  With 512 for
  // both -> now (search bit by bit), 500 equal values around the k-th: 812 rows of 4666 fp32 61 -> 21 us (42), 32 of 4666
  // 17.2 -> 11.2 (15.3), 1024 of 8192 65 -> 24 (43), 1024 of 32768 117 -> 74 (155).  exp(N(0, 1)) scores of every type never reach
  // the limits; uniform ones with one near zero do: 512 rows of 16384 48 -> 36.  Just above them the count is the dearer way:
  // 200 equal values in 1024 rows of 32768 88 -> 95.
  constexpr int kGather = VPT > 8 ? 256 : 128;
  static_assert(VPT % W == 0, "whole vectors");
  __shared__ __attribute__((aligned(16))) uint32_t hist[kBins];
  __shared__ __attribute__((aligned(16))) uint32_t cand[kGather];
  __shared__ uint32_t wave_a[kW], wave_b[kW];
  __shared__ uint32_t block_ties[J * kW];
  __shared__ uint32_t sh_bin, sh_above, sh_count, sh_key, sh_need, sh_ties, sh_gathered;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* s = scores + (int64_t)blockIdx.x * N;
  uint8_t* m = mask + (int64_t)blockIdx.x * N;
  const uint32_t kk = (uint32_t)min(max(k, 0), N);

  // Keys; 0 stands for a column past N (no key is 0: -inf, the smallest value, has a positive one).
  uint32_t u[VPT];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int col = (j * T + tid) * W;
    float v[W];
    if (col + W <= N) {
      __builtin_memcpy(v, s + col, 16);   // one load whatever the row's alignment
#pragma unroll
      for (int e = 0; e < W; ++e) u[j * W + e] = order_key(v[e]);
    } else {
#pragma unroll
      for (int e = 0; e < W; ++e) u[j * W + e] = (col + e < N) ? order_key(s[col + e]) : 0u;
    }
  }

  for (int i = tid; i < kBins; i += T) hist[i] = 0u;
  if (tid == 0) sh_gathered = 0u;
  uint32_t lo = 1u, range = 0xfffffffeu; // the k-th largest key is in [lo, lo + range]
  uint32_t need = kk;                    // and is the need-th largest of the `ties` keys in there
  uint32_t key = 0xffffffffu, ties = 0u; // k <= 0: nothing is kept
  while (kk > 0) {
    // the smallest and the largest key of the range (the smallest through its complement, where 0 is neutral)
    uint32_t hi = 0u, nlo = 0u;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const bool in = u[i] - lo <= range;
      hi = max(hi, in ? u[i] : 0u);
      nlo = max(nlo, in ? ~u[i] : 0u);
    }
    hi = wave_max(hi);
    nlo = wave_max(nlo);
    if (lane == 0) {
      wave_a[wave] = hi;
      wave_b[wave] = nlo;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kW; ++w) {
      hi = max(hi, wave_a[w]);
      nlo = max(nlo, wave_b[w]);
    }
    lo = ~nlo;
    range = hi - lo;
    if (range == 0u && ties > 0u) {   // one value many times over
      key = lo;
      break;
    }
    const int bits = range ? 32 - __builtin_clz(range) : 0;
    const int shift = max(bits - kBinBits, 0);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      // A bin that many lanes share (zeros, ties) serializes their atomics.  Where the first column of a vector shows
      // that, the lanes that agree with the first live one add theirs together, key by key; doing so always
      // costs 5 us on rows of 32768 columns.
      const bool in0 = u[j * W] - lo <= range;
      const uint64_t live0 = __builtin_amdgcn_ballot_w64(in0);
      const uint32_t bin0 = (u[j * W] - lo) >> shift;
      const uint32_t lead0 = __builtin_amdgcn_readlane(bin0, live0 ? __builtin_ctzll(live0) : 0);
      if (__builtin_popcountll(__builtin_amdgcn_ballot_w64(in0 && bin0 == lead0)) <= 8) {
#pragma unroll
        for (int e = 0; e < W; ++e) {
          const uint32_t d = u[j * W + e] - lo;
          if (d <= range) atomicAdd(&hist[d >> shift], 1u);
        }
      } else {
#pragma unroll
        for (int e = 0; e < W; ++e) {
          const uint32_t d = u[j * W + e] - lo, bin = d >> shift;
          const bool in = d <= range;
          const uint64_t live = __builtin_amdgcn_ballot_w64(in);
          const uint32_t lead = __builtin_amdgcn_readlane(bin, live ? __builtin_ctzll(live) : 0);
          const uint64_t same = __builtin_amdgcn_ballot_w64(in && bin == lead);
          if (same != 0 && lane == __builtin_ctzll(same)) atomicAdd(&hist[bin], (uint32_t)__builtin_popcountll(same));
          if (in && bin != lead) atomicAdd(&hist[bin], 1u);
        }
      }
    }
    __syncthreads();
    // thread t takes bins kBins - 1 - 2t and the one below: prefix sums are counts from the top
    const uint32_t h0 = hist[kBins - 1 - 2 * tid], h1 = hist[kBins - 2 - 2 * tid];
    const uint32_t incl = wave_scan(h0 + h1);
    if (lane == 63) wave_a[wave] = incl;
    __syncthreads();
    uint32_t above = incl - h0 - h1;
#pragma unroll
    for (int w = 0; w < kW; ++w) above += (w < wave) ? wave_a[w] : 0u;
    if (above < need && above + h0 >= need) {
      sh_bin = (uint32_t)(kBins - 1 - 2 * tid);
      sh_above = above;
      sh_count = h0;
    } else if (above + h0 < need && above + h0 + h1 >= need) {
      sh_bin = (uint32_t)(kBins - 2 - 2 * tid);
      sh_above = above + h0;
      sh_count = h1;
    }
    hist[kBins - 1 - 2 * tid] = 0u;
    hist[kBins - 2 - 2 * tid] = 0u;
    __syncthreads();
    ties = sh_count;
    need -= sh_above;
    lo += sh_bin << shift;
    range = min((1u << shift) - 1u, 0xffffffffu - lo);   // (past 2^32 it would take in the padding)
    if (shift == 0) {
      key = lo;
      break;
    }
    if (ties <= (uint32_t)kGather) {
      const uint32_t count = ties;
#pragma unroll
      for (int i = 0; i < VPT; ++i)
        if (u[i] - lo <= range) cand[atomicAdd(&sh_gathered, 1u)] = u[i];
      __syncthreads();
      if (tid < (int)count) {
        const uint32_t mine = cand[tid];
        uint32_t gt = 0, eq = 0;
        for (uint32_t i = 0; i < count; ++i) {
          const uint32_t o = cand[i];
          gt += o > mine ? 1u : 0u;
          eq += o == mine ? 1u : 0u;
        }
        if (gt < need && gt + eq >= need) {   // the same for every key that ties with it
          sh_key = mine;
          sh_need = need - gt;
          sh_ties = eq;
        }
      }
      __syncthreads();
      key = sh_key;
      need = sh_need;
      ties = sh_ties;
      break;
    }
  }
  // `key` is the key of the k-th largest element; `need` of the `ties` keys equal to it are kept
  if (tid == 0 && threshold) threshold[blockIdx.x] = key_value(key);

  const bool drop_ties = need < ties;   // uniform: some ties are dropped, rank them by column
  if (drop_ties) {
    // ties per block of 64 * W columns, in column order, then their exclusive prefix sums
#pragma unroll
    for (int j = 0; j < J; ++j) {
      uint32_t c = 0;
#pragma unroll
      for (int e = 0; e < W; ++e) c += u[j * W + e] == key ? 1u : 0u;
      c = wave_sum(c);
      if (lane == 0) block_ties[j * kW + wave] = c;
    }
    __syncthreads();
    if (wave == 0) {
      uint32_t base = 0;
      for (int i0 = 0; i0 < J * kW; i0 += 64) {
        const uint32_t c = (i0 + lane < J * kW) ? block_ties[i0 + lane] : 0u;
        const uint32_t incl = wave_scan(c);
        if (i0 + lane < J * kW) block_ties[i0 + lane] = base + incl - c;
        base += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int col = (j * T + tid) * W;
    uint32_t rank = 0u;   // ties in front of this thread's columns
    if (drop_ties) {
      uint32_t mine = 0;
#pragma unroll
      for (int e = 0; e < W; ++e) mine += u[j * W + e] == key ? 1u : 0u;
      rank = block_ties[j * kW + wave] + wave_scan(mine) - mine;
    }
    uint8_t out[W];
#pragma unroll
    for (int e = 0; e < W; ++e) {
      const bool eq = u[j * W + e] == key;
      out[e] = (kk > 0 && (u[j * W + e] > key || (eq && rank < need))) ? 1 : 0;
      if (drop_ties && eq) ++rank;
    }
    if (col + W <= N) {
      __builtin_memcpy(m + col, out, W);
    } else {
#pragma unroll
      for (int e = 0; e < W; ++e)
        if (col + e < N) m[col + e] = out[e];
    }
  }
}

// The same selection for 16-bit score rows, two keys to a register: the order of a 16-bit float is that of a 16-bit
// integer (sign and magnitude turned into two's complement, every NaN the largest one), so keys are made, compared, counted and
// turned into mask bytes by the packed 16-bit instructions and two counts always end it: the first over up to 8 * T
// equal bins of the range between the smallest and the largest key, the second over the values of the bin that holds the
// k-th largest one.  Bound by the vector instructions of the one CU that holds a row, then by the LDS atomics of the first count.
// Kernel time, 32 rows, this one against topk_mask_kernel on the widened values: 32768 columns fp16 15.1 -> 11.6 us, bf16
// 15.0 -> 11.1, 12000 fp16 13.1 -> 7.6, 8192 bf16 6.4 -> 5.2; 512 rows of 16384 26.5 -> 12.9, 640 of 4096 15.5 -> 9.9; with 85
// columns in a hundred equal 32768 21.6 -> 16.6, 512 rows of 16384 34 -> 17.
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef int16_t i16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u16x2 pk(uint32_t v) { return __builtin_bit_cast(u16x2, v); }
__device__ __forceinline__ uint32_t word(u16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ u16x2 both(uint32_t v) { return (u16x2){(uint16_t)v, (uint16_t)v}; }

// Keys of two elements: 1..0xffff in the order of the values, -0 and +0 one key, NaNs not yet in their place.
__device__ __forceinline__ uint32_t order_pair(uint32_t x) {
  const u16x2 neg = __builtin_bit_cast(u16x2, __builtin_bit_cast(i16x2, x) >> (int16_t)15);
  return word((pk(x & 0x7fff7fffu) ^ neg) - neg) ^ 0x80008000u;
}

// W4: vectors of eight columns per thread; ET: _Float16 or uint16_t (bf16 bits).
template <int T, int W4, typename ET>
__global__ __launch_bounds__(T) void topk16_mask_kernel(const ET* __restrict__ scores, uint8_t* __restrict__ mask,
                                                        float* __restrict__ threshold, int N, int k) {
  constexpr int kW = T / 64;
  constexpr int kBins = 8 * T, kBinBits = __builtin_ctz(kBins);
  constexpr uint32_t kInf = __is_same(ET, _Float16) ? 0x7c00u : 0x7f80u;
  static_assert(16 - kBinBits <= 6, "one lane per value of a bin");
  __shared__ __attribute__((aligned(16))) u32x4 hist[kBins / 4];
  __shared__ uint32_t fine[64];
  __shared__ uint32_t wave_a[kW], wave_b[kW];
  __shared__ uint32_t block_ties[W4 * kW];
  __shared__ uint32_t sh_bin, sh_above, sh_count;
  uint32_t* const bins = reinterpret_cast<uint32_t*>(hist);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const ET* s = scores + (int64_t)blockIdx.x * N;
  uint8_t* m = mask + (int64_t)blockIdx.x * N;
  const uint32_t kk = (uint32_t)min(max(k, 0), N);

  // 0 stands for a column past N
  uint32_t u[W4][4];
  u16x2 mag = both(0);
#pragma unroll
  for (int j = 0; j < W4; ++j) {
    const int col = (j * T + tid) * 8;
    if (col + 8 <= N) {
      __builtin_memcpy(u[j], s + col, 16);   // one load whatever the row's alignment
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) u[j][e] = 0u;
      if (col < N) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (col + e < N) u[j][e >> 1] |= (uint32_t)__builtin_bit_cast(uint16_t, s[col + e]) << (16 * (e & 1));
      }
    }
  }
  hist[2 * tid] = (u32x4){0u, 0u, 0u, 0u};
  hist[2 * tid + 1] = (u32x4){0u, 0u, 0u, 0u};
  if (tid < 64) fine[tid] = 0u;
  u16x2 most = both(0);   // as unsigned numbers: above infinity where there is a sign or a NaN
#pragma unroll
  for (int j = 0; j < W4; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) most = __builtin_elementwise_max(most, pk(u[j][e]));
  u16x2 hi = both(0), lo1 = both(0xffff);   // largest key, smallest key - 1 (where 0, no key, is the largest)
  if (__builtin_amdgcn_ballot_w64(most[0] > kInf || most[1] > kInf) == 0) {
    // Neither, which is what column sums, means and maxima are: such a number and the top bit is its key, three
    // instructions per pair where the general case takes twelve (a call with 32 rows of 32768 fp16 11.6 -> 9.9 us, 640 rows 34 -> 28.5, 32 of
    // 60000 20.6 -> 17.3; 8192 columns and fewer 0-5 %).
    u16x2 least = both(0x7fff);
#pragma unroll
    for (int j = 0; j < W4; ++j) {
      const int col = (j * T + tid) * 8;
      if (__builtin_amdgcn_ballot_w64(col + 8 > N) == 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          least = __builtin_elementwise_min(least, pk(u[j][e]));
          u[j][e] ^= 0x80008000u;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          uint32_t key = u[j][e] ^ 0x80008000u;
          if (col + 2 * e >= N) key = 0u;
          else if (col + 2 * e + 1 >= N) key &= 0xffffu;
          u[j][e] = key;
          lo1 = __builtin_elementwise_min(lo1, pk(key) - both(1));
        }
      }
    }
    if (tid * 8 < N) hi = pk(word(most) ^ 0x80008000u);
    lo1 = __builtin_elementwise_min(lo1, pk(word(least) ^ 0x80008000u) - both(1));
  } else {
#pragma unroll
    for (int j = 0; j < W4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) mag = __builtin_elementwise_max(mag, pk(u[j][e] & 0x7fff7fffu));
    const bool any_nan = __builtin_amdgcn_ballot_w64(mag[0] > kInf || mag[1] > kInf) != 0;
#pragma unroll
    for (int j = 0; j < W4; ++j) {
      const int col = (j * T + tid) * 8;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t x = u[j][e];
        uint32_t key = order_pair(x);
        if (any_nan) {
          const u16x2 over = __builtin_elementwise_min(__builtin_elementwise_sub_sat(pk(x & 0x7fff7fffu), both(kInf)), both(1));
          key |= word(both(0) - over);
        }
        if (col + 8 > N) {   // (the last vectors of the row)
          if (col + 2 * e >= N) key = 0u;
          else if (col + 2 * e + 1 >= N) key &= 0xffffu;
        }
        u[j][e] = key;
        hi = __builtin_elementwise_max(hi, pk(key));
        lo1 = __builtin_elementwise_min(lo1, pk(key) - both(1));
      }
    }
  }
  auto equals = [](const uint32_t(&v)[4], uint32_t x) {   // how many of eight 16-bit numbers are x
    u16x2 differ = both(0);
#pragma unroll
    for (int e = 0; e < 4; ++e) differ += __builtin_elementwise_min(pk(v[e]) ^ both(x), both(1));
    return 8u - (uint32_t)differ[0] - (uint32_t)differ[1];
  };
  uint32_t key = 0xffffu, need = kk, ties = 0u;   // k <= 0: nothing is kept
  if (kk > 0) {
    uint32_t top = wave_max(max((uint32_t)hi[0], (uint32_t)hi[1])), bottom = wave_max(0xffffu - min((uint32_t)lo1[0], (uint32_t)lo1[1]));
    if (lane == 0) {
      wave_a[wave] = top;
      wave_b[wave] = bottom;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kW; ++w) {
      top = max(top, wave_a[w]);
      bottom = max(bottom, wave_b[w]);
    }
    const uint32_t lo = 0x10000u - bottom;
    const uint32_t range = top - lo;
    const int bits = range ? 32 - __builtin_clz(range) : 0;
    const int shift = max(bits - kBinBits, 0);
    const u16x2 lo2 = both(lo), shift2 = both((uint32_t)shift);
#pragma unroll
    for (int j = 0; j < W4; ++j) {
      const int col = (j * T + tid) * 8;
      uint32_t b[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) b[e] = word((pk(u[j][e]) - lo2) >> shift2);
      // A bin that many lanes share (zeros, ties) serializes their atomics: where the first column of a vector shows that,
      // its keys in the bin of the first lane are added up by packed compares.
      const bool whole = col + 8 <= N;
      const uint64_t live = __builtin_amdgcn_ballot_w64(whole);
      const uint32_t lead = __builtin_amdgcn_readlane(b[0] & 0xffffu, live ? __builtin_ctzll(live) : 0);
      auto bin_of = [&](int e) { return (e & 1) ? b[e >> 1] >> 16 : b[e >> 1] & 0xffffu; };
      if (__builtin_popcountll(__builtin_amdgcn_ballot_w64(whole && (b[0] & 0xffffu) == lead)) <= 8) {
        if (whole) {
#pragma unroll
          for (int e = 0; e < 8; ++e) atomicAdd(&bins[bin_of(e)], 1u);
        }
      } else {
        const uint32_t c = wave_sum(whole ? equals(b, lead) : 0u);
        if (lane == 0) atomicAdd(&bins[lead], c);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (whole && bin_of(e) != lead) atomicAdd(&bins[bin_of(e)], 1u);
      }
      if (!whole && col < N) {   // the row's last columns
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (col + e < N) atomicAdd(&bins[bin_of(e)], 1u);
      }
    }
    __syncthreads();
    // thread t takes the eight bins from kBins - 1 - 8t down: prefix sums are counts from the top
    const u32x4 h1 = hist[kBins / 4 - 1 - 2 * tid], h0 = hist[kBins / 4 - 2 - 2 * tid];
    const uint32_t own = (h0[0] + h0[1] + h0[2] + h0[3]) + (h1[0] + h1[1] + h1[2] + h1[3]);
    const uint32_t incl = wave_scan(own);
    if (lane == 63) wave_a[wave] = incl;   // (read above before the last barrier)
    __syncthreads();
    uint32_t above = incl - own;
#pragma unroll
    for (int w = 0; w < kW; ++w) above += (w < wave) ? wave_a[w] : 0u;
    if (above < need && above + own >= need) {   // one thread of the workgroup
#pragma unroll
      for (int e = 7; e >= 0; --e) {
        const uint32_t c = e >= 4 ? h1[e - 4] : h0[e];
        if (above < need) {
          sh_bin = (uint32_t)(kBins - 8 - 8 * tid + e);
          sh_above = above;
          sh_count = c;
        }
        above += c;
      }
    }
    __syncthreads();
    const uint32_t bin = sh_bin;
    need -= sh_above;
    key = lo + (bin << shift);
    ties = sh_count;
    if (shift > 0) {
      // The bin's values are key .. key + low (0, a column past N, is none of them).
      const uint32_t low = min((1u << shift) - 1u, 0xffffu - key);
      const u16x2 base2 = both(key), low2 = both(low);
      u16x2 nearest[W4], least = both(0xffff);
#pragma unroll
      for (int j = 0; j < W4; ++j) {
        nearest[j] = both(0xffff);
#pragma unroll
        for (int e = 0; e < 4; ++e) nearest[j] = __builtin_elementwise_min(nearest[j], pk(u[j][e]) - base2);
        least = __builtin_elementwise_min(least, nearest[j]);
      }
      const uint32_t some = min((uint32_t)least[0], (uint32_t)least[1]);
      const uint64_t holds = __builtin_amdgcn_ballot_w64(some <= low);
      if (holds != 0) {
        // one value that the wave holds may be there many times over: those are added up by packed compares
        const uint32_t lead = __builtin_amdgcn_readlane(some, __builtin_ctzll(holds));
        uint32_t c = 0u;
#pragma unroll
        for (int j = 0; j < W4; ++j) {
          if (__builtin_amdgcn_ballot_w64(nearest[j][0] <= low || nearest[j][1] <= low) == 0) continue;
          u16x2 out = both(0);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            out += __builtin_elementwise_min(__builtin_elementwise_sub_sat(pk(u[j][e]) - base2, low2), both(1));
          const uint32_t same = equals(u[j], key + lead);
          c += same;
          if (__builtin_amdgcn_ballot_w64(8u - (uint32_t)out[0] - (uint32_t)out[1] != same) == 0) continue;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const uint32_t t = (((e & 1) ? u[j][e >> 1] >> 16 : u[j][e >> 1] & 0xffffu) - key) & 0xffffu;
            if (t <= low && t != lead) atomicAdd(&fine[t], 1u);
          }
        }
        c = wave_sum(c);
        if (lane == 0) atomicAdd(&fine[lead], c);
      }
      __syncthreads();
      // every wave looks for itself: lane l takes the value 63 - l of the bin
      const uint32_t f = fine[63 - lane], over = wave_scan(f) - f;
      const int at = __builtin_ctzll(__builtin_amdgcn_ballot_w64(over < need && over + f >= need));
      key += 63u - (uint32_t)at;
      ties = (uint32_t)__builtin_amdgcn_readlane((int)f, at);
      need -= (uint32_t)__builtin_amdgcn_readlane((int)over, at);
    }
  }
  // `key` is the key of the k-th largest element; `need` of the `ties` keys equal to it are kept
  if (tid == 0 && threshold) {
    const int v = (int)key - 0x8000;
    const uint16_t h = (uint16_t)(v < 0 ? 0x8000 - v : v);
    threshold[blockIdx.x] = key == 0xffffu ? __builtin_bit_cast(float, 0x7fffffffu) : widen<ET>(__builtin_bit_cast(ET, h));
  }

  const bool drop_ties = need < ties;   // uniform: some ties are dropped, rank them by column
  if (drop_ties) {
    // ties per block of 512 columns, in column order, then their exclusive prefix sums
#pragma unroll
    for (int j = 0; j < W4; ++j) {
      uint32_t c = equals(u[j], key);
      c = __builtin_amdgcn_ballot_w64(c != 0u) ? wave_sum(c) : 0u;
      if (lane == 0) block_ties[j * kW + wave] = c;
    }
    __syncthreads();
    if (wave == 0) {
      uint32_t base = 0;
      for (int i0 = 0; i0 < W4 * kW; i0 += 64) {
        const uint32_t c = (i0 + lane < W4 * kW) ? block_ties[i0 + lane] : 0u;
        const uint32_t incl = wave_scan(c);
        if (i0 + lane < W4 * kW) block_ties[i0 + lane] = base + incl - c;
        base += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
      }
    }
    __syncthreads();
  }
  // columns above `floor` are kept; ties are added where some are dropped.  (Nothing is above the key of k <= 0.)
  const u16x2 floor2 = both(drop_ties || kk == 0 ? key : key - 1u);
#pragma unroll
  for (int j = 0; j < W4; ++j) {
    const int col = (j * T + tid) * 8;
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = word(__builtin_elementwise_min(__builtin_elementwise_sub_sat(pk(u[j][e]), floor2), both(1)));
    if (drop_ties) {
      const uint32_t mine = equals(u[j], key);
      if (__builtin_amdgcn_ballot_w64(mine != 0u)) {
        uint32_t rank = block_ties[j * kW + wave] + wave_scan(mine) - mine;   // ties in front of this thread's columns
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t x = (e & 1) ? u[j][e >> 1] >> 16 : u[j][e >> 1] & 0xffffu;
          if (x == key) {
            if (rank < need) w[e >> 1] |= 1u << (16 * (e & 1));
            ++rank;
          }
        }
      }
    }
    const uint32_t out[2] = {__builtin_amdgcn_perm(w[1], w[0], 0x06040200u), __builtin_amdgcn_perm(w[3], w[2], 0x06040200u)};
    if (col + 8 <= N) {
      __builtin_memcpy(m + col, out, 8);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (col + e < N) m[col + e] = (uint8_t)(out[e >> 2] >> (8 * (e & 3)));
    }
  }
}

template <typename ET>
__global__ __launch_bounds__(kTopkThreads) void topk_mask_long_kernel(const ET* __restrict__ scores,
                                                                      uint8_t* __restrict__ mask,
                                                                      float* __restrict__ threshold, int N, int k) {
  constexpr int kW = kTopkThreads / 64;
  __shared__ uint32_t hist[256];
  __shared__ uint32_t sh_prefix, sh_need, sh_ties;
  __shared__ uint32_t wave_eq[kW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const ET* s = scores + (int64_t)blockIdx.x * N;
  uint8_t* m = mask + (int64_t)blockIdx.x * N;
  const uint32_t kk = (uint32_t)min(max(k, 0), N);
  uint32_t prefix = 0, decided = 0, need = kk;
  for (int pass = 0; pass < 4; ++pass) {
    const int shift = 24 - 8 * pass;
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    for (int j0 = 0; j0 < N; j0 += kTopkThreads) {
      const int j = j0 + tid;
      const uint32_t x = (j < N) ? order_key(widen<ET>(s[j])) : 0u;
      const bool live = (j < N) && ((x & decided) == prefix);
      const uint32_t d = (x >> shift) & 255u;
      const uint64_t lives = __builtin_amdgcn_ballot_w64(live);
      if (lives == 0) continue;
      const uint32_t d0 = __builtin_amdgcn_readlane(d, __builtin_ctzll(lives));
      if (__builtin_amdgcn_ballot_w64(live && d == d0) == lives) {   // one bin for the whole wave
        if (lane == 0) atomicAdd(&hist[d0], (uint32_t)__builtin_popcountll(lives));
      } else if (live) {
        atomicAdd(&hist[d], 1u);
      }
    }
    __syncthreads();
    if (tid < 64) {   // one wave walks the bins from the top: 4 bins per lane, suffix sums across lanes
      uint32_t h[4], tot = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        h[e] = hist[255 - (lane * 4 + e)];   // lane 0 holds the four largest digits
        tot += h[e];
      }
      uint32_t incl = tot;
#pragma unroll
      for (int dd = 1; dd < 64; dd <<= 1) {
        const uint32_t o = __shfl_up(incl, dd);
        if (lane >= dd) incl += o;
      }
      uint32_t above = incl - tot;    // keys in larger digits than this lane's
      // the digit where the running count first reaches `need`
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (above < need && above + h[e] >= need) {
          sh_prefix = prefix | ((uint32_t)(255 - (lane * 4 + e)) << shift);
          sh_need = need - above;
          sh_ties = h[e];
        }
        above += h[e];
      }
    }
    __syncthreads();
    if (need > 0) {
      prefix = sh_prefix;
      need = sh_need;
    } else {
      prefix |= 0xffu << shift;   // k == 0: nothing is kept, any threshold above every key will do
    }
    decided |= 0xffu << shift;
    __syncthreads();
  }
  // prefix is now the key of the k-th largest element; `need` of the sh_ties keys equal to it are kept
  const uint32_t T = prefix;
  const uint32_t ties = (kk > 0) ? sh_ties : 0u;
  if (tid == 0 && threshold) threshold[blockIdx.x] = key_value(T);
  const int per = (N + kTopkThreads - 1) / kTopkThreads;   // thread t writes columns [t*per, t*per + per)
  const int base = tid * per;
  uint32_t before = 0;
  if (need < ties) {
    uint32_t mine = 0;
    for (int i = 0; i < per; ++i) mine += (base + i < N && order_key(widen<ET>(s[base + i])) == T) ? 1u : 0u;
    before = ties_before(mine, wave_eq, lane, wave);
  }
  const bool keep_all_ties = need >= ties;
  for (int i = 0; i < per; ++i) {
    const int j = base + i;
    if (j >= N) break;
    const uint32_t x = order_key(widen<ET>(s[j]));
    const bool eq = x == T;
    m[j] = ((kk > 0) && ((x > T) || (eq && (keep_all_ties || before < need)))) ? 1 : 0;
    if (eq) ++before;
  }
}

// ---------------------------------------------------------------------------------------------
// Rows of more than 32768 columns with a workspace: a row is spread over workgroups of VPT * 1024
// columns (VPT = 32 keys per thread, in registers, when that still gives a workgroup per CU, else 8).  Radix select, eight bits per launch: launch PASS
// histograms digit PASS of the keys that match the digits chosen so far, one histogram per workgroup,
// written whole (no atomics in memory, nothing to clear, bitwise reproducible).  Every workgroup of the
// next launch adds up the row's histograms and repeats the choice of the digit, so no launch is needed
// for that.  The last launch chooses the fourth digit, finds the ties in front of its columns in the
// earlier workgroups' histograms of that digit, and writes the mask.

struct TopkState {
  uint32_t prefix;   // digits chosen so far, in place
  uint32_t need;     // how many keys to keep among those that match the prefix
  uint32_t ties;     // how many keys fell into the digit chosen last
  uint32_t pad;
};

// workspace: hist[2][rows][parts][256] followed by state[rows][4]
__host__ __device__ inline size_t topk_hist_words(int64_t rows, int parts) { return (size_t)rows * parts * 256; }

// The choice of digit `pass` for one row, by the whole workgroup: the bins of the row's `parts` histograms
// are added up, then one wave walks them from the top.  prev is the state before this digit.
__device__ __forceinline__ TopkState topk_choose(const uint32_t* __restrict__ hist_row, int parts, TopkState prev,
                                                 int pass, uint32_t* bins, TopkState* chosen, int tid, int lane) {
  const int shift = 24 - 8 * pass;
  if (tid < 256) {
    uint32_t v = 0;
    for (int q = 0; q < parts; ++q) v += hist_row[q * 256 + tid];
    bins[tid] = v;
  }
  if (tid == 0) *chosen = TopkState{prev.prefix | (0xffu << shift), 0u, 0u, 0u};   // need == 0: nothing is kept
  __syncthreads();
  if (tid < 64) {   // 4 bins per lane, lane 0 holds the four largest digits; suffix sums across lanes
    uint32_t h[4], tot = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      h[e] = bins[255 - (lane * 4 + e)];
      tot += h[e];
    }
    uint32_t incl = tot;
#pragma unroll
    for (int dd = 1; dd < 64; dd <<= 1) {
      const uint32_t o = __shfl_up(incl, dd);
      if (lane >= dd) incl += o;
    }
    uint32_t above = incl - tot;   // keys in larger digits than this lane's
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (above < prev.need && above + h[e] >= prev.need)   // true for exactly one bin when need > 0
        *chosen = TopkState{prev.prefix | ((uint32_t)(255 - (lane * 4 + e)) << shift), prev.need - above, h[e], 0u};
      above += h[e];
    }
  }
  __syncthreads();
  const TopkState out = *chosen;
  __syncthreads();   // bins and chosen may be written again
  return out;
}

// The VPT keys of a thread from column col0 on; columns past N get key 0 and valid bit 0.
template <int VPT, typename ET>
__device__ __forceinline__ uint32_t topk_load(const ET* __restrict__ s, int N, int col0, uint32_t u[VPT]) {
  if (col0 + VPT <= N) {
    constexpr int W = 16 / (int)sizeof(ET);
#pragma unroll
    for (int i = 0; i < VPT; i += W) {
      ET v[W];
      __builtin_memcpy(v, s + col0 + i, 16);   // one load whatever the row's alignment (520 rows of 58671 fp32, element by element 934 us, so 299)
#pragma unroll
      for (int e = 0; e < W; ++e) u[i + e] = order_key(widen<ET>(v[e]));
    }
    return VPT == 32 ? 0xffffffffu : (1u << (VPT & 31)) - 1u;
  }
  uint32_t valid = 0;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const bool in = col0 + i < N;
    u[i] = in ? order_key(widen<ET>(s[in ? col0 + i : 0])) : 0u;
    valid |= in ? (1u << i) : 0u;
  }
  return valid;
}

template <int PASS, int VPT, typename ET>
__global__ __launch_bounds__(kTopkThreads) void topk_spread_hist_kernel(const ET* __restrict__ scores,
                                                                        uint32_t* __restrict__ ws, int64_t rows,
                                                                        int N, int k, int parts) {
  __shared__ uint32_t bins[256];
  __shared__ uint32_t hist[256];
  __shared__ TopkState chosen;
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t row = blockIdx.x / parts;
  const int part = (int)(blockIdx.x - row * parts);
  const size_t words = topk_hist_words(rows, parts);
  TopkState* states = reinterpret_cast<TopkState*>(ws + 2 * words) + row * 4;
  uint32_t* mine = ws + (PASS & 1) * words + ((size_t)row * parts + part) * 256;

  uint32_t u[VPT];
  const ET* s = scores + row * N;
  const uint32_t valid = topk_load<VPT>(s, N, (part * kTopkThreads + tid) * VPT, u);

  TopkState st{0u, (uint32_t)min(max(k, 0), N), 0u, 0u};
  if (PASS > 0) {
    if (PASS > 1) st = states[PASS - 2];
    st = topk_choose(ws + ((PASS - 1) & 1) * words + (size_t)row * parts * 256, parts, st, PASS - 1, bins, &chosen,
                     tid, lane);
    if (part == 0 && tid == 0) states[PASS - 1] = st;
  }
  if (tid < 256) hist[tid] = 0;
  __syncthreads();
  constexpr uint32_t decided = PASS == 0 ? 0u : 0xffffffffu << (32 - 8 * PASS);
  constexpr int shift = 24 - 8 * PASS;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const bool live = ((valid >> i) & 1u) && ((u[i] & decided) == st.prefix);
    const uint32_t d = (u[i] >> shift) & 255u;
    const uint64_t lives = __builtin_amdgcn_ballot_w64(live);
    if (lives == 0) continue;
    const uint32_t d0 = __builtin_amdgcn_readlane(d, __builtin_ctzll(lives));
    if (__builtin_amdgcn_ballot_w64(live && d == d0) == lives) {   // one bin for the whole wave
      if (lane == 0) atomicAdd(&hist[d0], (uint32_t)__builtin_popcountll(lives));
    } else if (live) {
      atomicAdd(&hist[d], 1u);
    }
  }
  __syncthreads();
  if (tid < 256) mine[tid] = hist[tid];
}

template <int VPT, typename ET>
__global__ __launch_bounds__(kTopkThreads) void topk_spread_write_kernel(const ET* __restrict__ scores,
                                                                         uint8_t* __restrict__ mask,
                                                                         float* __restrict__ threshold,
                                                                         const uint32_t* __restrict__ ws, int64_t rows,
                                                                         int N, int k, int parts) {
  constexpr int kW = kTopkThreads / 64;
  __shared__ uint32_t bins[256];
  __shared__ TopkState chosen;
  __shared__ uint32_t wave_eq[kW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t row = blockIdx.x / parts;
  const int part = (int)(blockIdx.x - row * parts);
  const size_t words = topk_hist_words(rows, parts);
  const TopkState* states = reinterpret_cast<const TopkState*>(ws + 2 * words) + row * 4;
  const uint32_t* last = ws + words + (size_t)row * parts * 256;   // the histograms of digit 3 (3 & 1 == 1)

  uint32_t u[VPT];
  const ET* s = scores + row * N;
  const int col0 = (part * kTopkThreads + tid) * VPT;
  const uint32_t valid = topk_load<VPT>(s, N, col0, u);

  const uint32_t kk = (uint32_t)min(max(k, 0), N);
  const TopkState st = topk_choose(last, parts, states[2], 3, bins, &chosen, tid, lane);
  const uint32_t T = st.prefix, need = st.need, ties = (kk > 0) ? st.ties : 0u;
  if (part == 0 && tid == 0 && threshold) threshold[row] = key_value(T);

  uint32_t before = 0;
  if (need < ties) {   // uniform over the row: some ties are dropped, rank them by column
    uint32_t mine = 0;
#pragma unroll
    for (int i = 0; i < VPT; ++i) mine += (((valid >> i) & 1u) && u[i] == T) ? 1u : 0u;
    before = ties_before(mine, wave_eq, lane, wave);
    for (int q = 0; q < part; ++q) before += last[q * 256 + (T & 255u)];   // ties in the workgroups in front
  }
  const bool keep_all_ties = need >= ties;
  uint8_t* m = mask + row * N;
  const bool whole = valid == (VPT == 32 ? 0xffffffffu : (1u << (VPT & 31)) - 1u);
#pragma unroll
  for (int i0 = 0; i0 < VPT; i0 += 8) {
    uint64_t w = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int i = i0 + e;
      const bool eq = ((valid >> i) & 1u) && u[i] == T;
      const bool keep = (kk > 0) && ((u[i] > T) || (eq && (keep_all_ties || before < need)));
      if (eq) ++before;
      w |= (uint64_t)(keep ? 1 : 0) << (8 * e);
    }
    if (whole) {
      __builtin_memcpy(m + col0 + i0, &w, 8);   // (any alignment)
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if ((valid >> (i0 + e)) & 1u) m[col0 + i0 + e] = (uint8_t)(w >> (8 * e));
    }
  }
}

// ---------------------------------------------------------------------------------------------
thread_local char g_err[256] = "";

int fail(int code, const char* what) {
  snprintf(g_err, sizeof(g_err), "%s", what);
  return code;
}


// dims = sizes of the batch, head and row dimensions.  The stride of a dimension of size one is never
// used to form an address, so it may be anything (torch reports arbitrary strides there, and a slice of an
// expanded tensor keeps stride 0): only the strides that matter are checked.
int check_strides(const void* ptr, const int64_t s[4], const char* name, const int dims[3], int D, int esize) {
  if (s[3] != 1) {
    snprintf(g_err, sizeof(g_err), "%s: stride of the last dimension must be 1 (got %lld)", name, (long long)s[3]);
    return FCR_E_STRIDE;
  }
  const int al = 16 / esize;   // elements per 16 bytes
  bool ok = (reinterpret_cast<uintptr_t>(ptr) & 15) == 0;
  for (int i = 0; i < 3; ++i)
    if (dims[i] > 1 && (s[i] % al != 0 || s[i] < 0)) ok = false;
  if (dims[2] > 1 && s[2] * esize >= (1 << 25)) ok = false;
  if (!ok) {
    snprintf(g_err, sizeof(g_err),
             "%s: base pointer must be 16-byte aligned, batch/head/row strides non-negative multiples of 16 bytes (%d elements), row stride < 2^25 bytes",
             name, al);
    return FCR_E_STRIDE;
  }
  // Rows that overlap (an expanded operand has row stride 0) cannot be described by the buffer views
  // the kernels read through: the view of the rows from r on is (rows - r) * stride bytes long.
  if (dims[2] > 1 && s[2] < D) {
    snprintf(g_err, sizeof(g_err), "%s: row stride (%lld) must be at least D (%d) when there is more than one row",
             name, (long long)s[2], D);
    return FCR_E_STRIDE;
  }
  return 0;
}

// (b,h) pairs per launch group, a multiple of 8.  Without a mask all sweeps of a launch are equally
// long and about one workgroup per CU (256) keeps the tiles of a (b,h) together in time.  With the
// causal mask the longest-first order needs room to level the triangle: about 1024 workgroups and
// never fewer than 32 pairs (measured: smaller groups lose up to 8 % on 32 heads of 8192 rows,
// larger ones up to 11 % on 1024 heads of 2048 rows, whose operands then come from HBM per tile).
int head_group(int64_t bh, int64_t per_bh, bool causal) {
  const int cus = chip_cus();
  int64_t g = ((causal ? 4 * cus : cus) / per_bh) & ~7ll;
  const int64_t least = causal ? 32 : 8;
  if (g < least) g = least;
  return (int)(g < bh ? g : bh);
}

// Rows the kernels take: a multiple of 16 bytes, at most 1 KiB (and no product of D that could overflow).
bool row_width_ok(int dtype, int D) {
  const int esize = elem_bytes(dtype);
  return D >= 1 && D <= 64 * kMaxKStepsF32 / esize && (D * esize) % 16 == 0;
}

// The arguments of a launch over the queries or (by_keys) the keys; no HIP call.
int check_problem(const void* q, const void* k, int dtype, int B, int H, int M, int N, int D, const int64_t qs[4],
                  const int64_t ks[4], float scale, bool by_keys) {
  if (!q || !k || !qs || !ks) return fail(FCR_E_NULL, "null pointer argument");
  if (dtype != FCR_DTYPE_F16 && dtype != FCR_DTYPE_BF16 && dtype != FCR_DTYPE_F32)
    return fail(FCR_E_DTYPE, "dtype must be FCR_DTYPE_F16, FCR_DTYPE_BF16 or FCR_DTYPE_F32");
  if (B < 1 || H < 1 || M < 1 || N < 1) return fail(FCR_E_SHAPE, "B, H, M, N must be >= 1");
  const int esize = elem_bytes(dtype);
  if (!row_width_ok(dtype, D))
    return fail(FCR_E_SHAPE, esize == 2 ? "D must be a multiple of 8 in [8, 512]"
                                         : "D must be a multiple of 4 in [4, 256] for FCR_DTYPE_F32");
  if (M > (1 << 30) || N > (1 << 30)) return fail(FCR_E_SHAPE, "M and N must be <= 2^30");
  const int64_t bh = (int64_t)B * H;
  // a launch may have fewer than 2^32 threads: fewer than 2^24 workgroups of 256 (the finest tiling, 128 rows; f32_tile sees to it that
  // workgroups of 512 are half as many)
  if (bh * (((int64_t)(by_keys ? N : M) + 127) / 128) >= kMaxWorkgroups)
    return fail(FCR_E_SHAPE, "B*H*ceil(rows/128) must be below 2^24 workgroups");
  if (!isfinite(scale)) return fail(FCR_E_SCALE, "scale must be finite");
  const int qdims[3] = {B, H, M}, kdims[3] = {B, H, N};
  int rc = check_strides(q, qs, "q", qdims, D, esize);
  if (rc) return rc;
  return check_strides(k, ks, "k", kdims, D, esize);
}

// Rows of a launch's tiles and how many of its workgroups share a CU.
struct TileChoice {
  int rows, per_cu;
};
TileChoice tile_choice(int dtype, int D, int M, int N, int64_t bh, bool by_keys, int col_mode, bool causal) {
  const int ksteps = ksteps_of(dtype, D);
  if (in_parts(dtype, D)) {
    const F32Tile t = by_keys ? f32_col_tile(f32_ksteps(ksteps), col_mode == kModeBoth, M, N, bh, causal) : f32_row_tile(M, N, bh, causal);
    return TileChoice{t.rows(), 8 / t.waves};
  }
  const int per_cu = ksteps > kMaxKSteps ? 1 : 2;
  if (by_keys && half_tiles(dtype, D, N, bh)) return TileChoice{kWaves * 16, per_cu};
  return TileChoice{by_keys ? kWaves * 32 * col_tile_blocks(ksteps, col_mode, N, bh, causal)
                            : row_tile_rows(dtype, D, M, N, bh, causal), per_cu};
}

// Params::fill: see map_group.  Only for launches of one group, whose places are in order of length over the whole launch, and
// for kernels that run two workgroups per CU.  Per call, plain order and with the second helping backwards, workgroups per
// CU in brackets: 256-row tiles, 40 heads of 3258 (2.03) 141 -> 120 us, 48 of 2929 (2.25) 133 -> 117, 32 of 5120 (2.5) 236 -> 221,
// 32 of 5632 (2.75) 269 -> 263, but 40 of 4538 (2.81) 214 -> 216, 32 of 6656 (3.25) 339 -> 350; 128-row tiles, 12 heads of
// 5000 (1.9) 128 -> 106, 24 of 3072, sums and maxima (2.25) 79 -> 72, 32 of 3072 x 256 (3) 155 -> 150, 8 of 16384 (4) 530 -> 514,
// nothing lost beyond and within 1 % of it.  (All bf16 or fp16, D = 128 where none is named.)
int fill_places(const Params& p, const TileChoice& t, bool causal) {
  const int cus = chip_cus();
  if (!causal || p.splits > 1 || p.group != p.bh_count || p.total <= cus || t.per_cu < 2) return 0;
  return (int64_t)p.total * 4 <= (int64_t)cus * (t.rows > 128 ? 11 : 16) ? cus : 0;
}

int make_params(Params& p, const void* q, const void* k, int dtype, int B, int H, int M, int N, int D,
                const int64_t qs[4], const int64_t ks[4], float scale, bool by_keys, bool causal,
                int col_mode = kModeSum) {
  const int rc = check_problem(q, k, dtype, B, H, M, N, D, qs, ks, scale, by_keys);
  if (rc) return rc;
  const int esize = elem_bytes(dtype);
  const int64_t bh = (int64_t)B * H;
  // the device is first asked (for its CU count) here, after every argument check
  const int trows = tile_choice(dtype, D, M, N, bh, by_keys, col_mode, causal).rows;
  const int64_t tiles = ((by_keys ? N : M) + trows - 1) / trows;
  p.q = static_cast<const char*>(q);
  p.k = static_cast<const char*>(k);
  // a single row is given the stride of a dense one: the buffer views are sized rows * stride
  p.q_sb = B > 1 ? qs[0] * esize : 0; p.q_sh = H > 1 ? qs[1] * esize : 0; p.q_sr = M > 1 ? qs[2] * esize : D * esize;
  p.k_sb = B > 1 ? ks[0] * esize : 0; p.k_sh = H > 1 ? ks[1] * esize : 0; p.k_sr = N > 1 ? ks[2] * esize : D * esize;
  p.H = H; p.M = M; p.N = N;
  p.dgran = D * esize / 16;
  p.c = N > M ? N - M : 0;
  p.scale2 = (float)((double)scale * 1.4426950408889634);
  p.split_most = (float)(131072.0 / (std::fabs((double)scale * 1.4426950408889634) * std::sqrt((double)D)));
  p.tiles = (int)tiles;
  p.bh_count = (int)bh;
  p.total = (int)(bh * tiles);
  p.lse = nullptr;
  p.out = nullptr;
  p.out2 = nullptr;
  p.part = nullptr;
  p.splits = 1;
  p.fill = 0;
  p.stream_once = 0;
  p.out_fmt = FCR_DTYPE_F32;
  p.mean_from = -1;
  p.inv_m = 0.f;
  p.teams = 0;
  p.sync = nullptr;
  p.spin_limit = 0;
  p.col_tiles = p.col_group = p.row_blocks = p.col_blocks = p.parts = p.run_chunks = 0;
  return 0;
}

// Key ranges per row tile in the row kernel.  One sweep per workgroup when there is at least one
// workgroup per CU; otherwise the keys of a tile are split so that about two per CU run, each
// keeping at least four 64-key chunks.
int row_splits(int dtype, int B, int H, int M, int N, int D) {
  const int64_t chunks = (N + kChunk - 1) / kChunk;
  if (chunks < 16) return 1;
  // (fp32 launches in parts of at least one 128-row tile per CU are never split; the mask makes no difference below that)
  const int trows = in_parts(dtype, D) ? 128 : row_tile_rows(dtype, D, M, N, (int64_t)B * H, false);  // same with the mask when wgs < 256
  const int64_t wgs = (int64_t)B * H * ((M + trows - 1) / trows);
  const int cus = chip_cus();
  if (wgs >= cus) return 1;
  int64_t s = 2 * cus / wgs;
  if (s > chunks / 4) s = chunks / 4;
  if (s > 64) s = 64;
  return s < 1 ? 1 : (int)s;
}

// The single-sweep path (col_fused_kernel): 16-bit operands, rows of at most 256 bytes, at most 128 queries
// and enough keys for the sweep to matter.  A (b,h) pair is shared by `splits` workgroups of 512 keys each;
// teams * splits workgroups are launched, never more than the chip holds at once.
constexpr int kFusedMinChunks = 16;   // 1024 keys
struct FusedPlan {
  int qh;       // 1: 64 query rows per workgroup and 1024 keys per pair, 2: 128 rows and 512 keys
  int nq;       // groups of sixteen queries per wave: 4, or 2 (at most 32 queries) with 2048 keys per pair
  int splits, teams;
  int64_t part_at, sync_at;   // where the partial row values and the counters start in the workspace, in floats
  int64_t floats;             // workspace size
};
// Shape conditions only: the size of the workspace must not depend on the element type.
bool fused_shape(int64_t bh, int M, int N, FusedPlan& f) {
  const int64_t nchunks = ((int64_t)N + kChunk - 1) / kChunk;
  if (M > 2 * 64 || nchunks < kFusedMinChunks) return false;
  f.qh = M > 64 ? 2 : 1;
  const int cap = chip_cus();   // one workgroup per CU
  // With at most 32 queries a workgroup can keep the scores of 2048 keys of a pair, which spreads the time
  // between two sweeps over twice the keys, but it leaves half the workgroups per pair.  The choice is the
  // one with the least estimated time: rounds x (0.56 us per chunk + 4.5 us between sweeps).
  double best = 0.0;
  f.nq = 0;
  for (int nq = 4; nq >= 2; nq /= 2) {
    if (nq < 4 && (f.qh != 1 || M > 16 * nq)) continue;
    const int chunks = fused_chunks(f.qh, nq);
    const int64_t splits = (nchunks + chunks - 1) / chunks;
    if (splits > cap) continue;
    const int64_t teams = (cap / splits) < bh ? (cap / splits) : bh;
    const int64_t rounds = (bh + teams - 1) / teams;
    const int64_t swept = nchunks < chunks ? nchunks : chunks;
    const double cost = (double)rounds * (0.56 * (double)swept + 4.5);
    if (f.nq == 0 || cost < best) {
      best = cost;
      f.nq = nq;
      f.splits = (int)splits;
      f.teams = (int)teams;
    }
  }
  if (f.nq == 0) return false;
  f.part_at = (bh * M + 63) / 64 * 64;
  f.sync_at = f.part_at + 2 * (2ll * cap * 64 * f.qh);   // two sets of one 64-bit slot per row and workgroup
  f.floats = f.sync_at + 32;
  return true;
}

// The single sweep in workgroups of four waves, two per CU, for at most 32 queries in several rounds, where the caller's workspace
// has room for their slots (they follow the status word of the form above).  The rule, over 1500 shapes of 2 to 32 queries, 1024 to 65536
// keys and 4 to 1000 pairs in several rounds of eight waves, us per call of eight waves and of four: where eight waves keep four query groups
// four waves won everywhere (484 shapes, 0.81: 300 pairs of 32 x 2045 x 32, maxima, 35.9, 22.1; 128 of 32 x 5001 x 128, both, 51.7, 41.4; 300 of 2 x 1024 x 128
// 26.0, 21.6).  Where those keep two groups the rounds are the same, and what decides is the time between two sweeps against that of
// the loads: rows of more than 128 bytes 0.96 (512 pairs of 32 x 16384 x 128 is one of them), of 128 bytes 1.00, of 64 bytes 1.04 (64 of
// 31 x 15509 x 32 25.0, 28.6; 128 of 16 x 7672 x 32 23.9, 27.0); of 128 bytes and one eight-wave workgroup per pair, which exchanges nothing,
// 1.05 (444 of 17 x 1313 x 64 25.8, 29.0).  The last two keep eight waves.
struct FusedPairPlan {
  int splits, teams;   // teams 0: not this form
  int64_t part_at, floats;
};
FusedPairPlan fused_pair_plan(int64_t bh, int M, int N, int ksteps, const FusedPlan& f) {
  FusedPairPlan o{0, 0, f.sync_at + 32, f.floats};
  if (M > 32 || bh <= f.teams || (f.nq == 2 && ksteps <= 2 && (ksteps == 1 || f.splits == 1))) return o;
  const int cap = 2 * chip_cus();
  const int64_t nchunks = ((int64_t)N + kChunk - 1) / kChunk, chunks = kFusedSteps * 2, splits = (nchunks + chunks - 1) / chunks;
  if (splits > cap) return o;
  o.splits = (int)splits;
  o.teams = (int)((cap / splits) < bh ? cap / splits : bh);
  o.floats = o.part_at + 2 * (2ll * o.teams * o.splits * 32);
  return o;
}

// The single sweep's keys of a pair, dealt evenly to the workgroups of its team (p.splits: as few as can hold them), in steps of
// `chunks_per_step`; and to as many workgroups as there are CUs for where one round is all there is and that leaves a workgroup at most
// five eighths of its steps, two or more (a smaller part does not pay for the exchange, and in several rounds the next pair's loads run under it): 0.91
// to 0.94 of the time for 2850 such shapes.  To 64 at most, as every member reads every other's sums: one pair of 65 to 128 queries and 24576 to 32768 keys
// 18.0 us with as few as can hold them, 18.1 with a member per CU, 14.7 with 64, 14.6 with 96, 15.2 with 128; of 2 to 32 and 49152 to 65536 keys 17.2, 17.2, 14.8, 14.7 and
// 14.8.  Not where two query groups per wave hold twice the keys (1.05 for 85 shapes; the estimate that chose them counts on those).
void spread_keys(Params& p, int N, int chunks_per_step, int cap, bool may_widen) {
  const int steps = (N + chunks_per_step * kChunk - 1) / (chunks_per_step * kChunk);
  int per = (steps + p.splits - 1) / p.splits;
  if (may_widen && p.teams == p.bh_count) {
    const int places = cap / p.teams < 64 ? cap / p.teams : 64;
    int wide = (steps + places - 1) / places;
    if (wide < 2) wide = 2;
    if (8 * wide <= 5 * per) per = wide;
  }
  p.splits = (steps + per - 1) / per;
  p.run_chunks = per * chunks_per_step;
}

// The path for one query (one_query_*_kernel): sizes of its launches and its scratch, which lies behind everything
// fcr_lse_bytes asks for.  Any element type and any number of keys.
struct OneQueryPlan {
  int lanes;              // lanes per key row: the row's granules, rounded up to a power of two
  int splits, rows_wg;    // key ranges per pair and their length
  int64_t pitch;          // floats per pair of the score array
  int64_t part_at, scores_at, floats;   // where the pairs and the scores start and the workspace ends, in floats
};
OneQueryPlan one_query_plan(int dtype, int64_t bh, int N, int D, int64_t base_floats) {
  OneQueryPlan o;
  const int dgran = D * elem_bytes(dtype) / 16;
  for (o.lanes = 1; o.lanes < dgran;) o.lanes *= 2;
  const int64_t step = 4 * kOneLoads * (64 / o.lanes);   // keys a workgroup reads at a time
  // about 128 workgroups per CU, each with at least one step: they fit eight at a time, and many short ranges level
  // the end and read memory more nearly in order (default cache policy, 256 pairs of 9001 bf16 keys of 128: 16 per CU 120 us, 32: 118,
  // 64: 115, 128 and more: 112; token-major keys of 256 prefer 32: 237 against 243)
  int64_t splits = 128ll * chip_cus() / bh;
  const int64_t steps = (N + step - 1) / step;
  if (splits > steps) splits = steps;
  if (splits < 1) splits = 1;
  const int64_t steps_wg = (steps + splits - 1) / splits;
  o.rows_wg = (int)(steps_wg * step);
  o.splits = (int)((steps + steps_wg - 1) / steps_wg);
  o.pitch = ((int64_t)N + 63) / 64 * 64;
  o.part_at = (base_floats + 63) / 64 * 64;
  o.scores_at = o.part_at + (2 * bh * o.splits + 63) / 64 * 64;
  o.floats = o.scores_at + bh * o.pitch;
  return o;
}

// The path for pairs whose keys fit the registers of a workgroup (few_keys_kernel): up to 512 16-bit keys of 128, 256 of 256.  Against
// the two kernels, 11000 shapes of 1 to 1500 pairs, 2 to 8192 queries, 2 to 512 keys, all reductions, with and without the mask: 0.56 of their
// time where one launch does (below), 0.74 elsewhere.  Not taken for more than 128 keys where no two workgroups share a pair, sixteen chunks
// or more are done one behind the other (48 with at most 256 keys) and neither the pairs fill the chip nor the keys the registers (`filled`):
// two kernels -> here, 300 pairs of 5970 x 384 x 64, maxima, 262 -> 458 us, 257 of 4715 x 141 x 8 82 -> 153, 300 of 1831 x 400 x 96, both, 140 -> 205;
// nor for more than 256 keys of 64 bytes in such calls, whose time is the vector port's in both (1024 pairs of 2172 x 428 x 8, maxima, 215 -> 315).
// What that leaves out (526 shapes) takes 1.15 times as long here; of the others 2 % lose 3 % or more, most of them rows of 64 bytes against at
// most 128 keys.
// form -1: the other paths.
struct FewKeysPlan {
  int form;          // keys of a workgroup: 128 << form
  int splits;        // workgroups per pair
  int parts;         // sets of columns that they leave (16-bit operands: one each)
  int64_t part_at, floats;   // where the columns of the parts start and the workspace ends, in floats
};
// The same for fp32 operands in parts (few_keys_f32_kernel): up to 256 keys, in four waves up to 128 and in eight beyond; ks: k-steps of
// 32 d.  Against the two kernels, 11600 shapes of 1 to 1500 pairs, 40 to 8192 queries, all reductions, with and without the mask: 0.66 of
// their time where it is taken, 0.47 where several workgroups share a pair (2 pairs of 256 x 256 x 64 13.7 -> 8.9 us, 32 of 256 x 256 x 128 20.8 -> 11.9,
// 512 of them 77 -> 52, 4 of 4096 x 256 x 128 117 -> 17, 256 of them 480 -> 294).
// Below 1024 queries the path and the ranges of queries whose columns are added up apart (at most eight) follow from M, N and D alone, so that
// the bits of a result do not depend on the number of pairs; left out are rows of up to 128 bytes against so many queries that the sweeps, which stage
// four times the rows between two barriers, win for most numbers of pairs (206 of 900 x 172 x 48 1.15 times their time, 166 of 497 x 164 x 32 1.28).
// From 1024 on ranges are one to a workgroup, and long calls of short rows that fill neither the chip nor the registers are left out, as few_keys_plan
// does (`least`: 280 pairs of 5698 x 39 x 32, both, 199 -> 344; 137 of 7618 x 226 x 48 368 -> 479; 316 of 2605 x 14 x 32 93 -> 143).
// Of 30000 shapes that are taken (8 to 256 keys, D of 32 to 256; 0.579 of the time) 1.8 % lose 3 % or more, nearly all of them rows of D < 64 with 100 pairs or more (353 of 462 x 24 x 32, both,
// 24.3 -> 36.6; D = 64: 527 of 484 x 20 47 -> 59), where fewer pairs gain 10 to 25 %: the path must not follow from the number of pairs.  Two chunks (three of at most 128 keys) go to one workgroup, whose launch is
// the only one (2 pairs of 64 x 64 x 64 7.3 -> 6.5, but of 128 x 64 x 64 9.1 and 10.6).
FewKeysPlan few_keys_f32_plan(FewKeysPlan o, int64_t bh, int M, int N, int ks, bool both, int64_t base_floats) {
  if (N > 256) return o;
  const int form = N > 128 ? 1 : 0, rows = 16 * f32_groups(ks);
  const int64_t chunks = ((int64_t)M + rows - 1) / rows, places = (form == 1 ? 1 : 2) * (int64_t)chip_cus();
  const bool short_call = M < 1024;
  int64_t s = places / bh;
  if (s > chunks) s = chunks;
  if (s < 1 || chunks <= (form == 1 ? 2 : 3)) s = 1;
  const int64_t len = short_call ? (chunks + 7) / 8 : (chunks + s - 1) / s, parts = (chunks + len - 1) / len;   // (no part is empty)
  if (s > parts) s = parts;
  if (short_call) {
    if (ks == 1 ? chunks >= (form == 1 ? 8 : 16) : ks == 2 && form == 1 && chunks >= 16) return o;
  } else if (s <= 3) {
    // chunks one behind the other, and the share of the chip's workgroups and of their keys that is there
    const int64_t rounds = (bh * s + places - 1) / places, steps = rounds * ((chunks + s - 1) / s);
    const double filled = (double)(bh * s) / (double)(rounds * places) * N / (128 << form);
    double least = 0.0;
    if (form == 1) {
      if (ks == 1) least = 2.0;
      else if (ks == 2) least = steps >= 64 ? 0.85 : steps >= 32 ? 0.6 : 0.4;
      else if (steps >= 64) least = ks == 8 ? 0.3 : ks == 4 ? 0.4 : 0.5;
      else if (ks == 3) least = 0.4;
    } else if (ks == 1) {
      least = steps >= 64 ? 0.6 : steps >= 32 ? 0.4 : 0.3;
    } else if (ks == 2) {
      least = steps >= 64 ? 0.3 : steps >= 32 ? 0.2 : 0.1;
    } else if (ks > 4 && s == 1 && steps >= 64) {
      least = 0.1;
    }
    if (filled < least) return o;
  }
  o.form = form;
  o.splits = (int)s;
  o.parts = (int)parts;
  if (s > 1) {
    o.part_at = (base_floats + 63) / 64 * 64;
    o.floats = o.part_at + (both ? 2 : 1) * parts * bh * N;
  }
  return o;
}
FewKeysPlan few_keys_plan(int dtype, int B, int H, int M, int N, int D, bool both, int64_t base_floats) {
  FewKeysPlan o;
  o.form = -1;
  o.splits = o.parts = 1;
  o.part_at = o.floats = base_floats;
  const int ks = ksteps_of(dtype, D);
  const int64_t bh = (int64_t)B * H;
  if ((dtype == FCR_DTYPE_F32 ? !in_parts(dtype, D) : ks > kMaxKSteps) || M < 2 || B > 65535 || bh >= kMaxWorkgroups / 2) return o;   // (the grid's limits)
  if (dtype == FCR_DTYPE_F32) return few_keys_f32_plan(o, bh, M, N, f32_ksteps(ks), both, base_floats);
  const int groups = few_keys_groups(ks), most = groups == 4 ? 2 : 1;
  int form = 0;
  while (form <= most && N > (128 << form)) ++form;
  if (form > most) return o;
  o.form = form;
  const int waves = form == most ? 8 : 4;
  const int rows = 16 * few_keys_queries(ks);
  const int64_t chunks = ((int64_t)M + rows - 1) / rows;
  const int64_t places = (waves == 8 ? 1 : 2) * (int64_t)chip_cus();
  int64_t s = places / bh;
  if (s > chunks) s = chunks;
  if (s < 1) s = 1;
  // A few chunks go to one workgroup, whose launch is then the only one: 2 pairs of 64 x 64 x 128 8.8 -> 5.0 us per call, of 128 x 128 8.8 -> 6.1,
  // of 160 x 160 8.9 -> 8.4, but of 200 x 200 8.9 -> 11.0; rows of 512 bytes 100 x 100 8.8 -> 8.3, 128 x 128 8.7 -> 9.1; more than 256 keys
  // 96 x 500 x 64 8.9 -> 7.8, 128 x 500 x 128 10.4 -> 11.2.  (3840 shapes of all reductions, masks and up to 1500 pairs: two were slower.)
  if (chunks <= (form == 2 ? 3 : ks > 4 ? 7 : 5)) {
    s = 1;
  } else if (s == 1) {
    // chunks one behind the other, and the share of the chip's workgroups and of their keys that is there
    const int64_t rounds = (bh + places - 1) / places, steps = rounds * chunks;
    const double filled = (double)bh / (double)(rounds * places) * N / (128 << form);
    const bool many = steps >= 48;
    double least = 0.0;
    if (form == 2) least = steps < 16 ? 0.0 : ks == 1 ? 2.0 : ks == 2 ? (many ? 0.7 : 0.6) : many ? 0.5 : 0.4;
    else if (form == 1 && many) least = ks == 1 ? 0.6 : ks > 4 ? 0.45 : 0.0;
    if (filled < least) {
      o.form = -1;
      return o;
    }
  }
  o.splits = o.parts = (int)s;
  if (s > 1) {
    o.part_at = (base_floats + 63) / 64 * 64;
    o.floats = o.part_at + (both ? 2 : 1) * s * bh * N;
  }
  return o;
}

// Both sweeps in one launch (both_sweeps_kernel): 32-row blocks per wave of its row and its column tiles; row_blocks 0: two launches.
// The column sweeps start where row sweeps leave a CU, so a launch that does not fill its last round no longer costs a round twice, and
// where the mask gives row tiles that end early the column sweeps follow them.  What two launches have and one has not: keys split over workgroups where there are few
// row tiles, rounds that tiles fill exactly, both second helpings dealt backwards (map_group), and no words to fill, which counts in calls of 20 us.
// `rows` and `small`: tiles of 256 and of 128 rows per CU.  Figures: one launch's time against two's, of 30700 shapes of 1 to 2500 pairs, 130 to 9000 queries, 513 to 50000
// keys, fp16 and bf16, all reductions, as a geometric mean and the share that loses 3 % or more.  What is taken: 0.922, 1.7 % (0.845 below one round; 1.15 at worst); what the
// cuts below leave to two launches: 0.994, 21 % (1.39).  us, two launches -> one:
//   With the mask and at most 1.5 keys per query (`level`) the column sweeps can follow the row sweeps from the start: 0.911.  Rows of 129 to 256 bytes have 128-row tiles up
//   to 0.9 (11 of 4078 x 128 103 -> 68), 256-row ones for rows up to 1.9 (27 of 2240 65 -> 55), for both beyond (155 of 1538 151 -> 134); others 128-row tiles (10 of
//   1895 x 256 54 -> 41, 32 of 2048 79 -> 69, 259 of 626 x 64 41 -> 35).
//   With the mask and more keys than that 0.961, without it 0.929: no column can start before the rows of its pair end, so there has to be a row tile for every
//   CU (24 of 2893 x 128 144 -> 122, 18 of 7902 x 64 449 -> 359).
struct BothPlan {
  int row_blocks = 0, col_blocks = 0;
};
BothPlan both_plan(int dtype, int ksteps, int64_t bh, int M, int N, bool causal) {
  BothPlan o;
  // (a wait is bounded by polls, a microsecond or more each: row sweeps of up to 2^20 keys take a tenth of the default bound)
  if (dtype == FCR_DTYPE_F32 || ksteps > kMaxKSteps || M <= kSmallRows || M > (1 << 20) || N > (1 << 20)) return o;
  const int cus = chip_cus();
  const int64_t tiles = bh * ((M + 127) / 128), cols = bh * ((N + 127) / 128);   // of 128 rows
  if (tiles + cols >= kMaxWorkgroups / 2) return o;
  const double small = (double)tiles / cus, rows = (double)(bh * ((M + 255) / 256)) / cus;
  const bool longer = 2 * (int64_t)N > 3 * (int64_t)M, level = causal && !longer;
  auto within = [&](double from, double to) { return rows >= from && rows < to; };
  // few tiles, whose keys two launches split: 0.99, 28 %, and 1.006, 33 % (1 pair of 6891 x 8176 x 32 46 -> 64); the rest below 0.4 0.875
  if (level && ((small < 0.26 && 20 * (int64_t)N > 23 * (int64_t)M) || (small < 0.4 && bh == 1 && ksteps <= 3))) return o;
  // Multiples of eight pairs, which deal every die whole pairs, leave two launches less to gain: 0.999, 28 % between 0.9 and 2.7 rounds of 193 to 256 bytes (72 of
  // 840 x 128 26 -> 32; other numbers of pairs 0.947, 6 %), 0.985, 12 % of 129 to 192 (0.966, 5 %), 0.983, 8 % of more than 256 (0.969, 1 %).
  const bool whole = bh % 8 == 0 && level;
  if (whole && (ksteps > 4 ? within(1.3, 1.9) : ksteps == 4 ? within(0.9, 2.7) : ksteps == 3 && within(0.9, 4.0))) return o;
  // A few hundred queries against many keys: 0.997, 30 % (246 of 314 x 8281 x 96 387 -> 440: 256-row tiles, where two launches have three of 128); the rest of up to 384 queries 0.945.
  if (longer && M <= 384 && (ksteps <= 2 ? M <= 256 || rows >= 4.0 : ksteps <= 4 ? M > 256 : M <= 256 && rows >= 2.0)) return o;
  int nr = 1, nc = 1;
  if (ksteps > 4) {
    if (rows >= 5.0) return o;                                                   // 0.99 (216 pairs of 1562 x 256 290 -> 309)
    if (!level && small < 1.05) return o;
    if (longer && causal && N >= 11000 && rows < 2.0) return o;                  // 1.004, 10 % (17 of 6554 x 20777 x 256 1771 -> 1987); the rest 0.975
    if (!causal && rows < 1.0 && (small >= 1.5 || 10 * (int64_t)N < 9 * (int64_t)M)) return o;   // 0.994, 12 %; the rest below one round 0.895
  } else if (level && ksteps <= 2) {
    if (rows >= 16.0 || within(1.1, 2.7) || (rows >= 2.7 && N >= 10000)) return o;   // (61 of 2304 x 64 68 -> 75, 10 of 8777 138 -> 148)
    if (N < 700 && within(0.6, 1.1)) return o;                                   // 1.03, 56 % (58 of 671 x 562 x 32 14.1 -> 15.5); with more keys 0.814
  } else if (level) {
    if (rows >= 10.0 || within(2.1, 2.65) || (rows >= 2.65 && N >= 8000)) return o;  // as fast (48 of 2929 x 128 118 -> 120, 32 of 8192 468 -> 472)
    if (N >= 3400 && within(1.85, 2.1)) return o;                                // 0.97, 18 %; with fewer keys 0.936
    if (ksteps == 3 && within(1.0, 2.65)) return o;                              // 0.99, 21 % (25 of 4880 x 80 145 -> 168)
    if (N < 1000 && (ksteps == 3 ? within(0.6, 1.0) : within(0.9, 1.1))) return o;   // 0.99, 33 %, and 0.985, 39 %; with more keys 0.786 and 0.912
    nr = rows >= 0.9 ? 2 : 1;
    nc = rows >= 1.9 ? 2 : 1;
  } else {
    if (rows >= 10.0 || (longer && rows < (ksteps <= 2 ? 1.1 : 1.85))) return o; // (68 of 1090 x 8104 x 128 318 -> 334)
    if (!longer && (small < 1.02 || rows < (ksteps <= 2 ? 0.67 : 1.0))) return o;   // 0.997, 23 %, and 0.98, 26 % (5 of 7839 x 6211 x 128 148 -> 198); beyond 0.92
    if (!longer && ksteps <= 2 && small >= 1.5 && rows < 1.1) return o;
    if (ksteps > 2) {
      nr = rows >= 1.5 ? 2 : 1;
      nc = rows >= 1.85 ? 2 : 1;
    }
  }
  o.row_blocks = nr;
  o.col_blocks = nc;
  return o;
}

// Where the status word of both_sweeps_kernel stands in a workspace of fcr_workspace_bytes, in floats, for problems that take it with the mask or
// without (the size does not know which); -1 where there is none, as where few_keys_kernel is meant, whose columns may lie there.
// base_floats: what fcr_lse_bytes asks for.
constexpr int kStatusFloats = 32;
int64_t both_status_at(int dtype, int B, int H, int M, int N, int D, int64_t base_floats) {
  const int ksteps = ksteps_of(dtype, D);
  const int64_t bh = (int64_t)B * H;
  if (both_plan(dtype, ksteps, bh, M, N, true).row_blocks == 0 && both_plan(dtype, ksteps, bh, M, N, false).row_blocks == 0) return -1;
  return few_keys_plan(dtype, B, H, M, N, D, false, base_floats).form >= 0 ? -1 : (base_floats + 63) / 64 * 64;
}

int launched(const char* what) {
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) return 0;
  snprintf(g_err, sizeof(g_err), "%s launch failed: %s", what, hipGetErrorString(e));
  return (int)e;
}

// one row tile per (b,h) and at least 1 GiB of keys: stream them past the caches
inline bool keys_read_once(const Params& p) {
  return p.tiles == 1 && (int64_t)p.bh_count * p.N * p.dgran * 16 >= (1ll << 30);
}

template <int DT, int KS, int NB, bool ONCE>
void launch_lse_blocks(const Params& p, bool causal, hipStream_t s) {
  const dim3 grid(p.total), block(kThreads);
  if (causal) hipLaunchKernelGGL((row_lse_kernel<DT, KS, true, NB, ONCE>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((row_lse_kernel<DT, KS, false, NB, ONCE>), grid, block, 0, s, p);
}

template <int DT, int KS>
void launch_lse(const Params& p, bool causal, hipStream_t s) {
  if constexpr (DT == FCR_DTYPE_F32) {
    if (row_half_tiles(DT, p.dgran * 4, p.M, p.N, p.bh_count)) {
      if (keys_read_once(p)) return launch_lse_blocks<DT, KS, 0, true>(p, causal, s);
      return launch_lse_blocks<DT, KS, 0, false>(p, causal, s);
    }
  }
  if constexpr (KS <= 4) {
    if (row_blocks_per_wave(KS, p.M, p.N, p.bh_count, causal) == 2) return launch_lse_blocks<DT, KS, 2, false>(p, causal, s);
  }
  if (keys_read_once(p)) return launch_lse_blocks<DT, KS, 1, true>(p, causal, s);
  launch_lse_blocks<DT, KS, 1, false>(p, causal, s);
}

template <int DT, int KS, int MODE>
void launch_col_mode(const Params& p, bool causal, hipStream_t s) {
  const dim3 grid(p.total), block(kThreads);
  constexpr int NB = (MODE == kModeBoth && KS == 1) ? 1 : blocks_per_wave(KS);   // (see col_tile_blocks)
  if constexpr (DT == FCR_DTYPE_F32) {
    if (half_tiles(DT, p.dgran * 4, p.N, p.bh_count)) {
      if (causal) hipLaunchKernelGGL((col_reduce_kernel<DT, KS, true, MODE, 0>), grid, block, 0, s, p);
      else hipLaunchKernelGGL((col_reduce_kernel<DT, KS, false, MODE, 0>), grid, block, 0, s, p);
      return;
    }
  }
  if constexpr (NB == 2) {
    if (col_tile_blocks(KS, MODE, p.N, p.bh_count, causal) == 1) {
      if (causal) hipLaunchKernelGGL((col_reduce_kernel<DT, KS, true, MODE, 1>), grid, block, 0, s, p);
      else hipLaunchKernelGGL((col_reduce_kernel<DT, KS, false, MODE, 1>), grid, block, 0, s, p);
      return;
    }
  }
  if (causal) hipLaunchKernelGGL((col_reduce_kernel<DT, KS, true, MODE, NB>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((col_reduce_kernel<DT, KS, false, MODE, NB>), grid, block, 0, s, p);
}

template <int KS, int NW, int NG>
void launch_lse_f32_tile(const Params& p, bool causal, hipStream_t s) {
  const dim3 grid(p.total), block(64 * NW);
  if (keys_read_once(p)) {
    if (causal) hipLaunchKernelGGL((row_lse_f32_kernel<KS, true, NG, true, NW>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((row_lse_f32_kernel<KS, false, NG, true, NW>), grid, block, 0, s, p);
    return;
  }
  if (causal) hipLaunchKernelGGL((row_lse_f32_kernel<KS, true, NG, false, NW>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((row_lse_f32_kernel<KS, false, NG, false, NW>), grid, block, 0, s, p);
}

template <int KS>
void launch_lse_f32(const Params& p, bool causal, hipStream_t s) {
  const F32Tile t = f32_row_tile(p.M, p.N, p.bh_count, causal);
  if (t.waves == 4) t.groups == 1 ? launch_lse_f32_tile<KS, 4, 1>(p, causal, s) : launch_lse_f32_tile<KS, 4, 2>(p, causal, s);
  else t.groups == 1 ? launch_lse_f32_tile<KS, 8, 1>(p, causal, s) : launch_lse_f32_tile<KS, 8, 2>(p, causal, s);
}

template <int KS, int MODE, int NW, int NG>
void launch_col_f32_tile(const Params& p, bool causal, hipStream_t s) {
  const dim3 grid(p.total), block(64 * NW);
  if (causal) hipLaunchKernelGGL((col_reduce_f32_kernel<KS, true, MODE, NG, NW>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((col_reduce_f32_kernel<KS, false, MODE, NG, NW>), grid, block, 0, s, p);
}

template <int KS, int MODE>
void launch_col_f32_mode(const Params& p, bool causal, hipStream_t s) {
  const F32Tile t = f32_col_tile(KS, MODE == kModeBoth, p.M, p.N, p.bh_count, causal);
  if (t.waves == 4) t.groups == 1 ? launch_col_f32_tile<KS, MODE, 4, 1>(p, causal, s) : launch_col_f32_tile<KS, MODE, 4, 2>(p, causal, s);
  else t.groups == 1 ? launch_col_f32_tile<KS, MODE, 8, 1>(p, causal, s) : launch_col_f32_tile<KS, MODE, 8, 2>(p, causal, s);
}

template <int KS>
void launch_col_f32(const Params& p, bool causal, int mode, hipStream_t s) {
  if (mode == kModeSum) launch_col_f32_mode<KS, kModeSum>(p, causal, s);
  else if (mode == kModeMax) launch_col_f32_mode<KS, kModeMax>(p, causal, s);
  else launch_col_f32_mode<KS, kModeBoth>(p, causal, s);
}

template <int DT, int KS, int MODE, int NG>
void launch_col_small_groups(const Params& p, bool causal, hipStream_t s) {
  const dim3 grid(p.total), block(kThreads);
  if (causal) hipLaunchKernelGGL((col_small_kernel<DT, KS, true, MODE, NG>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((col_small_kernel<DT, KS, false, MODE, NG>), grid, block, 0, s, p);
}

template <int DT, int KS, int MODE>
void launch_col_small_mode(const Params& p, bool causal, hipStream_t s) {
  if (p.M <= 64) launch_col_small_groups<DT, KS, MODE, 4>(p, causal, s);
  else launch_col_small_groups<DT, KS, MODE, 8>(p, causal, s);
}

template <int DT, int KS>
void launch_col_small(const Params& p, bool causal, int mode, hipStream_t s) {
  if (mode == kModeSum) launch_col_small_mode<DT, KS, kModeSum>(p, causal, s);
  else if (mode == kModeMax) launch_col_small_mode<DT, KS, kModeMax>(p, causal, s);
  else launch_col_small_mode<DT, KS, kModeBoth>(p, causal, s);
}

// Workgroups of col_fused_kernel wait for each other, so all of a launch must be on the chip together: the
// host plans with two workgroups of 256 threads, or one of 512, per CU, and the launch is refused (the caller
// then takes the two-kernel path) if the runtime says that this build of the kernel does not fit that way.
template <class K>
bool fits_per_cu(K kernel, int threads, int want) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, 0) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return n >= want;
}

template <int DT, int KS, int MODE, int QH, int NQ, bool SKIP, int NW>
void launch_col_fused_form(const Params& p, bool causal, hipStream_t s) {
  const dim3 grid(p.total), block(64 * NW);
  static int fits[2] = {-1, -1};   // asked once per kernel (the answer depends on its registers and LDS, not on the device of a kind)
  int f = __atomic_load_n(&fits[causal], __ATOMIC_RELAXED);
  if (f < 0) {
    f = causal ? fits_per_cu(col_fused_kernel<DT, KS, true, MODE, QH, NQ, SKIP, NW>, 64 * NW, 8 / NW)
               : fits_per_cu(col_fused_kernel<DT, KS, false, MODE, QH, NQ, SKIP, NW>, 64 * NW, 8 / NW);
    __atomic_store_n(&fits[causal], f, __ATOMIC_RELAXED);
  }
  if (!f) {
    fcr_detail::fused_refused = true;
    return;
  }
  if (causal) hipLaunchKernelGGL((col_fused_kernel<DT, KS, true, MODE, QH, NQ, SKIP, NW>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((col_fused_kernel<DT, KS, false, MODE, QH, NQ, SKIP, NW>), grid, block, 0, s, p);
}

// More than 64 queries: where there is nothing to leave out the question alone costs (4 x 32 pairs of 89 x 4096 x 64
// 40.7 -> 42.6 us, 32 of 128 x 4096 x 128 17.6 -> 17.8), so the host asks it; elsewhere leaving chunks out takes 0.94 (maxima, both) of the time.
template <int DT, int KS, int MODE, int QH, int NQ, int NW>
void launch_col_fused_mode(const Params& p, bool causal, hipStream_t s) {
  if constexpr (QH == 2) {
    const int chunks = (p.N + kChunk - 1) / kChunk;
    if (p.run_chunks != fused_chunks(QH, NQ) || chunks % p.run_chunks != 0) return launch_col_fused_form<DT, KS, MODE, QH, NQ, true, NW>(p, causal, s);
    launch_col_fused_form<DT, KS, MODE, QH, NQ, false, NW>(p, causal, s);
  } else {
    launch_col_fused_form<DT, KS, MODE, QH, NQ, true, NW>(p, causal, s);
  }
}

template <int DT, int KS, int QH, int NQ, int NW>
void launch_col_fused_groups(const Params& p, bool causal, int m, hipStream_t s) {
  if (m == kModeSum) launch_col_fused_mode<DT, KS, kModeSum, QH, NQ, NW>(p, causal, s);
  else if (m == kModeMax) launch_col_fused_mode<DT, KS, kModeMax, QH, NQ, NW>(p, causal, s);
  else launch_col_fused_mode<DT, KS, kModeBoth, QH, NQ, NW>(p, causal, s);
}

// mode: kModeSum, kModeMax or kModeBoth, + 4 for more than 64 queries, + 8 for two groups of sixteen queries
// per wave, + 16 for that in four waves
template <int DT, int KS>
void launch_col_fused(const Params& p, bool causal, int mode, hipStream_t s) {
  const int m = mode & 3;
  if (mode & 4) launch_col_fused_groups<DT, KS, 2, 4, 8>(p, causal, m, s);
  else if (mode & 16) launch_col_fused_groups<DT, KS, 1, 2, 4>(p, causal, m, s);
  else if (mode & 8) launch_col_fused_groups<DT, KS, 1, 2, 8>(p, causal, m, s);
  else launch_col_fused_groups<DT, KS, 1, 4, 8>(p, causal, m, s);
}

template <int DT, int KS>
void launch_col(const Params& p, bool causal, int mode, hipStream_t s) {
  if (mode == kModeSum) launch_col_mode<DT, KS, kModeSum>(p, causal, s);
  else if (mode == kModeMax) launch_col_mode<DT, KS, kModeMax>(p, causal, s);
  else launch_col_mode<DT, KS, kModeBoth>(p, causal, s);
}

template <int DT, int KS, int MODE, int NG, int NW>
void launch_few_keys_form(const Params& p, bool causal, hipStream_t s) {
  const dim3 grid((unsigned)p.H, (unsigned)(p.bh_count / p.H), (unsigned)p.splits), block(64 * NW);
  if (causal) hipLaunchKernelGGL((few_keys_kernel<DT, KS, true, MODE, NG, NW>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((few_keys_kernel<DT, KS, false, MODE, NG, NW>), grid, block, 0, s, p);
}

template <int DT, int KS, int MODE>
void launch_few_keys_mode(const Params& p, bool causal, int form, hipStream_t s) {
  if (form == 0) return launch_few_keys_form<DT, KS, MODE, 2, 4>(p, causal, s);
  if constexpr (few_keys_groups(KS) == 2) {
    launch_few_keys_form<DT, KS, MODE, 2, 8>(p, causal, s);
  } else {
    if (form == 1) launch_few_keys_form<DT, KS, MODE, 4, 4>(p, causal, s);
    else launch_few_keys_form<DT, KS, MODE, 4, 8>(p, causal, s);
  }
}

template <int DT, int KS>
void launch_few_keys(const Params& p, bool causal, int mode, int form, hipStream_t s) {
  if (mode == kModeSum) launch_few_keys_mode<DT, KS, kModeSum>(p, causal, form, s);
  else if (mode == kModeMax) launch_few_keys_mode<DT, KS, kModeMax>(p, causal, form, s);
  else launch_few_keys_mode<DT, KS, kModeBoth>(p, causal, form, s);
}

template <int KS, int MODE, int NG, int NW>
void launch_few_keys_f32_form(const Params& p, bool causal, hipStream_t s) {
  const dim3 grid((unsigned)p.H, (unsigned)(p.bh_count / p.H), (unsigned)p.splits), block(64 * NW);
  if (causal) hipLaunchKernelGGL((few_keys_f32_kernel<KS, true, MODE, NG, NW>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((few_keys_f32_kernel<KS, false, MODE, NG, NW>), grid, block, 0, s, p);
}
template <int KS, int MODE>
void launch_few_keys_f32_mode(const Params& p, bool causal, int form, hipStream_t s) {
  if (form == 0) return launch_few_keys_f32_form<KS, MODE, 2, 4>(p, causal, s);
  launch_few_keys_f32_form<KS, MODE, 2, 8>(p, causal, s);
}
template <int KS>
void launch_few_keys_f32(const Params& p, bool causal, int mode, int form, hipStream_t s) {
  if (mode == kModeSum) launch_few_keys_f32_mode<KS, kModeSum>(p, causal, form, s);
  else if (mode == kModeMax) launch_few_keys_f32_mode<KS, kModeMax>(p, causal, form, s);
  else launch_few_keys_f32_mode<KS, kModeBoth>(p, causal, form, s);
}

template <int DT, int KS, int MODE, int NBR, int NBC>
void launch_both_tiles(const Params& p, bool causal, hipStream_t s) {
  const dim3 grid((unsigned)(((p.total + 7) & ~7) + p.bh_count * p.col_tiles)), block(kThreads);
  if (causal) hipLaunchKernelGGL((both_sweeps_kernel<DT, KS, true, MODE, NBR, NBC>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((both_sweeps_kernel<DT, KS, false, MODE, NBR, NBC>), grid, block, 0, s, p);
}
template <int DT, int KS, int MODE>
void launch_both_mode(const Params& p, bool causal, hipStream_t s) {
  if constexpr (KS == 3 || KS == 4) {
    if (p.row_blocks == 2 && p.col_blocks == 2) return launch_both_tiles<DT, KS, MODE, 2, 2>(p, causal, s);
    if (p.row_blocks == 2) return launch_both_tiles<DT, KS, MODE, 2, 1>(p, causal, s);
  }
  launch_both_tiles<DT, KS, MODE, 1, 1>(p, causal, s);
}
template <int DT, int KS>
void launch_both(const Params& p, bool causal, int mode, hipStream_t s) {
  if (mode == kModeSum) launch_both_mode<DT, KS, kModeSum>(p, causal, s);
  else if (mode == kModeMax) launch_both_mode<DT, KS, kModeMax>(p, causal, s);
  else launch_both_mode<DT, KS, kModeBoth>(p, causal, s);
}

#define FCR_DISPATCH_KS(DT, ksteps, CALL)                  \
  switch (ksteps) {                                        \
    case 1: CALL(DT, 1); break;                            \
    case 2: CALL(DT, 2); break;                            \
    case 3: CALL(DT, 3); break;                            \
    case 4: CALL(DT, 4); break;                            \
    case 5: CALL(DT, 5); break;                            \
    case 6: CALL(DT, 6); break;                            \
    case 7: CALL(DT, 7); break;                            \
    default: CALL(DT, 8); break;                           \
  }

// rows of more than 512 bytes: 9 to 16 k-steps
#define FCR_DISPATCH_KS_LONG(DT, ksteps, CALL)             \
  switch (ksteps) {                                        \
    case 9: CALL(DT, 9); break;                            \
    case 10: CALL(DT, 10); break;                          \
    case 11: CALL(DT, 11); break;                          \
    case 12: CALL(DT, 12); break;                          \
    case 13: CALL(DT, 13); break;                          \
    case 14: CALL(DT, 14); break;                          \
    case 15: CALL(DT, 15); break;                          \
    default: CALL(DT, 16); break;                          \
  }

#define FCR_DISPATCH_KS4(DT, ksteps, CALL)                 \
  switch (ksteps) {                                        \
    case 1: CALL(DT, 1); break;                            \
    case 2: CALL(DT, 2); break;                            \
    case 3: CALL(DT, 3); break;                            \
    default: CALL(DT, 4); break;                           \
  }

}  // namespace

// The sweeps of one element type (see the declarations at the top).
#define FCR_CALL_LSE(DT, KS) launch_lse<DT, KS>(p, causal, s)
#define FCR_CALL_COL(DT, KS) launch_col<DT, KS>(p, causal, mode, s)
#define FCR_CALL_COL_SMALL(DT, KS) launch_col_small<DT, KS>(p, causal, mode, s)
#define FCR_CALL_COL_FUSED(DT, KS) launch_col_fused<DT, KS>(p, causal, mode, s)
#define FCR_CALL_FEW_KEYS(DT, KS) launch_few_keys<DT, KS>(p, causal, mode, form, s)
#define FCR_SWEEPS_16BIT(NAME, DT)                                                                       \
  void fcr_detail::NAME(int which, const Params& p, int ksteps, bool causal, int mode, hipStream_t s) { \
    if (which == 0) { FCR_DISPATCH_KS(DT, ksteps, FCR_CALL_LSE) }                                        \
    else if (which == 1) { FCR_DISPATCH_KS(DT, ksteps, FCR_CALL_COL) }                                   \
    else { FCR_DISPATCH_KS4(DT, ksteps, FCR_CALL_COL_SMALL) }                                            \
  }
#if FCR_HAS(1)
FCR_SWEEPS_16BIT(sweeps_f16, FCR_DTYPE_F16)
#endif
#if FCR_HAS(2)
FCR_SWEEPS_16BIT(sweeps_bf16, FCR_DTYPE_BF16)
#endif
#if FCR_HAS(7)
void fcr_detail::sweeps_f16_single(const Params& p, int ksteps, bool causal, int mode, hipStream_t s) {
  FCR_DISPATCH_KS4(FCR_DTYPE_F16, ksteps, FCR_CALL_COL_FUSED)
}
#endif
#if FCR_HAS(8)
void fcr_detail::sweeps_bf16_single(const Params& p, int ksteps, bool causal, int mode, hipStream_t s) {
  FCR_DISPATCH_KS4(FCR_DTYPE_BF16, ksteps, FCR_CALL_COL_FUSED)
}
#endif
#if FCR_HAS(9)
void fcr_detail::sweeps_f16_few_keys(const Params& p, int ksteps, bool causal, int mode, int form, hipStream_t s) {
  FCR_DISPATCH_KS(FCR_DTYPE_F16, ksteps, FCR_CALL_FEW_KEYS)
}
#endif
#if FCR_HAS(10)
void fcr_detail::sweeps_bf16_few_keys(const Params& p, int ksteps, bool causal, int mode, int form, hipStream_t s) {
  FCR_DISPATCH_KS(FCR_DTYPE_BF16, ksteps, FCR_CALL_FEW_KEYS)
}
#endif
#define FCR_CALL_BOTH(DT, KS) launch_both<DT, KS>(p, causal, mode, s)
#if FCR_HAS(11)
void fcr_detail::sweeps_f16_both(const Params& p, int ksteps, bool causal, int mode, hipStream_t s) {
  FCR_DISPATCH_KS(FCR_DTYPE_F16, ksteps, FCR_CALL_BOTH)
}
#endif
#if FCR_HAS(12)
void fcr_detail::sweeps_bf16_both(const Params& p, int ksteps, bool causal, int mode, hipStream_t s) {
  FCR_DISPATCH_KS(FCR_DTYPE_BF16, ksteps, FCR_CALL_BOTH)
}
#endif
#if FCR_HAS(13)
void fcr_detail::sweeps_f32_few_keys(const Params& p, int ksteps, bool causal, int mode, int form, hipStream_t s) {
  switch (f32_ksteps(ksteps)) {
    case 1: launch_few_keys_f32<1>(p, causal, mode, form, s); break;
    case 2: launch_few_keys_f32<2>(p, causal, mode, form, s); break;
    case 3: launch_few_keys_f32<3>(p, causal, mode, form, s); break;
    case 4: launch_few_keys_f32<4>(p, causal, mode, form, s); break;
    case 5: launch_few_keys_f32<5>(p, causal, mode, form, s); break;
    case 6: launch_few_keys_f32<6>(p, causal, mode, form, s); break;
    case 7: launch_few_keys_f32<7>(p, causal, mode, form, s); break;
    default: launch_few_keys_f32<8>(p, causal, mode, form, s); break;
  }
}
#endif
#if FCR_HAS(3)
void fcr_detail::sweeps_f32(int which, const Params& p, int ksteps, bool causal, int mode, hipStream_t s) {
  if (!in_parts(FCR_DTYPE_F32, p.dgran * 4)) {
    constexpr int DT = FCR_DTYPE_F32;
    if (ksteps == 1) which == 0 ? launch_lse<DT, 1>(p, causal, s) : launch_col<DT, 1>(p, causal, mode, s);
    else which == 0 ? launch_lse<DT, 2>(p, causal, s) : launch_col<DT, 2>(p, causal, mode, s);
    return;
  }
  switch (f32_ksteps(ksteps)) {
    case 1: which == 0 ? launch_lse_f32<1>(p, causal, s) : launch_col_f32<1>(p, causal, mode, s); break;
    case 2: which == 0 ? launch_lse_f32<2>(p, causal, s) : launch_col_f32<2>(p, causal, mode, s); break;
    case 3: which == 0 ? launch_lse_f32<3>(p, causal, s) : launch_col_f32<3>(p, causal, mode, s); break;
    default: which == 0 ? launch_lse_f32<4>(p, causal, s) : launch_col_f32<4>(p, causal, mode, s); break;
  }
}
#endif
#if FCR_HAS(4)
void fcr_detail::sweeps_f32_long_rows(int which, const Params& p, int ksteps, bool causal, int mode, hipStream_t s) {
  switch (f32_ksteps(ksteps)) {
    case 5: which == 0 ? launch_lse_f32<5>(p, causal, s) : launch_col_f32<5>(p, causal, mode, s); break;
    case 6: which == 0 ? launch_lse_f32<6>(p, causal, s) : launch_col_f32<6>(p, causal, mode, s); break;
    case 7: which == 0 ? launch_lse_f32<7>(p, causal, s) : launch_col_f32<7>(p, causal, mode, s); break;
    default: which == 0 ? launch_lse_f32<8>(p, causal, s) : launch_col_f32<8>(p, causal, mode, s); break;
  }
}
#endif
#if FCR_HAS(5)
void fcr_detail::sweeps_f16_long_rows(int which, const Params& p, int ksteps, bool causal, int mode, hipStream_t s) {
  if (which == 0) { FCR_DISPATCH_KS_LONG(FCR_DTYPE_F16, ksteps, FCR_CALL_LSE) }
  else { FCR_DISPATCH_KS_LONG(FCR_DTYPE_F16, ksteps, FCR_CALL_COL) }
}
#endif
#if FCR_HAS(6)
void fcr_detail::sweeps_bf16_long_rows(int which, const Params& p, int ksteps, bool causal, int mode, hipStream_t s) {
  if (which == 0) { FCR_DISPATCH_KS_LONG(FCR_DTYPE_BF16, ksteps, FCR_CALL_LSE) }
  else { FCR_DISPATCH_KS_LONG(FCR_DTYPE_BF16, ksteps, FCR_CALL_COL) }
}
#endif
#undef FCR_CALL_LSE
#undef FCR_CALL_COL
#undef FCR_CALL_COL_SMALL
#undef FCR_CALL_COL_FUSED
#undef FCR_CALL_FEW_KEYS

#if FCR_HAS(0)
namespace {
// process-wide switches (fcr_set_option)
int g_single_sweep = 1;
long long g_wait_polls = 1ll << 20;

// sweeps of the element type `dtype`
void launch_sweeps(int dtype, int which, const Params& p, int ksteps, bool causal, int mode, hipStream_t s,
                   unsigned* zero = nullptr, int zero_words = 0) {
  if (zero_words > 0)
    hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)((zero_words + 1023) / 1024)), dim3(256), 0, s, zero, zero_words, p.sync);
  const bool long_rows = ksteps > kMaxKSteps;
  if (which == 3) {   // the single sweep: 16-bit elements, rows of at most 256 bytes
    if (dtype == FCR_DTYPE_F16) fcr_detail::sweeps_f16_single(p, ksteps, causal, mode, s);
    else fcr_detail::sweeps_bf16_single(p, ksteps, causal, mode, s);
    return;
  }
  if (dtype == FCR_DTYPE_F16) (long_rows ? fcr_detail::sweeps_f16_long_rows : fcr_detail::sweeps_f16)(which, p, ksteps, causal, mode, s);
  else if (dtype == FCR_DTYPE_BF16) (long_rows ? fcr_detail::sweeps_bf16_long_rows : fcr_detail::sweeps_bf16)(which, p, ksteps, causal, mode, s);
  else (long_rows ? fcr_detail::sweeps_f32_long_rows : fcr_detail::sweeps_f32)(which, p, ksteps, causal, mode, s);
}

template <int DT, bool ONCE>
void launch_one_query_scores(const Params& p, const OneQueryPlan& o, float* scores, hipStream_t s) {
  const dim3 grid((unsigned)p.total), block(256);
  switch (o.lanes) {
    case 1: hipLaunchKernelGGL((one_query_scores_kernel<DT, 1, ONCE>), grid, block, 0, s, p, scores, o.pitch, o.rows_wg); break;
    case 2: hipLaunchKernelGGL((one_query_scores_kernel<DT, 2, ONCE>), grid, block, 0, s, p, scores, o.pitch, o.rows_wg); break;
    case 4: hipLaunchKernelGGL((one_query_scores_kernel<DT, 4, ONCE>), grid, block, 0, s, p, scores, o.pitch, o.rows_wg); break;
    case 8: hipLaunchKernelGGL((one_query_scores_kernel<DT, 8, ONCE>), grid, block, 0, s, p, scores, o.pitch, o.rows_wg); break;
    case 16: hipLaunchKernelGGL((one_query_scores_kernel<DT, 16, ONCE>), grid, block, 0, s, p, scores, o.pitch, o.rows_wg); break;
    case 32: hipLaunchKernelGGL((one_query_scores_kernel<DT, 32, ONCE>), grid, block, 0, s, p, scores, o.pitch, o.rows_wg); break;
    default: hipLaunchKernelGGL((one_query_scores_kernel<DT, 64, ONCE>), grid, block, 0, s, p, scores, o.pitch, o.rows_wg); break;
  }
}
template <int DT>
void launch_one_query_scores(bool once, const Params& p, const OneQueryPlan& o, float* scores, hipStream_t s) {
  if (once) launch_one_query_scores<DT, true>(p, o, scores, s);
  else launch_one_query_scores<DT, false>(p, o, scores, s);
}

// Keys that a workgroup reads while the second launch of the other way would still be on its way to the device, 256 KiB, or, where
// the pairs are a workgroup for at least every other CU and no second round, 1 MiB.  us per call, two launches and one, bf16 keys of 128,
// calls queued behind each other: 8 pairs of 512 6.7, 4.8, of 1024 7.0, 6.5, but of 2048 7.0, 10.1; 100 of 1024 10.3, 6.8; 256 of 64 6.5, 3.7, of
// 512 10.4, 5.3, of 1024 15.5, 13.7, of 2048 25.1, 21.9, of 4096 46.4, 41.1, but of 8192 91.0, 94.5; 640 pairs of 512 17.8, 18.6.
// A load spans `lanes` granules whatever the row holds of them, and a few pairs wait for nothing but their loads: there rows of 17
// granules in 32 lanes count as 32 (keys of 136: 1 pair of 764 6.5, 8.1, 4 of 938 7.0, 9.4, 24 of 960 7.8, 9.6; of 320: 4 of 377 6.8, 8.8).
inline bool one_query_alone(const Params& p, int lanes) {
  const int cus = chip_cus();
  if (p.bh_count > cus || p.N > kOnePairKeys) return false;
  const int64_t bytes = (int64_t)p.N * p.dgran * 16, loaded = (int64_t)p.N * lanes * 16;
  if (2 * (int64_t)p.bh_count >= cus) return bytes <= 1 << 20;
  const int64_t most = 16 * (int64_t)p.bh_count < cus ? 256 << 10 : 4 * (int64_t)p.bh_count < cus ? 384 << 10 : 512 << 10;
  return bytes <= 256 << 10 && loaded <= most;
}

template <int DT>
void launch_one_query_pair(const Params& p, int lanes, int mode, hipStream_t s) {
  const dim3 grid((unsigned)p.bh_count), block(kOnePairThreads);
  switch (lanes) {
    case 1: hipLaunchKernelGGL((one_query_pair_kernel<DT, 1>), grid, block, 0, s, p, mode); break;
    case 2: hipLaunchKernelGGL((one_query_pair_kernel<DT, 2>), grid, block, 0, s, p, mode); break;
    case 4: hipLaunchKernelGGL((one_query_pair_kernel<DT, 4>), grid, block, 0, s, p, mode); break;
    case 8: hipLaunchKernelGGL((one_query_pair_kernel<DT, 8>), grid, block, 0, s, p, mode); break;
    case 16: hipLaunchKernelGGL((one_query_pair_kernel<DT, 16>), grid, block, 0, s, p, mode); break;
    case 32: hipLaunchKernelGGL((one_query_pair_kernel<DT, 32>), grid, block, 0, s, p, mode); break;
    default: hipLaunchKernelGGL((one_query_pair_kernel<DT, 64>), grid, block, 0, s, p, mode); break;
  }
}

int launch_one_query(Params& p, int dtype, const OneQueryPlan& o, float* ws, int mode, hipStream_t s) {
  if (one_query_alone(p, o.lanes)) {
    if (dtype == FCR_DTYPE_F16) launch_one_query_pair<FCR_DTYPE_F16>(p, o.lanes, mode, s);
    else if (dtype == FCR_DTYPE_BF16) launch_one_query_pair<FCR_DTYPE_BF16>(p, o.lanes, mode, s);
    else launch_one_query_pair<FCR_DTYPE_F32>(p, o.lanes, mode, s);
    return launched("one_query_pair_kernel");
  }
  float* const scores = ws + o.scores_at;
  p.part = ws + o.part_at;
  p.splits = o.splits;
  p.total = (int)(p.bh_count * (int64_t)o.splits);
  // Keys that pairs share by a stride of zero.  The heads of a batch entry follow each other and meet in the caches: no
  // non-temporal loads (8 x 32 x 9001 x 128 bf16 81 -> 56 us, fp32 164 -> 89).  Batch entries are all heads apart.  What the
  // eight L2s hold together still meets there (16 x 32 x 4096 bf16 63 -> 48, 64 x 8 x 16384 284 -> 138).  More than
  // that goes range by range through the whole batch, if it has a workgroup for every XCD (16 x 32 x 6000 bf16 113 -> 70,
  // fp32 236 -> 114; within the L2s the plain order is faster: 16 x 32 x 4096 x 64 bf16 26 against 32; 4 x 32 x 6000 bf16
  // 27 plain and non-temporal, 35 in this order).
  const int batch = p.bh_count / p.H;
  const bool by_heads = p.H > 1 && p.k_sh == 0, by_batch = !by_heads && batch > 1 && p.k_sb == 0;
  const bool fits = (int64_t)p.H * p.N * p.dgran * 16 <= (32ll << 20), beside = by_batch && !fits && batch >= 8;
  const bool once = !by_heads && !beside && !(by_batch && fits);
  p.group = beside ? batch : 1;
  if (dtype == FCR_DTYPE_F16) launch_one_query_scores<FCR_DTYPE_F16>(once, p, o, scores, s);
  else if (dtype == FCR_DTYPE_BF16) launch_one_query_scores<FCR_DTYPE_BF16>(once, p, o, scores, s);
  else launch_one_query_scores<FCR_DTYPE_F32>(once, p, o, scores, s);
  int rc = launched("one_query_scores_kernel");
  if (rc) return rc;
  p.tiles = (p.N + 256 * kOneCols - 1) / (256 * kOneCols);
  const dim3 grid((unsigned)(p.bh_count * (int64_t)p.tiles)), block(256);
  if (mode == kModeSum) hipLaunchKernelGGL(one_query_columns_kernel<kModeSum>, grid, block, 0, s, p, scores, o.pitch);
  else if (mode == kModeMax) hipLaunchKernelGGL(one_query_columns_kernel<kModeMax>, grid, block, 0, s, p, scores, o.pitch);
  else hipLaunchKernelGGL(one_query_columns_kernel<kModeBoth>, grid, block, 0, s, p, scores, o.pitch);
  return launched("one_query_columns_kernel");
}

int launch_both(Params& p, int dtype, int ksteps, const BothPlan& o, float* ws, int mode, bool causal, hipStream_t s) {
  p.lse = ws;
  p.row_blocks = o.row_blocks;
  p.col_blocks = o.col_blocks;
  const int row_rows = kWaves * 32 * o.row_blocks, col_rows = kWaves * 32 * o.col_blocks;
  p.tiles = (p.M + row_rows - 1) / row_rows;
  p.col_tiles = (p.N + col_rows - 1) / col_rows;
  p.total = p.bh_count * p.tiles;
  p.group = head_group(p.bh_count, p.tiles, causal);
  p.col_group = head_group(p.bh_count, p.col_tiles, causal);
  p.fill = fill_places(p, TileChoice{row_rows, 2}, causal);
  const long long polls = __atomic_load_n(&g_wait_polls, __ATOMIC_RELAXED);
  p.spin_limit = polls > 0x7fffffffll ? 0x7fffffff : (int)polls;
  const int64_t words = (int64_t)p.bh_count * p.M;
  hipLaunchKernelGGL(fill_words_kernel, dim3((unsigned)((words + 1023) / 1024)), dim3(256), 0, s, reinterpret_cast<unsigned*>(ws), words, kNotYet, p.sync);
  const int rc = launched("fill_words_kernel");
  if (rc) return rc;
  (dtype == FCR_DTYPE_F16 ? fcr_detail::sweeps_f16_both : fcr_detail::sweeps_bf16_both)(p, ksteps, causal, mode, s);
  return launched("both_sweeps_kernel");
}

int launch_few_keys(Params& p, int dtype, int ksteps, const FewKeysPlan& o, float* ws, int mode, bool causal, hipStream_t s) {
  p.lse = ws;
  Params sweep = p;
  sweep.splits = o.splits;
  sweep.parts = o.parts;
  if (o.splits > 1) {
    sweep.out = ws + o.part_at;
    sweep.out2 = ws + o.part_at + (mode == kModeBoth ? (int64_t)o.parts * p.bh_count * p.N : 0);
    sweep.out_fmt = FCR_DTYPE_F32;
    sweep.mean_from = -1;
  }
  (dtype == FCR_DTYPE_F32 ? fcr_detail::sweeps_f32_few_keys : dtype == FCR_DTYPE_F16 ? fcr_detail::sweeps_f16_few_keys : fcr_detail::sweeps_bf16_few_keys)(sweep, ksteps, causal, mode, o.form, s);
  const int rc = launched("few_keys_kernel");
  if (rc || o.splits == 1) return rc;
  p.part = ws + o.part_at;
  p.splits = o.parts;
  const dim3 grid((unsigned)((p.bh_count * (int64_t)p.N + 255) / 256)), block(256);
  if (mode == kModeSum) hipLaunchKernelGGL(merge_columns_kernel<kModeSum>, grid, block, 0, s, p);
  else if (mode == kModeMax) hipLaunchKernelGGL(merge_columns_kernel<kModeMax>, grid, block, 0, s, p);
  else hipLaunchKernelGGL(merge_columns_kernel<kModeBoth>, grid, block, 0, s, p);
  return launched("merge_columns_kernel");
}

template <int VPT, typename ET>
void launch_topk_spread(const ET* scores, uint8_t* mask, float* threshold, int64_t rows, int N, int k, uint32_t* w,
                        hipStream_t s) {
  const int parts = (N + VPT * kTopkThreads - 1) / (VPT * kTopkThreads);
  const dim3 grid((unsigned)(rows * parts)), block(kTopkThreads);
  hipLaunchKernelGGL((topk_spread_hist_kernel<0, VPT, ET>), grid, block, 0, s, scores, w, rows, N, k, parts);
  hipLaunchKernelGGL((topk_spread_hist_kernel<1, VPT, ET>), grid, block, 0, s, scores, w, rows, N, k, parts);
  hipLaunchKernelGGL((topk_spread_hist_kernel<2, VPT, ET>), grid, block, 0, s, scores, w, rows, N, k, parts);
  hipLaunchKernelGGL((topk_spread_hist_kernel<3, VPT, ET>), grid, block, 0, s, scores, w, rows, N, k, parts);
  hipLaunchKernelGGL((topk_spread_write_kernel<VPT, ET>), grid, block, 0, s, scores, mask, threshold, w, rows, N, k,
                     parts);
}

// The top-k launches for one element type: spread over workgroups when the caller brought enough scratch
// for a long row, else one workgroup per row.
template <int T, int W4, typename ET>
void launch_topk16(const ET* scores, uint8_t* mask, float* threshold, int64_t rows, int N, int k, hipStream_t s) {
  hipLaunchKernelGGL((topk16_mask_kernel<T, W4, ET>), dim3((unsigned)rows), dim3(T), 0, s, scores, mask, threshold, N, k);
}

template <typename ET>
int topk_any(const ET* scores, uint8_t* mask, float* threshold, int64_t rows, int N, int k, void* ws, size_t ws_bytes,
             hipStream_t s) {
  constexpr int T = kTopkThreads;
  if constexpr (sizeof(ET) == 2) {
    // up to kTopk16Columns fit the registers of one workgroup, eight to a 16-byte vector
    if (N <= 8 * 256) return launch_topk16<256, 1>(scores, mask, threshold, rows, N, k, s), 0;
    if (N <= 8 * T) return launch_topk16<T, 1>(scores, mask, threshold, rows, N, k, s), 0;
    if (N <= 16 * T) return launch_topk16<T, 2>(scores, mask, threshold, rows, N, k, s), 0;
    if (N <= 32 * T) return launch_topk16<T, 4>(scores, mask, threshold, rows, N, k, s), 0;
    if (N <= kTopk16Columns) return launch_topk16<T, 8>(scores, mask, threshold, rows, N, k, s), 0;
  }
  const size_t want = fcr_topk_bytes(rows, N);
  if (ws && want != 0 && ws_bytes >= want) {
    uint32_t* w = static_cast<uint32_t*>(ws);
    // 32 keys per thread while that leaves a workgroup per CU, else 8
    const int64_t coarse = rows * ((N + 32 * T - 1) / (32 * T));
    if (coarse >= chip_cus()) launch_topk_spread<32>(scores, mask, threshold, rows, N, k, w, s);
    else launch_topk_spread<8>(scores, mask, threshold, rows, N, k, w, s);
    return 0;
  }
  const dim3 grid((unsigned)rows), block(T);
  if constexpr (sizeof(ET) == 4) {
    if (N <= 32 * T) {
      if (N <= 8 * 256) hipLaunchKernelGGL((topk_mask_kernel<256, 8>), grid, dim3(256), 0, s, scores, mask, threshold, N, k);
      else if (N <= 8 * T) hipLaunchKernelGGL((topk_mask_kernel<T, 8>), grid, block, 0, s, scores, mask, threshold, N, k);
      else if (N <= 16 * T) hipLaunchKernelGGL((topk_mask_kernel<T, 16>), grid, block, 0, s, scores, mask, threshold, N, k);
      else hipLaunchKernelGGL((topk_mask_kernel<T, 32>), grid, block, 0, s, scores, mask, threshold, N, k);
      return 0;
    }
  }
  hipLaunchKernelGGL(topk_mask_long_kernel<ET>, grid, block, 0, s, scores, mask, threshold, N, k);
  return 0;
}
}  // namespace

namespace {
size_t fcr_lse_bytes_two_kernels(int B, int H, int M, int N) {
  // The most any row width asks for, so the size holds for every dtype and D.  Of one problem the widths differ
  // only in the tile height, 128 or 256 rows: four k-steps take 256 where any width does (one block costs them
  // the most), and the higher tile has the fewer workgroups, hence the most splits.  (Every call comes here.)
  const int splits = row_splits(FCR_DTYPE_F16, B, H, M, N, 128);
  const size_t rows = (size_t)B * (size_t)H * (size_t)M;
  return rows * sizeof(float) * (splits > 1 ? 1 + (size_t)splits : 1);
}

}  // namespace
thread_local bool fcr_detail::fused_refused = false;

extern "C" {

int fcr_version(void) { return FCR_VERSION; }

const char* fcr_last_error(void) { return g_err; }

size_t fcr_lse_bytes(int B, int H, int M, int N, int D) {
  if (B < 1 || H < 1 || M < 1 || N < 1 || D < 1) return 0;
  {
    // the single-sweep path keeps partial row values and its counters behind the row statistics
    FusedPlan f;
    if (fused_shape((int64_t)B * H, M, N, f)) {
      const size_t two_kernels = fcr_lse_bytes_two_kernels(B, H, M, N);
      const size_t one = (size_t)f.floats * sizeof(float);
      return one > two_kernels ? one : two_kernels;
    }
  }
  return fcr_lse_bytes_two_kernels(B, H, M, N);
}

namespace {
// status: a word to clear, or null
int row_lse_any(const void* q, const void* k, float* lse, unsigned* status, int dtype, int B, int H, int M, int N, int D,
                const int64_t q_strides[4], const int64_t k_strides[4], float scale, int causal, void* stream) {
  Params p;
  if (!lse) return fail(FCR_E_NULL, "null pointer argument");
  int rc = make_params(p, q, k, dtype, B, H, M, N, D, q_strides, k_strides, scale, false, causal != 0);
  if (rc) return rc;
  p.lse = lse;
  p.sync = status;
  p.splits = row_splits(dtype, B, H, M, N, D);
  p.part = lse + (int64_t)B * H * M;  // only touched when splits > 1 (see fcr_lse_bytes)
  p.total *= p.splits;
  const int ksteps = ksteps_of(dtype, D);
  p.group = head_group(p.bh_count, (int64_t)p.tiles * p.splits, causal != 0);
  p.fill = fill_places(p, tile_choice(dtype, D, M, N, p.bh_count, false, 0, causal != 0), causal != 0);
  hipStream_t s = static_cast<hipStream_t>(stream);
  launch_sweeps(dtype, 0, p, ksteps, causal != 0, 0, s);
  rc = launched("row_lse_kernel");
  if (rc || p.splits == 1) return rc;
  const int64_t rows = (int64_t)B * H * M;
  hipLaunchKernelGGL(lse_combine_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, s, p.part, lse, rows,
                     p.splits);
  return launched("lse_combine_kernel");
}
}  // namespace

int fcr_row_lse(const void* q, const void* k, float* lse, int dtype, int B, int H, int M, int N, int D,
                const int64_t q_strides[4], const int64_t k_strides[4], float scale, int causal,
                void* stream) {
  return row_lse_any(q, k, lse, nullptr, dtype, B, H, M, N, D, q_strides, k_strides, scale, causal, stream);
}

namespace {
// Element type of the results and whether the sums leave the kernel as means.
struct ResultSpec {
  int fmt = FCR_DTYPE_F32;
  bool mean = false;
};

int col_reduce_any(const void* q, const void* k, const float* lse, void* out, void* out2, int mode, int dtype,
                   int B, int H, int M, int N, int D, const int64_t q_strides[4], const int64_t k_strides[4],
                   float scale, int causal, void* stream, const ResultSpec& res = ResultSpec()) {
  Params p;
  if (!lse || !out || (mode == kModeBoth && !out2)) return fail(FCR_E_NULL, "null pointer argument");
  int rc = make_params(p, q, k, dtype, B, H, M, N, D, q_strides, k_strides, scale, true, causal != 0, mode);
  if (rc) return rc;
  p.group = head_group(p.bh_count, p.tiles, causal != 0);
  const int ksteps = ksteps_of(dtype, D);
  p.lse = const_cast<float*>(lse);
  p.out = out;
  p.out2 = out2;
  p.out_fmt = res.fmt;
  if (res.mean) {
    p.mean_from = causal ? p.c : N;
    p.inv_m = 1.0f / (float)M;
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  // (fp32 operands always take the general sweep, which splits them)
  if (M <= kSmallRows && ksteps <= 4 && dtype != FCR_DTYPE_F32) {
    // Few queries: the sweep with all of them resident in every wave and the keys streamed, if the
    // problem fills the chip that way: 512 to 1024 workgroups (at least two per CU), each sweeping at
    // least 16 chunks of keys, or 8 if that is what it takes.
    const int64_t nchunks = ((int64_t)N + kChunk - 1) / kChunk;
    int64_t splits = 0;
    const int cus = chip_cus();
    for (int64_t least = 16; least >= 8 && p.bh_count * splits < 2 * cus; least /= 2) {  // longer sweeps first
      splits = 4 * cus / p.bh_count;
      if (splits > nchunks / least) splits = nchunks / least;
      if (splits < 1) splits = 1;
      const int64_t per = (nchunks + splits - 1) / splits;
      splits = (nchunks + per - 1) / per;  // no empty ranges
    }
    if (p.bh_count * splits >= 2 * cus) {
      p.splits = (int)splits;
      p.total = (int)(p.bh_count * splits);
      p.group = head_group(p.bh_count, splits, false);
      p.stream_once = ((int64_t)p.bh_count * N * p.dgran * 16 >= (1ll << 30)) ? 1 : 0;
      launch_sweeps(dtype, 2, p, ksteps, causal != 0, mode, s);
      return launched("col_small_kernel");
    }
  }
  p.fill = fill_places(p, tile_choice(dtype, D, M, N, p.bh_count, true, mode, causal != 0), causal != 0);
  launch_sweeps(dtype, 1, p, ksteps, causal != 0, mode, s);
  return launched("col_reduce_kernel");
}
}  // namespace

int fcr_col_reduce(const void* q, const void* k, const float* lse, float* out, int dtype, int B, int H,
                   int M, int N, int D, const int64_t q_strides[4], const int64_t k_strides[4],
                   float scale, int reduction, int causal, void* stream) {
  if (reduction != FCR_REDUCE_SUM && reduction != FCR_REDUCE_MAX)
    return fail(FCR_E_REDUCTION, "reduction must be FCR_REDUCE_SUM or FCR_REDUCE_MAX");
  return col_reduce_any(q, k, lse, out, nullptr, reduction == FCR_REDUCE_MAX ? kModeMax : kModeSum, dtype, B, H, M,
                        N, D, q_strides, k_strides, scale, causal, stream);
}

int fcr_col_reduce_sum_max(const void* q, const void* k, const float* lse, float* out_sum, float* out_max,
                           int dtype, int B, int H, int M, int N, int D, const int64_t q_strides[4],
                           const int64_t k_strides[4], float scale, int causal, void* stream) {
  return col_reduce_any(q, k, lse, out_sum, out_max, kModeBoth, dtype, B, H, M, N, D, q_strides, k_strides, scale,
                        causal, stream);
}

size_t fcr_topk_bytes(int64_t rows, int N) {
  if (rows < 1 || N <= 32 * kTopkThreads || N > (1 << 30)) return 0;
  const int parts = (N + 8 * kTopkThreads - 1) / (8 * kTopkThreads);   // the finer of the two ways to cut a row
  if (rows * parts >= (1ll << 22)) return 0;   // more workgroups of 1024 threads than one launch may have
  return 2 * topk_hist_words(rows, parts) * sizeof(uint32_t) + (size_t)rows * 4 * sizeof(TopkState);
}
size_t fcr_topk_bytes_typed(int dtype, int64_t rows, int N) {
  if (dtype != FCR_DTYPE_F16 && dtype != FCR_DTYPE_BF16 && dtype != FCR_DTYPE_F32) return 0;
  return elem_bytes(dtype) == 2 && N <= kTopk16Columns ? 0 : fcr_topk_bytes(rows, N);
}

int fcr_topk_mask_typed(const void* scores, int dtype, uint8_t* mask, float* threshold, int64_t rows, int N, int k,
                        void* ws, size_t ws_bytes, void* stream) {
  if (!scores || !mask) return fail(FCR_E_NULL, "null pointer argument");
  if (dtype != FCR_DTYPE_F16 && dtype != FCR_DTYPE_BF16 && dtype != FCR_DTYPE_F32)
    return fail(FCR_E_DTYPE, "scores must be fp16, bf16 or fp32");
  // one workgroup of 1024 threads per row (or per part of a row), fewer than 2^32 threads per launch
  if (rows < 1 || rows >= (1ll << 22) || N < 1) return fail(FCR_E_SHAPE, "rows must be in [1, 2^22) and N >= 1");
  if (ws && (reinterpret_cast<uintptr_t>(ws) & 15) != 0)
    return fail(FCR_E_STRIDE, "the top-k workspace must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == FCR_DTYPE_F32) topk_any(static_cast<const float*>(scores), mask, threshold, rows, N, k, ws, ws_bytes, s);
  else if (dtype == FCR_DTYPE_F16) topk_any(static_cast<const _Float16*>(scores), mask, threshold, rows, N, k, ws, ws_bytes, s);
  else topk_any(static_cast<const uint16_t*>(scores), mask, threshold, rows, N, k, ws, ws_bytes, s);
  return launched("top-k kernels");
}

int fcr_topk_mask_ws(const float* scores, uint8_t* mask, float* threshold, int64_t rows, int N, int k, void* ws,
                     size_t ws_bytes, void* stream) {
  return fcr_topk_mask_typed(scores, FCR_DTYPE_F32, mask, threshold, rows, N, k, ws, ws_bytes, stream);
}

int fcr_topk_mask(const float* scores, uint8_t* mask, float* threshold, int64_t rows, int N, int k, void* stream) {
  return fcr_topk_mask_typed(scores, FCR_DTYPE_F32, mask, threshold, rows, N, k, nullptr, 0, stream);
}

int fcr_pack_f32(const float* src, void* dst, int64_t rows, int D, int terms, int is_key, void* stream) {
  if (!src || !dst) return fail(FCR_E_NULL, "null pointer argument");
  if (rows < 1 || D < 1) return fail(FCR_E_SHAPE, "rows and D must be >= 1");
  if (terms != 1 && terms != 3) return fail(FCR_E_SHAPE, "terms must be 1 or 3");
  const int dpad = (D + 7) / 8 * 8;
  if (terms * dpad > 32 * kMaxKSteps) return fail(FCR_E_SHAPE, "terms * D (padded to 8) must be <= 256");
  const int64_t n = rows * dpad;
  if ((n + 255) / 256 > 0x7fffffffll) return fail(FCR_E_SHAPE, "too many elements");
  hipLaunchKernelGGL(pack_f32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), src, static_cast<_Float16*>(dst), rows, D, dpad, terms,
                     is_key != 0);
  return launched("pack_f32_kernel");
}

namespace {
// Whether a stream is being captured, or that cannot be told.
bool is_capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) == hipSuccess && st == hipStreamCaptureStatusNone) return false;
  (void)hipGetLastError();
  return true;
}

// A single sweep expects the whole chip: its workgroups wait for each other, one of eight waves or two of four per CU.  Two of them issued on
// different streams could be dispatched side by side, each holding CUs the other needs, until their bounded
// waits run out.  So inside a process they are chained: a single sweep on another stream than the one before
// first waits (on the GPU; the host blocks only if that stream was destroyed or, once, was another thread's hipStreamPerThread) for an event recorded at the end of that stream.  Calls that
// stay on one stream pay nothing (an event behind every call costs 5 us of a 18 us call; on hipStreamPerThread there is one as soon as others follow there).  Not under stream
// capture (a graph carries no such edge; graphs holding single sweeps must not replay side by side on one GPU),
// not for other processes on the same GPU, and not for fcr_colreduce_static, whose calls must not overlap anyway.
// Where the order cannot be had the call takes the two kernels.
struct SweepOrder {
  hipEvent_t done = nullptr;
  hipStream_t last = nullptr;
  uint64_t thread = 0;      // of hipStreamPerThread, one handle for a stream of every thread: whose
  bool any = false;
  bool recorded = false;    // `done` stands behind the last launch
  bool mixed = false;       // other streams follow on hipStreamPerThread, where no other thread can record `done`: each launch there does
};
SweepOrder g_order[64];
std::mutex g_order_mu;

uint64_t thread_number() {   // (the address of a thread's own variable may come back with another thread)
  static std::atomic<uint64_t> count{0};
  static thread_local const uint64_t mine = ++count;
  return mine;
}

// Stream s waits for what is on the stream of the last single sweep.
bool wait_for_last(SweepOrder* o, hipStream_t s) {
  if (!o->recorded) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    hipError_t e = o->thread != 0 ? hipErrorInvalidHandle : hipStreamIsCapturing(o->last, &st);
    if (e == hipSuccess && st != hipStreamCaptureStatusNone) return false;   // (what it was given before the capture may still run)
    if (e == hipSuccess) e = hipEventRecord(o->done, o->last);
    if (e != hipSuccess) {   // the stream is gone or another thread's, its work perhaps still there: the host waits for the device, whoever captures meanwhile
      (void)hipGetLastError();
      o->mixed = o->mixed || o->thread != 0;
      hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
      if (hipThreadExchangeStreamCaptureMode(&mode) != hipSuccess) return false;
      e = hipDeviceSynchronize();
      (void)hipThreadExchangeStreamCaptureMode(&mode);
      return e == hipSuccess;
    }
  }
  return hipStreamWaitEvent(s, o->done, 0) == hipSuccess;
}

// Whether a single sweep may be launched on stream s; then `o` is the device's entry, locked until order_end, or null for a captured launch,
// which nothing orders.
bool order_begin(hipStream_t s, SweepOrder*& o) {
  o = nullptr;
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  if (st != hipStreamCaptureStatusNone) return true;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    (void)hipGetLastError();
    return false;
  }
  g_order_mu.lock();
  SweepOrder* const e = &g_order[dev];
  if (!e->done && hipEventCreateWithFlags(&e->done, hipEventDisableTiming) != hipSuccess) e->done = nullptr;
  const bool same = e->last == s && e->thread == (s == hipStreamPerThread ? thread_number() : 0);
  if (!e->done || (e->any && !same && !wait_for_last(e, s))) {
    (void)hipGetLastError();
    g_order_mu.unlock();
    return false;
  }
  o = e;
  return true;
}
void order_end(SweepOrder* o, hipStream_t s, bool launched_it) {
  if (!o) return;
  if (launched_it) {
    o->last = s;
    o->thread = s == hipStreamPerThread ? thread_number() : 0;
    o->any = true;
    o->recorded = o->mixed && o->thread != 0 && hipEventRecord(o->done, s) == hipSuccess;
    if (!o->recorded) (void)hipGetLastError();
  }
  g_order_mu.unlock();
}

// Both sweeps of a call, writing `out` in its final form.  ws_bytes = bytes the caller's workspace is known
// to have (0: what fcr_lse_bytes asks for), lse_bytes = what fcr_lse_bytes gives (if ws_bytes is known).  One query takes the path of its own where the workspace has room for
// its scores, few queries against many keys take the single sweep.
int whole_call(const void* q, const void* k, void* out, const ResultSpec& res, float* ws, size_t ws_bytes,
               size_t lse_bytes, int dtype, int B, int H, int M, int N, int D, const int64_t q_strides[4],
               const int64_t k_strides[4], float scale, int mode, int causal, void* stream, void* out2 = nullptr) {
  Params p;
  int rc = make_params(p, q, k, dtype, B, H, M, N, D, q_strides, k_strides, scale, true, causal != 0, mode);
  if (rc) return rc;
  const int ksteps = ksteps_of(dtype, D);
  const bool single = __atomic_load_n(&g_single_sweep, __ATOMIC_RELAXED) != 0;
  FusedPlan f;
  const bool fused = dtype != FCR_DTYPE_F32 && ksteps <= 4 && fused_shape(p.bh_count, M, N, f);
  p.out = out;
  p.out2 = out2;
  p.out_fmt = res.fmt;
  if (res.mean) {
    p.mean_from = causal ? p.c : N;
    p.inv_m = 1.0f / (float)M;
  }
  p.stream_once = ((int64_t)p.bh_count * N * p.dgran * 16 >= (1ll << 30)) ? 1 : 0;
  if (single && M == 1 && ws_bytes != 0) {   // (the mask hides nothing from the only query)
    const OneQueryPlan o = one_query_plan(dtype, p.bh_count, N, D, (int64_t)(lse_bytes / sizeof(float)));
    if ((size_t)o.floats * sizeof(float) <= ws_bytes) {
      p.lse = ws;
      p.sync = fused ? reinterpret_cast<unsigned*>(ws + f.sync_at) : nullptr;   // fcr_colreduce_status looks there
      return launch_one_query(p, dtype, o, ws, mode, static_cast<hipStream_t>(stream));
    }
  }
  if (single && ws_bytes != 0) {
    const FewKeysPlan o = few_keys_plan(dtype, B, H, M, N, D, mode == kModeBoth, (int64_t)(lse_bytes / sizeof(float)));
    // (the keys of a pair are read through one view: all rows of a workgroup below 2 GiB)
    if (o.form >= 0 && (size_t)o.floats * sizeof(float) <= ws_bytes && ((int64_t)128 << o.form) * p.k_sr <= 0x7fffffff)
      return launch_few_keys(p, dtype, ksteps, o, ws, mode, causal != 0, static_cast<hipStream_t>(stream));
  }
  if (single && fused) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    p.lse = ws;
    p.part = ws + f.part_at;
    p.sync = reinterpret_cast<unsigned*>(ws + f.sync_at);
    p.splits = f.splits;
    p.teams = f.teams;
    int form = (f.qh == 2 ? 4 : 0) | (f.nq == 2 ? 8 : 0), rows = f.qh == 2 ? 128 : 16 * f.nq;
    const FusedPairPlan two = fused_pair_plan(p.bh_count, M, N, ksteps, f);
    if (two.teams > 0 && (size_t)two.floats * sizeof(float) <= ws_bytes) {
      p.part = ws + two.part_at;
      p.splits = two.splits;
      p.teams = two.teams;
      form = 16;
      rows = 32;
    }
    spread_keys(p, N, form == 16 || f.qh == 2 ? 1 : 2, chip_cus(), f.nq == 4 && form != 16);
    // the slots that the launch polls (one set of them for one round) and the status word start at zero
    const int words = (p.bh_count > p.teams ? 2 : 1) * p.teams * p.splits * rows * 2;
    p.total = p.teams * p.splits;
    const long long polls = __atomic_load_n(&g_wait_polls, __ATOMIC_RELAXED);
    p.spin_limit = polls > 0x7fffffffll ? 0x7fffffff : (int)polls;
    SweepOrder* order;
    if (order_begin(s, order)) {
      fcr_detail::fused_refused = false;
      launch_sweeps(dtype, 3, p, ksteps, causal != 0, mode | form, s, reinterpret_cast<unsigned*>(p.part), words);
      const int lrc = fcr_detail::fused_refused ? 0 : launched("col_fused_kernel");
      order_end(order, s, !fcr_detail::fused_refused && lrc == 0);
      if (!fcr_detail::fused_refused) return lrc;
    }
  }
  unsigned* status = nullptr;
  if (ws_bytes != 0) {
    const int64_t at = both_status_at(dtype, B, H, M, N, D, (int64_t)(lse_bytes / sizeof(float)));
    if (at >= 0 && (size_t)(at + kStatusFloats) * sizeof(float) <= ws_bytes) status = reinterpret_cast<unsigned*>(ws + at);
  }
  if (single && !is_capturing(static_cast<hipStream_t>(stream))) {   // (a captured call keeps the bits of the two launches)
    const BothPlan o = both_plan(dtype, ksteps, p.bh_count, M, N, causal != 0);
    p.sync = status;
    if (o.row_blocks > 0) return launch_both(p, dtype, ksteps, o, ws, mode, causal != 0, static_cast<hipStream_t>(stream));
  }
  rc = row_lse_any(q, k, ws, status, dtype, B, H, M, N, D, q_strides, k_strides, scale, causal, stream);
  if (rc) return rc;
  rc = col_reduce_any(q, k, ws, out, out2, mode, dtype, B, H, M, N, D, q_strides, k_strides, scale, causal, stream,
                      res);
  if (rc || !single || !fused) return rc;
  // a single sweep that was not launched, so nobody waited: fcr_colreduce_status looks there (behind the kernels, whose partial results may lie there)
  hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(256), 0, static_cast<hipStream_t>(stream), nullptr, 0, reinterpret_cast<unsigned*>(ws + f.sync_at));
  return launched("zero_words_kernel");
}
}  // namespace

int fcr_colreduce_sum_max(const void* q, const void* k, float* out_sum, float* out_max, float* lse_ws, int dtype, int B,
                          int H, int M, int N, int D, const int64_t q_strides[4], const int64_t k_strides[4],
                          float scale, int causal, void* stream) {
  if (!out_sum || !out_max || !lse_ws) return fail(FCR_E_NULL, "null pointer argument");
  return whole_call(q, k, out_sum, ResultSpec(), lse_ws, 0, 0, dtype, B, H, M, N, D, q_strides, k_strides, scale, kModeBoth,
                    causal, stream, out_max);
}

int fcr_colreduce(const void* q, const void* k, float* out, float* lse_ws, int dtype, int B, int H, int M,
                  int N, int D, const int64_t q_strides[4], const int64_t k_strides[4], float scale,
                  int reduction, int causal, void* stream) {
  if (!out || !lse_ws) return fail(FCR_E_NULL, "null pointer argument");
  if (reduction != FCR_REDUCE_SUM && reduction != FCR_REDUCE_MAX)
    return fail(FCR_E_REDUCTION, "reduction must be FCR_REDUCE_SUM or FCR_REDUCE_MAX");
  return whole_call(q, k, out, ResultSpec(), lse_ws, 0, 0, dtype, B, H, M, N, D, q_strides, k_strides, scale,
                    reduction == FCR_REDUCE_MAX ? kModeMax : kModeSum, causal, stream);
}

// Scratch of fcr_colreduce_static: the row statistics and, for few query rows against many keys, the
// partial results of the split row sweep or the single sweep's partial values and counters.  One copy per
// GPU, held until the process ends.  Host code must not pass the array's name to a kernel (it is a
// host-side stand-in there): the device address is asked once per device and kept.
static __device__ __align__(256) unsigned char scratch[FCR_STATIC_SCRATCH_BYTES];

namespace {
int static_scratch(float** ptr) {
  static void* ptrs[64] = {};
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    snprintf(g_err, sizeof(g_err), "hipGetDevice failed: %s", hipGetErrorString(e));
    return (int)e;
  }
  if (dev < 0 || dev >= 64) return fail(FCR_E_SHAPE, "device ordinal must be below 64");
  void* p = __atomic_load_n(&ptrs[dev], __ATOMIC_ACQUIRE);
  if (!p) {
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));  // this device's copy of the array
    if (e != hipSuccess || !p) {
      snprintf(g_err, sizeof(g_err), "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
      return e != hipSuccess ? (int)e : (int)hipErrorInvalidSymbol;
    }
    __atomic_store_n(&ptrs[dev], p, __ATOMIC_RELEASE);
  }
  *ptr = static_cast<float*>(p);
  return 0;
}
}  // namespace

int fcr_colreduce_to(const void* q, const void* k, void* out, int out_dtype, float* lse_ws, int dtype, int B, int H,
                     int M, int N, int D, const int64_t q_strides[4], const int64_t k_strides[4], float scale,
                     int reduction, int causal, void* stream) {
  if (!out || !lse_ws) return fail(FCR_E_NULL, "null pointer argument");
  if (reduction != FCR_REDUCE_SUM && reduction != FCR_REDUCE_MAX && reduction != FCR_REDUCE_MEAN)
    return fail(FCR_E_REDUCTION, "reduction must be FCR_REDUCE_SUM, FCR_REDUCE_MAX or FCR_REDUCE_MEAN");
  if (out_dtype != FCR_DTYPE_F16 && out_dtype != FCR_DTYPE_BF16 && out_dtype != FCR_DTYPE_F32)
    return fail(FCR_E_DTYPE, "out_dtype must be FCR_DTYPE_F16, FCR_DTYPE_BF16 or FCR_DTYPE_F32");
  ResultSpec res;
  res.fmt = out_dtype;
  res.mean = reduction == FCR_REDUCE_MEAN;
  return whole_call(q, k, out, res, lse_ws, 0, 0, dtype, B, H, M, N, D, q_strides, k_strides, scale,
                    reduction == FCR_REDUCE_MAX ? kModeMax : kModeSum, causal, stream);
}

int fcr_colreduce_sum_max_to(const void* q, const void* k, void* out_sum, void* out_max, int out_dtype, float* lse_ws,
                             int dtype, int B, int H, int M, int N, int D, const int64_t q_strides[4],
                             const int64_t k_strides[4], float scale, int sum_reduction, int causal, void* stream) {
  if (!out_sum || !out_max || !lse_ws) return fail(FCR_E_NULL, "null pointer argument");
  if (sum_reduction != FCR_REDUCE_SUM && sum_reduction != FCR_REDUCE_MEAN)
    return fail(FCR_E_REDUCTION, "sum_reduction must be FCR_REDUCE_SUM or FCR_REDUCE_MEAN");
  if (out_dtype != FCR_DTYPE_F16 && out_dtype != FCR_DTYPE_BF16 && out_dtype != FCR_DTYPE_F32)
    return fail(FCR_E_DTYPE, "out_dtype must be FCR_DTYPE_F16, FCR_DTYPE_BF16 or FCR_DTYPE_F32");
  ResultSpec res;
  res.fmt = out_dtype;
  res.mean = sum_reduction == FCR_REDUCE_MEAN;
  return whole_call(q, k, out_sum, res, lse_ws, 0, 0, dtype, B, H, M, N, D, q_strides, k_strides, scale, kModeBoth, causal,
                    stream, out_max);
}

size_t fcr_workspace_bytes(int dtype, int B, int H, int M, int N, int D) {
  const size_t base = fcr_lse_bytes(B, H, M, N, D);
  if (base == 0 || (dtype != FCR_DTYPE_F16 && dtype != FCR_DTYPE_BF16 && dtype != FCR_DTYPE_F32)) return base;
  if (M == 1 && row_width_ok(dtype, D))   // (a row the call rejects has no plan: no power of two of 64 lanes or less)
    return (size_t)one_query_plan(dtype, (int64_t)B * H, N, D, (int64_t)(base / sizeof(float))).floats * sizeof(float);
  if (row_width_ok(dtype, D)) {
    const int64_t floats = (int64_t)(base / sizeof(float));
    int64_t most = few_keys_plan(dtype, B, H, M, N, D, true, floats).floats;   // (one result takes half of it)
    const int64_t status_at = both_status_at(dtype, B, H, M, N, D, floats);
    if (status_at >= 0 && status_at + kStatusFloats > most) most = status_at + kStatusFloats;
    FusedPlan f;
    if (dtype != FCR_DTYPE_F32 && ksteps_of(dtype, D) <= 4 && fused_shape((int64_t)B * H, M, N, f)) {
      const FusedPairPlan two = fused_pair_plan((int64_t)B * H, M, N, ksteps_of(dtype, D), f);
      if (two.floats > most) most = two.floats;
    }
    return (size_t)most * sizeof(float);
  }
  return base;
}

int fcr_colreduce_ws(const void* q, const void* k, void* out, void* out_max, int out_dtype, void* ws, size_t ws_bytes,
                     int dtype, int B, int H, int M, int N, int D, const int64_t q_strides[4],
                     const int64_t k_strides[4], float scale, int reduction, int causal, void* stream) {
  if (!out || !ws) return fail(FCR_E_NULL, "null pointer argument");
  if (reduction != FCR_REDUCE_SUM && reduction != FCR_REDUCE_MEAN && (reduction != FCR_REDUCE_MAX || out_max))
    return fail(FCR_E_REDUCTION, out_max ? "with out_max, reduction must be FCR_REDUCE_SUM or FCR_REDUCE_MEAN"
                                         : "reduction must be FCR_REDUCE_SUM, FCR_REDUCE_MAX or FCR_REDUCE_MEAN");
  if (out_dtype != FCR_DTYPE_F16 && out_dtype != FCR_DTYPE_BF16 && out_dtype != FCR_DTYPE_F32)
    return fail(FCR_E_DTYPE, "out_dtype must be FCR_DTYPE_F16, FCR_DTYPE_BF16 or FCR_DTYPE_F32");
  if ((reinterpret_cast<uintptr_t>(ws) & 15) != 0) return fail(FCR_E_STRIDE, "the workspace must be 16-byte aligned");
  // every argument of both launches first: the workspace's size depends on the device
  int rc = check_problem(q, k, dtype, B, H, M, N, D, q_strides, k_strides, scale, true);
  if (!rc) rc = check_problem(q, k, dtype, B, H, M, N, D, q_strides, k_strides, scale, false);
  if (rc) return rc;
  const size_t need = fcr_lse_bytes(B, H, M, N, D);
  if (ws_bytes < need) {
    snprintf(g_err, sizeof(g_err), "the workspace has %zu bytes, fcr_lse_bytes asks for %zu", ws_bytes, need);
    return FCR_E_SCRATCH;
  }
  ResultSpec res;
  res.fmt = out_dtype;
  res.mean = reduction == FCR_REDUCE_MEAN;
  const int mode = out_max ? kModeBoth : reduction == FCR_REDUCE_MAX ? kModeMax : kModeSum;
  return whole_call(q, k, out, res, static_cast<float*>(ws), ws_bytes, need, dtype, B, H, M, N, D, q_strides, k_strides,
                    scale, mode, causal, stream, out_max);
}

int fcr_colreduce_static(const void* q, const void* k, float* out, int dtype, int B, int H, int M, int N, int D,
                         const int64_t q_strides[4], const int64_t k_strides[4], float scale, int reduction,
                         int causal, void* stream) {
  if (!out) return fail(FCR_E_NULL, "null pointer argument");
  if (reduction != FCR_REDUCE_SUM && reduction != FCR_REDUCE_MAX)
    return fail(FCR_E_REDUCTION, "reduction must be FCR_REDUCE_SUM or FCR_REDUCE_MAX");
  // every argument check of the two kernels first (the last step of make_params asks the device for its
  // CU count; nothing else has touched it by then)
  Params p;
  int rc = make_params(p, q, k, dtype, B, H, M, N, D, q_strides, k_strides, scale, false, causal != 0);
  if (rc) return rc;
  const size_t need = fcr_lse_bytes(B, H, M, N, D);
  if (need > (size_t)FCR_STATIC_SCRATCH_BYTES) {
    snprintf(g_err, sizeof(g_err),
             "fcr_colreduce_static: this problem needs %zu bytes of scratch, the built-in buffer has %zu; "
             "use fcr_colreduce with a caller-provided buffer",
             need, (size_t)FCR_STATIC_SCRATCH_BYTES);
    return FCR_E_SCRATCH;
  }
  float* ws = nullptr;
  rc = static_scratch(&ws);
  if (rc) return rc;
  // The kernels write every value of the buffer they later read (the single sweep's counters are cleared by
  // a small kernel in front of it), so nothing has to be cleared here.
  return fcr_colreduce(q, k, out, ws, dtype, B, H, M, N, D, q_strides, k_strides, scale, reduction, causal, stream);
}

int fcr_set_option(int option, long long value) {
  if (option == FCR_OPT_SINGLE_SWEEP) {
    __atomic_store_n(&g_single_sweep, value != 0 ? 1 : 0, __ATOMIC_RELAXED);
    return 0;
  }
  if (option == FCR_OPT_WAIT_POLLS) {
    if (value < 0) return fail(FCR_E_SHAPE, "FCR_OPT_WAIT_POLLS must be >= 0");
    __atomic_store_n(&g_wait_polls, value, __ATOMIC_RELAXED);
    return 0;
  }
  return fail(FCR_E_SHAPE, "unknown option");
}

namespace {
// FCR_E_WAIT if the word on the device is set, once the stream's work is done.
int read_status(const unsigned* at, const char* text, hipStream_t s) {
  unsigned word = 0;
  hipError_t e = hipMemcpyAsync(&word, at, sizeof(word), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    snprintf(g_err, sizeof(g_err), "reading the status word failed: %s", hipGetErrorString(e));
    return (int)e;
  }
  return word != 0 ? fail(FCR_E_WAIT, text) : 0;
}
}  // namespace

int fcr_colreduce_status(const float* lse_ws, int dtype, int B, int H, int M, int N, int D, void* stream) {
  if (!lse_ws) return fail(FCR_E_NULL, "null pointer argument");
  if (B < 1 || H < 1 || M < 1 || N < 1 || D < 1) return fail(FCR_E_SHAPE, "B, H, M, N, D must be >= 1");
  FusedPlan f;
  if (dtype == FCR_DTYPE_F32 || ksteps_of(dtype, D) > 4 || !fused_shape((int64_t)B * H, M, N, f)) return 0;
  return read_status(reinterpret_cast<const unsigned*>(lse_ws + f.sync_at),
                     "a workgroup of the single sweep gave up waiting for its team; the columns of that (b,h) pair are NaN", static_cast<hipStream_t>(stream));
}

int fcr_colreduce_ws_status(const void* ws, size_t ws_bytes, int dtype, int B, int H, int M, int N, int D, void* stream) {
  const int rc = fcr_colreduce_status(static_cast<const float*>(ws), dtype, B, H, M, N, D, stream);
  if (rc || (dtype != FCR_DTYPE_F16 && dtype != FCR_DTYPE_BF16) || !row_width_ok(dtype, D)) return rc;
  const int64_t at = both_status_at(dtype, B, H, M, N, D, (int64_t)(fcr_lse_bytes(B, H, M, N, D) / sizeof(float)));
  if (at < 0 || (size_t)(at + kStatusFloats) * sizeof(float) > ws_bytes) return 0;
  return read_status(static_cast<const unsigned*>(ws) + at, "a column sweep gave up waiting for row statistics; its columns are NaN", static_cast<hipStream_t>(stream));
}

}  // extern "C"
#endif  // FCR_HAS(0)
