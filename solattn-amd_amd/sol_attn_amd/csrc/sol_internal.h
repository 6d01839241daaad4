// Host <-> kernel parameter blocks and internal launchers (not part of the C-ABI).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>

#include "sol_device.h"

namespace sol {

// Key tokens of batch entry b: klen[b] clamped to [1, T] when per-entry
// lengths are given (ragged indexed windows), else T.  The clamp keeps every
// access inside the [B, T]-shaped index and the NKB-padded buffers whatever
// the caller's lengths hold.
__device__ __forceinline__ int batch_tokens(const int32_t* klen, int b, int T) {
  return klen ? min(max(klen[b], 1), T) : T;
}

struct PoolParams {
  TokenRows k, v;
  const int32_t* klen;  // [B] key tokens per batch entry (<= Tk), or null: all Tk
  uint16_t* ctiles;  // [B, H, NCT, 2, 64 * D] centroid tiles, or null
  uint16_t* tiles;   // [B, H, NKB, 2, 64 * D] K / V block tiles (TileLayout), or null
  int32_t* block_rows;  // [B, NKB] or null (indexed keys only): the first row of each whole key block
                        // whose 64 keys are consecutive rows, -1 for the others; only those go to tiles
  float* ksum;       // [B, H, NCH, 2, D] chunk sums, null -> no moments
  float* mean;       // [B, H, D]
  float* var;        // [B, H, D]
  int B, H, Tk, NKB, NCT, NCHP;  // NCHP = 4 * NCT pooling chunks of 16 blocks
                                 // (NKB, NCT: for Tk; ragged entries use a prefix)
  int fold_in_attention;  // 1: no moments_kernel launch; the attention launch folds
                          // the chunk sums itself (AttnParams::ksum, folds_moments)
  int blocks_only;        // 1: centroid tiles only (pool_blocks_kernel; at most 16 key
                          // blocks, plain rows, no klen / tiles / ksum): the attention
                          // launch forms the moments from the tile (AttnParams::tile_moments)
};

// Key sequences whose moments the attention kernels fold from the pooling
// pass's chunk sums (AttnParams::ksum) instead of a moments_kernel launch:
// more than one 16-block chunk (one chunk's moments the pooling kernel writes
// itself) and fewer than 16 whole chunks, where moments_kernel's cascade is a
// plain sequential fold that one thread per feature repeats in a few adds.
inline bool folds_moments(int64_t nkb) { return nkb > kPoolChunk && nkb < 16 * kPoolChunk; }

// Full key covariance (covariance.hip): the full-covariance threshold
// experiment.  Partial sums over kCovSplit centroid ranges per (entry, head).
constexpr int kCovSplit = 16;

struct CovParams {
  const uint16_t* ctiles;  // [B, H, NCT, 2, 64 * D] centroid tiles (K halves read)
  const float* mean;       // [B, H, D] key centroid means
  const int32_t* klen;     // [B] key tokens per entry, or null: all Tk
  float* partial;          // [B, H, kCovSplit, D, D] workspace
  float* cov;              // [B, H, D, D]
  int B, H, Tk, NCT;
};

// Query-block pairing (pairing.hip).
constexpr int kMaxLag = 256;           // strides considered: 1 .. kMaxLag
constexpr int kMaxPairBlocks = 8192;   // query blocks per (entry, head) the lag kernel holds in LDS

struct PairParams {
  TokenRows q;
  float* qc;         // [B, H, NQB, D] FP32 query-block means (cascade order), or null
  float* means;      // [B, H, D, NQB] normalised query-block means
  float* lags;       // [B, H, D, kMaxLag] per-feature lag sums
  int32_t* strides;  // [B, H] chosen pairing stride
  int B, H, Tq, NQB;
};

struct AttnParams {
  TokenRows q;
  const int32_t* pair_stride;  // [B, H] query-block pairing stride, or null: adjacent pairs
  const int32_t* klen;         // [B] key tokens per batch entry (<= Tk), or null: all Tk
  const int64_t* out_index;    // [B, Tq] output rows of an [N, H, D] output, or null
  int64_t out_rows;            // N: rows of an out_index output (others are skipped)
  TokenRows k, v;              // key rows the kernels DMA straight into LDS (tiles null)
  const uint16_t* tiles;       // [B, H, NKB, 2, 64 * D] pooled block tiles, or null: rows of k / v
  const int32_t* block_rows;   // [B, NKB] with tiles, or null: key blocks read from rows of k / v instead
                               // (their first row; -1: from the tile)
  const uint16_t* ctiles;      // [B, H, NCT, 2, 64 * D] centroid tiles
  const float* mean;           // [B, H, D]
  const float* var;            // [B, H, D]
  const float* ksum;           // [B, H, NCH, 2, D] pooling chunk sums, or null: when set (mean / var
                               // null, folds_moments(NKB), no klen) the cutoff stage folds the moments
  int tile_moments;            // 1: mean / var null, NKB <= 16, no klen: the cutoff stage forms the
                               // moments from the K centroids of centroid tile 0
  const float* cov;            // [B, H, D, D] full key covariance, or null: diagonal (var)
  const int8_t* k8;            // [B, H, NKB, 64 * D] INT8 K tiles (quantised-QK experiment), or null
  const float* k8_scale;       // [B, H, NKB] their scales
  const uint8_t* protection;   // [B, NQB, NKB] or null
  uint16_t* out;               // [B, Tq, H, D], or [N, H, D] rows out_index
  int32_t* counts;             // [B, NQB, H] or null
  uint8_t* dbg_selected;       // [B, NQB, H, NKB] or null
  float* dbg_proxy;            // [B, NQB, H, NKB] or null
  float* dbg_cutoff;           // [B, NQB, H] or null
  int B, H, Tq, Tk, NQB, NKB, NCT;  // NKB, NCT: buffer strides for Tk
  float scale, scale_log2, beta;
  int force;          // 0 finite beta, 1 beta = -inf (all exact), 2 beta = +inf
  int local_blocks;   // < 0 disables the local band
  int kv_sink_blocks, q_sink_blocks;
  int workgroup_form;  // 0: by launch size; 1 / 2: query blocks per workgroup of
                       // sol_attention_kernel
  int splits;          // key-range parts per front (query-sink) tile, >= 1 (sol_task)
  float* partial;      // their partial states when splits > 1: rows [B H][front][G 64][D + 4]
  uint32_t* mask;      // [B, H, NQB, NW] routing decisions (route_kernel), bit j of word w = key block 32 w + j;
                       // null: the attention kernel routes tile by tile
  int NW;              // ceil(NKB / 32)
  const float* qc;     // [B, H, NQB, D] FP32 query-block means for route_kernel, or null (formed from Q)
  int head_xcds;       // workgroup map: XCDs a head's tiles are kept on (HeadMap), or 0: all (balanced_task)
  int32_t* order;      // [B H, NQB] with mask: the regular query tiles of a two-block launch in
                       // the order order_kernel deals them to the XCDs, or null: tile order
};

// Indexed-window protection (plan.hip).
struct PlanParams {
  const int64_t* rows;         // [W, nq] sorted original query rows
  const int64_t* keys;         // [W, nk] sorted original key indices
  const int32_t* key_lengths;  // [W] keys per window (clamped to nk), or null: nk
  const int64_t* ranges;       // [nranges, 2] protected ranges [a, b)
  uint8_t* out;                // [W, NQB, NKB]
  int64_t W, nq, nk, NQB, NKB, local;
  int nranges;
};

// INT8 K tiles of the quantised-QK experiment (quant.hip).
struct QuantParams {
  TokenRows k;
  const int32_t* klen;  // [B] key tokens per batch entry (<= Tk), or null: all Tk
  int8_t* k8;           // [B, H, NKB, 64 * D]
  float* scale;         // [B, H, NKB]
  int B, H, Tk, NKB;
  int shifted;          // partial last blocks as the rows-mode attention tiles hold them
};

// Key-split groups of sol_small_kernel for a launch of `blocks` query blocks
// (over all entries and heads) against nkb key blocks, or 0 when the launch
// takes sol_attention_kernel.  Small launches leave most SIMDs idle, so their
// time is one workgroup's tile chain: KS groups of two waves split it KS ways,
// four while a CU holds one workgroup (at most kSmallBlocks query blocks), two
// while it holds two, or for one or two key blocks at head_dim 128 (2 x 121 x 63
// keys x 32 heads 20.9 -> 18.8 us a call, 1,000 x 128 x 8 17.0 -> 15.0, 128 x 128 x 8
// 14.6 -> 14.8; at 64 four groups may pool the keys too).  A query-sink block's chain is every key block: with two
// or more of them, over keys of more than kSmallChain steps, the launch goes
// to the one-block kernel, whose sink tiles split over workgroups instead (a
// single sink block is not split there).
constexpr int64_t kSmallBlocks = 256;
constexpr int64_t kSmallChain = 8;  // at head_dim 128; twice that at 64
inline int small_key_split(int64_t blocks, int64_t nkb, int64_t q_sink_blocks, int64_t head_dim) {
  const int ks = blocks <= kSmallBlocks && !(head_dim == 128 && nkb <= 2) ? 4 : 2;
  if (blocks > 2 * kSmallBlocks || nkb > kMaxKeyBlocks) return 0;
  return q_sink_blocks < 2 || nkb <= kSmallChain * ks * (128 / head_dim) ? ks : 0;
}

// K and V bytes of one head's key blocks.
inline int64_t head_key_bytes(int64_t nkb, int64_t head_dim) { return nkb * kBlock * head_dim * 4; }

// Share of the key blocks that a query block selects, as the threshold aims at
// it: that of a normal above beta (force 1: beta = -inf, 2: +inf).
inline double selected_share(int force, double beta) {
  return force == 1 ? 1.0 : force == 2 ? 0.0 : 0.5 * std::erfc(beta / std::sqrt(2.0));
}

// One query block per workgroup (a K and a V slot each, four workgroups per
// CU at head_dim 128) or two (a ring of two slots, the union of the pair's
// blocks, two workgroups per CU); AttnParams::workgroup_form 0.  Two blocks
// stream fewer bytes, but a wave idles on the tiles only its partner selected.
// One block while at most half the key blocks are selected, these are no more
// than half the head's query blocks (the workgroups that share a key tile's
// read from the L2), and K and V are at most 12 MB per head, 5 MB of them
// selected.  us a call, two blocks -> one, video field and random: 2 x 4,096 x
// 16 heads x D128 beta 1 119 -> 102, 125 -> 100, beta 0 205 -> 192, 217 -> 194,
// beta -1 9% and 5% slower; 4,096 x 10,000 keys x 24 beta 1 193 -> 179, 219 ->
// 185, beta 0 3% slower in the field; 2,048 x 8,192 x 32 beta 1 8% slower in the
// field; 24,576 x 24 beta 1 1860 -> 1719, 1971 -> 1932, beta 0 7% and 1% slower.
// Indexed windows need no copies of their keys in the one-block form: while 70%
// are selected, or with at most 192 key blocks (two -> one: 21 x 4,032 x 24
// beta 0 13753 -> 11878, beta -1 1% slower, at D64 beta -inf 9480 -> 9793; 21 x
// 2,000 x 24 beta -inf 4815 -> 4372).
// Launches of fewer than 512 pairs (256 CUs x 2 workgroups) would leave CUs
// idle with two.
// INT8 scores (the experiment) have no one-slot form: at head_dim 128 a
// one-block workgroup holds a 64 KB ring too, so a CU has half the waves of the
// two-block form.  us per call, one block -> two: 2 x 4,096 x 16 heads beta 1
// 155 -> 132, beta 0 269 -> 208; 16,384 x 8 367 -> 315; 32,768 x 16 2417 ->
// 2058; 21 x 4,032 windows x 24 10258 -> 9304.  At 64, where the ring is 32 KB, it
// is one way or the other: 2 x 4,096 x 16 beta 1 83 -> 93, beta -inf 215 -> 175;
// 2 x 1,823 windows x 32 beta +inf 145 -> 138.
constexpr int64_t kOneBlockKeyBytes = int64_t(12) << 20;
constexpr double kOneBlockSelectedBytes = 5 << 20;
constexpr int64_t kSmallLaunchGroups = 512;
inline bool one_block_launch(int64_t bh, int64_t nqb, int64_t nkb, int64_t head_dim, double share, bool int8,
                             bool windows) {
  if (bh * ((nqb + 1) / 2) < kSmallLaunchGroups) return true;
  const int64_t bytes = head_key_bytes(nkb, head_dim);
  if (bytes > kOneBlockKeyBytes || int8) return false;
  if (windows) return share <= 0.7 || nkb <= 192;
  return share <= 0.5 && 2 * share * double(nkb) <= double(nqb) && share * double(bytes) <= kOneBlockSelectedBytes;
}

// XCDs per head of a one-block launch (HeadMap; 0: balanced_task, every head
// on all eight).  On fewer, more of an XCD's workgroups stream the same keys
// through its L2 -- heads alike, 1, 2, 4 XCDs and all: 19,003 tokens x 16 heads
// 654, 657, 692, 777 us a call, 8,192 x 24 212, 212, 227, 264, 2 x 4,096 x 16
// 100, 100, 108, 121 -- but an XCD's work is what its heads select, and heads
// do differ: with one of 16 heads at half the blocks and the others at 2% (19,003,
// beta 2) 640, 501, 379, 334 us, where two-block workgroups on the
// balanced map took 388.  So the fewest XCDs at which the most that one head can
// hold up its group is kUnevenMax times the average.  A head costs at least 8
// steps' time and its centroid tiles per query block, at most half the key
// blocks more (the threshold is at least the mean); one such head among a
// group's P and the launch's `heads`.  Over 140 inputs -- one dense head, a
// quarter, every fourth, random densities; 4,096 to 24,576 tokens, 8 to 32 heads
// -- the launches took 0.61 to 1.05 of the two-block form's time there (1.05: one
// dense head of 24 at 10,000 tokens and beta 2).  At 1.7 that call took 0.87, and 4,096
// queries x 10,000 keys x 24 heads 182 instead of 164 us.
constexpr double kUnevenMax = 1.75;
inline int xcds_per_head(int64_t heads, int64_t nkb) {
  const double base = 8.0 + double(nkb) / kBlock, more = 0.5 * double(nkb) / base;
  for (int xcds = 1; xcds <= 4; xcds *= 2) {
    const double group = double(heads) * xcds / 8.0;
    if ((more / group + 1.0) <= kUnevenMax * (more / double(heads) + 1.0)) return xcds;
  }
  return 0;
}

// With K and V per head far beyond the L2 a head's own XCDs gain nothing, and
// eight heads at a time no longer fit the 256 MB memory-side cache.
constexpr int64_t kHeadMapKeyBytes = int64_t(24) << 20;

hipError_t launch_pool(const PoolParams& p, int D, hipStream_t stream);
hipError_t launch_quantize_keys(const QuantParams& p, int D, hipStream_t stream);
hipError_t launch_route(const AttnParams& p, int D, hipStream_t stream);
hipError_t launch_sol(const AttnParams& p, int D, hipStream_t stream);
hipError_t launch_dense(const AttnParams& p, int D, hipStream_t stream);
hipError_t launch_pairing(const PairParams& p, int D, hipStream_t stream);
hipError_t launch_plan_protection(const PlanParams& p, hipStream_t stream);
hipError_t launch_covariance(const CovParams& p, int D, hipStream_t stream);

}  // namespace sol
