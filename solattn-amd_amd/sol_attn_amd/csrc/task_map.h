// Workgroup -> query-tile maps of the attention kernels: plain index
// arithmetic, for the kernels and for the host.
#pragma once

#include <cstdint>

namespace sol {

constexpr int kXcds = 8;

// Workgroup ids are dealt round-robin over the 8 XCDs.  The id -> (head, query
// tile) map keeps every XCD on the SAME head at the same time, each on its own
// contiguous slice of that head's query tiles: neighbouring tiles share that
// XCD's L2, and the tiles of one head (43 MB at 84,672 tokens) are the whole
// live set of the memory-side cache.  The first F ids (a SOL launch's
// query-sink tiles, sol_task) go ahead of that map; after them, XCD x's
// workgroups take, head after head, its slice of the head's R tiles: floor(R
// / 8) tiles, one more for the XCDs that the R mod 8 leftover tiles of each
// head are dealt to -- round-robin, continuing from the F front ids -- so that
// every XCD holds the same number of workgroups to within one.  (Equal
// ceil(R / 8) slices with the last XCD short left 7 XCDs a workgroup round
// more than the eighth when R mod 8 != 0, or when the front ids fell on
// them: at 32,768 tokens x 4 heads with 128-token sinks, 129 workgroups
// against 64 slots per XCD.)  Ids past an XCD's count return -1 (idle).
struct TileTask {
  int bh, tile;
  int split = 0;  // key-range part of a split front tile (sol_task)
};

// Regular workgroup id i >= F: (head, tile in [0, R)) as described above.
__host__ __device__ inline TileTask balanced_task(int i, int F, int heads, int R) {
  const int x = i % kXcds, k = i / kXcds;
  const int fx = F > x ? (F - x + kXcds - 1) / kXcds : 0;  // front ids of XCD x
  const int kr = k - fx;                                    // its regular index
  const int base = R / kXcds, rem = R % kXcds;
  const int r0 = ((x - F) % kXcds + kXcds) % kXcds;  // leftover e goes to XCD (F + e) % 8
  // XCD x's regular workgroups in heads [0, h).
  auto cum = [&](int h) {
    const int n = h * rem;
    return h * base + (n > r0 ? (n - 1 - r0) / kXcds + 1 : 0);
  };
  int h = R > 0 ? min(heads, int(int64_t(kr) * kXcds / R)) : heads;
  while (h > 0 && cum(h) > kr) --h;
  while (h < heads && cum(h + 1) <= kr) ++h;
  if (h >= heads || kr < 0) return TileTask{-1, 0};
  // Start of XCD x's slice of head h: the slices of XCDs 0 .. x-1, of which
  // those in [c, c + rem) (mod 8) hold one leftover tile more.
  const int c = (F + h * rem) % kXcds;
  const int extra_before = c + rem <= kXcds ? max(0, min(x, c + rem) - c)
                                            : max(0, x - c) + min(x, c + rem - kXcds);
  return TileTask{h, x * base + extra_before + (kr - cum(h))};
}

// Workgroups of a launch of F front ids and `heads` x R regular tiles: every
// XCD's count, rounded up, eight times.
__host__ __device__ inline unsigned balanced_grid(int F, int heads, int R) {
  const int64_t total = int64_t(F) + int64_t(heads) * R;
  return unsigned(kXcds * ((total + kXcds - 1) / kXcds));
}

// Start of XCD x's even share of n tasks in a row.
__host__ __device__ inline int xcd_start(int n, int x) { return n / kXcds * x + n % kXcds * x / kXcds; }

// The other map (`head_xcds` = 1, 2 or 4): every head -- (entry, head) pair --
// belongs to a group of that many XCDs, so that its keys are read into those
// L2s alone instead of all eight.  Whole rounds of heads are dealt to the 8 /
// head_xcds groups in turn, each round starting three groups further on (heads
// that cost alike at a regular distance, as those of a batch's entries, meet
// different groups); the tiles of the last, partial round are one list that is
// cut evenly over the XCDs.  A group's XCDs take a slice of a head's tiles each
// -- neighbouring tiles select much the same keys: dealt out one by one a video
// field of 19,003 tokens x 16 heads took 719 us a call, in slices 659 -- and the
// slices are passed round from head to head, as R need not divide evenly.
struct HeadMap {
  int xcds, groups;     // XCDs per group; groups
  int rounds, rest, R;  // whole rounds of heads, heads of the partial one, tiles per head
  __host__ __device__ HeadMap(int heads, int R, int xcds)
      : xcds(xcds), groups(kXcds / xcds), rounds(heads / groups), rest(heads % groups), R(R) {}
  // Start of slice s of a head's tiles, and the slice the m-th XCD takes in round r.
  __host__ __device__ int slice(int s) const { return R / xcds * s + R % xcds * s / xcds; }
  __host__ __device__ int turn(int m, int r) const { return (m + r) % xcds; }
  // Tiles of XCD x in the whole rounds (R in every `xcds` of them), and in all.
  __host__ __device__ int whole(int x) const {
    int n = rounds / xcds * R;
    for (int r = 0; r < rounds % xcds; ++r) n += slice(turn(x % xcds, r) + 1) - slice(turn(x % xcds, r));
    return n;
  }
  __host__ __device__ int count(int x) const { return whole(x) + xcd_start(rest * R, x + 1) - xcd_start(rest * R, x); }
  // The k-th tile of XCD x (-1: past its last one).
  __host__ __device__ TileTask task(int x, int k) const {
    if (k >= count(x)) return TileTask{-1, 0};
    const int w = whole(x);
    if (k >= w) {
      const uint32_t j = uint32_t(xcd_start(rest * R, x) + (k - w));
      return TileTask{rounds * groups + int(j / uint32_t(R)), int(j % uint32_t(R))};
    }
    const int m = x % xcds;
    int r = int(uint32_t(k) / uint32_t(R)) * xcds, t = int(uint32_t(k) % uint32_t(R));
    int s = m, n = slice(s + 1) - slice(s);  // round r is a whole cycle's first: turn(m, r) = m
    while (t >= n) {
      t -= n;
      s = turn(m, ++r);
      n = slice(s + 1) - slice(s);
    }
    return TileTask{r * groups + (x / xcds + 3 * r) % groups, slice(s) + t};
  }
};

// Workgroups of a HeadMap launch of F front ids and `heads` x R regular tiles:
// the fullest XCD's, eight times.
inline unsigned head_grid(int F, int heads, int R, int xcds) {
  const HeadMap map(heads, R, xcds);
  int most = 0;
  for (int x = 0; x < kXcds; ++x) {
    const int n = xcd_start(F, x + 1) - xcd_start(F, x) + map.count(x);
    most = n > most ? n : most;
  }
  return unsigned(kXcds) * unsigned(most);
}

// SOL launches dispatch the first `front` query tiles of every (entry, head)
// ahead of the rest, head-interleaved.  With query sinks those tiles hold the
// sink query blocks, whose workgroups stream every key block and run several
// times longer than the others; behind the regular map the last heads' ones
// would start late and set the kernel's end (2 x 4,096 tokens x 16 heads with
// 128-token sinks: 251 -> 163 us).  The first `split_tiles` of them (<=
// front) are `splits` workgroups each, one per key range (split_range), whose
// partial states sol_merge_kernel combines.  The remaining tiles follow
// balanced_task or, with head_xcds, HeadMap (whose front ids are shared out
// evenly).  In 32 bits: a launch has fewer than 2^31 workgroups.
__host__ __device__ inline TileTask sol_task(int i, int ntiles, int front, int split_tiles, int heads, int splits,
                                             int head_xcds) {
  if (head_xcds) {
    const int x = i % kXcds, k = i / kXcds;
    const int per = split_tiles * splits + (front - split_tiles);  // front ids per head
    const int F = per * heads;
    const int nf = xcd_start(F, x + 1) - xcd_start(F, x);
    if (k < nf) {
      const uint32_t j = uint32_t(xcd_start(F, x) + k);
      const int h = int(j / uint32_t(per)), e = int(j % uint32_t(per));
      if (e < split_tiles * splits) return TileTask{h, e / splits, e % splits};
      return TileTask{h, split_tiles + e - split_tiles * splits};
    }
    TileTask t = HeadMap(heads, ntiles - front, head_xcds).task(x, k - nf);
    t.tile += front;
    return t;
  }
  const int nsplit = split_tiles * heads * splits;
  if (i < nsplit) {
    const int j = i / heads;
    return TileTask{i % heads, j / splits, j % splits};
  }
  const int nrest = (front - split_tiles) * heads;
  if (i - nsplit < nrest) return TileTask{(i - nsplit) % heads, split_tiles + (i - nsplit) / heads};
  TileTask t = balanced_task(i, nsplit + nrest, heads, ntiles - front);
  t.tile += front;
  return t;
}

// Query-sink tiles split by key range (sol_task) when a launch is split: the
// tiles of sink blocks [0, 2 floor(q_sink_blocks / 2)).  With adjacent
// pairing those tiles hold sink blocks only, in either workgroup form, so
// whether a query block is split depends on its index alone and both forms
// stay bit-identical.  A split launch pairs adjacent blocks (it ignores
// pair_stride).
__host__ __device__ inline int sink_split_tiles(int splits, int q_sink_blocks, int G, int front) {
  return splits > 1 ? min(front, (q_sink_blocks / 2 * 2) / G) : 0;
}

}  // namespace sol
