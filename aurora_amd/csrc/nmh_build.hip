// NMH build on gfx950: replaces cudaRebuildNMH (src/kernels/rebuilder.cu:311-450).
//
// Result (bit-identical to the reference's canonical semantics): the tree
// order of the triangles.  Node k of the implicit heap owns tree positions
// 2k and 2k+1; its children are nodes 2k+1 and 2k+2.
//
// The reference sorts the whole array by (node label, min key) at every level
// (sortTriangles, rebuilder.cu:262-289) with two Thrust radix sorts, swaps the
// first maximum of the max key into slot +1 (rebuilder.cu:127-151), relabels
// nodes and emits child splits through a host round trip per level
// (rebuilder.cu:247-260).  Here:
//   * subtree sizes and offsets of the left-complete tree are closed forms
//     (desc_count), so split emission and all host synchronisation vanish;
//   * only the pending region is sorted; finished node pairs are not moved
//     again -- their final in-pair order, which the reference obtains by
//     re-sorting them at every later level, is computed once as a
//     lexicographic comparison of the later levels' keys (newest first; only
//     the last three levels can differ since axes cycle with period 3);
//   * while node groups are larger than one workgroup's LDS tile, a level is a
//     segmented stable LSD radix sort (8-bit digits; a pass is a launch for
//     the tile histograms and one that sums every tile's offsets, ranks with
//     wave ballots and scatters) followed by a
//     tiled first-maximum reduction and an emit pass that writes finished
//     pairs and compacts the remainders for the next level.  The digits are
//     those of key - (the group's smallest key), so a group whose keys span
//     fewer than 2^24 values needs 3 passes (2^16: 2, ...): the emit pass
//     records each tile's key range, and the next level's first scatter
//     reduces them to its group's (smallest key, passes);
//   * once every group fits (<= kSubT elements) one workgroup takes a whole
//     subtree and runs all remaining levels in LDS with a bitonic sort on
//     (group, key, position) composite keys.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "context.h"

namespace aur {
namespace {

constexpr uint32_t kTile = 2048;  // radix / emit tile (elements)
constexpr uint32_t kChunk = 32;   // tiles per chunk of the radix offset scan
// Levels with a group of more chunks than this (4.2M triangles) sum the chunks
// in a launch of their own: otherwise every tile of the group reads all of them.
// Device time per build with and without it: 10.76 and 10.91 ms at 10M, 24.0
// and 25.1 ms at 20M.  Limits of 24 and 120 differ by less than 1% at 1M to 20M.
constexpr uint32_t kScanChunks = 64;
constexpr uint32_t kSubT = 4096;  // max elements of an LDS-resident subtree
constexpr int kThreads = 256;
constexpr int kSubThreads = 1024;  // k_subtree

struct TileDesc {
  uint32_t start, count, child, group;
};
struct ChildDesc {
  uint32_t off, size, tb, te;
};
struct GroupDesc {
  uint32_t off, size, tb, te, cb, ce;  // tiles [tb, te), offset chunks [cb, ce)
};
struct SubGroup {
  uint32_t off, size, first, count;
};

// Order of a finished pair x, y of a level <= L - 2: whether y comes first.
// The reference re-sorts every finished pair at the later levels; only the
// last three can differ.  key(axis, element): the element's min key.
template <class Key>
__device__ __forceinline__ bool second_first(uint32_t x, uint32_t y, int level, int L, Key key) {
  const int lo = max(level + 1, L - 3);
  for (int lev = L - 1; lev >= lo; --lev) {
    const auto kx = key(lev % 3, x), ky = key(lev % 3, y);
    if (ky < kx) return true;
    if (kx < ky) return false;
  }
  return false;
}

// bb: triangle bounds (min, max), [axis][triangle].
__device__ inline void write_pair(uint32_t h, uint32_t x, uint32_t y, int level, int L,
                                  const float2* __restrict__ bb, uint32_t N,
                                  uint32_t* __restrict__ P) {
  const bool swap = second_first(x, y, level, L, [&](int a, uint32_t i) { return bb[(size_t)a * N + i].x; });
  P[2 * (size_t)h] = swap ? y : x;
  P[2 * (size_t)h + 1] = swap ? x : y;
}

// computeTriangleBounds (rebuilder.cu:72-91), (min, max) pairs [axis][triangle]:
// one 8-byte load gives both keys of a triangle on an axis.
// With V also the identity order with the axis-0 max keys (the sort's payload)
// and the first level's axis-0 sort keys K.
__global__ void k_bounds(const float* __restrict__ v, uint32_t N, float2* __restrict__ bb, uint2* __restrict__ V,
                         uint32_t* __restrict__ K) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const float* p = v + (size_t)i * 9;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float2 b = make_float2(fminf(fminf(p[3 * a], p[3 * a + 1]), p[3 * a + 2]),
                                 fmaxf(fmaxf(p[3 * a], p[3 * a + 1]), p[3 * a + 2]));
    bb[(size_t)a * N + i] = b;
    if (a == 0 && V) {
      V[i] = make_uint2(i, fkey(b.y));
      K[i] = fkey(b.x);
    }
  }
}

// Indices read back from device arrays are clamped to [0, N) before they
// address another array: a defect then shows up as a wrong tree in the parity
// tests, never as an out-of-bounds access.
__device__ __forceinline__ uint32_t clampi(uint32_t i, uint32_t N) { return i < N ? i : N - 1; }

// Radix passes a group needs: its keys minus the smallest, k - r.x, span
// [0, r.y - r.x]; digits above the span's top byte are zero in every key, and
// a stable sort by a digit that is equal for all keys keeps the order.  Pass
// 0 runs for every group (its digit, (k - r.x) & 255, is a rotation of the
// key's low byte, and the group's range is known only after the pass's
// histograms).  Pass p of a level moves the groups with group_passes > p,
// from buffer p & 1 to the other, so a group's sorted data ends in buffer
// group_passes & 1.  Kernels read a tile's (smallest key, passes) as
// TP[tile] (by block index, so the load does not wait for the tile's
// descriptor).
__device__ __forceinline__ uint32_t group_passes(uint2 r) {
  const uint32_t d = r.y - r.x;
  return d < 0x10000u ? (d < 0x100u ? 1u : 2u) : (d < 0x1000000u ? 3u : 4u);
}

__global__ void k_fill0(uint32_t* __restrict__ p, uint32_t N) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < N) p[i] = 0;
}

// Inclusive scan of one value per thread over the 256 threads (4 waves):
// shuffles within each wave, then the wave totals through LDS.
__device__ __forceinline__ uint32_t block_incl_scan256(uint32_t v, uint32_t* __restrict__ wsum) {
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t u = __shfl_up(v, off);
    if (lane >= (uint32_t)off) v += u;
  }
  if (lane == 63) wsum[wave] = v;
  __syncthreads();
  for (uint32_t w = 0; w < wave; ++w) v += wsum[w];
  return v;
}

// Key range of a group, by a block: from the previous level's emit tiles of the
// group's parent node (prev_children[group], tile ranges TR), or the full range
// on the first level (prev_children null).
__device__ __forceinline__ uint2 group_range(const ChildDesc* __restrict__ prev_children, uint32_t group,
                                             const uint2* __restrict__ TR) {
  __shared__ uint32_t rmin[kThreads / 64], rmax[kThreads / 64];
  if (!prev_children) return make_uint2(0u, 0xFFFFFFFFu);  // uniform: a kernel argument
  const ChildDesc pc = prev_children[group];
  uint32_t mn = 0xFFFFFFFFu, mx = 0u;
  for (uint32_t t = pc.tb + threadIdx.x; t < pc.te; t += kThreads) {
    const uint2 tr = TR[t];
    mn = min(mn, tr.x);
    mx = max(mx, tr.y);
  }
  for (int off = 32; off > 0; off >>= 1) {
    mn = min(mn, (uint32_t)__shfl_xor(mn, off));
    mx = max(mx, (uint32_t)__shfl_xor(mx, off));
  }
  if ((threadIdx.x & 63u) == 0) {
    rmin[threadIdx.x >> 6] = mn;
    rmax[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  uint2 r = make_uint2(rmin[0], rmax[0]);
#pragma unroll
  for (int w = 1; w < kThreads / 64; ++w) r = make_uint2(min(r.x, rmin[w]), max(r.y, rmax[w]));
  return r;
}

// f(row, R[row][threadIdx.x]) for the rows [b, e) of 256 counts, eight loads in
// flight (the last eight repeat a row rather than go one at a time).
template <class F>
__device__ __forceinline__ void each_row(const uint32_t* __restrict__ R, uint32_t b, uint32_t e, F&& f) {
  for (uint32_t r = b; r < e; r += 8) {
    uint32_t v[8];
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u) v[u] = R[(size_t)min(r + u, e - 1) * 256 + threadIdx.x];
#pragma unroll
    for (uint32_t u = 0; u < 8; ++u)
      if (r + u < e) f(r + u, v[u]);
  }
}

// Exclusive sum over the digits before digit threadIdx.x of `total`, in the
// order of (digit - rot) & 255.  s: 256 words of LDS.
__device__ __forceinline__ uint32_t digit_offset(uint32_t total, uint32_t rot, uint32_t* s, uint32_t* wsum) {
  const uint32_t sp = (threadIdx.x - rot) & 255u;
  s[sp] = total;
  __syncthreads();
  const uint32_t own = s[threadIdx.x];
  s[threadIdx.x] = block_incl_scan256(own, wsum) - own;
  __syncthreads();
  return s[sp];
}

// Per-tile digit histogram H[tile][digit], also added into its chunk's digit
// counts CS[chunk][digit] (integer atomics: the sums are exact whatever the
// order).  CS starts at zero: all of it before the first level, and the rows of
// the next pass's counts (CSnext) are zeroed here, by the first tile of each
// chunk.  Pass 0 counts the key's low byte (indexed so; k_radix_scatter and
// k_radix_group_scan order the digits).
__global__ __launch_bounds__(kThreads) void k_radix_hist(const TileDesc* __restrict__ tiles,
                                                         const GroupDesc* __restrict__ groups,
                                                         const uint2* __restrict__ TP,
                                                         const uint32_t* __restrict__ K,
                                                         uint32_t pass,
                                                         uint32_t* __restrict__ H,
                                                         uint32_t* __restrict__ CS,
                                                         uint32_t* __restrict__ CSnext) {
  __shared__ uint32_t h[256];
  const TileDesc t = tiles[blockIdx.x];
  const GroupDesc g = groups[t.group];
  const uint32_t in_group = blockIdx.x - g.tb, chunk = g.cb + in_group / kChunk;
  if (in_group % kChunk == 0) CSnext[(size_t)chunk * 256 + threadIdx.x] = 0u;
  uint32_t kmin = 0;
  if (pass > 0) {
    const uint2 tp = TP[blockIdx.x];
    if (tp.y <= pass) return;  // uniform per block
    kmin = tp.x;
  }
  const uint32_t shift = 8u * pass;
  h[threadIdx.x] = 0;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < t.count; i += kThreads)
    atomicAdd(&h[((K[t.start + i] - kmin) >> shift) & 255u], 1u);
  __syncthreads();
  const uint32_t v = h[threadIdx.x];
  H[(size_t)blockIdx.x * 256 + threadIdx.x] = v;
  if (v) atomicAdd(&CS[(size_t)chunk * 256 + threadIdx.x], v);
}

// For levels with groups of many chunks (kScanChunks).  Per group: exclusive
// digit offsets of the group (digit-major), and the base B[chunk][digit] of
// every chunk of the group (the counts of the group's earlier chunks added).
// Pass 0 first sets the group's key range: GP[group] and TP[tile] of the group
// take (smallest key, passes).  Its digits are the keys' low bytes, scanned in
// the order of (low byte - smallest key) & 255.
__global__ __launch_bounds__(kThreads) void k_radix_group_scan(const GroupDesc* __restrict__ groups,
                                                               uint2* __restrict__ GP,
                                                               uint2* __restrict__ TP,
                                                               const ChildDesc* __restrict__ prev_children,
                                                               const uint2* __restrict__ TR,
                                                               uint32_t pass,
                                                               const uint32_t* __restrict__ S,
                                                               uint32_t* __restrict__ B) {
  __shared__ uint32_t s[256], wsum[kThreads / 64];
  const uint32_t d = threadIdx.x;
  uint32_t rot = 0;  // scan position of digit d: (d - rot) & 255
  const GroupDesc g = groups[blockIdx.x];
  if (pass > 0 && GP[blockIdx.x].y <= pass) return;  // uniform per block
  // the group's digit counts first: their loads then overlap the range's
  uint32_t total = 0;
#pragma unroll 8
  for (uint32_t c = g.cb; c < g.ce; ++c) total += S[(size_t)c * 256 + d];
  if (pass == 0) {
    const uint2 r = group_range(prev_children, blockIdx.x, TR);
    const uint2 gp = make_uint2(r.x, group_passes(r));
    if (d == 0) GP[blockIdx.x] = gp;
    for (uint32_t t = g.tb + d; t < g.te; t += kThreads) TP[t] = gp;
    rot = r.x & 255u;
  }
  uint32_t run = g.off + digit_offset(total, rot, s, wsum);
#pragma unroll 8
  for (uint32_t c = g.cb; c < g.ce; ++c) {
    B[(size_t)c * 256 + d] = run;
    run += S[(size_t)c * 256 + d];
  }
}

// Stable scatter of one 2048-element tile, staged through LDS.  Ranking:
// wave w owns the tile's elements [512w, 512w + 512) in rounds of 64; lanes
// with the same digit are found with 8 ballots, and the wave keeps its
// running count per digit in its own LDS row (read, then written by the
// digit's first lane, in the wave's program order: no workgroup barrier per
// round).  Each element (key and 8-byte payload) then lands in LDS at its
// digit-sorted tile position, and the tile is written out in that order: a
// digit's run is one contiguous store at the tile's output offset for the
// digit.  (Ranking in rounds of 256 elements across the
// workgroup, with four barriers per round, took 20-35% longer; staging only
// a 16-bit tile index and re-reading the payload at write-out measured 6%
// slower despite the smaller LDS footprint.)
// The tile's output offsets: the group's digit offsets and the counts of the
// group's earlier chunks (from the chunks' counts CS, or with B as
// k_radix_group_scan left them), and the counts of the chunk's earlier tiles.
// Without B, pass 0 also sets the tile's (smallest key, passes), TP[tile].
// They are summed here, once per tile and after the ranking (the payload's
// loads are then still in flight behind it), because two launches for them, per
// group and per chunk, cost 9 us of a pass of 29 at 1M triangles and not less
// at 10M (1.35 -> 1.17 ms and 11.0 -> 10.9 ms of device time per build; before
// the ranking: 11.1).
__global__ __launch_bounds__(kThreads) void k_radix_scatter(
    const TileDesc* __restrict__ tiles, const GroupDesc* __restrict__ groups, uint2* __restrict__ TP,
    const ChildDesc* __restrict__ prev_children, const uint2* __restrict__ TR,
    const uint32_t* __restrict__ Kin, const uint2* __restrict__ Vin, uint32_t pass,
    const uint32_t* __restrict__ H, const uint32_t* __restrict__ CS, const uint32_t* __restrict__ B,
    uint32_t m, uint32_t* __restrict__ Kout, uint2* __restrict__ Vout) {
  constexpr uint32_t kWaves = kThreads / 64;
  constexpr uint32_t kRounds = kTile / kThreads;  // rounds of 64 per wave
  __shared__ uint32_t sk[kTile];
  __shared__ uint2 sv[kTile];
  __shared__ uint32_t wc[kWaves][256];  // per-wave running digit counts, then tile positions
  __shared__ uint32_t delta[256];       // output position - tile position, per digit
  __shared__ uint32_t wsum[kWaves];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const TileDesc t = tiles[blockIdx.x];
  uint32_t kmin = 0;  // pass 0: the low byte itself (the offsets follow the group's digit order)
  if (pass > 0) {
    const uint2 tp = TP[blockIdx.x];
    if (tp.y <= pass) return;  // uniform per block
    kmin = tp.x;
  }
  const uint32_t shift = 8u * pass;
#pragma unroll
  for (uint32_t q = 0; q < 4; ++q) wc[wave][q * 64 + lane] = 0;
  const uint32_t w0 = wave * (kRounds * 64);
  uint32_t k[kRounds], loc[kRounds];
  uint2 v[kRounds];
#pragma unroll
  for (uint32_t r = 0; r < kRounds; ++r) {
    const uint32_t i = w0 + r * 64 + lane;
    const bool valid = i < t.count;
    k[r] = valid ? Kin[t.start + i] : 0u;
    v[r] = valid ? Vin[t.start + i] : make_uint2(0u, 0u);
  }
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (uint32_t r = 0; r < kRounds; ++r) {
    const bool valid = w0 + r * 64 + lane < t.count;
    const uint32_t dg = ((k[r] - kmin) >> shift) & 255u;
    uint64_t mask = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bool bit = (dg >> b) & 1u;
      const uint64_t bb = __ballot(bit);
      mask &= bit ? bb : ~bb;
    }
    const uint32_t rank = __popcll(mask & lt_mask);
    const uint32_t off = wc[wave][dg];
    if (valid && rank == 0) wc[wave][dg] = off + (uint32_t)__popcll(mask);
    loc[r] = off + rank;
  }
  // thread tid = digit d: the tile's output offset
  const GroupDesc g = groups[t.group];
  const uint32_t in_group = blockIdx.x - g.tb, chunk = g.cb + in_group / kChunk;
  uint32_t base = 0;
  if (B) {
    base = B[(size_t)chunk * 256 + tid];
  } else {
    uint32_t total = 0;
    each_row(CS, g.cb, g.ce, [&](uint32_t c, uint32_t v) {
      total += v;
      base += c < chunk ? v : 0u;
    });
    uint32_t rot = 0;
    if (pass == 0) {
      const uint2 r = group_range(prev_children, t.group, TR);
      if (tid == 0) TP[blockIdx.x] = make_uint2(r.x, group_passes(r));
      rot = r.x & 255u;
    }
    base += g.off + digit_offset(total, rot, delta, wsum);
  }
  each_row(H, blockIdx.x - in_group % kChunk, blockIdx.x, [&](uint32_t, uint32_t v) { base += v; });
  __syncthreads();
  // thread tid = digit d: the tile's count, its first tile position, and
  // the first tile position of each wave's elements with digit d
  uint32_t c[kWaves], cnt = 0;
#pragma unroll
  for (uint32_t w = 0; w < kWaves; ++w) {
    c[w] = wc[w][tid];
    cnt += c[w];
  }
  const uint32_t first = block_incl_scan256(cnt, wsum) - cnt;
  {
    uint32_t run = first;
#pragma unroll
    for (uint32_t w = 0; w < kWaves; ++w) {
      wc[w][tid] = run;
      run += c[w];
    }
  }
  delta[tid] = base - first;
  __syncthreads();
#pragma unroll
  for (uint32_t r = 0; r < kRounds; ++r) {
    if (w0 + r * 64 + lane < t.count) {
      const uint32_t pos = wc[wave][((k[r] - kmin) >> shift) & 255u] + loc[r];
      if (pos < kTile) {
        sk[pos] = k[r];
        sv[pos] = v[r];
      }
    }
  }
  __syncthreads();
  const uint32_t n_out = min(t.count, kTile);
  for (uint32_t j = tid; j < n_out; j += kThreads) {
    const uint32_t key = sk[j];
    const uint32_t pos = delta[((key - kmin) >> shift) & 255u] + j;
    if (pos < m) {
      Kout[pos] = key;
      Vout[pos] = sv[j];
    }
  }
}

// First maximum of the max key over child positions [off+1, off+size)
// restricted to this tile: (key, position), key 0 = none.  The group's sorted
// data is in V0 or V1 (group_passes).
__global__ __launch_bounds__(kThreads) void k_argmax_partial(const TileDesc* __restrict__ tiles,
                                                             const ChildDesc* __restrict__ children,
                                                             const uint2* __restrict__ TP,
                                                             const uint2* __restrict__ V0,
                                                             const uint2* __restrict__ V1,
                                                             uint2* __restrict__ partial) {
  __shared__ uint32_t sk[kThreads / 64], sp[kThreads / 64];
  const TileDesc t = tiles[blockIdx.x];
  const ChildDesc c = children[t.child];
  const uint2* __restrict__ V = (TP[blockIdx.x].y & 1u) ? V1 : V0;
  const uint32_t lo = max(t.start, c.off + 1), hi = t.start + t.count;
  uint32_t bk = 0, bp = 0xFFFFFFFFu;
  for (uint32_t i = lo + threadIdx.x; i < hi; i += kThreads) {
    const uint32_t k = V[i].y;  // the element's max key, carried by the sort
    if (k > bk) {
      bk = k;
      bp = i;
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    const uint32_t ok = __shfl_xor(bk, off), op = __shfl_xor(bp, off);
    if (ok > bk || (ok == bk && op < bp)) {
      bk = ok;
      bp = op;
    }
  }
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  if (lane == 0) {
    sk[wave] = bk;
    sp[wave] = bp;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kThreads / 64; ++w)
      if (sk[w] > bk || (sk[w] == bk && sp[w] < bp)) {
        bk = sk[w];
        bp = sp[w];
      }
    partial[blockIdx.x] = make_uint2(bk, bp);
  }
}

// (max key, lowest position) over a child's tiles, by a block: every block of
// k_emit takes its own, as a launch for it cost 4 us a level (8 at 10M).
__device__ __forceinline__ uint32_t child_argmax(const ChildDesc& d, const uint2* __restrict__ partial) {
  __shared__ uint2 best[kThreads / 64];
  uint2 b = make_uint2(0u, 0xFFFFFFFFu);
  const auto take = [&](uint2 p) {
    if (p.x > b.x || (p.x == b.x && p.y < b.y)) b = p;
  };
  for (uint32_t t = d.tb + threadIdx.x; t < d.te; t += kThreads) take(partial[t]);
  for (int off = 32; off > 0; off >>= 1)
    take(make_uint2((uint32_t)__shfl_xor(b.x, off), (uint32_t)__shfl_xor(b.y, off)));
  if ((threadIdx.x & 63u) == 0) best[threadIdx.x >> 6] = b;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kThreads / 64; ++w) take(best[w]);
  return b.y;
}

// Writes finished pairs (tree positions 2h, 2h+1) and compacts remainders
// (read from V0 or V1 as the group's sort left them, written to Vnext); with
// Knext, also the next level's sort keys and max keys of the compacted
// remainders (one 8-byte load of their bounds on the next axis), and the
// tile's (smallest, largest) key in TR[tile] ((~0, 0) if it has none).  A
// tile's remainders all go to the next level's group of the tile's node.
// With orig (the last level before the subtree phase),
// the remainders are renumbered instead: position dst takes the place of
// triangle id val, orig[dst] = val, and its bounds on all three axes go to
// bbR[axis][dst] (mR per axis), so that every subtree group reads one
// contiguous window of bounds.
__global__ __launch_bounds__(kThreads) void k_emit(const TileDesc* __restrict__ tiles,
                                                   const ChildDesc* __restrict__ children,
                                                   const uint2* __restrict__ partial,
                                                   const uint2* __restrict__ TP,
                                                   const uint2* __restrict__ V0,
                                                   const uint2* __restrict__ V1,
                                                   uint2* __restrict__ Vnext, uint32_t first,
                                                   int level, int L, const float2* __restrict__ bb,
                                                   uint32_t N, uint32_t* __restrict__ P,
                                                   uint32_t* __restrict__ Knext,
                                                   uint2* __restrict__ TR,
                                                   float2* __restrict__ bbR, uint32_t* __restrict__ orig,
                                                   uint32_t mR) {
  const TileDesc t = tiles[blockIdx.x];
  const ChildDesc c = children[t.child];
  const uint2* __restrict__ V = (TP[blockIdx.x].y & 1u) ? V1 : V0;
  const float2* bnext = bb + (size_t)((level + 1) % 3) * N;
  uint32_t am = child_argmax(c, partial);
  if (am <= c.off || am >= c.off + c.size) am = c.off + 1;  // cannot happen for sizes >= 2
  uint32_t kmin = 0xFFFFFFFFu, kmax = 0u;
  for (uint32_t r = threadIdx.x; r < t.count; r += kThreads) {
    const uint32_t i = t.start + r;
    if (i == c.off) {
      write_pair(first + t.child, clampi(V[c.off].x, N), clampi(V[am].x, N), level, L, bb, N, P);
    } else if (i >= c.off + 2) {
      const uint32_t val = clampi((i == am) ? V[c.off + 1].x : V[i].x, N);
      const uint32_t dst = i - 2 * (t.child + 1);
      if (Knext) {
        const float2 b = bnext[val];
        const uint32_t key = fkey(b.x);
        Knext[dst] = key;
        Vnext[dst] = make_uint2(val, fkey(b.y));
        kmin = min(kmin, key);
        kmax = max(kmax, key);
      } else if (orig) {
        const float2 b0 = bb[val], b1 = bb[(size_t)N + val], b2 = bb[2 * (size_t)N + val];
        if (dst < mR) {
          orig[dst] = val;
          bbR[dst] = b0;
          bbR[(size_t)mR + dst] = b1;
          bbR[2 * (size_t)mR + dst] = b2;
        }
        Vnext[dst] = make_uint2(dst, 0u);
      } else {
        Vnext[dst] = make_uint2(val, 0u);
      }
    }
  }
  if (Knext) {  // uniform: a kernel argument
    __shared__ uint32_t rmin[kThreads / 64], rmax[kThreads / 64];
    for (int off = 32; off > 0; off >>= 1) {
      kmin = min(kmin, (uint32_t)__shfl_xor(kmin, off));
      kmax = max(kmax, (uint32_t)__shfl_xor(kmax, off));
    }
    if ((threadIdx.x & 63u) == 0) {
      rmin[threadIdx.x >> 6] = kmin;
      rmax[threadIdx.x >> 6] = kmax;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int w = 1; w < kThreads / 64; ++w) {
        kmin = min(kmin, rmin[w]);
        kmax = max(kmax, rmax[w]);
      }
      TR[blockIdx.x] = make_uint2(kmin, kmax);
    }
  }
}

// The keys of sort_slots: positive normal doubles, which v_min_f64 and
// v_max_f64 order as their bits and return unchanged.
constexpr unsigned long long kSlotKey = 1ull << 62, kSlotEnd = 0x7FEull << 52;

// LDS position of entry i.  Linear over xor and a permutation of each aligned
// run of 32 entries; the passes below, whose lanes read entries 4t + const at
// the small distances, then meet each bank pair once per half wave.
__device__ __forceinline__ uint32_t slot_pos(uint32_t i) { return i ^ ((i >> 2) & 31u) ^ ((i >> 5) & 1u); }

// Bitonic sort of each aligned run of S entries (S a power of two >= 2) of the
// entries [0, span), entry i at K[slot_pos(i)], ascending.  A run holds at most
// `fill` entries, then kSlotEnd.  A merge begins by comparing mirrored entries:
// every comparison then has the same direction, one minimum and one maximum,
// and the ends stay where they are, so that comparisons with them are left out.
// What binds is the chain of passes, each of which reads and writes LDS (4096
// entries: 512 cycles at 128 bytes per cycle) and waits for it.  A pass takes
// two stages of four entries per thread in registers, and the first stage of an
// odd number of them goes alone: 41 passes for 4096 entries instead of 78.
// Wave w owns entries [256w, 256w + 256) in every pass whose distances are at
// most 128, so a wave barrier orders those.  (2584 triangles, one group: 184 us
// with 64-bit compares and selects and entry i at K[i], 144 with minima and
// maxima and slot_pos, 139 with `fill`.  Three stages of eight entries in 28
// passes leave half of the waves without work: 158 us.)
__device__ __forceinline__ void sort_slots(double* K, uint32_t span, uint32_t S, uint32_t fill) {
  static_assert(kSubThreads == kSubT / 4, "four entries per thread");
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const auto order = [](double& x, double& y) {
    double lo, hi;  // no canonicalisation before the minimum: never NaN
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(x), "v"(y));
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(x), "v"(y));
    x = lo;
    y = hi;
  };
  const auto barrier = [](bool wave_only) {
    if (wave_only) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
      __syncthreads();
    }
  };
  // runs of 2 or 4
  if (4 * tid < span) {
    const uint32_t p = slot_pos(4 * tid);
    double x0 = K[p], x1 = K[p ^ slot_pos(1)], x2 = K[p ^ slot_pos(2)], x3 = K[p ^ slot_pos(3)];
    order(x0, x1);
    order(x2, x3);
    if (S > 2) {
      order(x0, x3);
      order(x1, x2);
      order(x0, x1);
      order(x2, x3);
    }
    K[p] = x0;
    K[p ^ slot_pos(1)] = x1;
    K[p ^ slot_pos(2)] = x2;
    K[p ^ slot_pos(3)] = x3;
  }
  barrier(S > 4);
  for (uint32_t k = 8; k <= S; k <<= 1) {
    uint32_t j = k >> 1, mirror = k - 1;
    if (__builtin_ctz(k) & 1) {
#pragma unroll
      for (uint32_t r = 0; r < 2; ++r) {
        const uint32_t t = 2 * (tid & ~63u) + 64 * r + lane;
        const uint32_t i = ((t & ~(j - 1)) << 1) | (t & (j - 1));
        if (i < span && (i & (S - 1)) < fill) {
          const uint32_t p = slot_pos(i), q = p ^ slot_pos(mirror);
          double x = K[p], y = K[q];
          order(x, y);
          K[p] = x;
          K[q] = y;
        }
      }
      barrier(j <= 128);
      j >>= 1;
      mirror = 0;
    }
    for (; j > 1; j >>= 2) {
      const uint32_t h = j >> 1;
      const uint32_t i = ((tid & ~(h - 1)) << 2) | (tid & (h - 1));
      if (i < span && (i & (S - 1)) + h < fill) {
        // distances (j, h): entries i, i + h and their partners, which are
        // mirrored within the run of k in a merge's first stage
        const uint32_t far = mirror ? mirror : j;
        const uint32_t p0 = slot_pos(i), p1 = p0 ^ slot_pos(h);
        const uint32_t p2 = p0 ^ slot_pos(mirror ? far ^ h : far), p3 = p0 ^ slot_pos(mirror ? far : far ^ h);
        double x0 = K[p0], x1 = K[p1], x2 = K[p2], x3 = K[p3];
        if (mirror) {
          order(x0, x3);
          order(x1, x2);
        } else {
          order(x0, x2);
          order(x1, x3);
        }
        order(x0, x1);
        order(x2, x3);
        K[p0] = x0;
        K[p1] = x1;
        K[p2] = x2;
        K[p3] = x3;
      }
      mirror = 0;
      // after (2, 1): the next size 2k starts with distance k
      const uint32_t jn = j > 2 ? j >> 2 : k;
      barrier(j <= 128 && jn <= 128 && !(j == 2 && k == S));
    }
  }
}

// One workgroup per group: all remaining levels of the group's subtree(s),
// in LDS.  Elements are their positions in the group's window of bb (the
// bounds in position order: written by the last k_emit, or the input order of
// a tree that starts here); orig (optional) maps positions to triangle ids
// where the tree order is written.
//
// A level sorts each sort group, the remainder of one node of the previous
// level: a range of its own in the sorted order of that level, holding the
// nodes 2q and 2q + 1 of this one.  Group q is sorted in its own slot of S
// entries, S the power of two that holds the first (largest) group.  The
// slots fit kSubT = T: the workgroup's first group has at most T triangles, so its
// parent heads at most T/2 + 1 nodes; in a left-complete tree the leftmost
// node r levels below then heads at most T/2^(r+1) + 1, its children hold at
// most T/2^r triangles, and there are at most 2^r groups at that depth.
//
// A group is one chain of dependent steps (the passes of the sorts, 230 over
// the 12 levels of 4096 elements, and eight barriers a level), so its latency
// is the launch for trees of up to a million triangles: 139 us for the 2584 of
// one group, 133 us for the 256 groups of 1M.  1024 threads take a pass in one
// step, and the keys of all axes are in LDS (six dwords per element), so that
// no level waits for global memory; the triangle ids of a level's pairs, read
// from orig, are stored one level later.
// 146 KB of LDS: one group of 16 waves per CU.  Groups of 2048, two per CU,
// take 112 us at 1M but leave one more level to the radix passes (then of 130
// us): a build of 1M triangles took 1.70 ms instead of 1.62, of 10M 11.3 ms on
// the device instead of 11.0, and a tree of 2050 to 4096
// triangles, which is one group here, 0.30 ms instead of 0.18.
__global__ __launch_bounds__(kSubThreads, 4) void k_subtree(const SubGroup* __restrict__ groups,
                                                            const float2* __restrict__ bb,
                                                            uint32_t N, uint32_t n, int L,
                                                            int level0, uint32_t* __restrict__ P,
                                                            const uint32_t* __restrict__ orig) {
  constexpr uint32_t T = kSubT;
  constexpr uint32_t kPer = T / kSubThreads;        // elements per thread
  constexpr uint32_t kNodes = T / 2 / kSubThreads;  // nodes per thread
  constexpr uint32_t kPosBits = 12;
  static_assert(1u << kPosBits == T, "");
  __shared__ uint32_t kmin[3][T], kmax[3][T];
  __shared__ double K[T];
  __shared__ uint16_t E[T];
  __shared__ uint16_t nodeOff[T / 2 + 1];
  __shared__ uint16_t nodeArg[T / 2];
  // once the sorted order is read out, the sort buffer holds the sorted
  // elements (E2) and their max keys (MK)
  uint32_t* E2 = reinterpret_cast<uint32_t*>(K);
  uint32_t* MK = E2 + T;

  const SubGroup g = groups[blockIdx.x];
  const uint32_t tid = threadIdx.x;
  uint32_t m = min(g.size, T);
  for (uint32_t i = tid; i < m; i += kSubThreads) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float2 b = bb[(size_t)a * N + g.off + i];
      kmin[a][i] = fkey(b.x);
      kmax[a][i] = fkey(b.y);
    }
    E[i] = (uint16_t)i;
  }
  uint32_t f = g.first, c = g.count;
  // the pairs of this thread's nodes of the previous level: written once
  // their ids are here
  bool held[kNodes];
  uint32_t held_h[kNodes], held_x[kNodes], held_y[kNodes];
#pragma unroll
  for (uint32_t r = 0; r < kNodes; ++r) held[r] = false;
  const auto put = [&](uint32_t r, uint32_t h, uint32_t x, uint32_t y) {
    held[r] = true;
    held_h[r] = h;
    held_x[r] = orig ? orig[g.off + x] : g.off + x;
    held_y[r] = orig ? orig[g.off + y] : g.off + y;
  };
  const auto flush = [&]() {
#pragma unroll
    for (uint32_t r = 0; r < kNodes; ++r) {
      if (held[r]) {
        P[2 * (size_t)held_h[r]] = held_x[r];
        P[2 * (size_t)held_h[r] + 1] = held_y[r];
      }
      held[r] = false;
    }
  };
  for (int level = level0; level < L && m > 0; ++level) {
    const int a = level % 3;
    for (uint32_t j = tid; j <= c; j += kSubThreads) nodeOff[j] = (uint16_t)(2u * desc_count32(f, f + j, n));
    __syncthreads();
    // sort groups q < ng = the nodes' pairs, entry p of group q in slot entry
    // q * S + p (kSlotEnd beyond the group's size)
    const uint32_t ng = (c + 1) / 2, size0 = nodeOff[min(2u, c)];
    const uint32_t ls = size0 > 2 ? 32u - (uint32_t)__clz((int)(size0 - 1)) : 1u, S = 1u << ls;
    const uint32_t span = min(ng << ls, T);
#pragma unroll
    for (uint32_t r = 0; r < kPer; ++r) {
      const uint32_t sl = tid + r * kSubThreads;
      if (sl >= span) break;
      const uint32_t q = sl >> ls, p = sl & (S - 1), o = nodeOff[2 * q];
      const uint32_t i = o + p;
      K[slot_pos(sl)] = __longlong_as_double((long long)(
          i < nodeOff[min(2 * q + 2, c)] ? kSlotKey | ((unsigned long long)kmin[a][E[i]] << kPosBits) | p : kSlotEnd));
    }
    flush();
    __syncthreads();
    sort_slots(K, span, S, size0);
    const bool last = level == L - 1;
    // sorted entry p of group q is sorted position nodeOff[2q] + p
    uint32_t ev[kPer], kv[kPer], at[kPer];
#pragma unroll
    for (uint32_t r = 0; r < kPer; ++r) {
      const uint32_t sl = tid + r * kSubThreads;
      ev[r] = kv[r] = 0;
      at[r] = ~0u;
      if (sl < span) {
        const uint32_t q = sl >> ls, o = nodeOff[2 * q], i = o + (sl & (S - 1));
        if (i < nodeOff[min(2 * q + 2, c)]) {
          at[r] = i;
          ev[r] = E[min(o + ((uint32_t)__double_as_longlong(K[slot_pos(sl)]) & ((1u << kPosBits) - 1)), m - 1)];
          kv[r] = kmax[a][ev[r]];
        }
      }
    }
    __syncthreads();  // every sorted slot is read: E2 and MK overwrite them
#pragma unroll
    for (uint32_t r = 0; r < kPer; ++r)
      if (at[r] != ~0u) {
        E2[at[r]] = ev[r];
        MK[at[r]] = kv[r];
      }
    __syncthreads();
    if (last) {
#pragma unroll
      for (uint32_t r = 0; r < kNodes; ++r) {
        const uint32_t j = tid + r * kSubThreads;
        if (j < c) put(r, f + j, E2[nodeOff[j]], E2[nodeOff[j] + 1]);
      }
      break;
    }
    // first maximum of the max key over each node's [o + 1, e): W lanes per
    // node, as many as there are threads for
    uint32_t lw = 6;
    while (lw > 0 && (c << lw) > kSubThreads) --lw;
    const uint32_t W = 1u << lw;
    for (uint32_t j0 = 0; j0 < c; j0 += kSubThreads >> lw) {
      const uint32_t j = j0 + (tid >> lw), w = tid & (W - 1);
      uint32_t bk = 0, bp = 0xFFFFFFFFu, o = 0, e = 0;
      if (j < c) {
        o = nodeOff[j];
        e = nodeOff[j + 1];
        for (uint32_t i = o + 1 + w; i < e; i += W) {
          const uint32_t k = MK[i];
          if (k > bk) {
            bk = k;
            bp = i;
          }
        }
      }
      for (uint32_t off = W >> 1; off > 0; off >>= 1) {
        const uint32_t ok = __shfl_xor(bk, off), op = __shfl_xor(bp, off);
        if (ok > bk || (ok == bk && op < bp)) {
          bk = ok;
          bp = op;
        }
      }
      if (j < c && w == 0) nodeArg[j] = (uint16_t)((bp > o && bp < e) ? bp : o + 1);  // sizes are >= 2
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < kNodes; ++r) {
      const uint32_t j = tid + r * kSubThreads;
      if (j < c) {
        const uint32_t x = E2[nodeOff[j]], y = E2[nodeArg[j]];
        const bool swap = second_first(x, y, level, L, [&](int ax, uint32_t i) { return kmin[ax][i]; });
        put(r, f + j, swap ? y : x, swap ? x : y);
      }
    }
    // compaction: the node of a sorted position is one of its group's two
#pragma unroll
    for (uint32_t r = 0; r < kPer; ++r) {
      const uint32_t i = at[r];
      if (i == ~0u) continue;
      uint32_t j = 2u * ((tid + r * kSubThreads) >> ls);
      if (j + 1 < c && i >= nodeOff[j + 1]) ++j;
      if (i >= nodeOff[j] + 2u)
        E[i - 2 * (j + 1)] = (uint16_t)((i == nodeArg[j]) ? E2[nodeOff[j] + 1] : ev[r]);
    }
    __syncthreads();
    m -= 2 * c;
    const uint64_t nf = 2ull * f + 1;
    if (nf >= n) break;
    const uint64_t nc = std::min<uint64_t>(2ull * c, n - nf);
    f = (uint32_t)nf;
    c = (uint32_t)nc;
  }
  flush();
}

// applyIndices (rebuilder.cu:217-245): gather every per-triangle array.
__global__ void k_gather_geometry(const uint32_t* __restrict__ P, uint32_t N,
                                  const float* __restrict__ iv, const float* __restrict__ in,
                                  const float* __restrict__ iuv, const uint16_t* __restrict__ ish,
                                  float* __restrict__ ov, float* __restrict__ on,
                                  float* __restrict__ ouv, uint16_t* __restrict__ osh) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const size_t s = clampi(P[i], N);
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    ov[(size_t)i * 9 + k] = iv[s * 9 + k];
    on[(size_t)i * 9 + k] = in[s * 9 + k];
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) ouv[(size_t)i * 6 + k] = iuv[s * 6 + k];
  osh[i] = ish[s];
}

__device__ inline void slab_of(const float* v, int a, float& lo, float& hi) {
  // intersect.cuh:25-33, 109-111 over the node's two triangles
  const float* p = v;
  const float* q = v + 9;
  lo = fminf(fminf(fminf(p[3 * a], p[3 * a + 1]), p[3 * a + 2]),
             fminf(fminf(q[3 * a], q[3 * a + 1]), q[3 * a + 2]));
  hi = fmaxf(fmaxf(fmaxf(p[3 * a], p[3 * a + 1]), p[3 * a + 2]),
             fmaxf(fmaxf(q[3 * a], q[3 * a + 1]), q[3 * a + 2]));
}

// Traversal records (common.h): thread K writes record K, of node K - 1.
// Record 0 also goes to host memory (root).
__global__ void k_node_records(const float* __restrict__ v, uint32_t n, NodeRec* __restrict__ nodes,
                               NodeRec* __restrict__ root) {
  const uint32_t K = blockIdx.x * blockDim.x + threadIdx.x;
  if (K > n) return;
  NodeRec r = {};
  if (K == 0) {
    slab_of(v, 0, r.cslab[0], r.cslab[1]);
    nodes[0] = r;
    *root = r;
    return;
  }
  const uint32_t k = K - 1;
  const float* p = v + (size_t)k * 18;  // points layout, two triangles
  const uint32_t d = depth_of(k);
  const int ca = (int)((d + 1) % 3);
  const uint64_t cl = 2ull * k + 1;
  r.cslab[0] = r.cslab[2] = kNoSlab;
  r.cslab[1] = r.cslab[3] = -kNoSlab;
  if (cl < n) slab_of(v + cl * 18, ca, r.cslab[0], r.cslab[1]);
  if (cl + 1 < n) slab_of(v + (cl + 1) * 18, ca, r.cslab[2], r.cslab[3]);
  bool normal = true;
#pragma unroll
  for (int c = 0; c < 4; ++c) normal = normal && normal_coord(r.cslab[c]);
  // the group's extent: the two triangles on every axis, and the slabs of
  // the parent and the grandparent on theirs (the node's own is its triangles').
  // A slab 2^15 times as large as a triangle of the node and 2^8 times the
  // extent of both (under a ground plane or a sky dome) is left out: the halves
  // could not hold the triangle in its units, and in the triangles' own the test
  // works for the rays that meet the node near them.
  float extent = 0.0f, coord = 0.0f, larger[2] = {0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < 18; ++i)
    if (i % 3) larger[i / 9] = fmaxf(larger[i / 9], fabsf(p[i] - p[i - i % 3]));
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    float lo, hi;
    slab_of(p, a, lo, hi);
    extent = fmaxf(extent, hi - lo);
    coord = fmaxf(coord, fmaxf(fabsf(lo), fabsf(hi)));
  }
  uint32_t anc = k;
  const float limit = fmaxf(0x1p8f * extent, 0x1p15f * fminf(larger[0], larger[1]));
  for (uint32_t up = 1; up <= 2 && up <= d; ++up) {
    float lo, hi;
    anc = (anc - 1) / 2;
    slab_of(v + (size_t)anc * 18, (int)((d - up) % 3), lo, hi);
    if (hi - lo <= limit) extent = fmaxf(extent, hi - lo);
  }
  int ex = 0;
  (void)frexpf(extent, &ex);  // extent < 2^ex
  const bool reject = coord <= kRejectCoord && extent >= kRejectScaleMin && extent <= kRejectScaleMax;
  const float unit = reject ? ldexpf(1.0f, -ex) : __builtin_inff(), scale = 2.0f * unit;
  float size[2], edge[2][6];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const float* q = p + 9 * t;
    size[t] = 0x1p-10f;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float e1 = q[3 * a + 1] - q[3 * a], e2 = q[3 * a + 2] - q[3 * a];
      edge[t][a] = reject ? e1 * unit : 0.0f;
      edge[t][3 + a] = reject ? e2 * unit : 0.0f;
      size[t] = fmaxf(size[t], fmaxf(fabsf(edge[t][a]), fabsf(edge[t][3 + a])));
    }
    size[t] *= 1.0f + 0x1p-10f;  // not below after rounding to half
  }
#pragma unroll
  for (int c = 0; c < 6; ++c) r.e[c] = half2v{(_Float16)edge[0][c], (_Float16)edge[1][c]};
  float dv[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    r.ref[a] = reject ? p[3 * a] * scale : 0.0f;
    dv[a] = reject ? (p[9 + 3 * a] - p[3 * a]) * scale : 0.0f;
  }
  r.dxy = half2v{(_Float16)dv[0], (_Float16)dv[1]};
  r.dz_a = half2v{(_Float16)dv[2], (_Float16)size[0]};
  const half2v sb = {(_Float16)size[1], (_Float16)0.0f};
  r.scale_b = __float_as_uint(scale) | (normal ? 0u : kNodeSlabsOdd) | __builtin_bit_cast(uint32_t, sb);
  nodes[K] = r;
}

// cudaGenerateTB (utility.cu:136-180).
__global__ void k_generate_tb(const float* __restrict__ normals, uint32_t N,
                              float* __restrict__ tangents, float* __restrict__ bitangents) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const V3 up = mk(0.0f, 1.0f, 0.0f), fwd = mk(0.0f, 0.0f, 1.0f);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const V3 nv = ld3(normals + (size_t)i * 9 + 3 * k);
    V3 T = cross(nv, up);
    if (length(T) < kEpsilon) T = cross(nv, fwd);
    const V3 B = cross(nv, T);
    float* tp = tangents + (size_t)i * 9 + 3 * k;
    float* bp = bitangents + (size_t)i * 9 + 3 * k;
    tp[0] = T.x;
    tp[1] = T.y;
    tp[2] = T.z;
    bp[0] = B.x;
    bp[1] = B.y;
    bp[2] = B.z;
  }
}

inline uint32_t blocks(uint64_t n, uint32_t b) { return (uint32_t)((n + b - 1) / b); }

// Above this much, a build's scratch is freed when it ends.
constexpr size_t kKeepScratch = 256ull << 20;

}  // namespace

struct LevelPlan {
  int level;
  uint32_t m, first, ngroups, ntiles;
  size_t child_base, group_base, tile_base;
  bool scan;  // k_radix_group_scan runs
};

struct BuildPlan {
  uint32_t count = 0;  // triangles (0: none)
  int L = 0, level0 = 0;
  uint32_t nsub = 0;
  size_t max_tiles = 1, max_groups = 1, max_chunks = 1;
  std::vector<LevelPlan> levels;
  std::vector<uint8_t> image;  // every descriptor array; empty once on the device
  size_t at_tiles = 0, at_children = 0, at_groups = 0, at_sub = 0;
};

// Queues the tangent frames of the tree-order normals.
static aur_status launch_tb(aur_context* ctx) {
  const uint32_t N = ctx->count;
  AUR_HIP(ctx, ctx->tangents.reserve((size_t)N * 9));
  AUR_HIP(ctx, ctx->bitangents.reserve((size_t)N * 9));
  k_generate_tb<<<blocks(N, 256), 256, 0, ctx->stream>>>(ctx->normals.p, N, ctx->tangents.p,
                                                         ctx->bitangents.p);
  AUR_LAUNCH_CHECK(ctx, "k_generate_tb");
  return AUR_OK;
}

aur_status generate_tb(aur_context* ctx) {
  if (!ctx->built) return ctx->fail(AUR_ERR_STATE, "generate_tb: geometry not built");
  const aur_status st = launch_tb(ctx);
  ctx->has_tb = ctx->has_tb || st == AUR_OK;
  return st;
}

// The host's part of a build: it depends on the triangle count alone, so the
// context keeps the last one and its device copy.
static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

void make_plan(uint32_t N, BuildPlan& bp) {
  const uint32_t n = N / 2;
  int L = 0;
  for (uint32_t x = n; x; x >>= 1) ++L;  // log2i(n) + 1
  int level0 = 0;
  if (N > kSubT) {
    level0 = L - 1;
    for (int l = 1; l < L; ++l) {
      const uint64_t fp = (1ull << (l - 1)) - 1;  // first node of the parent level
      const uint64_t maxg = 2 * desc_count(fp, fp + 1, n) - 2;
      if (maxg <= kSubT) {
        level0 = l;
        break;
      }
    }
  }
  std::vector<TileDesc> tiles;
  std::vector<ChildDesc> children;
  std::vector<GroupDesc> groups;
  uint32_t chunk_count = 0;  // chunks of kChunk tiles of one group, per level
  std::vector<LevelPlan>& plan = bp.levels;
  plan.clear();
  size_t max_tiles = 1, max_groups = 1, max_chunks = 1;
  for (int l = 0; l < level0; ++l) {
    LevelPlan lp{};
    lp.level = l;
    lp.first = (uint32_t)((1ull << l) - 1);
    const uint64_t last = std::min<uint64_t>((2ull << l) - 1, n);
    lp.m = (uint32_t)(N - 2ull * lp.first);
    lp.child_base = children.size();
    lp.group_base = groups.size();
    lp.tile_base = tiles.size();
    uint64_t off = 0;
    int64_t cur_parent = -1;
    for (uint64_t h = lp.first; h < last; ++h) {
      const uint64_t size = 2 * desc_count(h, h + 1, n);
      const int64_t parent = l == 0 ? 0 : (int64_t)((h - 1) / 2);
      if (parent != cur_parent) {
        if (!groups.empty() && groups.size() > lp.group_base) groups.back().te = (uint32_t)(tiles.size() - lp.tile_base);
        groups.push_back(GroupDesc{(uint32_t)off, 0, (uint32_t)(tiles.size() - lp.tile_base), 0, 0, 0});
        cur_parent = parent;
      }
      GroupDesc& g = groups.back();
      g.size += (uint32_t)size;
      ChildDesc cd{(uint32_t)off, (uint32_t)size, (uint32_t)(tiles.size() - lp.tile_base), 0};
      for (uint64_t st = 0; st < size; st += kTile)
        tiles.push_back(TileDesc{(uint32_t)(off + st), (uint32_t)std::min<uint64_t>(kTile, size - st),
                                 (uint32_t)(h - lp.first),
                                 (uint32_t)(groups.size() - 1 - lp.group_base)});
      cd.te = (uint32_t)(tiles.size() - lp.tile_base);
      children.push_back(cd);
      off += size;
    }
    groups.back().te = (uint32_t)(tiles.size() - lp.tile_base);
    lp.ngroups = (uint32_t)(groups.size() - lp.group_base);
    lp.ntiles = (uint32_t)(tiles.size() - lp.tile_base);
    chunk_count = 0;
    for (size_t gi = lp.group_base; gi < groups.size(); ++gi) {
      GroupDesc& g = groups[gi];
      g.cb = chunk_count;
      chunk_count += (g.te - g.tb + kChunk - 1) / kChunk;
      g.ce = chunk_count;
      lp.scan = lp.scan || g.ce - g.cb > kScanChunks;
    }
    max_chunks = std::max<size_t>(max_chunks, chunk_count);
    max_tiles = std::max<size_t>(max_tiles, lp.ntiles);
    max_groups = std::max<size_t>(max_groups, lp.ngroups);
    plan.push_back(lp);
  }
  std::vector<SubGroup> sub;
  if (level0 == 0) {
    sub.push_back(SubGroup{0, N, 0, 1});
  } else {
    const uint64_t fp = (1ull << (level0 - 1)) - 1;
    const uint64_t lastp = std::min<uint64_t>((1ull << level0) - 1, n);
    const uint64_t fc = (1ull << level0) - 1;
    for (uint64_t p = fp; p < lastp; ++p) {
      const uint64_t c0 = 2 * p + 1;
      if (c0 >= n) break;
      const uint64_t c1 = std::min<uint64_t>(c0 + 2, n);
      const uint64_t off = 2 * desc_count(fc, c0, n);
      const uint64_t size = 2 * desc_count(c0, c1, n);
      sub.push_back(SubGroup{(uint32_t)off, (uint32_t)size, (uint32_t)c0, (uint32_t)(c1 - c0)});
    }
  }
  bp.count = N;
  bp.L = L;
  bp.level0 = level0;
  bp.nsub = (uint32_t)sub.size();
  bp.max_tiles = max_tiles;
  bp.max_groups = max_groups;
  bp.max_chunks = max_chunks;
  // one image of every descriptor array, 256-byte aligned
  bp.image.clear();
  const auto put = [&](const void* p, size_t bytes) {
    const size_t at = bp.image.size();
    bp.image.resize(align256(at + std::max<size_t>(bytes, 1)));
    if (bytes) memcpy(bp.image.data() + at, p, bytes);
    return at;
  };
  bp.at_tiles = put(tiles.data(), tiles.size() * sizeof(TileDesc));
  bp.at_children = put(children.data(), children.size() * sizeof(ChildDesc));
  bp.at_groups = put(groups.data(), groups.size() * sizeof(GroupDesc));
  bp.at_sub = put(sub.data(), sub.size() * sizeof(SubGroup));
}

aur_status nmh_build(aur_context* ctx, aur_build_stats* stats, bool tangents) {
  const uint32_t N = ctx->count;
  if (N < 2 || (N & 1u)) return ctx->fail(AUR_ERR_STATE, "rebuild: no even-sized geometry uploaded");
  const uint32_t n = N / 2;
  hipStream_t s = ctx->stream;
  if (!ctx->build_plan) ctx->build_plan = std::make_unique<BuildPlan>();
  BuildPlan& bp = *ctx->build_plan;
  if (bp.count != N) {
    bp.count = 0;  // until the device copy is whole
    BuildPlan next;
    make_plan(N, next);
    AUR_HIP(ctx, ctx->build_desc.reserve(next.image.size()));
    AUR_HIP(ctx, hipMemcpyAsync(ctx->build_desc.p, next.image.data(), next.image.size(), hipMemcpyHostToDevice, s));
    AUR_HIP(ctx, hipStreamSynchronize(s));
    next.image = std::vector<uint8_t>();
    bp = std::move(next);
  }
  const int L = bp.L, level0 = bp.level0;
  const std::vector<LevelPlan>& plan = bp.levels;
  const auto desc = [&](size_t at) { return ctx->build_desc.p + at; };
  const TileDesc* dtiles = reinterpret_cast<const TileDesc*>(desc(bp.at_tiles));
  const ChildDesc* dchildren = reinterpret_cast<const ChildDesc*>(desc(bp.at_children));
  const GroupDesc* dgroups = reinterpret_cast<const GroupDesc*>(desc(bp.at_groups));
  const SubGroup* dsub = reinterpret_cast<const SubGroup*>(desc(bp.at_sub));

  // ---- device scratch, one allocation ----
  // pending triangles when the subtree phase starts
  const uint32_t m0 = level0 > 0 ? (uint32_t)(N - 2 * ((1ull << level0) - 1)) : N;
  size_t ws = 0;
  const auto take = [&](size_t bytes) {
    const size_t at = ws;
    ws = align256(ws + bytes);
    return at;
  };
  const bool large = !plan.empty();  // levels of groups above one workgroup's LDS
  const size_t at_bb = take((size_t)3 * N * sizeof(float2));  // (min, max) per axis and triangle
  // the same for the subtree phase's pending region, by position
  const size_t at_bbR = take(large ? (size_t)3 * m0 * sizeof(float2) : 0);
  // sort payload (triangle id, max key on the level's axis): the level's
  // input, the other side of the radix passes, and the emit pass's output
  const size_t vb = large ? (size_t)N * sizeof(uint2) : 0, kb = large ? (size_t)N * sizeof(uint32_t) : 0;
  const size_t at_V[3] = {take(vb), take(vb), take(vb)}, at_K[2] = {take(kb), take(kb)};
  const size_t tb = large ? bp.max_tiles : 0, cb = large ? bp.max_chunks : 0, nb = large ? bp.max_groups : 0;
  // (smallest key, passes) per group and tile, emit tiles' key ranges, passes
  // per offset chunk, first maxima
  const size_t at_GP = take(nb * sizeof(uint2)), at_TP = take(tb * sizeof(uint2)), at_TR = take(tb * sizeof(uint2));
  const size_t at_partial = take(tb * sizeof(uint2)), at_H = take(tb * 256 * 4);
  const size_t at_CS = take(2 * cb * 256 * 4), at_CB = take(cb * 256 * 4);  // CS: this pass's and the next's
  AUR_HIP(ctx, ctx->build_scratch.reserve(ws));
  AUR_HIP(ctx, ctx->perm.reserve(N));
  const auto u2 = [&](size_t at) { return reinterpret_cast<uint2*>(ctx->build_scratch.p + at); };
  const auto u1 = [&](size_t at) { return reinterpret_cast<uint32_t*>(ctx->build_scratch.p + at); };
  float2* const bb = reinterpret_cast<float2*>(ctx->build_scratch.p + at_bb);
  float2* const bbR = reinterpret_cast<float2*>(ctx->build_scratch.p + at_bbR);
  uint2 *const GP = u2(at_GP), *const TP = u2(at_TP), *const TR = u2(at_TR), *const partial = u2(at_partial);
  uint32_t *const Ka = u1(at_K[0]), *const Kb = u1(at_K[1]), *const H = u1(at_H), *const CB = u1(at_CB);
  uint32_t* const CS[2] = {u1(at_CS), u1(at_CS) + cb * 256};

  hipEvent_t& e0 = ctx->build_event[0];
  hipEvent_t& e1 = ctx->build_event[1];
  if (!e0) AUR_HIP(ctx, hipEventCreate(&e0));
  if (!e1) AUR_HIP(ctx, hipEventCreate(&e1));
  AUR_HIP(ctx, hipEventRecord(e0, s));

  // level 0's keys come with the identity order; every later level's keys
  // and max keys are gathered by the previous level's emit pass
  uint2* Vcur = u2(at_V[0]);  // the level's input (k_bounds', then the previous emit's output)
  uint2* Valt = u2(at_V[1]);  // the other side of the radix passes
  uint2* Vout = u2(at_V[2]);  // the emit pass's output
  k_bounds<<<blocks(N, 256), 256, 0, s>>>(ctx->in_vertices.p, N, bb, large ? Vcur : nullptr, Ka);
  if (large) k_fill0<<<blocks(bp.max_chunks * 256, 256), 256, 0, s>>>(CS[0], (uint32_t)(bp.max_chunks * 256));
  for (size_t li = 0; li < plan.size(); ++li) {
    const LevelPlan& lp = plan[li];
    const TileDesc* tl = dtiles + lp.tile_base;
    const ChildDesc* ch = dchildren + lp.child_base;
    const GroupDesc* gr = dgroups + lp.group_base;
    // the previous level's nodes: group g of this level is node g's remainder
    const ChildDesc* prev = li == 0 ? nullptr : dchildren + plan[li - 1].child_base;
    uint32_t *kin = Ka, *kout = Kb;
    uint2 *vin = Vcur, *vout = Valt;
    // every launch of a pass skips the groups that need fewer passes
    for (uint32_t pass = 0; pass < 4; ++pass) {
      uint32_t* const cs = CS[pass & 1];
      k_radix_hist<<<lp.ntiles, kThreads, 0, s>>>(tl, gr, TP, kin, pass, H, cs, CS[~pass & 1]);
      if (lp.scan) k_radix_group_scan<<<lp.ngroups, kThreads, 0, s>>>(gr, GP, TP, prev, TR, pass, cs, CB);
      k_radix_scatter<<<lp.ntiles, kThreads, 0, s>>>(tl, gr, TP, prev, TR, kin, vin, pass, H, cs,
                                                     lp.scan ? CB : nullptr, lp.m, kout, vout);
      std::swap(kin, kout);
      std::swap(vin, vout);
    }
    // each group's sorted data is in Vcur or Valt (group_passes); the keys
    // are not read again, so Ka takes the next level's
    const bool last = li + 1 == plan.size();
    k_argmax_partial<<<lp.ntiles, kThreads, 0, s>>>(tl, ch, TP, Vcur, Valt, partial);
    k_emit<<<lp.ntiles, kThreads, 0, s>>>(tl, ch, partial, TP, Vcur, Valt, Vout, lp.first, lp.level, L,
                                          bb, N, ctx->perm.p, last ? nullptr : Ka, TR,
                                          last ? bbR : nullptr, last ? Ka : nullptr, m0);
    // rotate: the emit output is the next level's input
    uint2* const free_buf = Vcur;
    Vcur = Vout;
    Vout = Valt;
    Valt = free_buf;
  }
  AUR_LAUNCH_CHECK(ctx, "nmh level kernels");
  // the subtree phase, on positions renumbered by the last k_emit if levels
  // came before it
  k_subtree<<<bp.nsub, kSubThreads, 0, s>>>(dsub, large ? bbR : bb, m0, n, L, level0, ctx->perm.p,
                                            large ? Ka : nullptr);
  AUR_LAUNCH_CHECK(ctx, "k_subtree");

  // pinned once per context, while the GPU builds: 0.1 ms
  if (!ctx->root_host) AUR_HIP(ctx, hipHostMalloc((void**)&ctx->root_host, sizeof(NodeRec)));
  AUR_HIP(ctx, ctx->vertices.reserve((size_t)N * 9));
  AUR_HIP(ctx, ctx->normals.reserve((size_t)N * 9));
  AUR_HIP(ctx, ctx->texcoords.reserve((size_t)N * 6));
  AUR_HIP(ctx, ctx->shader_ids.reserve(N));
  AUR_HIP(ctx, ctx->nodes.reserve((size_t)n + 1));
  AUR_HIP(ctx, ctx->trace_work.reserve((size_t)kTraceWorkSets * kWorkWords));
  k_gather_geometry<<<blocks(N, 256), 256, 0, s>>>(ctx->perm.p, N, ctx->in_vertices.p,
                                                   ctx->in_normals.p, ctx->in_texcoords.p,
                                                   ctx->in_shader_ids.p, ctx->vertices.p,
                                                   ctx->normals.p, ctx->texcoords.p,
                                                   ctx->shader_ids.p);
  k_node_records<<<blocks((uint64_t)n + 1, 256), 256, 0, s>>>(ctx->vertices.p, n, ctx->nodes.p, ctx->root_host);
  AUR_LAUNCH_CHECK(ctx, "gather/node records");
  AUR_HIP(ctx, hipEventRecord(e1, s));
  const aur_status tangents_status = tangents ? launch_tb(ctx) : AUR_OK;
  AUR_HIP(ctx, hipStreamSynchronize(s));
  float ms = 0.0f;
  AUR_HIP(ctx, hipEventElapsedTime(&ms, e0, e1));
  // record 0, for launches that start every ray at the root without reading it
  ctx->root_lo = ctx->root_host->cslab[0];
  ctx->root_hi = ctx->root_host->cslab[1];
  // A rebuild of the same size (an edit, a deforming mesh) finds its scratch
  // in place.  Beyond the limit (about 3.3M triangles) the build outweighs the
  // allocation.
  if (ws > kKeepScratch) ctx->build_scratch.release();
  ctx->levels = (uint32_t)L;
  ctx->built = true;
  ctx->has_tb = tangents && tangents_status == AUR_OK;
  if (stats) {
    stats->count = N;
    stats->levels = (uint32_t)L;
    stats->build_ms = ms;
  }
  return tangents_status;
}

}  // namespace aur

aur_context::aur_context() = default;
aur_context::~aur_context() {
  for (hipEvent_t e : build_event)
    if (e) (void)hipEventDestroy(e);
  if (root_host) (void)hipHostFree(root_host);
}
