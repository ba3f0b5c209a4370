// Ground planes for gfx950: the reference's binned per-cell plane fit and a
// batched point-level plane RANSAC.
//
// 1. sloam_ground_planes -- sloam::sloam::binGroundPoints + Plane::Plane /
//    Plane::computeModel (sloam/src/core/sloam.cpp:330-386, 391-400;
//    sloam/src/objects/plane.cpp:3-17, 96-128; utils.h:9-28):
//      bin      one thread per point: 2-D radius in float (pow_2 squares in
//               double and rounds to float), angle atan2f, radius / angle bins
//               in double.  Few cells (up to 255, of moderate size): a stable
//               partition by cell, each cell's lowest points selected by its
//               fit workgroup.  Otherwise keys (cell, index) and (cell, z) for
//               two stable radix sorts (radix.hip).  Both give each cell's
//               points in input order and in increasing z (ties: input order)
//      fit      one workgroup per cell: the bottom floor(size / retainNum)
//               points by z when retainNum < size (else all points, input
//               order); float centroid summed sequentially in that order as
//               the reference does; FP64 covariance of the float-centred
//               points; FP64 Jacobi: normal = smallest eigenvector (the
//               reference's JacobiSVD U[:,2]); features = the first
//               numGroundFeatures points
// 2. sloam_plane_plan_* -- point-level plane RANSAC (no counterpart in the
//    reference, which fits each cell by SVD without RANSAC): Philox4x32-10
//    samples of 3 points, plane through them in FP32, inlier |n.p + d| < thr
//    counted by wavefront ballot; best = max count, lowest index; FP64 PCA
//    refit over the inliers.  Large sets are cut into chunks that several
//    workgroups score and refit.  Predicate: Plane::distance(const PointT&)
//    (sloam/src/objects/plane.cpp:136-151) for a unit normal.
#include <cstring>

#include "common.hpp"

#include <algorithm>
#include <cmath>
#include <new>
#include <numeric>
#include <vector>

namespace {

constexpr int kGB = 256;
constexpr double kPiDef = 3.14159265;  // PIDEF, sloam/include/helpers/definitions.h:28
constexpr int kCentroidTile = 2048;

// unsigned key in the order of the floats' <, -0 and +0 equal (so that their
// ties keep input order, as std::stable_sort with < does)
__device__ inline uint32_t orderable(float f) {
  const uint32_t u = __float_as_uint(f == 0.0f ? 0.0f : f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

struct GroundCfgDev {
  int R, T, n_cells, nf;
  double min_d, max_d, retain_num;
  float ox, oy;
};

// Cell of a point, n_cells outside the grid (after every cell in the sorts).
__device__ inline int ground_cell(const float4& p, const GroundCfgDev& cfg) {
  if (!(isfinite(p.x) && isfinite(p.y) && isfinite(p.z))) return cfg.n_cells;
  const float dx = cfg.ox - p.x, dy = cfg.oy - p.y;
  const float a = (float)((double)dx * (double)dx);
  const float b = (float)((double)dy * (double)dy);
  const double r = (double)sqrtf(a + b);
  if (!(r < cfg.max_d && r > cfg.min_d)) return cfg.n_cells;
  const double th = (double)atan2f(p.y - cfg.oy, p.x - cfg.ox);
  int rb = (int)floor(r / (cfg.max_d / (double)cfg.R));
  int tb = (int)floor((kPiDef + th) / (2 * kPiDef / (double)cfg.T));
  rb = max(0, min(rb, cfg.R - 1));
  tb = max(0, min(tb, cfg.T - 1));
  return rb * cfg.T + tb;
}

// ---- few cells: one stable partition by cell, then a selection per cell ------
// (sloam_ground_planes chooses it: at most kSelCells cells, and cells of a size
// whose kept points one workgroup can select.)
constexpr int kSelCells = 255;   // cells (and the outside) are one 8-bit digit
constexpr int kSelTile = 1024;   // points per workgroup of the partition
constexpr int kSelWave = kSelTile / (kGB / 64);  // consecutive points per wave
constexpr int kSelKeys = 4096;   // points of a cell whose keys are held in LDS
constexpr int kSelCand = 2048;   // of them sorted at once
constexpr int kSelBins = kGB;
constexpr int kSelRank = 512;    // up to here sorted by counting smaller ones
// larger cells: threads, bins of the threshold's search, points of its bin
// that are sorted along, loads of a thread in flight
constexpr int kBigB = 1024;
constexpr int kBigW = kBigB / 64;
constexpr int kBigBins = 2048;
constexpr int kBigSlack = 8192;
constexpr int kBigAhead = 16;
// average points per cell up to which the selection is taken (more: two radix
// sorts; a workgroup re-reads a larger cell from L2 several times)
constexpr int kSelAvg = 16384;

// cells of one tile's points, and the tile's count of every cell in
// table[cell][tile] (rows of `stride`)
__global__ __launch_bounds__(kGB) void ground_cells_kernel(const float4* __restrict__ pts, int cap,
                                                           const int32_t* __restrict__ d_n,
                                                           GroundCfgDev cfg, int stride,
                                                           uint8_t* __restrict__ cell,
                                                           int32_t* __restrict__ table) {
  __shared__ int h[kGB];
  const int n = min(d_n ? *d_n : cap, cap);
  const int base = blockIdx.x * kSelTile;
  if (base >= n) return;
  h[threadIdx.x] = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kSelTile / kGB; ++j) {
    const int i = base + j * kGB + (int)threadIdx.x;
    if (i < n) {
      const int c = ground_cell(pts[i], cfg);
      cell[i] = (uint8_t)c;
      atomicAdd(&h[c], 1);
    }
  }
  __syncthreads();
  if ((int)threadIdx.x <= cfg.n_cells)
    table[(size_t)threadIdx.x * stride + blockIdx.x] = h[threadIdx.x];
}

// Stable partition of the points by cell: index and orderable z of each, the
// cells' offsets.  Every workgroup sums the table's rows over the tiles in use
// (exclusive scan over cells, tiles before its own), ranks its points with
// ballots over the digit's `bits` bits, and each wave owns consecutive points
// so that the workgroup meets only twice.  With the selection below it
// replaces a sort by cell and a sort by (cell, z): 6 radix passes of two
// launches each, 100 us of a 350 us front end at 128 x 2048.
__global__ __launch_bounds__(kGB) void ground_part_kernel(
    const float4* __restrict__ pts, int cap, const int32_t* __restrict__ d_n, GroundCfgDev cfg,
    int stride, int bits, const uint8_t* __restrict__ cell, const int32_t* __restrict__ table,
    int32_t* __restrict__ idx, uint32_t* __restrict__ zkey, int32_t* __restrict__ offsets) {
  __shared__ int first[kGB], wc[kGB / 64][kGB], wtot[kGB / 64];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int n = min(d_n ? *d_n : cap, cap);
  const int base = blockIdx.x * kSelTile;
  if (base >= n && blockIdx.x > 0) return;
  constexpr int kR = kSelWave / 64;
  float z[kR];
  int c[kR], rank[kR];
#pragma unroll
  for (int r = 0; r < kR; ++r) {
    const int i = base + wave * kSelWave + r * 64 + lane;
    c[r] = -1;
    z[r] = 0.f;
    if (i < n) {
      c[r] = cell[i];
      z[r] = pts[i].z;
    }
  }
  const int tiles = (n + kSelTile - 1) / kSelTile;
  int tot = 0, before = 0;
  if (t <= cfg.n_cells) {
    const int4* row = reinterpret_cast<const int4*>(table + (size_t)t * stride);
    const int me = blockIdx.x;
#pragma unroll 4
    for (int q = 0; q < (tiles + 3) / 4; ++q) {
      const int4 v = row[q];
      const int b = 4 * q;
      const int c0 = v.x, c1 = b + 1 < tiles ? v.y : 0, c2 = b + 2 < tiles ? v.z : 0,
                c3 = b + 3 < tiles ? v.w : 0;
      tot += c0 + c1 + c2 + c3;
      before += (b < me ? c0 : 0) + (b + 1 < me ? c1 : 0) + (b + 2 < me ? c2 : 0) +
                (b + 3 < me ? c3 : 0);
    }
  }
  int s = tot;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(s, o, 64);
    if (lane >= o) s += u;
  }
  if (lane == 63) wtot[wave] = s;
#pragma unroll
  for (int w = 0; w < kGB / 64; ++w) wc[w][t] = 0;
  __syncthreads();
  int wo = 0;
#pragma unroll
  for (int w = 0; w < kGB / 64; ++w) wo += w < wave ? wtot[w] : 0;
  const int start = wo + s - tot;
  first[t] = start + before;
  if (blockIdx.x == 0 && t <= cfg.n_cells) offsets[t] = start;
  const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int r = 0; r < kR; ++r) {
    uint64_t peers = __builtin_amdgcn_ballot_w64(c[r] >= 0);
    for (int b = 0; b < bits; ++b) {
      const bool bit = (c[r] >> b) & 1;
      const uint64_t m = __builtin_amdgcn_ballot_w64(c[r] >= 0 && bit);
      peers &= bit ? m : ~m;
    }
    const int p = __builtin_popcountll(peers & lt);
    rank[r] = 0;
    if (c[r] >= 0) {
      rank[r] = wc[wave][c[r]] + p;
      __builtin_amdgcn_wave_barrier();
      if (p == 0) wc[wave][c[r]] += __builtin_popcountll(peers);
    }
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kR; ++r) {
    if (c[r] < 0 || c[r] >= cfg.n_cells) continue;
    int dest = first[c[r]] + rank[r];
    for (int w = 0; w < wave; ++w) dest += wc[w][c[r]];
    idx[dest] = base + wave * kSelWave + r * 64 + lane;
    zkey[dest] = orderable(z[r]);
  }
}

struct GroundSel {
  uint32_t keys[kSelKeys];
  unsigned long long cand[kSelCand];
  int hist[kSelBins];
  uint32_t wmin[kGB / 64], wmax[kGB / 64];
  int wtot[kGB / 64];
  int n_cand, bin, count, mode;
};

// The first k points by (z, input order) of a cell of s <= kSelKeys points,
// k <= s, as input indices into list.  Rounds of at most kSelCand points: the
// pending keys' range is cut into 256 bins, the bins that reach k (or as many
// as fit) are gathered and sorted as (key, position) pairs; a first bin that
// does not fit is cut again, down to one key, whose points follow in input
// order.  The usual cell (a few thousand points, 5 % kept) takes one round of
// ~100 candidates.
__device__ inline void ground_select(const uint32_t* __restrict__ gkey,
                                     const int32_t* __restrict__ gidx, int s, int k,
                                     int32_t* __restrict__ list, GroundSel& L) {
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  for (int i = t; i < s; i += kGB) L.keys[i] = gkey[i];
  __syncthreads();
  unsigned long long lo = 0;  // smallest pending key
  int done = 0;
  while (done < k) {
    const int rem = k - done;
    uint32_t kmin = 0xffffffffu, kmax = 0u;
    for (int i = t; i < s; i += kGB) {
      const uint32_t q = L.keys[i];
      if (q >= lo) {
        kmin = min(kmin, q);
        kmax = max(kmax, q);
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      kmin = min(kmin, (uint32_t)__shfl_xor((int)kmin, o, 64));
      kmax = max(kmax, (uint32_t)__shfl_xor((int)kmax, o, 64));
    }
    if (lane == 0) {
      L.wmin[wave] = kmin;
      L.wmax[wave] = kmax;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kGB / 64; ++w) {
      kmin = min(kmin, L.wmin[w]);
      kmax = max(kmax, L.wmax[w]);
    }
    int shift, mode, bin;
    for (;;) {
      const uint32_t span = kmax - kmin;
      shift = span >> 8 ? 24 - __builtin_clz(span) : 0;  // (span >> shift) < 256
      L.hist[t] = 0;
      if (t == 0) {
        L.n_cand = 0;
        L.mode = 3;
        L.bin = kSelBins - 1;
      }
      __syncthreads();
      for (int i = t; i < s; i += kGB) {
        const uint32_t q = L.keys[i];
        if (q >= kmin && q <= kmax) atomicAdd(&L.hist[(q - kmin) >> shift], 1);
      }
      __syncthreads();
      const int h = L.hist[t];
      int c = h;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int u = __shfl_up(c, o, 64);
        if (lane >= o) c += u;
      }
      if (lane == 63) L.wtot[wave] = c;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < kGB / 64; ++w) c += w < wave ? L.wtot[w] : 0;
      // c: points up to and in bin t.  One thread at most finds each case.
      const int prev = c - h;
      if (h > 0 && c <= kSelCand) {
        // the bin that reaches the remaining count ...
        if (prev < rem && c >= rem) {
          L.mode = 1;
          L.bin = t;
        }
      } else if (h > 0 && prev < rem) {
        if (prev > 0 && prev <= kSelCand) {
          L.mode = 1;  // ... or the bins before the first that does not fit
          L.bin = t - 1;
        } else if (prev == 0) {
          L.mode = 2;  // the first bin alone does not fit
          L.bin = t;
        }
      }
      __syncthreads();
      mode = L.mode;
      bin = L.bin;
      __syncthreads();
      if (mode != 2 || shift == 0) break;
      kmin += (uint32_t)bin << shift;
      kmax = min(kmax, kmin + ((1u << shift) - 1u));
    }
    if (mode == 2) {
      // more points of one key than are sorted at once: in input order
      const uint32_t v = kmin + (uint32_t)bin;
      int got = 0;
      for (int i0 = 0; i0 < s && got < rem; i0 += kGB) {
        const int i = i0 + t;
        const bool f = i < s && L.keys[i] == v;
        const uint64_t b = __builtin_amdgcn_ballot_w64(f);
        if (lane == 0) L.wtot[wave] = __builtin_popcountll(b);
        __syncthreads();
        int off = got + __builtin_popcountll(b & ((1ull << lane) - 1ull));
        for (int w = 0; w < kGB / 64; ++w) {
          off += w < wave ? L.wtot[w] : 0;
          got += L.wtot[w];
        }
        if (f && off < rem) list[done + off] = gidx[i];
        __syncthreads();
      }
      done += min(got, rem);
      lo = (unsigned long long)v + 1ull;
      continue;
    }
    // gather the bins up to `bin` and sort them by (key, position)
    const unsigned long long bound =  // exclusive
        min((unsigned long long)kmin + ((unsigned long long)(bin + 1) << shift),
            (unsigned long long)kmax + 1ull);
    for (int i = t; i < s; i += kGB) {
      const uint32_t q = L.keys[i];
      if (q >= kmin && q < bound) {
        const int o = atomicAdd(&L.n_cand, 1);
        L.cand[o] = ((unsigned long long)q << 32) | (unsigned)i;
      }
    }
    __syncthreads();
    const int C = L.n_cand;
    const int take = min(C, rem);
    if (C <= kSelRank) {
      for (int e = t; e < C; e += kGB) {
        const unsigned long long me = L.cand[e];
        int r = 0;
        for (int j = 0; j < C; ++j) r += L.cand[j] < me ? 1 : 0;
        if (r < take) list[done + r] = gidx[(uint32_t)me];
      }
    } else {
      int P = 2 * kSelRank;
      while (P < C) P <<= 1;
      for (int e = C + t; e < P; e += kGB) L.cand[e] = ~0ull;
      for (int size = 2; size <= P; size <<= 1)
        for (int step = size >> 1; step > 0; step >>= 1) {
          __syncthreads();
          for (int e = t; e < P / 2; e += kGB) {
            const int a = 2 * e - (e & (step - 1)), b = a + step;
            const unsigned long long x = L.cand[a], y = L.cand[b];
            if ((x > y) == ((a & size) == 0)) {
              L.cand[a] = y;
              L.cand[b] = x;
            }
          }
        }
      __syncthreads();
      for (int e = t; e < take; e += kGB) list[done + e] = gidx[(uint32_t)L.cand[e]];
    }
    done += take;
    lo = bound;
    __syncthreads();
  }
  __syncthreads();
}

struct GroundBig {
  int hist[kBigBins];
  int wc[kBigW][256];
  uint32_t wmin[kBigW], wmax[kBigW];
  int wtot[kBigW], bin, prev, count;
};

// Memory of a large cell's sort: two arrays of (key, position) pairs.
struct GroundPairs {
  uint32_t *key, *key2;
  int32_t *pos, *pos2;
};

// inclusive wave scan
__device__ inline int ground_scan(int v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  return v;
}

// Calls f(position, key) for the points [b, e) of a wave in order, 64 at a
// time (key valid below e only), kBigAhead loads in flight.
template <typename F>
__device__ inline void ground_walk(const uint32_t* key, int b, int e, F f) {
  const int lane = threadIdx.x & 63;
  for (int i0 = b; i0 < e; i0 += 64 * kBigAhead) {
    uint32_t q[kBigAhead];
#pragma unroll
    for (int u = 0; u < kBigAhead; ++u) q[u] = key[min(i0 + 64 * u + lane, e - 1)];
#pragma unroll
    for (int u = 0; u < kBigAhead; ++u)
      if (i0 + 64 * u < e) f(i0 + 64 * u + lane, q[u]);
  }
}

// The same for a cell of more than kSelKeys points, by kBigB threads, in a
// bounded number of passes over the s keys whatever their distribution and k:
// the range of the keys; the bin of the k-th key (cut again, at most twice,
// while it holds more than kBigSlack points of more than one key; of one key
// only the missing points are taken, the first in input order); the points up
// to that bin in input order, each wave over consecutive ones; and a stable
// sort of those, 8 bits a pass over the bits in which they differ.  Latency
// and the LDS adds of one CU bound it (a pass over 262,144 keys 20 us, with
// the adds 54).  262,144 points in one cell, 5 % kept, the whole call: 352 us;
// in rounds of kSelCand points over all keys 4,709, by two radix sorts of the
// cloud (ground_sort) 444.  65,536 points: 119 / 443 / 187.
__device__ inline void ground_select_big(const uint32_t* __restrict__ gkey,
                                         const int32_t* __restrict__ gidx, int s, int k,
                                         int32_t* list, GroundPairs pairs, GroundBig& L) {
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint64_t below_lane = (1ull << lane) - 1ull;
  // a wave's share of n points: consecutive, in multiples of 64
  auto share = [&](int n, int& b, int& e) {
    const int per = (n + kBigB - 1) / kBigB * 64;
    b = min(n, wave * per);
    e = min(n, b + per);
  };
  int wb, we;
  share(s, wb, we);
  // smallest and largest of the waves' values, on every thread
  auto extremes = [&](uint32_t& a, uint32_t& b) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      a = min(a, (uint32_t)__shfl_xor((int)a, o, 64));
      b = max(b, (uint32_t)__shfl_xor((int)b, o, 64));
    }
    if (lane == 0) {
      L.wmin[wave] = a;
      L.wmax[wave] = b;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kBigW; ++w) {
      a = min(a, L.wmin[w]);
      b = max(b, L.wmax[w]);
    }
  };
  uint32_t kmin = 0xffffffffu, kmax = 0u;
  ground_walk(gkey, wb, we, [&](int, uint32_t q) {  // past the end: the last key again
    kmin = min(kmin, q);
    kmax = max(kmax, q);
  });
  extremes(kmin, kmax);
  // [lo, hi]: the bin of the k-th key, with `inside` points and `before`
  // smaller ones
  uint32_t lo = kmin, hi = kmax;
  int before = 0, inside = s;
  while (lo < hi && inside > kBigSlack && before + inside > k) {
    const int shift = max(0, 21 - (int)__builtin_clz(hi - lo));  // ((hi - lo) >> shift) < kBigBins
    for (int i = t; i < kBigBins; i += kBigB) L.hist[i] = 0;
    __syncthreads();
    uint32_t first = 0xffffffffu, last = 0u;
    ground_walk(gkey, wb, we, [&](int i, uint32_t q) {
      if (i < we && q >= lo && q <= hi) {
        first = min(first, q);
        last = max(last, q);
        atomicAdd(&L.hist[(q - lo) >> shift], 1);
      }
    });
    extremes(first, last);
    if (first == last) {  // one key's points
      lo = hi = first;
      break;
    }
    constexpr int kPer = kBigBins / kBigB;
    int h[kPer], mine = 0;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      h[j] = L.hist[kPer * t + j];
      mine += h[j];
    }
    int c = ground_scan(mine, lane);
    if (lane == 63) L.wtot[wave] = c;
    __syncthreads();
    for (int w = 0; w < wave; ++w) c += L.wtot[w];
    c += before - mine;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      if (c < k && c + h[j] >= k) {  // one thread finds it
        L.bin = kPer * t + j;
        L.prev = c;
        L.count = h[j];
      }
      c += h[j];
    }
    __syncthreads();
    before = L.prev;
    inside = L.count;
    lo += (uint32_t)L.bin << shift;
    hi = min(hi, lo + ((1u << shift) - 1u));
    __syncthreads();
  }
  __syncthreads();
  // The smaller points and the bin's (of one key's only those missing), as
  // (key - kmin, position), each wave's at the start of its own share.
  int quota = inside;  // of the wave
  if (lo == hi && before + inside > k) {
    int n_in = 0;
    ground_walk(gkey, wb, we, [&](int i, uint32_t q) {
      n_in += __builtin_popcountll(__builtin_amdgcn_ballot_w64(i < we && q == lo));
    });
    if (lane == 0) L.wtot[wave] = n_in;
    __syncthreads();
    quota = k - before;
    for (int w = 0; w < wave; ++w) quota -= L.wtot[w];
    quota = max(quota, 0);
  }
  int n = 0, n_in = 0;
  ground_walk(gkey, wb, we, [&](int i, uint32_t q) {
    const bool lt = i < we && q < lo, in = i < we && q >= lo && q <= hi;
    const uint64_t bi = __builtin_amdgcn_ballot_w64(in);
    const bool take = lt || (in && n_in + __builtin_popcountll(bi & below_lane) < quota);
    const uint64_t bt = __builtin_amdgcn_ballot_w64(take);
    const int dest = wb + n + __builtin_popcountll(bt & below_lane);
    if (take) {
      pairs.key[dest] = q - kmin;
      pairs.pos[dest] = i;
    }
    n += __builtin_popcountll(bt);
    n_in += __builtin_popcountll(bi);
  });
  const uint32_t range = hi - kmin;
  const int bits = range ? 32 - (int)__builtin_clz(range) : 1;
  int cb = wb, ce = wb + n;  // the wave's part of the pass's input
  for (int bit = 0; bit < bits; bit += 8) {
    for (int i = t; i < kBigW * 256; i += kBigB) L.wc[i >> 8][i & 255] = 0;
    __syncthreads();  // the pairs, too
    ground_walk(pairs.key, cb, ce, [&](int i, uint32_t q) {
      if (i < ce) atomicAdd(&L.wc[wave][(q >> bit) & 255], 1);
    });
    __syncthreads();
    int tot = 0;
    if (t < 256) {
#pragma unroll
      for (int w = 0; w < kBigW; ++w) {
        const int c = L.wc[w][t];
        L.wc[w][t] = tot;
        tot += c;
      }
    }
    int off = ground_scan(tot, lane);
    if (lane == 63) L.wtot[wave] = off;
    __syncthreads();
    if (t < 256) {
      off -= tot;
      for (int w = 0; w < wave; ++w) off += L.wtot[w];
#pragma unroll
      for (int w = 0; w < kBigW; ++w) L.wc[w][t] += off;
    }
    const int C = L.wtot[0] + L.wtot[1] + L.wtot[2] + L.wtot[3];
    __syncthreads();
    for (int i0 = cb; i0 < ce; i0 += 64 * kBigAhead) {
      uint32_t qs[kBigAhead];
      int32_t vs[kBigAhead];
#pragma unroll
      for (int u = 0; u < kBigAhead; ++u) {
        const int i = min(i0 + 64 * u + lane, ce - 1);
        qs[u] = pairs.key[i];
        vs[u] = pairs.pos[i];
      }
#pragma unroll
      for (int u = 0; u < kBigAhead; ++u) {
        if (i0 + 64 * u >= ce) break;
        const bool act = i0 + 64 * u + lane < ce;
        const int d = (qs[u] >> bit) & 255;
        uint64_t peers = __builtin_amdgcn_ballot_w64(act);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
          const uint64_t m = __builtin_amdgcn_ballot_w64(act && ((d >> b) & 1));
          peers &= (d >> b) & 1 ? m : ~m;
        }
        const int r = __builtin_popcountll(peers & below_lane);
        if (act) {
          const int dest = L.wc[wave][d] + r;
          __builtin_amdgcn_wave_barrier();
          if (r == 0) L.wc[wave][d] += __builtin_popcountll(peers);
          pairs.key2[dest] = qs[u];
          pairs.pos2[dest] = vs[u];
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
    share(C, cb, ce);
    pairs = {pairs.key2, pairs.key, pairs.pos2, pairs.pos};
    __syncthreads();
  }
#pragma unroll 4
  for (int j = t; j < k; j += kBigB) list[j] = gidx[pairs.pos[j]];
  __syncthreads();
}

// points per workgroup of ground_bin; cells counted in LDS up to kBinLds cells
constexpr int kBinPts = 2048;
constexpr int kBinLds = 4096;

__global__ __launch_bounds__(kGB) void ground_bin_kernel(
    const float4* __restrict__ pts, int cap, const int32_t* __restrict__ d_n, GroundCfgDev cfg,
    unsigned long long* __restrict__ key_idx, unsigned long long* __restrict__ key_z,
    int32_t* __restrict__ vals_idx, int32_t* __restrict__ vals_z, int32_t* __restrict__ counts) {
  // per-workgroup cell counts in LDS, one global atomic per non-empty cell
  // (all points of a scan fall in few cells: per-point global atomics on the
  // same counters serialise)
  __shared__ int hcount[kBinLds];
  const bool lds = cfg.n_cells <= kBinLds;
  if (lds)
    for (int c = threadIdx.x; c < cfg.n_cells; c += kGB) hcount[c] = 0;
  __syncthreads();
  const int n = min(d_n ? *d_n : cap, cap);
  const int base = blockIdx.x * kBinPts;
  for (int j = threadIdx.x; j < kBinPts; j += kGB) {
    const int i = base + j;
    if (i >= n) break;  // the sorts stop at n
    const float4 p = pts[i];
    const float z = p.z;
    const unsigned long long cell = (unsigned long long)ground_cell(p, cfg);
    if ((int)cell < cfg.n_cells) {
      if (lds)
        atomicAdd(&hcount[(int)cell], 1);
      else
        atomicAdd(counts + cell, 1);
    }
    // (cell) and (cell, z): the stable sort keeps input order within equal keys
    key_idx[i] = cell;
    key_z[i] = (cell << 32) | (unsigned long long)orderable(z);
    vals_idx[i] = i;
    vals_z[i] = i;
  }
  __syncthreads();
  if (lds)
    for (int c = threadIdx.x; c < cfg.n_cells; c += kGB) {
      const int v = hcount[c];
      if (v) atomicAdd(counts + c, v);
    }
}

__global__ __launch_bounds__(kGB) void ground_offsets_kernel(const int32_t* __restrict__ counts,
                                                             int n_cells,
                                                             int32_t* __restrict__ offsets) {
  // one workgroup; n_cells is small (radii x theta bins)
  __shared__ int carry;
  __shared__ int wtot[kGB / 64];
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int base = 0; base < n_cells; base += kGB) {
    const int i = base + (int)threadIdx.x;
    const int v = i < n_cells ? counts[i] : 0;
    int s = v;
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(s, o, 64);
      if (lane >= o) s += t;
    }
    if (lane == 63) wtot[wave] = s;
    __syncthreads();
    int woff = 0;
    for (int w = 0; w < wave; ++w) woff += wtot[w];
    const int excl = carry + woff + s - v;
    if (i < n_cells) offsets[i] = excl;
    __syncthreads();
    if (threadIdx.x == kGB - 1) carry = excl + v;
    __syncthreads();
  }
  if (threadIdx.x == 0) offsets[n_cells] = carry;
}

template <int K>
__device__ inline void gsum(double (&v)[K], double* lds) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = sl_wave_sum(v[k]);
  __syncthreads();
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < K; ++k) lds[wave * K + k] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K; ++k) {
    double t = lds[k];
    for (int w = 1; w < kGB / 64; ++w) t += lds[w * K + k];
    v[k] = t;
  }
  __syncthreads();
}

// info: {valid, kept, binned, 0}; model: plane[4], centroid[3], unused.
// offsets (nullable): the cells' exclusive prefix of counts; without it
// (few cells) each workgroup adds the counts of the cells before its own.
// kSelect: by_idx and zkey are the points partitioned by cell, by_z receives
// the cell's kept points where they are the lowest by z; pairs are the sort
// buffers of the large cells, which all kBigB threads select (the first kGB do
// the rest).
template <bool kSelect>
__global__ __launch_bounds__(kSelect ? kBigB : kGB) void ground_fit_kernel(
    const float4* __restrict__ pts, const int32_t* __restrict__ counts,
    const int32_t* __restrict__ offsets,
    const int32_t* __restrict__ by_idx, int32_t* __restrict__ by_z,
    const uint32_t* __restrict__ zkey, GroundPairs pairs, GroundCfgDev cfg,
    int4* __restrict__ info, double* __restrict__ model, float4* __restrict__ features,
    int32_t* __restrict__ kept_index, int32_t* __restrict__ kept_offsets) {
  // the selection's memory serves the centroid's tiles afterwards
  struct Tiles {
    float v[3][kCentroidTile];
  };
  constexpr size_t kLds =
      kSelect ? std::max({sizeof(GroundSel), sizeof(GroundBig), sizeof(Tiles)}) : sizeof(Tiles);
  __shared__ __align__(16) unsigned char lds[kLds];
  float(*tile)[kCentroidTile] = reinterpret_cast<Tiles*>(lds)->v;
  __shared__ double red[(kGB / 64) * 6];
  __shared__ float cen[3];
  const int c = blockIdx.x;
  int off, s;
  if (offsets) {
    off = offsets[c];
    s = offsets[c + 1] - off;
  } else {
    off = 0;
    for (int i = 0; i < c; ++i) off += counts[i];
    s = counts[c];
  }
  int k = s;
  const int32_t* list = by_idx + off;
  if (cfg.retain_num < (double)s) {
    k = (int)((double)s / cfg.retain_num);
    k = min(k, s);
    list = by_z + off;
  }
  bool listed = false;  // kept_index holds the cell's points
  if constexpr (kSelect) {
    const bool reduced = cfg.retain_num < (double)s, big = reduced && s > kSelKeys;
    if (big) {
      ground_select_big(zkey + off, by_idx + off, s, k, by_z + off,
                        {pairs.key + off, pairs.key2 + off, pairs.pos + off, pairs.pos2 + off},
                        *reinterpret_cast<GroundBig*>(lds));
      if (kept_index)
        for (int j = threadIdx.x; j < s; j += kBigB) kept_index[off + j] = j < k ? list[j] : -1;
      listed = true;
    }
    if (threadIdx.x >= kGB) return;  // no barrier waits for waves that ended
    if (reduced && !big)
      ground_select(zkey + off, by_idx + off, s, k, by_z + off,
                    *reinterpret_cast<GroundSel*>(lds));
  }
  const bool valid = k >= cfg.nf && k > 0;
  double* out = model + 8 * (size_t)c;
  if (kept_index) {
    // the cell's kept points, in the order used (slots past k hold -1)
    if (!listed)
      for (int j = threadIdx.x; j < s; j += kGB) kept_index[off + j] = j < k ? list[j] : -1;
    if (threadIdx.x == 0) {
      kept_offsets[c] = off;
      if (c == cfg.n_cells - 1) kept_offsets[cfg.n_cells] = off + s;
    }
  }
  if (!valid) {
    if (threadIdx.x == 0) {
      info[c] = make_int4(0, k, s, 0);
      for (int i = 0; i < 8; ++i) out[i] = 0.0;
    }
    return;
  }
  // centroid: sequential float sums in list order (the reference's
  // computeCentroid), staged through LDS tiles
  float sum = 0.f;  // lane 0: x, 1: y, 2: z
  for (int t0 = 0; t0 < k; t0 += kCentroidTile) {
    const int tn = min(kCentroidTile, k - t0);
    __syncthreads();
#pragma unroll 4
    for (int j = threadIdx.x; j < tn; j += kGB) {
      const float4 p = pts[list[t0 + j]];
      tile[0][j] = p.x;
      tile[1][j] = p.y;
      tile[2][j] = p.z;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
      const float* row = tile[threadIdx.x];
      const float4* row4 = reinterpret_cast<const float4*>(row);
      float4 v[4];  // the next sixteen
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = row4[u];
      int j = 0;
      for (; j + 16 <= tn; j += 16) {
        const int ahead = min(j + 16, kCentroidTile - 16) / 4;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float4 q = v[u];
          v[u] = row4[ahead + u];
          sum = (((sum + q.x) + q.y) + q.z) + q.w;
        }
      }
      for (; j < tn; ++j) sum = sum + row[j];
    }
  }
  if (threadIdx.x < 3) cen[threadIdx.x] = (float)((double)sum / (double)k);
  __syncthreads();
  const float cx = cen[0], cy = cen[1], cz = cen[2];
  double S[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll 2
  for (int j = threadIdx.x; j < k; j += kGB) {
    const float4 p = pts[list[j]];
    const double x = (double)(p.x - cx), y = (double)(p.y - cy), z = (double)(p.z - cz);
    S[0] += x * x;
    S[1] += x * y;
    S[2] += x * z;
    S[3] += y * y;
    S[4] += y * z;
    S[5] += z * z;
  }
  gsum<6>(S, red);
  for (int j = threadIdx.x; j < cfg.nf; j += kGB) features[(size_t)c * cfg.nf + j] = pts[list[j]];
  if (threadIdx.x != 0) return;
  double w[3], V[3][3], nrm[3];
  sl_eig3(S, w, V);
  const int kmin = sl_argmin3(w);
  nrm[0] = kmin == 0 ? V[0][0] : (kmin == 1 ? V[0][1] : V[0][2]);
  nrm[1] = kmin == 0 ? V[1][0] : (kmin == 1 ? V[1][1] : V[1][2]);
  nrm[2] = kmin == 0 ? V[2][0] : (kmin == 1 ? V[2][1] : V[2][2]);
  // orientation: upward (z > 0); a horizontal normal falls back to the
  // largest-|component|-positive rule
  if (nrm[2] < 0.0) {
    nrm[0] = -nrm[0];
    nrm[1] = -nrm[1];
    nrm[2] = -nrm[2];
  }
  if (nrm[2] == 0.0) sl_sign_normalise(nrm);
  const double d = -(nrm[0] * (double)cx + nrm[1] * (double)cy + nrm[2] * (double)cz);
  out[0] = nrm[0];
  out[1] = nrm[1];
  out[2] = nrm[2];
  out[3] = d;
  out[4] = (double)cx;
  out[5] = (double)cy;
  out[6] = (double)cz;
  out[7] = 0.0;
  info[c] = make_int4(1, k, s, 0);
}

// ---------------------------------------------------------------------------
// batched plane RANSAC
// ---------------------------------------------------------------------------
constexpr int kPlB = 256;
constexpr int kPlW = kPlB / 64;
constexpr int kPlHB = 8;
constexpr int kPlTile = 1024;
constexpr int kPlHyps = 64;         // hypotheses per score workgroup
constexpr int kPlScore = 1024;      // points per score chunk
constexpr int kPlScoreMax = 65536;  // score workgroups a batch is cut into at most
constexpr int kPlRefit = 2048;      // points per refit chunk
constexpr int kPlMaxChunks = 256;   // refit chunks per set at most

struct PlFrame {
  float m[3];
  int32_t n;
};

struct PlHyp {
  float nx, ny, nz, d;  // unit normal and offset in the local frame (p - m)
  int valid;
};

__device__ inline PlHyp plane_hyp(const float a[3], const float b[3], const float c[3]) {
  PlHyp h;
  const float ux = b[0] - a[0], uy = b[1] - a[1], uz = b[2] - a[2];
  const float vx = c[0] - a[0], vy = c[1] - a[1], vz = c[2] - a[2];
  float nx = uy * vz - uz * vy;
  float ny = uz * vx - ux * vz;
  float nz = ux * vy - uy * vx;
  const float len = sqrtf(nx * nx + ny * ny + nz * nz);
  h.valid = len > 0.0f ? 1 : 0;  // false for a degenerate triangle or NaN
  if (h.valid) {
    nx = nx / len;
    ny = ny / len;
    nz = nz / len;
    h.nx = nx;
    h.ny = ny;
    h.nz = nz;
    h.d = -((nx * a[0] + ny * a[1]) + nz * a[2]);
  } else {
    h.nx = h.ny = h.nz = 0.f;
    h.d = INFINITY;  // |t| < thr never holds
  }
  return h;
}

__device__ inline PlHyp plane_hyp_for(const float* __restrict__ P, int n, int set, int hidx,
                                      const PlFrame& f, uint32_t k0, uint32_t k1, uint32_t tag,
                                      int32_t idx[3]) {
  SlU4 ctr = {(uint32_t)hidx, (uint32_t)set, tag, 0u};
  const SlU4 x = sl_philox4x32_10(ctr, k0, k1);
  sl_draw3(x.x, x.y, x.z, (uint32_t)n, &idx[0], &idx[1], &idx[2]);
  float q[3][3];
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int c = 0; c < 3; ++c) q[j][c] = P[3 * (size_t)idx[j] + c] - f.m[c];
  return plane_hyp(q[0], q[1], q[2]);
}

__device__ inline bool plane_inlier(float x, float y, float z, const PlHyp& h, float thr) {
  const float t = __builtin_fmaf(h.nx, x, __builtin_fmaf(h.ny, y, __builtin_fmaf(h.nz, z, h.d)));
  return fabsf(t) < thr;
}

// The sets are cut twice: into score chunks (the points one workgroup scores
// kPlHyps hypotheses on) and into refit chunks (kPlRefit points or more, at
// most kPlMaxChunks a set).  A chunk is {set, first point, points, chunks of
// the set << 16 | chunk index} with the points relative to the set; an empty
// set has one empty chunk.
struct PlChunk {
  int set, first, n, of;
  __device__ int count() const { return (int)((uint32_t)of >> 16); }
  __device__ int index() const { return of & 0xffff; }
};

// Bounding box of a refit chunk (6 floats per chunk); zeroes what the next
// kernels accumulate into: the set's counts (its first chunk's workgroup),
// the arrival counters of the refit and the mask words.
__global__ __launch_bounds__(kPlB) void plane_box_kernel(
    const float* __restrict__ xyz, const int32_t* __restrict__ offsets,
    const PlChunk* __restrict__ chunks, int n_hyp, float* __restrict__ box,
    int32_t* __restrict__ counts, int2* __restrict__ arrived, uint32_t* __restrict__ mask,
    long long mask_words) {
  __shared__ float red[kPlW][6];
  const PlChunk ck = chunks[blockIdx.x];
  const float* P = xyz + 3 * ((size_t)offsets[ck.set] + ck.first);
  float mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int i = threadIdx.x; i < ck.n; i += kPlB)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float q = P[3 * (size_t)i + k];
      mn[k] = fminf(mn[k], q);
      mx[k] = fmaxf(mx[k], q);
    }
  if (ck.index() == 0) {
    for (int h = threadIdx.x; h < n_hyp; h += kPlB) counts[(size_t)ck.set * n_hyp + h] = 0;
    if (threadIdx.x == 0) arrived[ck.set] = make_int2(0, 0);
  }
  if (mask)
    for (long long w = (long long)blockIdx.x * kPlB + threadIdx.x; w < mask_words;
         w += (long long)gridDim.x * kPlB)
      mask[w] = 0u;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      mn[k] = fminf(mn[k], __shfl_xor(mn[k], o, 64));
      mx[k] = fmaxf(mx[k], __shfl_xor(mx[k], o, 64));
    }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0)
    for (int k = 0; k < 3; ++k) {
      red[wave][k] = mn[k];
      red[wave][3 + k] = mx[k];
    }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int k = threadIdx.x;
    float a = red[0][k];
    for (int w = 1; w < kPlW; ++w) a = k < 3 ? fminf(a, red[w][k]) : fmaxf(a, red[w][k]);
    box[6 * (size_t)blockIdx.x + k] = a;
  }
}

// The set's frame from the boxes of its R refit chunks (minima and maxima:
// the order does not matter), by every thread of the workgroup.
__device__ inline PlFrame plane_frame(const float* __restrict__ box, int R, int n,
                                      float (*red)[6]) {
  float v[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
  for (int r = threadIdx.x; r < R; r += kPlB)
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const float q = box[6 * (size_t)r + k];
      v[k] = k < 3 ? fminf(v[k], q) : fmaxf(v[k], q);
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const float q = __shfl_xor(v[k], o, 64);
      v[k] = k < 3 ? fminf(v[k], q) : fmaxf(v[k], q);
    }
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int k = 0; k < 6; ++k) red[threadIdx.x >> 6][k] = v[k];
  __syncthreads();
  PlFrame f;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    float a = red[0][k], b = red[0][3 + k];
    for (int w = 1; w < kPlW; ++w) {
      a = fminf(a, red[w][k]);
      b = fmaxf(b, red[w][3 + k]);
    }
    f.m[k] = n > 0 ? 0.5f * (a + b) : 0.0f;
  }
  f.n = n;
  return f;
}

// Inlier counts of kPlHyps hypotheses (blockIdx.y) over one score chunk.
// A set's chunks add their counts with integer atomics (any order gives the
// same counts); a set of one chunk stores them.  A workgroup per set and 256
// hypotheses, as before, left a scan's ground (one set) on one CU: 457 us at
// 27,001 points x 200 hypotheses, and the largest patch of a batch set its
// time (339 us at 300 sets of 40..20,000 points); in chunks of 1,024 points x
// 64 hypotheses the two take 10.7 us (launch and gather latency) and 29 us
// (17 us of VALU issue, 12 of them the 3 FMA + 1 compare per point and
// hypothesis).
__global__ __launch_bounds__(kPlB) void plane_score_kernel(
    const float* __restrict__ xyz, const int32_t* __restrict__ offsets,
    const float* __restrict__ box, const int2* __restrict__ set_chunks,
    const PlChunk* __restrict__ chunks, int n_hyp, float thr, uint32_t k0, uint32_t k1,
    uint32_t tag, PlFrame* __restrict__ frames, int32_t* __restrict__ counts,
    int32_t* __restrict__ samples) {
  __shared__ float4 hp[kPlHyps];
  __shared__ float sx[kPlTile], sy[kPlTile], sz[kPlTile];
  __shared__ int cnt[kPlHyps];
  __shared__ float red[kPlW][6];
  const PlChunk ck = chunks[blockIdx.x];
  const int c = ck.set, h0 = blockIdx.y * kPlHyps, hc = min(kPlHyps, n_hyp - h0);
  const int off = offsets[c];
  const int n = offsets[c + 1] - off;
  const float* P = xyz + 3 * (size_t)off;
  const int2 sc = set_chunks[c];
  const PlFrame f = plane_frame(box + 6 * (size_t)sc.x, sc.y, n, red);
  if (ck.index() == 0 && blockIdx.y == 0 && threadIdx.x == 0) frames[c] = f;
  if (threadIdx.x < kPlHyps) {
    const int t = threadIdx.x;
    float4 prm = make_float4(0.f, 0.f, 0.f, INFINITY);
    if (t < hc) {
      int32_t idx[3] = {-1, -1, -1};
      if (n >= 3) {
        const PlHyp h = plane_hyp_for(P, n, c, h0 + t, f, k0, k1, tag, idx);
        prm = make_float4(h.nx, h.ny, h.nz, h.d);
      }
      if (samples && ck.index() == 0) {
        int32_t* o = samples + 3 * ((size_t)c * n_hyp + h0 + t);
        o[0] = idx[0];
        o[1] = idx[1];
        o[2] = idx[2];
      }
    }
    hp[t] = prm;
    cnt[t] = 0;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  constexpr int hpw = kPlHyps / kPlW;  // hypotheses per wave
  for (int t0 = 0; t0 < ck.n; t0 += kPlTile) {
    const int tn = min(kPlTile, ck.n - t0);
    const int tn64 = (tn + 63) & ~63;
    __syncthreads();
    for (int i = threadIdx.x; i < tn64; i += kPlB) {
      float x = NAN, y = 0.f, z = 0.f;
      if (i < tn) {
        const float* q = P + 3 * ((size_t)ck.first + t0 + i);
        x = q[0] - f.m[0];
        y = q[1] - f.m[1];
        z = q[2] - f.m[2];
      }
      sx[i] = x;
      sy[i] = y;
      sz[i] = z;
    }
    __syncthreads();
#pragma unroll
    for (int hb = 0; hb < hpw; hb += kPlHB) {
      const int hbase = wave * hpw + hb;
      if (hbase >= hc) break;
      float NX[kPlHB], NY[kPlHB], NZ[kPlHB], D[kPlHB];
      int cc[kPlHB];
#pragma unroll
      for (int j = 0; j < kPlHB; ++j) {
        const float4 q = hp[hbase + j];
        NX[j] = q.x;
        NY[j] = q.y;
        NZ[j] = q.z;
        D[j] = q.w;
        cc[j] = 0;
      }
      for (int i0 = 0; i0 < tn64; i0 += 64) {
        const int i = i0 + lane;
        const float x = sx[i], y = sy[i], z = sz[i];
#pragma unroll
        for (int j = 0; j < kPlHB; ++j) {
          const float t = __builtin_fmaf(NX[j], x, __builtin_fmaf(NY[j], y,
                                                                  __builtin_fmaf(NZ[j], z, D[j])));
          cc[j] += __builtin_popcountll(__builtin_amdgcn_ballot_w64(fabsf(t) < thr));
        }
      }
      if (lane == 0)
#pragma unroll
        for (int j = 0; j < kPlHB; ++j) cnt[hbase + j] += cc[j];
    }
  }
  __syncthreads();
  if ((int)threadIdx.x < hc) {
    int32_t* o = counts + (size_t)c * n_hyp + h0 + threadIdx.x;
    const int v = cnt[threadIdx.x];
    if (ck.count() == 1)
      *o = v;
    else if (v)
      atomicAdd(o, v);
  }
}

// Sum of K doubles per thread over the workgroup, every thread gets it
// (waves, then the waves in order).
template <int K>
__device__ inline void plane_sum(double (&v)[K], double* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < K; ++k) v[k] = sl_wave_sum(v[k]);
  __syncthreads();
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < K; ++k) red[wave * K + k] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K; ++k) {
    double t = red[k];
    for (int w = 1; w < kPlW; ++w) t += red[w * K + k];
    v[k] = t;
  }
}

// Best hypothesis of a set (max count, lowest index), by every thread.
__device__ inline int plane_best(const int32_t* __restrict__ counts, int n_hyp, int n,
                                 long long* redk) {
  long long key = -1;
  for (int h = threadIdx.x; h < n_hyp; h += kPlB) {
    const long long kk = ((long long)counts[h] << 32) | (long long)(0xFFFFFFFFu - (uint32_t)h);
    key = kk > key ? kk : key;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const long long other = __shfl_xor(key, o, 64);
    key = other > key ? other : key;
  }
  if ((threadIdx.x & 63) == 0) redk[threadIdx.x >> 6] = key;
  __syncthreads();
  key = redk[0];
  for (int w = 1; w < kPlW; ++w) key = redk[w] > key ? redk[w] : key;
  return n >= 3 ? (int)(0xFFFFFFFFu - (uint32_t)(key & 0xFFFFFFFFll)) : -1;
}

// kPlAhead points per thread, loaded before any is used (the loads overlap),
// from i0 on in strides of the workgroup; NaN past n.
constexpr int kPlAhead = 4;
__device__ inline void plane_load(const float* __restrict__ P, int i0, int n,
                                  float (&q)[kPlAhead][3]) {
#pragma unroll
  for (int j = 0; j < kPlAhead; ++j) {
    const int i = i0 + j * kPlB + (int)threadIdx.x;
#pragma unroll
    for (int k = 0; k < 3; ++k) q[j][k] = i >= 0 && i < n ? P[3 * (size_t)i + k] : NAN;
  }
}

// Covariance (FP64, about mu) of the inliers of h among a chunk's points.
__device__ inline void plane_cov(const float* __restrict__ P, int n, const PlFrame& f,
                                 const PlHyp& h, float thr, const double mu[3], double (&S)[6]) {
#pragma unroll
  for (int k = 0; k < 6; ++k) S[k] = 0.0;
  for (int i0 = 0; i0 < n; i0 += kPlAhead * kPlB) {
    float q[kPlAhead][3];
    plane_load(P, i0, n, q);
#pragma unroll
    for (int j = 0; j < kPlAhead; ++j) {
      if (!plane_inlier(q[j][0] - f.m[0], q[j][1] - f.m[1], q[j][2] - f.m[2], h, thr)) continue;
      const double x = ((double)q[j][0] - (double)f.m[0]) - mu[0];
      const double y = ((double)q[j][1] - (double)f.m[1]) - mu[1];
      const double z = ((double)q[j][2] - (double)f.m[2]) - mu[2];
      S[0] += x * x;
      S[1] += x * y;
      S[2] += x * z;
      S[3] += y * y;
      S[4] += y * z;
      S[5] += z * z;
    }
  }
}

// Unit normal, offset and centroid of the plane of covariance S about mu.
__device__ inline void plane_solve(const double (&S)[6], const double mu[3], const PlFrame& f,
                                   double pl[7]) {
  double w3[3], V[3][3], nrm[3];
  sl_eig3(S, w3, V);
  const int kmin = sl_argmin3(w3);
  nrm[0] = kmin == 0 ? V[0][0] : (kmin == 1 ? V[0][1] : V[0][2]);
  nrm[1] = kmin == 0 ? V[1][0] : (kmin == 1 ? V[1][1] : V[1][2]);
  nrm[2] = kmin == 0 ? V[2][0] : (kmin == 1 ? V[2][1] : V[2][2]);
  if (nrm[2] < 0.0) {
    nrm[0] = -nrm[0];
    nrm[1] = -nrm[1];
    nrm[2] = -nrm[2];
  }
  if (nrm[2] == 0.0) sl_sign_normalise(nrm);
  const double cxyz[3] = {(double)f.m[0] + mu[0], (double)f.m[1] + mu[1], (double)f.m[2] + mu[2]};
  pl[0] = nrm[0];
  pl[1] = nrm[1];
  pl[2] = nrm[2];
  pl[3] = -(nrm[0] * cxyz[0] + nrm[1] * cxyz[1] + nrm[2] * cxyz[2]);
  pl[4] = cxyz[0];
  pl[5] = cxyz[1];
  pl[6] = cxyz[2];
}

// The refitted plane of covariance S about mu: unit normal, offset, centroid,
// by the first wave (the FP64 eigen-solve of four waves at once held the
// SIMDs longer than its own latency), every thread gets it.
__device__ inline void plane_from_cov(const double (&S)[6], const double mu[3], const PlFrame& f,
                                      double* lds, double pl[7]) {
  __syncthreads();
  if (threadIdx.x < 64) {
    plane_solve(S, mu, f, pl);
    if (threadIdx.x == 0)
      for (int i = 0; i < 7; ++i) lds[i] = pl[i];
  }
  __syncthreads();
  for (int i = 0; i < 7; ++i) pl[i] = lds[i];
}

// Inliers of the refitted plane (FP64) among a chunk's points, this thread's.
__device__ inline int plane_recount(const float* __restrict__ P, int n, const double pl[7],
                                    float thr) {
  int k = 0;
  for (int i0 = 0; i0 < n; i0 += kPlAhead * kPlB) {
    float q[kPlAhead][3];
    plane_load(P, i0, n, q);
#pragma unroll
    for (int j = 0; j < kPlAhead; ++j) {
      const double t = pl[0] * (double)q[j][0] + pl[1] * (double)q[j][1] +
                       pl[2] * (double)q[j][2] + pl[3];
      k += fabs(t) < (double)thr ? 1 : 0;  // false for the NaN past n
    }
  }
  return k;
}

__device__ inline int plane_sum_int(int v, int* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  int t = red[0];
  for (int w = 1; w < kPlW; ++w) t += red[w];
  return t;
}

// model: plane[4] (unit normal, z >= 0 orientation), centroid[3], inliers of
// the refitted plane.
//
// Mask, centroid and covariance sums of one refit chunk.  A set of one chunk (up to
// kPlRefit points) is finished here; of a larger one each chunk's sums go to
// part, for plane_finish.  90 us by one workgroup
// for a 27,001-point set, 9 + 11 us by fourteen.
__global__ __launch_bounds__(kPlB) void plane_refit_kernel(
    const float* __restrict__ xyz, const int32_t* __restrict__ offsets,
    const PlFrame* __restrict__ frames, const PlChunk* __restrict__ chunks,
    const int32_t* __restrict__ counts, int n_hyp, float thr, uint32_t k0, uint32_t k1,
    uint32_t tag, double* __restrict__ part, PlHyp* __restrict__ best_hyp,
    uint32_t* __restrict__ mask, int32_t* __restrict__ best_out, double* __restrict__ model) {
  __shared__ double red[kPlW * 6];
  __shared__ long long redk[kPlW];
  __shared__ int redi[kPlW];
  __shared__ PlHyp best_h;
  const PlChunk ck = chunks[blockIdx.x];
  const int c = ck.set;
  const int off = offsets[c];
  const int n = offsets[c + 1] - off;
  const float* P = xyz + 3 * (size_t)off;
  const PlFrame f = frames[c];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double* out = model + 8 * (size_t)c;
  const int best = plane_best(counts + (size_t)c * n_hyp, n_hyp, n, redk);
  if (threadIdx.x == 0) {
    if (best >= 0) {
      int32_t idx[3];
      best_h = plane_hyp_for(P, n, c, best, f, k0, k1, tag, idx);
    } else {
      best_h.valid = 0;
      best_h.nx = best_h.ny = best_h.nz = 0.f;
      best_h.d = INFINITY;
    }
    if (ck.index() == 0) {
      if (best_out) best_out[c] = best;
      best_hyp[c] = best_h;
    }
  }
  __syncthreads();
  const PlHyp h = best_h;
  // mask + centroid (FP64, relative to m)
  double acc[4] = {0, 0, 0, 0};
  const int gs = off + ck.first, gend = gs + ck.n;
  for (int gb = (gs & ~63); gb < gend; gb += kPlAhead * kPlB) {
    float q[kPlAhead][3];
    plane_load(xyz + 3 * (size_t)gs, gb - gs, ck.n, q);
#pragma unroll
    for (int j = 0; j < kPlAhead; ++j) {
      const bool in =
          plane_inlier(q[j][0] - f.m[0], q[j][1] - f.m[1], q[j][2] - f.m[2], h, thr);
      const uint64_t b = __builtin_amdgcn_ballot_w64(in);
      if (mask && lane == 0 && b) {
        const int w0 = (gb + j * kPlB + wave * 64) >> 5;
        if ((uint32_t)b) atomicOr(mask + w0, (uint32_t)b);
        if ((uint32_t)(b >> 32)) atomicOr(mask + w0 + 1, (uint32_t)(b >> 32));
      }
      if (in) {
        acc[0] += (double)q[j][0] - (double)f.m[0];
        acc[1] += (double)q[j][1] - (double)f.m[1];
        acc[2] += (double)q[j][2] - (double)f.m[2];
        acc[3] += 1.0;
      }
    }
  }
  plane_sum<4>(acc, red);
  const double k = acc[3];
  const bool whole = ck.count() == 1;
  if (whole && (k < 3.0 || !h.valid)) {
    if (threadIdx.x == 0) {
      for (int i = 0; i < 7; ++i) out[i] = 0.0;
      out[7] = k;
    }
    return;
  }
  const double mu[3] = {acc[0] / k, acc[1] / k, acc[2] / k};
  double S[6], pl[7];
  plane_cov(P + 3 * (size_t)ck.first, ck.n, f, h, thr, mu, S);
  plane_sum<6>(S, red);
  if (!whole) {
    double* o = part + 10 * (size_t)blockIdx.x;
    if (threadIdx.x == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = acc[i];
#pragma unroll
      for (int i = 0; i < 6; ++i) o[4 + i] = k > 0.0 ? S[i] : 0.0;
    }
    return;
  }
  plane_from_cov(S, mu, f, red, pl);
  const int t = plane_sum_int(plane_recount(P, n, pl, thr), redi);
  if (threadIdx.x == 0) {
    for (int i = 0; i < 7; ++i) out[i] = pl[i];
    out[7] = (double)t;
  }
}

// The sets of several chunks: the plane of the chunks' sums (the covariance
// about the common mean is the sum over the chunks of their own, each about
// its own mean, plus n_r d_r d_r' with d_r the distance of the means; FP64,
// in chunk order of a fixed tree), solved by every chunk's workgroup, and
// each chunk's share of its inliers; the chunk that arrives last writes the
// record.
__global__ __launch_bounds__(kPlB) void plane_finish_kernel(
    const float* __restrict__ xyz, const int32_t* __restrict__ offsets,
    const PlFrame* __restrict__ frames, const int2* __restrict__ set_chunks,
    const PlChunk* __restrict__ chunks, float thr, const PlHyp* __restrict__ best_hyp,
    const double* __restrict__ part, int2* __restrict__ arrived, double* __restrict__ model) {
  __shared__ double red[kPlW * 6];
  __shared__ int redi[kPlW];
  static_assert(kPlMaxChunks <= kPlB, "one thread per chunk");
  const PlChunk ck = chunks[blockIdx.x];
  if (ck.count() == 1) return;
  const int R = ck.count();
  const double* sp = part + 10 * ((size_t)set_chunks[ck.set].x + threadIdx.x);
  const bool mine = (int)threadIdx.x < R;
  double* out = model + 8 * (size_t)ck.set;
  double own[4], acc[4], S[6], pl[7];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = own[i] = mine ? sp[i] : 0.0;
#pragma unroll
  for (int i = 0; i < 6; ++i) S[i] = mine ? sp[4 + i] : 0.0;
  plane_sum<4>(acc, red);
  const double k = acc[3];
  if (k < 3.0 || !best_hyp[ck.set].valid) {
    if (ck.index() == 0 && threadIdx.x == 0) {
      for (int i = 0; i < 7; ++i) out[i] = 0.0;
      out[7] = k;
    }
    return;
  }
  const double mu[3] = {acc[0] / k, acc[1] / k, acc[2] / k};
  if (own[3] > 0.0) {
    const double x = own[0] / own[3] - mu[0], y = own[1] / own[3] - mu[1],
                 z = own[2] / own[3] - mu[2];
    S[0] += own[3] * (x * x);
    S[1] += own[3] * (x * y);
    S[2] += own[3] * (x * z);
    S[3] += own[3] * (y * y);
    S[4] += own[3] * (y * z);
    S[5] += own[3] * (z * z);
  }
  plane_sum<6>(S, red);
  plane_from_cov(S, mu, frames[ck.set], red, pl);
  const int t = plane_sum_int(
      plane_recount(xyz + 3 * ((size_t)offsets[ck.set] + ck.first), ck.n, pl, thr), redi);
  if (threadIdx.x != 0) return;
  atomicAdd(&arrived[ck.set].x, t);
  __threadfence();
  if (atomicAdd(&arrived[ck.set].y, 1) != R - 1) return;
  __threadfence();
  for (int i = 0; i < 7; ++i) out[i] = pl[i];
  out[7] = (double)atomicAdd(&arrived[ck.set].x, 0);
}

}  // namespace

struct sloam_plane_plan {
  sloam_ctx* ctx = nullptr;
  sloam_plane_fit_cfg cfg{};
  int32_t n_sets = 0;
  int64_t n_points = 0;
  int n_score = 0, n_refit = 0;  // chunks
  bool multi = false;            // some set has several refit chunks
  void* d_mem = nullptr;         // holds the tables and buffers below
  PlChunk* d_score = nullptr;    // largest sets first
  PlChunk* d_refit = nullptr;    // in set order
  int2* d_sets = nullptr;        // per set {first refit chunk, refit chunks}
  float* d_box = nullptr;        // 6 per refit chunk
  double* d_part = nullptr;      // 10 per refit chunk: centroid sums, covariance
  PlHyp* d_best_hyp = nullptr;   // per set, what the refit hands to the finish
  int2* d_arrived = nullptr;     // per set {inliers, chunks done}
  PlFrame* d_frames = nullptr;
  int32_t* d_counts = nullptr;
};

extern "C" {

int sloam_ground_planes(sloam_ctx* ctx, const float* d_points, int32_t capacity,
                        const int32_t* d_count, const sloam_ground_cfg* cfg, int32_t* d_cell_info,
                        double* d_cell_model, float* d_features, int32_t* d_kept_offsets,
                        int32_t* d_kept_index) {
  if (!ctx || !cfg || !d_cell_info || !d_cell_model || capacity < 0) return SLOAM_ERR_INVALID_ARG;
  if (cfg->radii_bins < 1 || cfg->theta_bins < 1 || !(cfg->retain_thresh > 0.0) ||
      cfg->num_features < 0)
    return SLOAM_ERR_INVALID_ARG;
  const int n_cells = cfg->radii_bins * cfg->theta_bins;
  if (n_cells > 65535) return SLOAM_ERR_TOO_LARGE;
  if (cfg->num_features > 0 && !d_features) return SLOAM_ERR_INVALID_ARG;
  if (capacity > 0 && !d_points) return SLOAM_ERR_INVALID_ARG;
  if ((d_kept_index != nullptr) != (d_kept_offsets != nullptr)) return SLOAM_ERR_INVALID_ARG;
  SLOAM_HIP(ctx, hipSetDevice(ctx->device));
  GroundCfgDev dc;
  dc.R = cfg->radii_bins;
  dc.T = cfg->theta_bins;
  dc.n_cells = n_cells;
  dc.nf = cfg->num_features;
  dc.min_d = cfg->min_dist;
  dc.max_d = cfg->max_dist;
  dc.retain_num = 1.0 / cfg->retain_thresh;
  dc.ox = cfg->origin[0];
  dc.oy = cfg->origin[1];
  const int cap = std::max(capacity, 1);
  // Partition by cell + selection per cell where the cells are one digit and
  // a cell of average size keeps at most one round of candidates and is not so
  // large that one workgroup's passes over it cost more than sorting.  36
  // cells, 5 % kept, 54,000 of 262,144 points: 51 us against 140; all 262,144:
  // 68 / 156, and with all of them in one cell 352 / 444.  250 cells, all
  // 500,000 points kept: 128 / 220, with 50,521 in one cell 836 / 1,080; 80
  // cells, 1,048,576 points in one: 1,633 / 1,628.  (The worst seen: 262,144
  // points of three heights in one cell, 447 / 421.)
  const bool select = capacity > 0 && n_cells <= kSelCells &&
                      (double)cap <= dc.retain_num * (double)kSelCand * (double)n_cells &&
                      (double)cap <= (double)kSelAvg * (double)n_cells;
  // scratch: 2 key arrays + a sort buffer each, 2 value arrays + a sort
  // buffer each, counts, offsets, sort histogram
  const int sel_tiles = (cap + kSelTile - 1) / kSelTile, sel_stride = (sel_tiles + 3) & ~3;
  const size_t kb =
      std::max(sizeof(unsigned long long) * (size_t)cap,
               select ? sizeof(int32_t) * (size_t)(n_cells + 1) * (size_t)sel_stride : 0);
  const size_t vb = sizeof(int32_t) * (size_t)cap;
  const size_t cb = sizeof(int32_t) * (size_t)(n_cells + 1);
  const size_t hb = sizeof(int32_t) * sloam_radix_hist_ints(cap);
  auto al = [](size_t x) { return (x + 255) / 256 * 256; };
  const size_t need = 4 * al(kb) + 4 * al(vb) + 2 * al(cb) + al(hb);
  void* base = nullptr;
  int st = sloam_ctx_scratch(ctx, 1, need, &base);
  if (st) return st;
  char* q = (char*)base;
  auto take = [&](size_t b) {
    char* r = q;
    q += al(b);
    return (void*)r;
  };
  unsigned long long* kA = (unsigned long long*)take(kb);
  unsigned long long* kB = (unsigned long long*)take(kb);
  unsigned long long* kT = (unsigned long long*)take(kb);
  unsigned long long* kT2 = (unsigned long long*)take(kb);
  int32_t* vA = (int32_t*)take(vb);
  int32_t* vB = (int32_t*)take(vb);
  int32_t* vT = (int32_t*)take(vb);
  int32_t* vT2 = (int32_t*)take(vb);
  // the two sorted value arrays (where each sort's last pass leaves them)
  int32_t* by_idx = vA;
  int32_t* by_z = vB;
  int32_t* counts = (int32_t*)take(cb);
  int32_t* offs = (int32_t*)take(cb);
  int32_t* hist = (int32_t*)take(hb);
  if (select) {
    uint8_t* cell = (uint8_t*)kA;
    int32_t* table = (int32_t*)kB;  // (n_cells + 1) rows of stride tiles
    uint32_t* zkey = (uint32_t*)kT;
    const GroundPairs pairs{zkey + cap, (uint32_t*)kT2, vT, vT2};
    int bits = 1;
    while ((1 << bits) <= n_cells) ++bits;
    const float4* pts = reinterpret_cast<const float4*>(d_points);
    {
      SloamKernelScope ks(ctx, "ground_bin");
      hipLaunchKernelGGL(ground_cells_kernel, dim3(sel_tiles), dim3(kGB), 0, ctx->stream, pts,
                         capacity, d_count, dc, sel_stride, cell, table);
    }
    {
      SloamKernelScope ks(ctx, "ground_sort");
      hipLaunchKernelGGL(ground_part_kernel, dim3(sel_tiles), dim3(kGB), 0, ctx->stream, pts,
                         capacity, d_count, dc, sel_stride, bits, cell, table, vA, zkey, offs);
    }
    {
      SloamKernelScope ks(ctx, "ground_fit");
      hipLaunchKernelGGL(ground_fit_kernel<true>, dim3(n_cells), dim3(kBigB), 0, ctx->stream, pts,
                         counts, offs, vA, vB, zkey, pairs, dc, reinterpret_cast<int4*>(d_cell_info),
                         d_cell_model, reinterpret_cast<float4*>(d_features), d_kept_index,
                         d_kept_offsets);
    }
    SLOAM_HIP(ctx, hipGetLastError());
    return SLOAM_OK;
  }
  st = sloam_fill_u32(ctx, (uint32_t*)counts, (size_t)n_cells, 0u);
  if (st) return st;
  {
    SloamKernelScope ks(ctx, "ground_bin");
    if (capacity > 0)
      hipLaunchKernelGGL(ground_bin_kernel, dim3((capacity + kBinPts - 1) / kBinPts), dim3(kGB), 0,
                         ctx->stream, reinterpret_cast<const float4*>(d_points), capacity,
                         d_count, dc, kA, kB, vA, vB, counts);
  }
  SLOAM_HIP(ctx, hipGetLastError());
  if (capacity > 0) {
    SloamKernelScope ks(ctx, "ground_sort");
    // cell ids 0..n_cells (n_cells: outside the grid) in cell_bits bits; the
    // (cell, z) keys hold the orderable z in the low 32 bits
    int cell_bits = 1;
    while ((1 << cell_bits) <= n_cells) ++cell_bits;
    unsigned long long* sorted_keys = nullptr;
    st = sloam_radix_sort(ctx, kA, vA, kT, vT, capacity, 0, cell_bits, d_count, hist, &sorted_keys,
                          &by_idx);
    if (st) return st;
    st = sloam_radix_sort(ctx, kB, vB, kT2, vT2, capacity, 0, 32 + cell_bits, d_count, hist,
                          &sorted_keys,
                          &by_z);
    if (st) return st;
  }
  {
    SloamKernelScope ks(ctx, "ground_fit");
    // a few hundred cells: each fit workgroup adds the counts before its cell
    const bool prefix = n_cells > kGB;
    if (prefix)
      hipLaunchKernelGGL(ground_offsets_kernel, dim3(1), dim3(kGB), 0, ctx->stream, counts,
                         n_cells, offs);
    hipLaunchKernelGGL(ground_fit_kernel<false>, dim3(n_cells), dim3(kGB), 0, ctx->stream,
                       reinterpret_cast<const float4*>(d_points), counts,
                       prefix ? offs : nullptr, by_idx, by_z, (const uint32_t*)nullptr, GroundPairs{},
                       dc,
                       reinterpret_cast<int4*>(d_cell_info), d_cell_model,
                       reinterpret_cast<float4*>(d_features), d_kept_index, d_kept_offsets);
  }
  SLOAM_HIP(ctx, hipGetLastError());
  return SLOAM_OK;
}

int sloam_plane_plan_create(sloam_ctx* ctx, const int32_t* h_offsets, int32_t n_sets,
                            const sloam_plane_fit_cfg* cfg, sloam_plane_plan** out) {
  if (!ctx || !h_offsets || !cfg || !out || n_sets < 0) return SLOAM_ERR_INVALID_ARG;
  *out = nullptr;
  if (cfg->n_hyp < 1 || cfg->n_hyp > (1 << 20) || !(cfg->thr > 0.0f)) return SLOAM_ERR_INVALID_ARG;
  if (h_offsets[0] != 0) return SLOAM_ERR_INVALID_ARG;
  for (int i = 0; i < n_sets; ++i)
    if (h_offsets[i + 1] < h_offsets[i]) return SLOAM_ERR_INVALID_ARG;
  SLOAM_HIP(ctx, hipSetDevice(ctx->device));
  sloam_plane_plan* p = new (std::nothrow) sloam_plane_plan();
  if (!p) return SLOAM_ERR_ALLOC;
  p->ctx = ctx;
  p->cfg = *cfg;
  p->n_sets = n_sets;
  p->n_points = h_offsets[n_sets];
  const int n_y = (cfg->n_hyp + kPlHyps - 1) / kPlHyps;
  // set c's chunks of `chunk` points (one empty chunk for an empty set)
  auto cut = [&](std::vector<PlChunk>& v, int c, int64_t chunk) {
    const int len = h_offsets[c + 1] - h_offsets[c];
    const int R = (int)std::max<int64_t>(1, (len + chunk - 1) / chunk);
    for (int r = 0; r < R; ++r) {
      const int64_t b = r * chunk, e = std::min<int64_t>(len, b + chunk);
      v.push_back(PlChunk{c, (int)b, (int)(e - b), (R << 16) | r});
    }
    return R;
  };
  std::vector<PlChunk> refit, score;
  std::vector<int2> sets(n_sets);
  for (int c = 0; c < n_sets; ++c) {
    const int64_t len = h_offsets[c + 1] - h_offsets[c];
    const int64_t even = (len + kPlMaxChunks - 1) / kPlMaxChunks;
    const int first = (int)refit.size();
    const int R = cut(refit, c, std::max<int64_t>(kPlRefit, (even + 63) / 64 * 64));
    sets[c] = make_int2(first, R);
    p->multi = p->multi || R > 1;
  }
  // score chunks of kPlScore points, of more where that would cut the batch
  // into over kPlScoreMax workgroups (the hypotheses are made once per chunk)
  // or a set into over 2^15 - 1 chunks
  int64_t chunk = kPlScore;
  while ((p->n_points / chunk) * n_y > kPlScoreMax || p->n_points / chunk > 32766) chunk *= 2;
  std::vector<int> order(n_sets);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
    return (h_offsets[a + 1] - h_offsets[a]) > (h_offsets[b + 1] - h_offsets[b]);
  });
  for (int c : order) cut(score, c, chunk);
  p->n_score = (int)score.size();
  p->n_refit = (int)refit.size();
  // one allocation: the three tables (uploaded in one copy), then the rest
  auto al = [](size_t x) { return (x + 255) / 256 * 256; };
  const size_t sb = al(sizeof(PlChunk) * score.size()), rb = al(sizeof(PlChunk) * refit.size()),
               tb = al(sizeof(int2) * sets.size()), bb = al(sizeof(float) * 6 * refit.size()),
               pb = al(sizeof(double) * 10 * refit.size()), hb = al(sizeof(PlHyp) * n_sets),
               ab = al(sizeof(int2) * n_sets), fb = al(sizeof(PlFrame) * n_sets),
               cb = al(sizeof(int32_t) * (size_t)n_sets * cfg->n_hyp);
  int st = sloam_dev_alloc(ctx, &p->d_mem, sb + rb + tb + bb + pb + hb + ab + fb + cb);
  if (!st && n_sets > 0) {
    std::vector<char> tables(sb + rb + tb);
    std::memcpy(tables.data(), score.data(), sizeof(PlChunk) * score.size());
    std::memcpy(tables.data() + sb, refit.data(), sizeof(PlChunk) * refit.size());
    std::memcpy(tables.data() + sb + rb, sets.data(), sizeof(int2) * sets.size());
    const hipError_t e = hipMemcpy(p->d_mem, tables.data(), tables.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) st = sloam_record_hip_error(ctx, e, "hipMemcpy(plane chunks)");
  }
  if (st) {
    sloam_plane_plan_destroy(p);
    return st;
  }
  char* q = static_cast<char*>(p->d_mem);
  auto take = [&](size_t bytes) {
    char* r = q;
    q += bytes;
    return (void*)r;
  };
  p->d_score = (PlChunk*)take(sb);
  p->d_refit = (PlChunk*)take(rb);
  p->d_sets = (int2*)take(tb);
  p->d_box = (float*)take(bb);
  p->d_part = (double*)take(pb);
  p->d_best_hyp = (PlHyp*)take(hb);
  p->d_arrived = (int2*)take(ab);
  p->d_frames = (PlFrame*)take(fb);
  p->d_counts = (int32_t*)take(cb);
  *out = p;
  return SLOAM_OK;
}

void sloam_plane_plan_destroy(sloam_plane_plan* p) {
  if (!p) return;
  sloam_dev_free(p->d_mem);
  delete p;
}

int sloam_plane_plan_exec(sloam_plane_plan* p, const float* d_xyz, const int32_t* d_offsets,
                          int32_t* d_counts, int32_t* d_samples, uint32_t* d_mask,
                          int32_t* d_best, double* d_model) {
  if (!p || !d_offsets || !d_model || (p->n_points > 0 && !d_xyz)) return SLOAM_ERR_INVALID_ARG;
  sloam_ctx* ctx = p->ctx;
  if (p->n_sets == 0) return SLOAM_OK;
  SLOAM_HIP(ctx, hipSetDevice(ctx->device));
  const uint32_t k0 = (uint32_t)p->cfg.seed, k1 = (uint32_t)(p->cfg.seed >> 32);
  const uint32_t tag = (uint32_t)p->cfg.stream_tag;
  int32_t* counts = d_counts ? d_counts : p->d_counts;
  const int H = p->cfg.n_hyp;
  const float thr = p->cfg.thr;
  const dim3 block(kPlB), chunks(p->n_refit);
  {
    SloamKernelScope ks(ctx, "plane_seed");
    hipLaunchKernelGGL(plane_box_kernel, chunks, block, 0, ctx->stream, d_xyz, d_offsets,
                       p->d_refit, H, p->d_box, counts, p->d_arrived, d_mask,
                       (long long)((p->n_points + 31) / 32));
  }
  SLOAM_HIP(ctx, hipGetLastError());
  {
    SloamKernelScope ks(ctx, "plane_score");
    hipLaunchKernelGGL(plane_score_kernel, dim3(p->n_score, (H + kPlHyps - 1) / kPlHyps), block, 0,
                       ctx->stream, d_xyz, d_offsets, p->d_box, p->d_sets, p->d_score, H, thr, k0,
                       k1, tag, p->d_frames, counts, d_samples);
  }
  SLOAM_HIP(ctx, hipGetLastError());
  {
    SloamKernelScope ks(ctx, "plane_refit");
    hipLaunchKernelGGL(plane_refit_kernel, chunks, block, 0, ctx->stream, d_xyz, d_offsets,
                       p->d_frames, p->d_refit, counts, H, thr, k0, k1, tag, p->d_part,
                       p->d_best_hyp, d_mask, d_best, d_model);
    if (p->multi)
      hipLaunchKernelGGL(plane_finish_kernel, chunks, block, 0, ctx->stream, d_xyz, d_offsets,
                         p->d_frames, p->d_sets, p->d_refit, thr, p->d_best_hyp, p->d_part,
                         p->d_arrived, d_model);
  }
  SLOAM_HIP(ctx, hipGetLastError());
  return SLOAM_OK;
}

}  // extern "C"
