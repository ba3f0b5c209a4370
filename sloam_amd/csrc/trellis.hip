// Tree instance front end for gfx950: organized connected components of the
// tree cloud and per-beam tree vertices (sloam/src/segmentation/trellis.cpp:
// 15-132, Instance::findClusters / findTrees / computeVertexProperties).
//
//   tr_tile             connected components inside tiles of 64 x 16 pixels: a
//                       pixel (finite x) joins its left and upper neighbours
//                       when their float distance is < the cluster threshold;
//                       the runs of a row come from one ballot, the rows are
//                       joined by union-find in LDS.  Each tile component's
//                       first pixel holds its size and bounding box
//   tr_border           unions across the tile borders (global, larger root
//                       under the smaller with atomicMin), so every root is
//                       its component's smallest pixel index, i.e. its first
//                       pixel in row-major order
//   tr_flatten          every pixel's root; the tile components add size and
//                       box to their root's; roots per block
//   tr_number           roots ranked in pixel order give the component
//                       numbers; the last workgroup lists the components with
//                       more than 80 points and their rows.  A component is
//                       4-connected, so each row of its box is one beam of
//                       the tree: no sort is needed to find them
//   tr_label            (labels asked for) the component number per pixel
//   tr_vertex           one workgroup per beam: its points in column order,
//                       medians of x, y, z, the points within 0.2 m of the
//                       median in (z, y, x, column) order, radius of the
//                       first / last
//   tr_assemble         one workgroup: vertices per tree (> 16 kept, first
//                       56), tree / vertex / point offsets
//   tr_copy             the vertex records and their kept points to the output
//
// Seven launches and about 100 us at 128 x 2048 with 36,000 tree pixels; a
// union-find over single pixels, ranks by three block scans and a radix sort of
// all pixels by component took nineteen and 220 us.
#include "common.hpp"

#include <algorithm>

namespace {

constexpr int kTB = 256;        // pixel kernels
constexpr int kTileW = 64;      // a wave holds a row of a tile
constexpr int kTileH = 16;
constexpr int kItems = 1024;    // pixels per block of the root numbering
constexpr int kAsm = 1024;      // assemble workgroup
constexpr int kSegLds = 1024;   // beam points staged in LDS (larger beams read HBM)
constexpr int kVtxBlocks = 2048;  // workgroups of the grid-stride vertex / copy kernels

struct TrCfgDev {
  int H, W, N;
  float thr, max_dist;
  int min_label_points, min_row_points, min_vertices, max_vertices;
  double radius_scale;
  int cap_trees, cap_vertices, cap_points;
};

// scratch counters: components, beams of the kept components, kept
// components, points handed out to beams, workgroups done
enum { kCntComps = 0, kCntSegs, kCntKept, kCntAlloc, kCntDone, kCntN = 8 };

// A kept component: its first pixel, number, last row, rows; first beam, columns.
struct TrComp {
  int root, id, row1, rows;
  int seg0, col0, col1, pad;
};

__device__ inline int ld_relaxed(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline int uf_find(int* L, int a) {
  int p = ld_relaxed(L + a);
  while (p != a) {
    a = p;
    p = ld_relaxed(L + a);
  }
  return a;
}

// Parents only decrease (L[x] <= x); a retry happens only when another lane
// lowered the parent meanwhile, so the loop ends.
__device__ inline void uf_union(int* L, int a, int b) {
  bool done = false;
  while (!done) {
    a = uf_find(L, a);
    b = uf_find(L, b);
    if (a < b) {
      const int old = atomicMin(L + b, a);
      done = (old == b);
      b = old;
    } else if (b < a) {
      const int old = atomicMin(L + a, b);
      done = (old == a);
      a = old;
    } else {
      done = true;
    }
  }
}

// float distance as pcl::euclideanDistance: sqrt((dx^2 + dy^2) + dz^2)
__device__ inline float dist3(float ax, float ay, float az, float bx, float by, float bz) {
  const float dx = ax - bx;
  const float dy = ay - by;
  const float dz = az - bz;
  return sqrtf(dx * dx + dy * dy + dz * dz);
}

__device__ inline bool linked(const float4& a, const float4& b, float thr) {
  return isfinite(a.x) && isfinite(b.x) && dist3(a.x, a.y, a.z, b.x, b.y, b.z) < thr;
}

// union-find over a tile's pixels in LDS, as uf_find / uf_union
__device__ inline int lds_find(int* L, int a) {
  int p = __hip_atomic_load(L + a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  while (p != a) {
    a = p;
    p = __hip_atomic_load(L + a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  return a;
}

__device__ inline void lds_union(int* L, int a, int b) {
  bool done = false;
  while (!done) {
    a = lds_find(L, a);
    b = lds_find(L, b);
    if (a == b) return;
    const int hi = max(a, b), lo = min(a, b);
    const int old = atomicMin(L + hi, lo);
    done = old == hi;
    a = old;
    b = lo;
  }
}

// size (0 except at the first pixel of a tile component), row1 / col0 / col1:
// the component's last row and columns, written at its first pixel only
struct TrBox {
  int* size;
  int* row1;
  int* col0;
  int* col1;
};

// first lane of this lane's run: the highest lane at or below it that is not
// linked to its left (bit 0 of left is 0)
__device__ inline int run_start(uint64_t left, int lane) {
  return 63 - __builtin_clzll(~left & (~0ull >> (63 - lane)));
}

__global__ __launch_bounds__(kTB) void tr_tile_kernel(const float4* __restrict__ cloud,
                                                      TrCfgDev cfg, int* __restrict__ L, TrBox box,
                                                      int* __restrict__ counters) {
  constexpr int kRows = kTileH / (kTB / 64);  // rows per wave
  __shared__ int lab[kTileW * kTileH], size[kTileW * kTileH], row1[kTileW * kTileH],
      col0[kTileW * kTileH], col1[kTileW * kTileH];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = blockIdx.x * kTileW + lane;
  const int r0 = blockIdx.y * kTileH;
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < kCntN) counters[threadIdx.x] = 0;
  auto point = [&](int r) {
    return r >= 0 && r < cfg.H && c < cfg.W ? cloud[(size_t)r * cfg.W + c]
                                            : make_float4(NAN, NAN, NAN, 0.f);
  };
  auto left_bits = [&](const float4& p) {
    float4 q;
    q.x = __shfl_up(p.x, 1, 64);
    q.y = __shfl_up(p.y, 1, 64);
    q.z = __shfl_up(p.z, 1, 64);
    return __builtin_amdgcn_ballot_w64(lane > 0 && linked(p, q, cfg.thr));
  };
  // the wave's rows and the one above them (inside the tile)
  float4 p[kRows + 1];
#pragma unroll
  for (int j = 0; j <= kRows; ++j) {
    const int rl = wave * kRows + j - 1;
    p[j] = rl < 0 ? make_float4(NAN, NAN, NAN, 0.f) : point(r0 + rl);
  }
  uint64_t left[kRows + 1], up[kRows];
#pragma unroll
  for (int j = 0; j <= kRows; ++j) left[j] = left_bits(p[j]);
#pragma unroll
  for (int j = 0; j < kRows; ++j)
    up[j] = __builtin_amdgcn_ballot_w64(linked(p[j + 1], p[j], cfg.thr));
#pragma unroll
  for (int j = 0; j < kRows; ++j) {
    const int l = (wave * kRows + j) * kTileW + lane;
    lab[l] = isfinite(p[j + 1].x) ? (wave * kRows + j) * kTileW + run_start(left[j + 1], lane) : -1;
    size[l] = 0;
    row1[l] = col1[l] = -1;
    col0[l] = kTileW;
  }
  __syncthreads();
  // one union per pair of touching runs: the first linked pixel of each
  // stretch in which both rows' runs go on
#pragma unroll
  for (int j = 0; j < kRows; ++j) {
    const uint64_t again = (up[j] << 1) & left[j + 1] & left[j];
    if (((up[j] & ~again) >> lane) & 1ull) {
      const int r = wave * kRows + j;
      lds_union(lab, r * kTileW + run_start(left[j + 1], lane),
                (r - 1) * kTileW + run_start(left[j], lane));
    }
  }
  __syncthreads();
  int root[kRows];
#pragma unroll
  for (int j = 0; j < kRows; ++j) {
    const int r = wave * kRows + j;
    root[j] = -1;
    if (isfinite(p[j + 1].x)) {
      root[j] = lds_find(lab, r * kTileW + run_start(left[j + 1], lane));
      if (!((left[j + 1] >> lane) & 1ull)) {  // one lane per run
        const int len = 1 + __builtin_ctzll(~((left[j + 1] >> lane) >> 1));
        atomicAdd(&size[root[j]], len);
        atomicMax(&row1[root[j]], r);
        atomicMin(&col0[root[j]], lane);
        atomicMax(&col1[root[j]], lane + len - 1);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kRows; ++j) {
    const int l = (wave * kRows + j) * kTileW + lane, r = r0 + wave * kRows + j;
    if (r >= cfg.H || c >= cfg.W) continue;
    const size_t at = (size_t)r * cfg.W + c;
    const bool first = root[j] == l;
    L[at] = root[j] < 0 ? -1
                        : (r0 + root[j] / kTileW) * cfg.W + (int)blockIdx.x * kTileW +
                              root[j] % kTileW;
    box.size[at] = first ? size[l] : 0;
    if (first) {
      box.row1[at] = r0 + row1[l];
      box.col0[at] = blockIdx.x * kTileW + col0[l];
      box.col1[at] = blockIdx.x * kTileW + col1[l];
    }
  }
}

// thread: a pixel of a tile's first row (below the first tile row) or first
// column (right of the first tile column)
__global__ __launch_bounds__(kTB) void tr_border_kernel(const float4* __restrict__ cloud,
                                                        TrCfgDev cfg, int* L) {
  const int t = blockIdx.x * kTB + threadIdx.x;
  const int rows = (cfg.H - 1) / kTileH, cols = (cfg.W - 1) / kTileW;
  if (t < rows * cfg.W) {
    const int c = t % cfg.W, r = (t / cfg.W + 1) * kTileH;
    const int p = r * cfg.W + c, q = p - cfg.W;
    const float4 a = cloud[p], b = cloud[q];
    if (!linked(a, b, cfg.thr)) return;
    if (c % kTileW != 0) {
      // joined already where both rows' runs and the link go on from the left
      const float4 al = cloud[p - 1], bl = cloud[q - 1];
      if (linked(al, bl, cfg.thr) && linked(a, al, cfg.thr) && linked(b, bl, cfg.thr)) return;
    }
    uf_union(L, p, q);
  } else if (t < rows * cfg.W + cols * cfg.H) {
    const int u = t - rows * cfg.W;
    const int r = u % cfg.H, c = (u / cfg.H + 1) * kTileW;
    const int p = r * cfg.W + c;
    const float4 a = cloud[p], b = cloud[p - 1];
    if (!linked(a, b, cfg.thr)) return;
    if (r % kTileH != 0) {
      const float4 au = cloud[p - cfg.W], bu = cloud[p - cfg.W - 1];
      if (linked(au, bu, cfg.thr) && linked(a, au, cfg.thr) && linked(b, bu, cfg.thr)) return;
    }
    uf_union(L, p, p - 1);
  }
}

// --- ordered compaction helpers (blocks of kItems items) --------------------

// inclusive wave scan
__device__ inline int wave_incl(int v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(v, o, 64);
    if (lane >= o) v += t;
  }
  return v;
}

// exclusive scan over the workgroup (NT threads); *total gets the sum.  All
// threads must call it.
template <int NT>
__device__ inline int block_excl(int v, int* wtot, int* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int s = wave_incl(v, lane);
  if (lane == 63) wtot[wave] = s;
  __syncthreads();
  int off = 0, all = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) {
    const int t = wtot[w];
    off += (w < wave) ? t : 0;
    all += t;
  }
  __syncthreads();
  *total = all;
  return off + s - v;
}

// Roots of kItems pixels per block, and their number.
__global__ __launch_bounds__(kTB) void tr_flatten_kernel(int N, const int* __restrict__ L,
                                                         int* __restrict__ root, TrBox box,
                                                         int* __restrict__ block_roots) {
  __shared__ int wsum[kTB / 64];
  const int base = blockIdx.x * kItems;
  int n = 0;
#pragma unroll
  for (int j = 0; j < kItems / kTB; ++j) {
    const int p = base + j * kTB + (int)threadIdx.x;
    if (p >= N) continue;
    int r = L[p];
    if (r >= 0) {
      for (int q = L[r]; q != r; q = L[r]) r = q;
      n += r == p ? 1 : 0;
      const int sz = box.size[p];
      if (sz > 0 && r != p) {
        atomicAdd(box.size + r, sz);
        atomicMax(box.row1 + r, box.row1[p]);
        atomicMin(box.col0 + r, box.col0[p]);
        atomicMax(box.col1 + r, box.col1[p]);
      }
    }
    root[p] = r;
  }
  for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = n;
  __syncthreads();
  if (threadIdx.x == 0) {
    int t = 0;
    for (int w = 0; w < kTB / 64; ++w) t += wsum[w];
    block_roots[blockIdx.x] = t;
  }
}

// Numbers the roots in pixel order (id, only at the roots); each block lists
// its kept components' roots, kept[block * kItems ..], and their number and
// rows; the last block to finish lays out the components and beams in order.
__global__ __launch_bounds__(kTB) void tr_number_kernel(
    const int* __restrict__ root, TrBox box, TrCfgDev cfg, const int* __restrict__ block_roots,
    int* __restrict__ id, int* __restrict__ kept, int2* __restrict__ block_kept,
    TrComp* __restrict__ comps, int* __restrict__ seg_comp, int* __restrict__ counters) {
  __shared__ int wtot[kTB / 64];
  __shared__ int s_rows, s_last;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int base = blockIdx.x * kItems;
  if (threadIdx.x == 0) s_rows = 0;
  // roots before this block
  int mine = 0;
  for (int b = threadIdx.x; b < (int)blockIdx.x; b += kTB) mine += block_roots[b];
  int run;
  block_excl<kTB>(mine, wtot, &run);
  int nk = 0;
  for (int j0 = 0; j0 < kItems; j0 += kTB) {
    const int p = base + j0 + (int)threadIdx.x;
    const bool is_root = p < cfg.N && root[p] == p;
    int all, all_k;
    const int e = block_excl<kTB>(is_root ? 1 : 0, wtot, &all);
    if (is_root) id[p] = run + e;
    const bool keep = is_root && box.size[p] > cfg.min_label_points;
    const int k = block_excl<kTB>(keep ? 1 : 0, wtot, &all_k);
    if (keep) {
      kept[base + nk + k] = p;
      atomicAdd(&s_rows, box.row1[p] - p / cfg.W + 1);
    }
    run += all;
    nk += all_k;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    block_kept[blockIdx.x] = make_int2(nk, s_rows);
    if (blockIdx.x == gridDim.x - 1) counters[kCntComps] = run;
    __threadfence();
    s_last = atomicAdd(counters + kCntDone, 1) == (int)gridDim.x - 1 ? 1 : 0;
    __threadfence();
  }
  __syncthreads();
  if (!s_last) return;
  int K = 0, S = 0;
  for (int b0 = 0; b0 < (int)gridDim.x; b0 += kTB) {
    const int b = b0 + (int)threadIdx.x;
    const int2 v = b < (int)gridDim.x ? block_kept[b] : make_int2(0, 0);
    int ak, as;
    int k = K + block_excl<kTB>(v.x, wtot, &ak);
    int s = S + block_excl<kTB>(v.y, wtot, &as);
    for (int j = 0; j < v.x; ++j, ++k) {
      const int p = kept[b * kItems + j];
      TrComp o;
      o.root = p;
      o.id = id[p];
      o.row1 = box.row1[p];
      o.rows = o.row1 - p / cfg.W + 1;
      o.seg0 = s;
      o.col0 = box.col0[p];
      o.col1 = box.col1[p];
      o.pad = 0;
      comps[k] = o;
      s += o.rows;
    }
    K += ak;
    S += as;
  }
  if (threadIdx.x == 0) {
    counters[kCntKept] = K;
    counters[kCntSegs] = S;
  }
  __syncthreads();
  for (int k = wave; k < K; k += kTB / 64) {
    const int s0 = comps[k].seg0, rows = comps[k].rows;
    for (int j = lane; j < rows; j += 64) seg_comp[s0 + j] = k;
  }
}

// label[p] = component id of pixel p (-1: no component)
__global__ __launch_bounds__(kTB) void tr_label_kernel(const int* __restrict__ root,
                                                       const int* __restrict__ id, int N,
                                                       int* __restrict__ label) {
  const int p = blockIdx.x * kTB + threadIdx.x;
  if (p >= N) return;
  const int r = root[p];
  label[p] = r < 0 ? -1 : id[r];
}

// --- vertices ----------------------------------------------------------------

struct SegOut {
  float4 med;     // median x, y, z; w unused
  double radius;
  int valid, m;
  int start, pad;  // kept points in tmp
};

// (z, y, x, column) lexicographic order of two beam points
__device__ inline bool zless(const float4& a, int ca, const float4& b, int cb) {
  if (a.z != b.z) return a.z < b.z;
  if (a.y != b.y) return a.y < b.y;
  if (a.x != b.x) return a.x < b.x;
  return ca < cb;
}

__device__ inline float axis_of(const float4& p, int a) { return a == 0 ? p.x : (a == 1 ? p.y : p.z); }

// unsigned key in the order of the floats' <, -0 and +0 equal
__device__ inline uint32_t order_key(float f) {
  const uint32_t u = __float_as_uint(f == 0.0f ? 0.0f : f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Ascending bitonic sort of P (a power of two) items in LDS by the whole
// workgroup; less(a, b) a strict order.  Barriers before, between and after.
template <typename T, typename Less>
__device__ inline void bitonic(T* v, int P, Less less) {
  for (int size = 2; size <= P; size <<= 1)
    for (int step = size >> 1; step > 0; step >>= 1) {
      __syncthreads();
      for (int e = threadIdx.x; e < P / 2; e += kTB) {
        const int a = 2 * e - (e & (step - 1)), b = a + step;
        const T x = v[a], y = v[b];
        const bool up = (a & size) == 0;
        if (up ? less(y, x) : less(x, y)) {
          v[a] = y;
          v[b] = x;
        }
      }
    }
  __syncthreads();
}

__device__ inline int pow2_from(int n, int least) {
  int P = least;
  while (P < n) P <<= 1;
  return P;
}

// One workgroup per beam (component k, one row).  Beams of up to 256 points (a
// trunk 1.5 m away covers 180 columns of 2048) rank every point against all
// the others from LDS, one point per thread; up to kSegLds points are sorted
// in LDS; longer ones rank from memory.  With one wave per beam and a rank
// loop per axis the few longest beams set the kernel's time: 59 us for the
// 1,400 beams of a 128 x 2048 scan.
__global__ __launch_bounds__(kTB) void tr_vertex_kernel(
    const float4* __restrict__ cloud, const int* __restrict__ root,
    const int* __restrict__ seg_comp, const TrComp* __restrict__ comps,
    int* __restrict__ counters, TrCfgDev cfg, SegOut* __restrict__ seg_out,
    int* __restrict__ cols, float4* __restrict__ tmp) {
  constexpr int kWaves = kTB / 64;
  __shared__ float4 sp[kSegLds];
  __shared__ int sc[kSegLds];
  __shared__ unsigned long long srt[kSegLds];
  __shared__ unsigned long long keepw[kSegLds / 64];
  __shared__ int wcount[kWaves];
  __shared__ int s_base, s_m;
  __shared__ float s_med[3];
  __shared__ float4 s_first, s_last;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int S = counters[kCntSegs];
  for (int s = blockIdx.x; s < S; s += gridDim.x) {
    const TrComp comp = comps[seg_comp[s]];
    const int row = comp.row1 - (s - comp.seg0);
    const float4* line = cloud + (size_t)row * cfg.W;
    const int* rline = root + (size_t)row * cfg.W;
    // the beam's points in column order
    auto gather = [&](auto put) {
      int run = 0;
      for (int c0 = comp.col0; c0 <= comp.col1; c0 += kTB) {
        const int c = c0 + t;
        const bool in = c <= comp.col1 && rline[c] == comp.root;
        const uint64_t b = __builtin_amdgcn_ballot_w64(in);
        if (lane == 0) wcount[wave] = __builtin_popcountll(b);
        __syncthreads();
        int off = run + __builtin_popcountll(b & ((1ull << lane) - 1ull));
        for (int w = 0; w < kWaves; ++w) {
          off += w < wave ? wcount[w] : 0;
          run += wcount[w];
        }
        if (in) put(off, c);
        __syncthreads();
      }
      return run;
    };
    const int n = gather([&](int j, int c) {
      if (j < kSegLds) {
        sc[j] = c;
        sp[j] = line[c];
      }
    });
    SegOut o;
    o.med = make_float4(0.f, 0.f, 0.f, 0.f);
    o.radius = 0.0;
    o.valid = 0;
    o.m = 0;
    o.start = 0;
    o.pad = 0;
    if (n > cfg.min_row_points) {
      const bool in_lds = n <= kSegLds;
      if (t == 0) {
        s_base = atomicAdd(counters + kCntAlloc, n);
        s_m = 0;
        s_med[0] = s_med[1] = s_med[2] = 0.f;
      }
      __syncthreads();
      const int base = s_base;
      if (!in_lds) {
        gather([&](int j, int c) { cols[base + j] = c; });
        __syncthreads();
      }
      auto C = [&](int j) -> int { return in_lds ? sc[j] : cols[base + j]; };
      auto P = [&](int j) -> float4 { return in_lds ? sp[j] : line[cols[base + j]]; };
      // medians: the element of rank floor(n / 2) by (value, index)
      const int mid = n / 2;
      if (n <= kTB || !in_lds) {
        for (int i = t; i < n; i += kTB) {
          const float4 v = P(i);
          int rx = 0, ry = 0, rz = 0;
          for (int j = 0; j < n; ++j) {
            const float4 q = P(j);
            rx += (q.x < v.x || (q.x == v.x && j < i)) ? 1 : 0;
            ry += (q.y < v.y || (q.y == v.y && j < i)) ? 1 : 0;
            rz += (q.z < v.z || (q.z == v.z && j < i)) ? 1 : 0;
          }
          if (rx == mid) s_med[0] = v.x;
          if (ry == mid) s_med[1] = v.y;
          if (rz == mid) s_med[2] = v.z;
        }
      } else {
        const int Q = pow2_from(n, 2 * kTB);
        for (int a = 0; a < 3; ++a) {
          for (int j = t; j < Q; j += kTB)
            srt[j] = j < n ? ((unsigned long long)order_key(axis_of(sp[j], a)) << 32) | (unsigned)j
                           : ~0ull;
          bitonic(srt, Q, [](unsigned long long x, unsigned long long y) { return x < y; });
          if (t == 0) s_med[a] = axis_of(sp[(uint32_t)srt[mid]], a);
          __syncthreads();
        }
      }
      __syncthreads();
      const float med[3] = {s_med[0], s_med[1], s_med[2]};
      // kept points
      auto near = [&](const float4& p) {
        return dist3(p.x, p.y, p.z, med[0], med[1], med[2]) < cfg.max_dist;
      };
      int mw = 0;
      for (int i0 = 0; i0 < n; i0 += kTB) {
        const int i = i0 + t;
        const uint64_t b = __builtin_amdgcn_ballot_w64(i < n && near(P(i)));
        if (in_lds && lane == 0) keepw[(i0 >> 6) + wave] = b;
        mw += __builtin_popcountll(b);
      }
      if (lane == 0 && mw) atomicAdd(&s_m, mw);
      __syncthreads();
      const int m = s_m;
      o.med = make_float4(med[0], med[1], med[2], 0.f);
      o.m = m;
      o.start = base;
      if (m > 1) {
        auto place = [&](int rank, const float4& p) {
          tmp[base + rank] = p;
          if (rank == 0) s_first = p;
          if (rank == m - 1) s_last = p;
        };
        if (n <= kTB) {
          if (t < n && ((keepw[wave] >> lane) & 1ull)) {
            const float4 p = sp[t];
            const int ci = sc[t];
            int rank = 0;
            for (int w = 0; w <= (n - 1) >> 6; ++w)
              for (uint64_t b = keepw[w]; b != 0; b &= b - 1) {
                const int j = 64 * w + (int)__builtin_ctzll(b);
                rank += zless(sp[j], sc[j], p, ci) ? 1 : 0;
              }
            place(rank, p);
          }
        } else if (in_lds) {
          // kept indices, then sorted (index -1: past the end)
          const int Q = pow2_from(m, 2);
          int before = 0;
          for (int w = 0; w < wave; ++w) before += __builtin_popcountll(keepw[w]);
          for (int i0 = 0; i0 < n; i0 += kTB) {
            const int i = i0 + t;
            const uint64_t b = i0 + 64 * wave < n ? keepw[(i0 >> 6) + wave] : 0ull;
            if (i < n && ((b >> lane) & 1ull))
              srt[before + __builtin_popcountll(b & ((1ull << lane) - 1ull))] = (unsigned)i;
            for (int w = wave; w < wave + kWaves; ++w)
              before += i0 + 64 * w < n ? __builtin_popcountll(keepw[(i0 >> 6) + w]) : 0;
          }
          for (int j = m + t; j < Q; j += kTB) srt[j] = ~0ull;
          bitonic(srt, Q, [&](unsigned long long x, unsigned long long y) {
            if (x == ~0ull) return false;
            if (y == ~0ull) return true;
            return zless(sp[x], sc[x], sp[y], sc[y]);
          });
          for (int j = t; j < m; j += kTB) place(j, sp[srt[j]]);
        } else {
          for (int i = t; i < n; i += kTB) {
            const float4 p = P(i);
            if (!near(p)) continue;
            const int ci = C(i);
            int rank = 0;
            for (int j = 0; j < n; ++j) {
              const float4 q = P(j);
              if (near(q) && zless(q, C(j), p, ci)) ++rank;
            }
            place(rank, p);
          }
        }
        __syncthreads();
        o.radius = cfg.radius_scale * (double)dist3(s_first.x, s_first.y, s_first.z, s_last.x,
                                                    s_last.y, s_last.z);
        o.valid = 1;
      }
      __syncthreads();  // LDS reused by the next beam
    }
    if (t == 0) seg_out[s] = o;
  }
}

// --- assembly ----------------------------------------------------------------

// One workgroup.  A wave per component ranks its valid vertices and adds up
// their points (the first max_vertices); a scan over the components then
// gives the trees' vertex and point offsets.  Per beam: rank in its tree (-1:
// not used) and first point relative to the tree's; per component: first
// vertex (-1: no tree) and first point.
__global__ __launch_bounds__(kAsm) void tr_assemble_kernel(
    const TrComp* __restrict__ comps, const SegOut* __restrict__ seg_out,
    const int* __restrict__ counters, TrCfgDev cfg, int2* __restrict__ seg_at,
    int2* __restrict__ comp_at, int32_t* __restrict__ tree_offsets,
    int32_t* __restrict__ point_offsets, int32_t* __restrict__ out_counts) {
  __shared__ int wtot[kAsm / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int K = counters[kCntKept];
  for (int k = wave; k < K; k += kAsm / 64) {
    const int s0 = comps[k].seg0, rows = comps[k].rows;
    int nv = 0, np = 0;
    for (int j0 = 0; j0 < rows; j0 += 64) {
      const int j = j0 + lane;
      int valid = 0, m = 0;
      if (j < rows) {
        valid = seg_out[s0 + j].valid;
        m = seg_out[s0 + j].m;
      }
      const uint64_t b = __builtin_amdgcn_ballot_w64(valid != 0);
      const int rank = nv + __builtin_popcountll(b & ((1ull << lane) - 1ull));
      const bool use = valid && rank < cfg.max_vertices;
      const int incl = wave_incl(use ? m : 0, lane);
      if (j < rows) seg_at[s0 + j] = make_int2(use ? rank : -1, np + incl - (use ? m : 0));
      nv += __builtin_popcountll(b);
      np += __shfl(incl, 63, 64);
    }
    if (lane == 0) comp_at[k] = make_int2(nv, np);
  }
  __syncthreads();
  int ct = 0, cv = 0, cp = 0;
  for (int k0 = 0; k0 < K; k0 += kAsm) {
    const int k = k0 + (int)threadIdx.x;
    const int2 v = k < K ? comp_at[k] : make_int2(0, 0);
    const bool tree = k < K && v.x > cfg.min_vertices;
    int at, av, ap;
    const int et = block_excl<kAsm>(tree ? 1 : 0, wtot, &at);
    const int ev = block_excl<kAsm>(tree ? min(v.x, cfg.max_vertices) : 0, wtot, &av);
    const int ep = block_excl<kAsm>(tree ? v.y : 0, wtot, &ap);
    if (k < K) comp_at[k] = make_int2(tree ? cv + ev : -1, cp + ep);
    if (tree && ct + et < cfg.cap_trees) tree_offsets[ct + et] = cv + ev;
    ct += at;
    cv += av;
    cp += ap;
  }
  if (threadIdx.x == 0) {
    const bool over = ct > cfg.cap_trees || cv > cfg.cap_vertices || cp > cfg.cap_points;
    if (!over) {
      tree_offsets[ct] = cv;
      point_offsets[cv] = cp;
    }
    out_counts[0] = ct;
    out_counts[1] = cv;
    out_counts[2] = cp;
    out_counts[3] = counters[kCntComps];
    out_counts[4] = over ? 1 : 0;
    out_counts[5] = counters[kCntSegs];
  }
}

// The used beams' vertex records and points, one wave per beam.
__global__ __launch_bounds__(64) void tr_copy_kernel(
    const int* __restrict__ seg_comp, const TrComp* __restrict__ comps,
    const int* __restrict__ counters, const SegOut* __restrict__ seg_out,
    const int2* __restrict__ seg_at, const int2* __restrict__ comp_at, TrCfgDev cfg,
    const float4* __restrict__ tmp, int32_t* __restrict__ vertex_int,
    double* __restrict__ vertex_f64, int32_t* __restrict__ point_offsets,
    float4* __restrict__ points) {
  const int S = counters[kCntSegs];
  for (int s = blockIdx.x; s < S; s += gridDim.x) {
    const int k = seg_comp[s];
    const int2 a = seg_at[s], b = comp_at[k];
    if (a.x < 0 || b.x < 0) continue;
    const int vi = b.x + a.x, po = b.y + a.y;
    if (vi >= cfg.cap_vertices) continue;
    const SegOut o = seg_out[s];
    if (threadIdx.x == 0) {
      vertex_int[4 * (size_t)vi + 0] = comps[k].id;
      vertex_int[4 * (size_t)vi + 1] = comps[k].row1 - (s - comps[k].seg0);
      vertex_int[4 * (size_t)vi + 2] = o.m;
      vertex_int[4 * (size_t)vi + 3] = 1;
      vertex_f64[4 * (size_t)vi + 0] = o.radius;
      vertex_f64[4 * (size_t)vi + 1] = (double)o.med.x;
      vertex_f64[4 * (size_t)vi + 2] = (double)o.med.y;
      vertex_f64[4 * (size_t)vi + 3] = (double)o.med.z;
      point_offsets[vi] = po;
    }
    if (po + o.m > cfg.cap_points) continue;
    for (int j = threadIdx.x; j < o.m; j += 64) points[po + j] = tmp[o.start + j];
  }
}

}  // namespace

extern "C" {

int sloam_trellis(sloam_ctx* ctx, const float* d_cloud, int32_t height, int32_t width,
                  const sloam_trellis_cfg* cfg, int32_t* d_labels, int32_t cap_trees,
                  int32_t cap_vertices, int32_t cap_points, int32_t* d_tree_offsets,
                  int32_t* d_vertex_int, double* d_vertex_f64, int32_t* d_point_offsets,
                  float* d_points, int32_t* d_counts) {
  if (!ctx || !cfg || !d_counts || height < 0 || width < 0) return SLOAM_ERR_INVALID_ARG;
  if (cap_trees < 0 || cap_vertices < 0 || cap_points < 0) return SLOAM_ERR_INVALID_ARG;
  if (!d_tree_offsets || !d_vertex_int || !d_vertex_f64 || !d_point_offsets ||
      (cap_points > 0 && !d_points))
    return SLOAM_ERR_INVALID_ARG;
  if (cfg->min_row_points < 0 || cfg->max_vertices < 0 || cfg->min_label_points < 0)
    return SLOAM_ERR_INVALID_ARG;
  const long long N64 = (long long)height * (long long)width;
  if (height > 65535 || width > 65535 || N64 >= (1ll << 20)) return SLOAM_ERR_TOO_LARGE;
  const int N = (int)N64;
  if (N > 0 && !d_cloud) return SLOAM_ERR_INVALID_ARG;
  SLOAM_HIP(ctx, hipSetDevice(ctx->device));
  TrCfgDev dc;
  dc.H = height;
  dc.W = width;
  dc.N = N;
  dc.thr = cfg->cluster_dist;
  dc.max_dist = cfg->max_dist_to_centroid;
  dc.min_label_points = cfg->min_label_points;
  dc.min_row_points = cfg->min_row_points;
  dc.min_vertices = cfg->min_vertices;
  dc.max_vertices = cfg->max_vertices;
  dc.radius_scale = cfg->radius_scale;
  dc.cap_trees = cap_trees;
  dc.cap_vertices = cap_vertices;
  dc.cap_points = cap_points;
  const int n1 = std::max(N, 1);
  const int n_blocks = (n1 + kItems - 1) / kItems;
  // kept components hold more than min_label_points pixels each, beams at
  // least one
  const size_t n_comps = (size_t)n1 / ((size_t)dc.min_label_points + 1) + 1;
  auto al = [](size_t x) { return (x + 255) / 256 * 256; };
  const size_t ib = sizeof(int) * (size_t)n1;
  const size_t need = 10 * al(ib) + al(sizeof(int2) * (size_t)n1) +
                      al(sizeof(TrComp) * n_comps) + al(sizeof(int2) * n_comps) +
                      al(sizeof(SegOut) * (size_t)n1) + al(sizeof(float4) * (size_t)n1) +
                      al(sizeof(int) * (size_t)n_blocks) + al(sizeof(int2) * (size_t)n_blocks) +
                      al(sizeof(int) * kCntN);
  void* base = nullptr;
  int st = sloam_ctx_scratch(ctx, 2, need, &base);
  if (st) return st;
  char* q = (char*)base;
  auto take = [&](size_t b) {
    char* r = q;
    q += al(b);
    return (void*)r;
  };
  int* L = (int*)take(ib);
  int* root = (int*)take(ib);
  int* id = (int*)take(ib);
  TrBox box;
  box.size = (int*)take(ib);
  box.row1 = (int*)take(ib);
  box.col0 = (int*)take(ib);
  box.col1 = (int*)take(ib);
  int* kept = (int*)take(ib);
  int* seg_comp = (int*)take(ib);
  int* cols = (int*)take(ib);
  int2* seg_at = (int2*)take(sizeof(int2) * (size_t)n1);
  TrComp* comps = (TrComp*)take(sizeof(TrComp) * n_comps);
  int2* comp_at = (int2*)take(sizeof(int2) * n_comps);
  SegOut* seg_out = (SegOut*)take(sizeof(SegOut) * (size_t)n1);
  float4* tmp = (float4*)take(sizeof(float4) * (size_t)n1);
  int* block_roots = (int*)take(sizeof(int) * (size_t)n_blocks);
  int2* block_kept = (int2*)take(sizeof(int2) * (size_t)n_blocks);
  int* counters = (int*)take(sizeof(int) * kCntN);
  const float4* cloud = reinterpret_cast<const float4*>(d_cloud);
  if (N == 0) {
    st = sloam_fill_u32(ctx, (uint32_t*)counters, kCntN, 0u);
    if (st) return st;
  }
  if (N > 0) {
    {
      SloamKernelScope ks(ctx, "trellis_cc");
      const int n_border =
          (height - 1) / kTileH * width + (width - 1) / kTileW * height;
      hipLaunchKernelGGL(tr_tile_kernel,
                         dim3((width + kTileW - 1) / kTileW, (height + kTileH - 1) / kTileH),
                         dim3(kTB), 0, ctx->stream, cloud, dc, L, box, counters);
      if (n_border > 0)
        hipLaunchKernelGGL(tr_border_kernel, dim3((n_border + kTB - 1) / kTB), dim3(kTB), 0,
                           ctx->stream, cloud, dc, L);
      hipLaunchKernelGGL(tr_flatten_kernel, dim3(n_blocks), dim3(kTB), 0, ctx->stream, N, L, root,
                         box, block_roots);
      hipLaunchKernelGGL(tr_number_kernel, dim3(n_blocks), dim3(kTB), 0, ctx->stream, root, box,
                         dc, block_roots, id, kept, block_kept, comps, seg_comp, counters);
      if (d_labels)
        hipLaunchKernelGGL(tr_label_kernel, dim3((N + kTB - 1) / kTB), dim3(kTB), 0, ctx->stream,
                           root, id, N, d_labels);
    }
    SLOAM_HIP(ctx, hipGetLastError());
    {
      SloamKernelScope ks(ctx, "trellis_vertex");
      hipLaunchKernelGGL(tr_vertex_kernel, dim3(std::min(kVtxBlocks, N)), dim3(kTB), 0,
                         ctx->stream, cloud, root, seg_comp, comps, counters, dc, seg_out, cols,
                         tmp);
    }
    SLOAM_HIP(ctx, hipGetLastError());
  }
  {
    SloamKernelScope ks(ctx, "trellis_assemble");
    hipLaunchKernelGGL(tr_assemble_kernel, dim3(1), dim3(kAsm), 0, ctx->stream, comps, seg_out,
                       counters, dc, seg_at, comp_at, d_tree_offsets, d_point_offsets, d_counts);
    if (N > 0)
      hipLaunchKernelGGL(tr_copy_kernel, dim3(std::min(kVtxBlocks, N)), dim3(64), 0, ctx->stream,
                         seg_comp, comps, counters, seg_out, seg_at, comp_at, dc, tmp,
                         d_vertex_int, d_vertex_f64, d_point_offsets,
                         reinterpret_cast<float4*>(d_points));
  }
  SLOAM_HIP(ctx, hipGetLastError());
  return SLOAM_OK;
}

}  // extern "C"
