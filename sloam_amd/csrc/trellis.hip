// Tree instance front end for gfx950: organized connected components of the
// tree cloud and per-beam tree vertices (sloam/src/segmentation/trellis.cpp:
// 15-132, Instance::findClusters / findTrees / computeVertexProperties).
//
//   tr_tile             connected components inside tiles of 64 x 32 pixels: a
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
//   tr_number           roots ranked in pixel order give the component numbers
//   tr_layout           one workgroup: the components with more than 80
//                       points and their rows.  A component is 4-connected,
//                       so each row of its box is one beam of the tree: no
//                       sort is needed to find them
//   tr_label            (labels asked for) the component number per pixel
//   tr_vertex           a wave per beam: its points in column order,
//                       medians of x, y, z, the points within 0.2 m of the
//                       median in (z, y, x, column) order, radius of the
//                       first / last
//   tr_assemble         one workgroup: vertices per tree (> 16 kept, first
//                       56), tree / vertex / point offsets
//   tr_copy             the vertex records and their kept points to the output
//
// Eight launches and about 77 us at 128 x 2048 with 36,000 tree pixels; a
// union-find over single pixels, ranks by three block scans and a radix sort of
// all pixels by component took nineteen and 220 us.
#include "common.hpp"

#include <algorithm>

namespace {

constexpr int kTB = 256;        // pixel kernels
constexpr int kTileB = 512;     // tile kernel
constexpr int kTileW = 64;      // a wave holds a row of a tile
constexpr int kTileH = 32;
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

// scratch counters: components, beams of the kept components, kept components
enum { kCntComps = 0, kCntSegs, kCntKept, kCntN = 8 };

// A kept component: its first pixel, number, last row, rows; first beam,
// columns; points before it and its beams so far (one counter per component:
// one for all beams serialised them)
struct TrComp {
  int root, id, row1, rows;
  int seg0, col0, col1, alloc;
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

__global__ __launch_bounds__(kTileB) void tr_tile_kernel(const float4* __restrict__ cloud,
                                                      TrCfgDev cfg, int* __restrict__ L, TrBox box,
                                                      int* __restrict__ counters) {
  constexpr int kRows = kTileH / (kTileB / 64);  // rows per wave
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

// The same for up to three counts below 2^21 each, packed.
__device__ inline uint64_t pack3(int a, int b, int c) {
  return (uint64_t)a | ((uint64_t)b << 21) | ((uint64_t)c << 42);
}
__device__ inline int unpack3(uint64_t v, int i) { return (int)((v >> (21 * i)) & 0x1fffff); }

template <int NT>
__device__ inline uint64_t block_excl3(uint64_t v, unsigned long long* wtot, uint64_t* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint64_t s = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t t = __shfl_up((unsigned long long)s, o, 64);
    if (lane >= o) s += t;
  }
  if (lane == 63) wtot[wave] = s;
  __syncthreads();
  uint64_t off = 0, all = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) {
    const uint64_t t = wtot[w];
    off += w < wave ? t : 0;
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
// its kept components' roots, kept[block * kItems ..], and their number.
__global__ __launch_bounds__(kTB) void tr_number_kernel(
    const int* __restrict__ root, TrBox box, TrCfgDev cfg, const int* __restrict__ block_roots,
    int* __restrict__ id, int* __restrict__ kept, int* __restrict__ block_kept,
    int* __restrict__ counters) {
  constexpr int kPer = kItems / kTB;  // consecutive pixels per thread
  __shared__ int wtot[kTB / 64];
  const int base = blockIdx.x * kItems;
  // roots before this block
  int mine = 0;
  for (int b = threadIdx.x; b < (int)blockIdx.x; b += kTB) mine += block_roots[b];
  int run, nk = 0;
  block_excl<kTB>(mine, wtot, &run);
  if (block_roots[blockIdx.x] > 0) {
    const int p0 = base + kPer * (int)threadIdx.x;
    int n = 0;  // roots + 65536 x kept ones
    int size[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      size[j] = p0 + j < cfg.N && root[p0 + j] == p0 + j ? box.size[p0 + j] : -1;
      n += size[j] < 0 ? 0 : (size[j] > cfg.min_label_points ? 65537 : 1);
    }
    int all;
    const int e = block_excl<kTB>(n, wtot, &all);
    int i = run + (e & 65535), k = e >> 16;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      if (size[j] < 0) continue;
      const int p = p0 + j;
      id[p] = i++;
      if (size[j] > cfg.min_label_points) kept[base + k++] = p;
    }
    run += all & 65535;
    nk = all >> 16;
  }
  if (threadIdx.x == 0) {
    block_kept[blockIdx.x] = nk;
    if (blockIdx.x == gridDim.x - 1) counters[kCntComps] = run;
  }
}

// The kept components and their beams in order, one workgroup, a thread per
// component (found by bisection of the blocks' prefix in LDS).  As the last
// workgroup of tr_number, behind a fence in each of its workgroups, this took
// longer than a launch of its own.
__global__ __launch_bounds__(kAsm) void tr_layout_kernel(
    TrBox box, TrCfgDev cfg, int n_blocks, const int* __restrict__ id,
    const int* __restrict__ kept, const int* __restrict__ block_kept, TrComp* __restrict__ comps,
    int* __restrict__ seg_comp, int* __restrict__ counters) {
  __shared__ int wtot[kAsm / 64];
  __shared__ unsigned long long wtot3[kAsm / 64];
  __shared__ int first[kAsm + 1];  // kept components before each block
  const int t = threadIdx.x;
  int K;
  const int e = block_excl<kAsm>(t < n_blocks ? block_kept[t] : 0, wtot, &K);
  first[t] = e;
  if (t == 0) first[kAsm] = K;
  __syncthreads();
  int S = 0, P = 0;
  for (int k0 = 0; k0 < K; k0 += kAsm) {
    const int k = k0 + t;
    TrComp o;
    int size = 0;
    o.rows = 0;
    if (k < K) {
      int lo = 0, hi = kAsm;  // first[lo] <= k < first[hi]
#pragma unroll
      for (int it = 0; it < 10; ++it) {
        const int mid = (lo + hi) >> 1;
        if (first[mid] <= k)
          lo = mid;
        else
          hi = mid;
      }
      const int p = kept[lo * kItems + (k - first[lo])];
      o.root = p;
      o.id = id[p];
      o.row1 = box.row1[p];
      o.rows = o.row1 - p / cfg.W + 1;
      o.col0 = box.col0[p];
      o.col1 = box.col1[p];
      size = box.size[p];
    }
    uint64_t all;
    const uint64_t at = block_excl3<kAsm>(pack3(o.rows, size, 0), wtot3, &all);
    if (k < K) {
      o.seg0 = S + unpack3(at, 0);
      o.alloc = P + unpack3(at, 1);
      comps[k] = o;
      for (int r = 0; r < o.rows; ++r) seg_comp[o.seg0 + r] = k;
    }
    S += unpack3(all, 0);
    P += unpack3(all, 1);
  }
  if (t == 0) {
    counters[kCntKept] = K;
    counters[kCntSegs] = S;
  }
}
static_assert(kAsm == 1024 && (1 << 20) / kItems <= kAsm, "a thread per block, ten bisections");

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

struct BeamLds {
  float4 sp[kSegLds];
  int sc[kSegLds];
  unsigned long long srt[kSegLds];
  unsigned long long keepw[kSegLds / 64];
  int wcount[kTB / 64];
  int base, m;
  float med[3];
  float4 first, last;
};

// A beam by the whole workgroup.  Up to kSegLds points are sorted in LDS;
// longer beams rank every point against all the others from memory.
__device__ inline void beam_block(const float4* __restrict__ cloud, const int* __restrict__ root,
                                  const TrComp& comp, int row, int* alloc, const TrCfgDev& cfg,
                                  SegOut* __restrict__ out, int* __restrict__ cols,
                                  float4* __restrict__ tmp, BeamLds& B) {
  constexpr int kWaves = kTB / 64;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const float4* line = cloud + (size_t)row * cfg.W;
  const int* rline = root + (size_t)row * cfg.W;
  // the beam's points in column order
  auto gather = [&](auto put) {
    int run = 0;
    for (int c0 = comp.col0; c0 <= comp.col1; c0 += kTB) {
      const int c = c0 + t;
      const bool in = c <= comp.col1 && rline[c] == comp.root;
      const uint64_t b = __builtin_amdgcn_ballot_w64(in);
      if (lane == 0) B.wcount[wave] = __builtin_popcountll(b);
      __syncthreads();
      int off = run + __builtin_popcountll(b & ((1ull << lane) - 1ull));
      for (int w = 0; w < kWaves; ++w) {
        off += w < wave ? B.wcount[w] : 0;
        run += B.wcount[w];
      }
      if (in) put(off, c);
      __syncthreads();
    }
    return run;
  };
  const int n = gather([&](int j, int c) {
    if (j < kSegLds) {
      B.sc[j] = c;
      B.sp[j] = line[c];
    }
  });
  const bool in_lds = n <= kSegLds;
  if (t == 0) {
    B.base = atomicAdd(alloc, n);
    B.m = 0;
    B.med[0] = B.med[1] = B.med[2] = 0.f;
  }
  __syncthreads();
  const int base = B.base;
  if (!in_lds) {
    gather([&](int j, int c) { cols[base + j] = c; });
    __syncthreads();
  }
  auto C = [&](int j) -> int { return in_lds ? B.sc[j] : cols[base + j]; };
  auto P = [&](int j) -> float4 { return in_lds ? B.sp[j] : line[cols[base + j]]; };
  // medians: the element of rank floor(n / 2) by (value, index)
  const int mid = n / 2;
  if (!in_lds) {
    for (int i = t; i < n; i += kTB) {
      const float4 v = P(i);
      int rx = 0, ry = 0, rz = 0;
      for (int j = 0; j < n; ++j) {
        const float4 q = P(j);
        rx += (q.x < v.x || (q.x == v.x && j < i)) ? 1 : 0;
        ry += (q.y < v.y || (q.y == v.y && j < i)) ? 1 : 0;
        rz += (q.z < v.z || (q.z == v.z && j < i)) ? 1 : 0;
      }
      if (rx == mid) B.med[0] = v.x;
      if (ry == mid) B.med[1] = v.y;
      if (rz == mid) B.med[2] = v.z;
    }
  } else {
    const int Q = pow2_from(n, 2);
    for (int a = 0; a < 3; ++a) {
      for (int j = t; j < Q; j += kTB)
        B.srt[j] =
            j < n ? ((unsigned long long)order_key(axis_of(B.sp[j], a)) << 32) | (unsigned)j
                  : ~0ull;
      bitonic(B.srt, Q, [](unsigned long long x, unsigned long long y) { return x < y; });
      if (t == 0) B.med[a] = axis_of(B.sp[(uint32_t)B.srt[mid]], a);
      __syncthreads();
    }
  }
  __syncthreads();
  const float med[3] = {B.med[0], B.med[1], B.med[2]};
  auto near = [&](const float4& p) {
    return dist3(p.x, p.y, p.z, med[0], med[1], med[2]) < cfg.max_dist;
  };
  int mw = 0;
  for (int i0 = 0; i0 < n; i0 += kTB) {
    const int i = i0 + t;
    const uint64_t b = __builtin_amdgcn_ballot_w64(i < n && near(P(i)));
    if (in_lds && lane == 0) B.keepw[(i0 >> 6) + wave] = b;
    mw += __builtin_popcountll(b);
  }
  if (lane == 0 && mw) atomicAdd(&B.m, mw);
  __syncthreads();
  const int m = B.m;
  if (m > 1) {
    auto place = [&](int rank, const float4& p) {
      tmp[base + rank] = p;
      if (rank == 0) B.first = p;
      if (rank == m - 1) B.last = p;
    };
    if (in_lds) {
      // kept indices, then sorted (all ones: past the end)
      const int Q = pow2_from(m, 2);
      int before = 0;
      for (int w = 0; w < wave; ++w) before += 64 * w < n ? __builtin_popcountll(B.keepw[w]) : 0;
      for (int i0 = 0; i0 < n; i0 += kTB) {
        const int i = i0 + t;
        const uint64_t b = i0 + 64 * wave < n ? B.keepw[(i0 >> 6) + wave] : 0ull;
        if (i < n && ((b >> lane) & 1ull))
          B.srt[before + __builtin_popcountll(b & ((1ull << lane) - 1ull))] = (unsigned)i;
        for (int w = wave; w < wave + kWaves; ++w)
          before += i0 + 64 * w < n ? __builtin_popcountll(B.keepw[(i0 >> 6) + w]) : 0;
      }
      for (int j = m + t; j < Q; j += kTB) B.srt[j] = ~0ull;
      bitonic(B.srt, Q, [&](unsigned long long x, unsigned long long y) {
        if (x == ~0ull) return false;
        if (y == ~0ull) return true;
        return zless(B.sp[x], B.sc[x], B.sp[y], B.sc[y]);
      });
      for (int j = t; j < m; j += kTB) place(j, B.sp[B.srt[j]]);
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
  }
  if (t == 0) {
    SegOut o;
    o.med = make_float4(med[0], med[1], med[2], 0.f);
    o.radius = m > 1 ? cfg.radius_scale * (double)dist3(B.first.x, B.first.y, B.first.z,
                                                        B.last.x, B.last.y, B.last.z)
                     : 0.0;
    o.valid = m > 1 ? 1 : 0;
    o.m = m;
    o.start = base;
    o.pad = 0;
    *out = o;
  }
  __syncthreads();  // LDS is reused
}

// A beam of n <= kWaveBeam points (LDS, column order, padded with infinities
// to a multiple of kRankStep) by one wave, kWaveBeam / 64 points per lane.
// Every point is ranked against all the others, kRankStep LDS reads in flight
// (the columns increase with the index, so ties go by index).
constexpr int kWaveBeam = 128;
constexpr int kRankStep = 8;
__device__ inline void beam_wave(const float4* sp, int n, int* alloc, const TrCfgDev& cfg,
                                 SegOut* __restrict__ out, float4* __restrict__ tmp) {
  constexpr int kPer = kWaveBeam / 64;
  const int lane = threadIdx.x & 63;
  int base = 0;
  if (lane == 0) base = atomicAdd(alloc, n);
  float4 v[kPer];
#pragma unroll
  for (int u = 0; u < kPer; ++u)
    v[u] = 64 * u + lane < n ? sp[64 * u + lane] : make_float4(NAN, NAN, NAN, 0.f);
  const int mid = n / 2;
  float med[3] = {0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    if (64 * u >= n) break;
    const int i = 64 * u + lane;
    int rx = 0, ry = 0, rz = 0;
    for (int j0 = 0; j0 < n; j0 += kRankStep) {
      float4 q[kRankStep];
#pragma unroll
      for (int e = 0; e < kRankStep; ++e) q[e] = sp[j0 + e];
#pragma unroll
      for (int e = 0; e < kRankStep; ++e) {
        const bool before = j0 + e < i;
        rx += (q[e].x < v[u].x || (q[e].x == v[u].x && before)) ? 1 : 0;
        ry += (q[e].y < v[u].y || (q[e].y == v[u].y && before)) ? 1 : 0;
        rz += (q[e].z < v[u].z || (q[e].z == v[u].z && before)) ? 1 : 0;
      }
    }
    const uint64_t bx = __builtin_amdgcn_ballot_w64(i < n && rx == mid);
    const uint64_t by = __builtin_amdgcn_ballot_w64(i < n && ry == mid);
    const uint64_t bz = __builtin_amdgcn_ballot_w64(i < n && rz == mid);
    if (bx) med[0] = __shfl(v[u].x, (int)__builtin_ctzll(bx), 64);
    if (by) med[1] = __shfl(v[u].y, (int)__builtin_ctzll(by), 64);
    if (bz) med[2] = __shfl(v[u].z, (int)__builtin_ctzll(bz), 64);
  }
  uint64_t keep[kPer];
  int m = 0;
#pragma unroll
  for (int u = 0; u < kPer; ++u) {
    keep[u] = __builtin_amdgcn_ballot_w64(
        64 * u + lane < n &&
        dist3(v[u].x, v[u].y, v[u].z, med[0], med[1], med[2]) < cfg.max_dist);
    m += __builtin_popcountll(keep[u]);
  }
  base = __shfl(base, 0, 64);
  SegOut o;
  o.med = make_float4(med[0], med[1], med[2], 0.f);
  o.radius = 0.0;
  o.valid = 0;
  o.m = m;
  o.start = base;
  o.pad = 0;
  if (m > 1) {
    float4 first = make_float4(0.f, 0.f, 0.f, 0.f), last = first;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      if (keep[u] == 0) continue;
      const int i = 64 * u + lane;
      int rank = 0;
      for (int j0 = 0; j0 < n; j0 += kRankStep) {
        float4 q[kRankStep];
#pragma unroll
        for (int e = 0; e < kRankStep; ++e) q[e] = sp[j0 + e];
#pragma unroll
        for (int e = 0; e < kRankStep; ++e) {
          const int j = j0 + e;
          uint64_t kw = keep[0];
#pragma unroll
          for (int x = 1; x < kPer; ++x) kw = j >= 64 * x ? keep[x] : kw;
          const bool kj = ((kw >> (j & 63)) & 1ull) != 0;  // uniform
          rank += kj && zless(q[e], j, v[u], i) ? 1 : 0;
        }
      }
      const bool mine = ((keep[u] >> lane) & 1ull) != 0;
      if (mine) tmp[base + rank] = v[u];
      const uint64_t bf = __builtin_amdgcn_ballot_w64(mine && rank == 0);
      const uint64_t bl = __builtin_amdgcn_ballot_w64(mine && rank == m - 1);
      if (bf) {
        const int l = (int)__builtin_ctzll(bf);
        first = make_float4(__shfl(v[u].x, l, 64), __shfl(v[u].y, l, 64), __shfl(v[u].z, l, 64),
                            0.f);
      }
      if (bl) {
        const int l = (int)__builtin_ctzll(bl);
        last = make_float4(__shfl(v[u].x, l, 64), __shfl(v[u].y, l, 64), __shfl(v[u].z, l, 64),
                           0.f);
      }
    }
    o.radius = cfg.radius_scale * (double)dist3(first.x, first.y, first.z, last.x, last.y, last.z);
    o.valid = 1;
  }
  if (lane == 0) *out = o;
}

// A wave per beam (component k, one row); beams of more than kWaveBeam points
// (a trunk 1.5 m away covers 180 columns of 2048) then take the workgroup.
// 1,955 beams of a 128 x 2048 scan (half of them under 10 points, the longest
// 68): 23 us, by the longest beams' rank loops; 41 us with a workgroup per beam
// and one counter for the points of all beams, 59 us with a wave per beam and a
// rank loop per axis.
__global__ __launch_bounds__(kTB) void tr_vertex_kernel(
    const float4* __restrict__ cloud, const int* __restrict__ root,
    const int* __restrict__ seg_comp, TrComp* __restrict__ comps,
    const int* __restrict__ counters, TrCfgDev cfg, SegOut* __restrict__ seg_out,
    int* __restrict__ cols, float4* __restrict__ tmp) {
  constexpr int kWaves = kTB / 64;
  __shared__ BeamLds B;
  __shared__ int s_long[kWaves];
  static_assert(kWaves * (kWaveBeam + kRankStep) <= kSegLds, "the waves' parts of the LDS stage");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int S = counters[kCntSegs];
  for (int s0 = blockIdx.x * kWaves; s0 < S; s0 += gridDim.x * kWaves) {
    const int s = s0 + wave;
    int is_long = 0;
    if (s < S) {
      const int k = seg_comp[s];
      const TrComp comp = comps[k];
      const int row = comp.row1 - (s - comp.seg0);
      const float4* line = cloud + (size_t)row * cfg.W;
      const int* rline = root + (size_t)row * cfg.W;
      float4* sp = B.sp + wave * (kWaveBeam + kRankStep);
      int n = 0;
      for (int c0 = comp.col0; c0 <= comp.col1; c0 += 64) {
        const int c = c0 + lane;
        const bool in = c <= comp.col1 && rline[c] == comp.root;
        const uint64_t b = __builtin_amdgcn_ballot_w64(in);
        const int off = n + __builtin_popcountll(b & ((1ull << lane) - 1ull));
        if (in && off < kWaveBeam) sp[off] = line[c];
        n += __builtin_popcountll(b);
      }
      if (n <= cfg.min_row_points) {
        if (lane == 0) {
          SegOut o;
          o.med = make_float4(0.f, 0.f, 0.f, 0.f);
          o.radius = 0.0;
          o.valid = o.m = o.start = o.pad = 0;
          seg_out[s] = o;
        }
      } else if (n <= kWaveBeam) {
        if (lane < kRankStep) sp[n + lane] = make_float4(INFINITY, INFINITY, INFINITY, 0.f);
        __builtin_amdgcn_wave_barrier();
        beam_wave(sp, n, &comps[k].alloc, cfg, seg_out + s, tmp);
      } else {
        is_long = 1;
      }
    }
    if (lane == 0) s_long[wave] = is_long;
    __syncthreads();
    for (int w = 0; w < kWaves; ++w) {
      if (!s_long[w]) continue;
      const int k = seg_comp[s0 + w];
      const TrComp comp = comps[k];
      beam_block(cloud, root, comp, comp.row1 - (s0 + w - comp.seg0), &comps[k].alloc, cfg,
                 seg_out + s0 + w, cols, tmp, B);
    }
    __syncthreads();
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
  __shared__ unsigned long long wtot[kAsm / 64];
  __shared__ int2 s_comp[kAsm];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int K = counters[kCntKept];
  constexpr int kWaves = kAsm / 64;
  constexpr int kAhead = 4;  // components per wave whose loads are in flight
  for (int k0 = wave; k0 < K; k0 += kWaves * kAhead) {
    int s0[kAhead], rows[kAhead], nv[kAhead], np[kAhead], most = 0;
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int k = k0 + u * kWaves;
      s0[u] = k < K ? comps[k].seg0 : 0;
      rows[u] = k < K ? comps[k].rows : 0;
      nv[u] = np[u] = 0;
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u) most = max(most, rows[u]);
    for (int j0 = 0; j0 < most; j0 += 64) {
      const int j = j0 + lane;
      int valid[kAhead], m[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        valid[u] = j < rows[u] ? seg_out[s0[u] + j].valid : 0;
        m[u] = j < rows[u] ? seg_out[s0[u] + j].m : 0;
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const uint64_t b = __builtin_amdgcn_ballot_w64(valid[u] != 0);
        const int rank = nv[u] + __builtin_popcountll(b & ((1ull << lane) - 1ull));
        const bool use = valid[u] && rank < cfg.max_vertices;
        const int incl = wave_incl(use ? m[u] : 0, lane);
        if (j < rows[u])
          seg_at[s0[u] + j] = make_int2(use ? rank : -1, np[u] + incl - (use ? m[u] : 0));
        nv[u] += __builtin_popcountll(b);
        np[u] += __shfl(incl, 63, 64);
      }
    }
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      if (lane == 0 && k0 + u * kWaves < K) {
        if (k0 + u * kWaves < kAsm)
          s_comp[k0 + u * kWaves] = make_int2(nv[u], np[u]);
        else
          comp_at[k0 + u * kWaves] = make_int2(nv[u], np[u]);
      }
  }
  __syncthreads();
  int ct = 0, cv = 0, cp = 0;
  for (int k0 = 0; k0 < K; k0 += kAsm) {
    const int k = k0 + (int)threadIdx.x;
    const int2 v = k >= K ? make_int2(0, 0) : (k < kAsm ? s_comp[k] : comp_at[k]);
    const bool tree = k < K && v.x > cfg.min_vertices;
    uint64_t all;
    const uint64_t e = block_excl3<kAsm>(
        tree ? pack3(1, min(v.x, cfg.max_vertices), v.y) : 0ull, wtot, &all);
    const int vi = cv + unpack3(e, 1), ti = ct + unpack3(e, 0);
    if (k < K) comp_at[k] = make_int2(tree ? vi : -1, cp + unpack3(e, 2));
    if (tree && ti < cfg.cap_trees) tree_offsets[ti] = vi;
    ct += unpack3(all, 0);
    cv += unpack3(all, 1);
    cp += unpack3(all, 2);
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

// The used beams' vertex records and points, one wave per beam; medians
// (nullable): 3 floats per vertex for the line fits.
__global__ __launch_bounds__(64) void tr_copy_kernel(
    const int* __restrict__ seg_comp, const TrComp* __restrict__ comps,
    const int* __restrict__ counters, const SegOut* __restrict__ seg_out,
    const int2* __restrict__ seg_at, const int2* __restrict__ comp_at, TrCfgDev cfg,
    const float4* __restrict__ tmp, int32_t* __restrict__ vertex_int,
    double* __restrict__ vertex_f64, int32_t* __restrict__ point_offsets,
    float4* __restrict__ points, float* __restrict__ medians) {
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
      if (medians) {
        medians[3 * (size_t)vi + 0] = o.med.x;
        medians[3 * (size_t)vi + 1] = o.med.y;
        medians[3 * (size_t)vi + 2] = o.med.z;
      }
    }
    if (po + o.m > cfg.cap_points) continue;
    for (int j = threadIdx.x; j < o.m; j += 64) points[po + j] = tmp[o.start + j];
  }
}

}  // namespace

int sloam_trellis_medians(sloam_ctx* ctx, const float* d_cloud, int32_t height, int32_t width,
                          const sloam_trellis_cfg* cfg, int32_t* d_labels, int32_t cap_trees,
                          int32_t cap_vertices, int32_t cap_points, int32_t* d_tree_offsets,
                          int32_t* d_vertex_int, double* d_vertex_f64, int32_t* d_point_offsets,
                          float* d_points, int32_t* d_counts, float* d_medians) {
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
                      2 * al(sizeof(int) * (size_t)n_blocks) +
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
  int* block_kept = (int*)take(sizeof(int) * (size_t)n_blocks);
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
                         dim3(kTileB), 0, ctx->stream, cloud, dc, L, box, counters);
      if (n_border > 0)
        hipLaunchKernelGGL(tr_border_kernel, dim3((n_border + kTB - 1) / kTB), dim3(kTB), 0,
                           ctx->stream, cloud, dc, L);
      hipLaunchKernelGGL(tr_flatten_kernel, dim3(n_blocks), dim3(kTB), 0, ctx->stream, N, L, root,
                         box, block_roots);
      hipLaunchKernelGGL(tr_number_kernel, dim3(n_blocks), dim3(kTB), 0, ctx->stream, root, box,
                         dc, block_roots, id, kept, block_kept, counters);
      hipLaunchKernelGGL(tr_layout_kernel, dim3(1), dim3(kAsm), 0, ctx->stream, box, dc, n_blocks,
                         id, kept, block_kept, comps, seg_comp, counters);
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
                         reinterpret_cast<float4*>(d_points), d_medians);
  }
  SLOAM_HIP(ctx, hipGetLastError());
  return SLOAM_OK;
}

extern "C" {

int sloam_trellis(sloam_ctx* ctx, const float* d_cloud, int32_t height, int32_t width,
                  const sloam_trellis_cfg* cfg, int32_t* d_labels, int32_t cap_trees,
                  int32_t cap_vertices, int32_t cap_points, int32_t* d_tree_offsets,
                  int32_t* d_vertex_int, double* d_vertex_f64, int32_t* d_point_offsets,
                  float* d_points, int32_t* d_counts) {
  return sloam_trellis_medians(ctx, d_cloud, height, width, cfg, d_labels, cap_trees, cap_vertices,
                               cap_points, d_tree_offsets, d_vertex_int, d_vertex_f64,
                               d_point_offsets, d_points, d_counts, nullptr);
}

}  // extern "C"
