// Batched point-level cylinder RANSAC for gfx950.
//
// Three kernels per batch (all on the context stream):
//   cyl_seed    one workgroup per cluster: bounding-box centre m, integer-exact
//               covariance sums, FP64 Jacobi eigen-solve -> seed axis and an
//               FP32 basis (e1, e2) of the plane orthogonal to it.
//   cyl_score   one workgroup per (cluster, hypothesis chunk), clusters largest
//               first: builds the chunk's hypotheses into LDS, streams the
//               cluster's points through LDS tiles as (u, v, s = u^2 + v^2) and
//               counts inliers with a wavefront ballot + popcount, 64 points per
//               compare, eight hypotheses per pass over a tile.
//   cyl_refit   one workgroup per cluster (one wave for small clusters, launches
//               per step for large ones): best hypothesis (max count, lowest
//               index), inlier bit mask, LO-RANSAC refit (Gauss-Newton on the
//               5-parameter geometric cylinder residual with inlier
//               re-selection; FP32 residuals, TwoSum sums, FP64 solve).
//
// The inlier predicate is the reference's point-to-cylinder distance
// (sloam/src/objects/cylinder.cpp:196-203, Cylinder::distance(const PointT&)):
// | ||(p - c) x a|| - r | < thr for a unit axis a.  With (u, v) the coordinates
// of p in the plane orthogonal to a and (cu, cv) the circle centre,
// ||(p - c) x a||^2 = (u - cu)^2 + (v - cv)^2 = s + A u + B v + K with
// A = -2 cu, B = -2 cv, K = cu^2 + cv^2, so the test becomes
// L < fma(u, A, fma(v, B, s)) < U with L = (r - thr)^2 - K (or -inf when
// r <= thr) and U = (r + thr)^2 - K: two FMAs, a clamp and a compare per pair.
#include "common.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <new>
#include <numeric>
#include <tuple>

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kHB = 8;  // hypotheses held in registers per pass over a tile
constexpr int kSeedPts = 8;  // points of a thread in flight in cyl_seed
// clusters from which on the seed axes have a launch of their own (200: 122 us
// for 121 without, 500: 123 / 125, 1200: 127 / 132, 4096: 589 / 606)
constexpr int kAxisClusters = 384;
constexpr int kScoreFill = 2048;  // score workgroups that fill the chip (8 a CU)
constexpr int kMaxLds = 65536;  // LDS bytes per workgroup this kernel asks for

struct CylFrame {
  float m[3];
  float e1[3];
  float e2[3];
  int32_t n;
  double axis[3];
  double reserved;
};

struct HypOut {
  float A, B, L, U;  // predicate parameters
  float cu, cv, r;   // circle in the local frame
  int valid;
};

// the same of a point relative to the frame centre
__device__ inline void rel_uvs(const CylFrame& f, const float d[3], float* u, float* v,
                               float* s) {
  const float uu = (d[0] * f.e1[0] + d[1] * f.e1[1]) + d[2] * f.e1[2];
  const float vv = (d[0] * f.e2[0] + d[1] * f.e2[1]) + d[2] * f.e2[2];
  *u = uu;
  *v = vv;
  *s = uu * uu + vv * vv;
}

__device__ inline void local_uvs(const CylFrame& f, float x, float y, float z, float* u, float* v,
                                 float* s) {
  const float d[3] = {x - f.m[0], y - f.m[1], z - f.m[2]};
  rel_uvs(f, d, u, v, s);
}

// Predicate parameters of the circle (cu, cv, r) of the local plane.
__device__ inline HypOut hyp_from_circle(float cu, float cv, float r, float thr,
                                         float max_radius) {
  HypOut h;
  h.cu = cu;
  h.cv = cv;
  h.r = r;
  h.valid = (r <= max_radius) ? 1 : 0;  // false for NaN / inf (degenerate triangle)
  if (h.valid) {
    h.A = -2.0f * h.cu;
    h.B = -2.0f * h.cv;
    const float K = h.cu * h.cu + h.cv * h.cv;
    const float hi = r + thr;
    h.U = hi * hi - K;
    const float lo = r - thr;
    h.L = lo > 0.0f ? lo * lo - K : -INFINITY;
  } else {
    h.A = 0.0f;
    h.B = 0.0f;
    h.L = INFINITY;
    h.U = -INFINITY;
  }
  return h;
}

// Circumcircle of three points of the local plane and the predicate parameters.
__device__ inline HypOut make_hyp(float ua, float va, float ub, float vb, float uc, float vc,
                                  float thr, float max_radius) {
  const float bx = ub - ua;
  const float by = vb - va;
  const float cx = uc - ua;
  const float cy = vc - va;
  const float d = 2.0f * (bx * cy - by * cx);
  const float b2 = bx * bx + by * by;
  const float c2 = cx * cx + cy * cy;
  const float ox = (cy * b2 - by * c2) / d;
  const float oy = (bx * c2 - cx * b2) / d;
  const float r = sqrtf(ox * ox + oy * oy);
  return hyp_from_circle(ua + ox, va + oy, r, thr, max_radius);
}

// A proposed circle (centre in the local frame, radius) as a hypothesis.
__device__ inline HypOut proposal_hyp(const CylFrame& f, const float* prop, float thr,
                                      float max_radius) {
  float cu, cv, s;
  local_uvs(f, prop[3], prop[4], prop[5], &cu, &cv, &s);
  return hyp_from_circle(cu, cv, prop[6], thr, max_radius);
}

// Hypothesis h of cluster c: the proposal for h == 0 when the cluster has a
// valid one (prop_c != nullptr), else the circumcircle of a Philox sample.
__device__ inline HypOut hyp_for(const float* __restrict__ P, int n, int c, int h,
                                 const CylFrame& f, float thr, float max_radius, uint32_t k0,
                                 uint32_t k1, uint32_t tag, int32_t idx[3],
                                 const float* prop_c) {
  if (prop_c && h == 0) {
    idx[0] = idx[1] = idx[2] = -1;
    return proposal_hyp(f, prop_c, thr, max_radius);
  }
  SlU4 ctr = {(uint32_t)h, (uint32_t)c, tag, 0u};
  const SlU4 x = sl_philox4x32_10(ctr, k0, k1);
  sl_draw3(x.x, x.y, x.z, (uint32_t)n, &idx[0], &idx[1], &idx[2]);
  float u[3], v[3], s;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float* q = P + 3 * (size_t)idx[k];
    local_uvs(f, q[0], q[1], q[2], &u[k], &v[k], &s);
  }
  return make_hyp(u[0], v[0], u[1], v[1], u[2], v[2], thr, max_radius);
}

__device__ inline bool is_inlier(float u, float v, float s, const HypOut& h) {
  const float t = __builtin_fmaf(u, h.A, __builtin_fmaf(v, h.B, s));
  return (t > h.L) && (t < h.U);
}

// ---------------------------------------------------------------------------
// seed: bounding-box centre, integer covariance, FP64 Jacobi, basis
// ---------------------------------------------------------------------------
// prop (nullable): proposals (SLOAM_PN_PROPOSAL_STRIDE floats per cluster);
// a valid proposal's circle, taken into the cluster's seed frame, is
// hypothesis 0.  active (nullable): clusters with active[c] == 0 are skipped.
__device__ inline const float* cluster_prop(const float* prop, int c) {
  if (!prop) return nullptr;
  const float* q = prop + (size_t)c * SLOAM_PN_PROPOSAL_STRIDE;
  return q[7] > 0.0f ? q : nullptr;
}

// Axis and basis of n points from the sums t of their quantised offsets and
// of the products (xx, xy, xz, yy, yz, zz).
__device__ inline void seed_axis(const long long (&t)[9], int n, CylFrame& f) {
  f.n = n;
  f.reserved = 0.0;
  double axis[3] = {0.0, 0.0, 1.0};
  if (n >= 2) {
    const double dn = (double)n;
    const double S0 = (double)t[0], S1 = (double)t[1], S2 = (double)t[2];
    double a6[6];
    a6[0] = (double)t[3] - S0 * S0 / dn;
    a6[1] = (double)t[4] - S0 * S1 / dn;
    a6[2] = (double)t[5] - S0 * S2 / dn;
    a6[3] = (double)t[6] - S1 * S1 / dn;
    a6[4] = (double)t[7] - S1 * S2 / dn;
    a6[5] = (double)t[8] - S2 * S2 / dn;
    double w[3], V[3][3];
    sl_eig3(a6, w, V);
    sl_eigvec(V, sl_argmax3(w), axis);
  }
  double e1[3], e2[3];
  sl_basis(axis, e1, e2);
  for (int k = 0; k < 3; ++k) {
    f.axis[k] = axis[k];
    f.e1[k] = (float)e1[k];
    f.e2[k] = (float)e2[k];
  }
}

// Two passes over the points, kSeedPts of them in flight a thread (one pass
// over memory up to 2048 points), then the eigen-solver, a serial chain of
// about 7 us: sums (nullable) takes the sums instead, and cyl_axis solves a
// large batch a lane each.  13.5e6 points in 1500 clusters (162 MB, the larger
// ones read twice): 121 us with a point in flight and 64-bit products, 66 now;
// 4096 clusters, 4.4e6 points: 59 -> 37; a keyframe's 12: 11.7 -> 9.
//
// order (nullable): the cluster of each workgroup, -1 for padding (the plans'
// largest-first order dealt to the XCDs as the scoring work list deals them,
// so a cluster's points are read through the L2 its scoring will read them
// through); without it workgroup b seeds cluster b
__global__ __launch_bounds__(kBlock) void cyl_seed_kernel(const float* __restrict__ xyz,
                                                          const int32_t* __restrict__ offsets,
                                                          int n_clusters,
                                                          const int32_t* __restrict__ active,
                                                          const int32_t* __restrict__ bcnt,
                                                          CylFrame* __restrict__ frames,
                                                          long long* __restrict__ sums,
                                                          const int32_t* __restrict__ order) {
  __shared__ float red_f[kWaves][6];
  __shared__ long long red_i[kWaves][9];
  const int c = order ? order[blockIdx.x] : (int)blockIdx.x;
  if (c < 0 || c >= n_clusters || (bcnt && c >= bcnt[0])) return;
  if (active && !active[c]) return;
  const int off = offsets[c];
  const int n = offsets[c + 1] - off;
  const float* P = xyz + 3 * (size_t)off;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;

  float mn[3] = {INFINITY, INFINITY, INFINITY};
  float mx[3] = {-INFINITY, -INFINITY, -INFINITY};
  float px[kSeedPts][3];
  // points first + kBlock j + thread; past the end the last point again
  auto load = [&](int first) {
#pragma unroll
    for (int j = 0; j < kSeedPts; ++j) {
      const float* q = P + 3 * (size_t)min(first + kBlock * j + (int)threadIdx.x, n - 1);
#pragma unroll
      for (int k = 0; k < 3; ++k) px[j][k] = q[k];
    }
  };
  for (int first = 0; first < n; first += kBlock * kSeedPts) {
    load(first);
#pragma unroll
    for (int j = 0; j < kSeedPts; ++j)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        mn[k] = fminf(mn[k], px[j][k]);
        mx[k] = fmaxf(mx[k], px[j][k]);
      }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    mn[k] = sl_wave_extreme<false>(mn[k]);
    mx[k] = sl_wave_extreme<true>(mx[k]);
  }
  if (lane == 0) {
    for (int k = 0; k < 3; ++k) {
      red_f[wave][k] = mn[k];
      red_f[wave][3 + k] = mx[k];
    }
  }
  __syncthreads();
  float m[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    float a = red_f[0][k], b = red_f[0][3 + k];
    for (int w = 1; w < kWaves; ++w) {
      a = fminf(a, red_f[w][k]);
      b = fmaxf(b, red_f[w][3 + k]);
    }
    m[k] = n > 0 ? 0.5f * (a + b) : 0.0f;
  }

  // integer-exact sums of q = rint((p - m) * 2^16), |q| < 2^23
  long long s[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int first = 0; first < n; first += kBlock * kSeedPts) {
    if (n > kBlock * kSeedPts) load(first);
    int32_t s1[3] = {0, 0, 0};
#pragma unroll
    for (int j = 0; j < kSeedPts; ++j) {
      if (first + kBlock * j >= n) break;
      int32_t q[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        double d = rint(((double)px[j][k] - (double)m[k]) * 65536.0);
        if (d > 8388607.0) d = 8388607.0;
        if (d < -8388607.0) d = -8388607.0;
        q[k] = first + kBlock * j + (int)threadIdx.x < n ? (int32_t)d : 0;
        s1[k] += q[k];
      }
      s[3] += (int64_t)q[0] * q[0];
      s[4] += (int64_t)q[0] * q[1];
      s[5] += (int64_t)q[0] * q[2];
      s[6] += (int64_t)q[1] * q[1];
      s[7] += (int64_t)q[1] * q[2];
      s[8] += (int64_t)q[2] * q[2];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) s[k] += s1[k];
  }
#pragma unroll
  for (int k = 0; k < 9; ++k) s[k] = sl_wave_sum_i64(s[k]);
  if (lane == 0)
    for (int k = 0; k < 9; ++k) red_i[wave][k] = s[k];
  __syncthreads();
  if (threadIdx.x != 0) return;
  long long t[9];
  for (int k = 0; k < 9; ++k) {
    t[k] = red_i[0][k];
    for (int w = 1; w < kWaves; ++w) t[k] += red_i[w][k];
  }
  if (sums) {
    CylFrame& f = frames[c];
    for (int k = 0; k < 3; ++k) f.m[k] = m[k];
    for (int k = 0; k < 9; ++k) sums[9 * (size_t)c + k] = t[k];
    return;
  }
  CylFrame f;
  for (int k = 0; k < 3; ++k) f.m[k] = m[k];
  seed_axis(t, n, f);
  frames[c] = f;
}

// The axes of a batch whose sums cyl_seed left in `sums`, a lane per cluster.
__global__ __launch_bounds__(64) void cyl_axis_kernel(const int32_t* __restrict__ offsets,
                                                      int n_clusters,
                                                      const int32_t* __restrict__ active,
                                                      const long long* __restrict__ sums,
                                                      CylFrame* __restrict__ frames) {
  const int c = blockIdx.x * 64 + (int)threadIdx.x;
  if (c >= n_clusters || (active && !active[c])) return;
  long long t[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) t[k] = sums[9 * (size_t)c + k];
  CylFrame f = frames[c];
  seed_axis(t, offsets[c + 1] - offsets[c], f);
  frames[c] = f;
}

// ---------------------------------------------------------------------------
// score: hypotheses x points, ballot/popcount inlier counts
//
// L < t < U is tested as med3(t, L', U') == t with L' the next float above L
// and U' the next below U: one VALU instruction and one compare, as two
// compares are, but one lane mask instead of two, so the scalar unit, shared
// by the CU's four SIMDs, has two operations per 64 pairs (count, add) instead
// of three (and).  2000 clusters x 1024 hypotheses, 2.20e9 pairs: 255 -> 227
// us.  (The product on v_mfma_f32_4x4x1_16b, which rounds like fmaf, takes a
// fifth longer: it does not overlap the VALU.)  Bound by VALU issue: the four
// instructions alone, without scalar or LDS work, take 4.8 ns per 64 pairs and
// SIMD (an FMA about two cycles, a clamp or compare about four, two waves' at
// once in part; the clock falls to 2.2 GHz under them).  The whole kernel takes
// 5.4 to 6.0 on 13.5e6 points, where an eighth of its vector instructions make
// hypotheses and local coordinates, and 7.5 on 2.0e6 points.
// work item = {cluster, first hypothesis, hypothesis count, unused}
// LDS: hyp params [hcap] float4 | counts [hcap] int | u,v,s [tile] float
// ---------------------------------------------------------------------------
// The next float above x (NaN and +inf stay).
__device__ inline float next_up(float x) {
  if (!(x < INFINITY)) return x;
  const int b = __float_as_int(x);
  return x == 0.0f ? __int_as_float(1) : __int_as_float(x > 0.0f ? b + 1 : b - 1);
}

// Score parameters {A, B, L', U'} of a hypothesis; one whose band holds no
// float (or that is invalid) gets A = B = 0 and L' = U' = -1: t is then
// s >= 0, never -1.
__device__ inline float4 score_params(const HypOut& h) {
  const float lo = next_up(h.L), hi = -next_up(-h.U);
  return lo <= hi ? make_float4(h.A, h.B, lo, hi) : make_float4(0.f, 0.f, -1.f, -1.f);
}

__global__ __launch_bounds__(kBlock) void cyl_score_kernel(
    const float* __restrict__ xyz, const int32_t* __restrict__ offsets,
    const CylFrame* __restrict__ frames, const int4* __restrict__ work, int n_hyp, int hcap,
    int tile, float thr, float max_radius, uint32_t k0, uint32_t k1, uint32_t tag,
    const float* __restrict__ prop, const int32_t* __restrict__ active,
    const int32_t* __restrict__ bcnt, int32_t* __restrict__ counts,
    int32_t* __restrict__ samples) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  if (bcnt && (int)blockIdx.x >= bcnt[1]) return;  // past the batch's work items
  float4* hp = reinterpret_cast<float4*>(smem_raw);
  int* cnt = reinterpret_cast<int*>(hp + hcap);
  float* su = reinterpret_cast<float*>(cnt + hcap);
  float* sv = su + tile;
  float* ss = sv + tile;

  const int4 w = work[blockIdx.x];
  const int c = w.x, h0 = w.y, hc = w.z;
  if (c < 0) return;  // padding of the per-XCD work order
  if (active && !active[c]) return;
  const float* pc = cluster_prop(prop, c);
  const int off = offsets[c];
  const int n = offsets[c + 1] - off;
  const float* P = xyz + 3 * (size_t)off;
  const CylFrame f = frames[c];

  for (int t = threadIdx.x; t < hcap; t += kBlock) {
    float4 prm = make_float4(0.f, 0.f, -1.f, -1.f);
    if (t < hc && n >= 3) {
      int32_t idx[3];
      const HypOut h = hyp_for(P, n, c, h0 + t, f, thr, max_radius, k0, k1, tag, idx, pc);
      prm = score_params(h);
      if (samples) {
        int32_t* o = samples + 3 * ((size_t)c * n_hyp + h0 + t);
        o[0] = idx[0];
        o[1] = idx[1];
        o[2] = idx[2];
      }
    } else if (t < hc && samples) {
      int32_t* o = samples + 3 * ((size_t)c * n_hyp + h0 + t);
      o[0] = -1;
      o[1] = -1;
      o[2] = -1;
    }
    hp[t] = prm;
    cnt[t] = 0;
  }

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int hpw = hcap / kWaves;  // hypotheses per wave (multiple of kHB)

  for (int t0 = 0; t0 < n; t0 += tile) {
    const int tn = min(tile, n - t0);
    const int tn64 = (tn + 63) & ~63;
    __syncthreads();
    for (int i = threadIdx.x; i < tn64; i += kBlock) {
      float u = 0.f, v = 0.f, s = NAN;
      if (i < tn) {
        const float* q = P + 3 * (size_t)(t0 + i);
        local_uvs(f, q[0], q[1], q[2], &u, &v, &s);
      }
      su[i] = u;
      sv[i] = v;
      ss[i] = s;
    }
    __syncthreads();
    for (int hb = 0; hb < hpw; hb += kHB) {
      const int hbase = wave * hpw + hb;
      if (hbase >= hc) break;
      float A[kHB], B[kHB], L[kHB], U[kHB];
      int cc[kHB];
#pragma unroll
      for (int j = 0; j < kHB; ++j) {
        const float4 q = hp[hbase + j];
        A[j] = q.x;
        B[j] = q.y;
        L[j] = q.z;
        U[j] = q.w;
        cc[j] = 0;
      }
      // uniform trip count: i0 lives in a scalar register, the compares write
      // scalar lane masks that are popcounted on the SALU.  All eight masks
      // before the first count (scheduled mask by mask through one register,
      // each compare waits for the count before it: 48 cycles per 64 pairs).
      for (int i0 = 0; i0 < tn64; i0 += 64) {
        const int i = i0 + lane;
        const float u = su[i];
        const float v = sv[i];
        const float s = ss[i];
        uint64_t in[kHB];
        float t[kHB], m[kHB];
#pragma unroll
        for (int j = 0; j < kHB; ++j) {
          t[j] = __builtin_fmaf(u, A[j], __builtin_fmaf(v, B[j], s));
          m[j] = __builtin_amdgcn_fmed3f(t[j], L[j], U[j]);
        }
#pragma unroll
        for (int j = 0; j < kHB; ++j) in[j] = __builtin_amdgcn_ballot_w64(m[j] == t[j]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kHB; ++j) cc[j] += __builtin_popcountll(in[j]);
      }
      if (lane == 0) {
#pragma unroll
        for (int j = 0; j < kHB; ++j) cnt[hbase + j] += cc[j];
      }
    }
  }
  __syncthreads();
  for (int t = threadIdx.x; t < hc; t += kBlock) counts[(size_t)c * n_hyp + h0 + t] = cnt[t];
}

// ---------------------------------------------------------------------------
// refit: best hypothesis, mask, LO-RANSAC cylinder refit with FP32 residuals
// and Jacobians, compensated FP32 sums and an FP64 5x5 solve.
//
// Rounds of Gauss-Newton steps on the 5-parameter geometric cylinder residual
//   d_i = ||(p_i - c) - ((p_i - c).a) a|| - r
// over the round's inliers: the FP32 inliers of the best hypothesis in round
// 0, |d_i| < thr under the model at the start of the round afterwards.
// Output record: root[3], ray[3], radius, inliers.
//
// Every cluster is cut into chunks of kRefitChunk points; the sums of a step
// are made per chunk by kRefitBlock threads: per point, in FP32, w, h,
// rho = ||w||, d = rho - r, n = w / rho and J = (-h n.e1, -h n.e2, -n.e1,
// -n.e2, -1); each thread adds its points' J J^T and J d terms with FMAs, the
// chunk's threads' values are added with TwoSum in groups of kRefitGroup
// threads (thread order, then group order) into one (sum, error) pair per
// term; the solve adds the chunks' pairs in chunk order and solves the
// normal equations in FP64.  The order of every addition is fixed (no
// atomics on values), so results do not depend on scheduling; the oracle
// restates the same arithmetic.  Two launch forms give the same bits:
//   team      (batches of clusters of up to 8,192 points, one-chunk clusters
//             of the others, and every counted plan)
//             cyl_refit_team: a wave or a workgroup walks every step of one
//             cluster over its chunks, its first wave solving between steps
//   per step  (the other clusters)  cyl_refit_init (best hypothesis, inlier
//             mask, round-0 membership bits, initial model), then per Gauss-Newton
//             step cyl_refit_step (one workgroup per chunk) and
//             cyl_refit_solve (one wave per cluster: lane q sums term q over
//             the chunks, lane 0 solves), then cyl_refit_final (the final
//             inliers' centroid sums per chunk) and cyl_refit_finish (the
//             output record, one wave per cluster)
// The kernels of the per-step form read the previous launch's results (no
// fences between workgroups inside a launch).
// ---------------------------------------------------------------------------
constexpr int kRefitBlock = 256;
constexpr int kRefitPerThread = 8;
constexpr int kRefitChunk = kRefitBlock * kRefitPerThread;
constexpr int kRefitGroup = 32;
constexpr int kRefitGroups = kRefitBlock / kRefitGroup;
constexpr int kRefitTerms = 20;  // 15 of J J^T (upper triangle), 5 of J d
// largest cluster the plans take (points), and its chunks
constexpr int kRefitMaxPoints = 1 << 17;
constexpr int kRefitMaxChunks = kRefitMaxPoints / kRefitChunk;
// A host-planned batch whose clusters have up to this many chunks goes to
// cyl_refit_team.  A batch with larger ones has a launch per step (every chunk
// of every cluster in parallel) for all of several chunks: the launches are
// paid anyway (600 clusters of 2000..12000 points: 334 us for 380 with only
// those above 4 chunks in them; without launches, 2000 clusters of up to 3
// chunks take 336 us, with launches for 3 chunks 395).  Counted plans (a
// keyframe's trees) always take the teams
constexpr int kRefitTeamChunks = 4;
// batches of up to this many clusters have a workgroup for each (four a CU)
constexpr int kRefitTeamBlocks = 1024;
// clusters (one wave each) per workgroup of the per-cluster solve and finish
constexpr int kRefitWaveClusters = 4;

enum RefitStatus : int32_t {
  kRefitActive = 0,    // Gauss-Newton steps continue
  kRefitStopped = 1,   // no more steps (too few inliers, radius <= 0)
  kRefitInvalid = 2,   // record already written as invalid
  kRefitInactive = 3,  // cluster not part of this run
};

// Per-cluster refit state.  The FP32 copy of the model and the basis of the
// plane orthogonal to its axis are made whenever the FP64 model changes.
struct RefitState {
  double a[3], c[3], r;  // axis, axis point (relative to the frame centre), radius
  double e1[3], e2[3];   // basis of the plane orthogonal to the axis
  float af[3], cf[3], rf, e1f[3], e2f[3];
  int32_t status;
  int32_t skip_round;  // round whose remaining steps are skipped (failed solve), -1
  int32_t rounds, iters;
};

struct Comp2 {
  float s, e;  // value s + e
};

// s + e = a + b exactly (TwoSum)
__device__ inline void two_sum(float a, float b, float& s, float& e) {
  s = a + b;
  const float bb = s - a;
  e = (a - (s - bb)) + (b - bb);
}

__device__ inline void comp_add(Comp2& acc, float x) {
  float s, e;
  two_sum(acc.s, x, s, e);
  acc.s = s;
  acc.e = acc.e + e;
}

__device__ inline void comp_add(Comp2& acc, const Comp2& x) {
  float s, e;
  two_sum(acc.s, x.s, s, e);
  acc.s = s;
  acc.e = acc.e + (e + x.e);
}

template <int K>
struct RefitRed {
  float v[K][kRefitGroups][kRefitGroup + 1];  // +1: group chains read distinct banks
  Comp2 grp[K][kRefitGroups];
};

// The chunk's (sum, error) pair of each of K per-thread values, into out[K]
// (global): TwoSum chains over kRefitGroup threads, then over the groups.
template <int K>
__device__ inline void chunk_partial(const float (&g)[K], RefitRed<K>& r, Comp2* out) {
  const int t = threadIdx.x;
  const int tg = t / kRefitGroup, tl = t % kRefitGroup;
#pragma unroll
  for (int k = 0; k < K; ++k) r.v[k][tg][tl] = g[k];
  __syncthreads();
  if (t < K * kRefitGroups) {
    const int k = t / kRefitGroups, q = t % kRefitGroups;
    Comp2 s = {0.0f, 0.0f};
    for (int j = 0; j < kRefitGroup; ++j) comp_add(s, r.v[k][q][j]);
    r.grp[k][q] = s;
  }
  __syncthreads();
  if (t < K) {
    Comp2 s = {0.0f, 0.0f};
#pragma unroll
    for (int q = 0; q < kRefitGroups; ++q) comp_add(s, r.grp[t][q]);
    out[t] = s;
  }
}

// Sum of one int per thread over the workgroup (every thread gets it).
__device__ inline int block_sum_int(int v, int* lds) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  int s = 0;
#pragma unroll
  for (int w = 0; w < kRefitBlock / 64; ++w) s += lds[w];
  return s;
}

// The basis of the FP64 model and the FP32 copy of both.
__device__ inline void refit_model_f32(RefitState& S) {
  sl_basis(S.a, S.e1, S.e2);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    S.af[i] = (float)S.a[i];
    S.cf[i] = (float)S.c[i];
    S.e1f[i] = (float)S.e1[i];
    S.e2f[i] = (float)S.e2[i];
  }
  S.rf = (float)S.r;
}

// Of N points x (relative to the frame centre): w, the part of the offset to
// the model's axis point orthogonal to the axis, h along it, rho = |w| and
// 1 / rho.  Together, so that their chains overlap.
template <int N>
__device__ inline void refit_dist(const RefitState& S, const float (&x)[N][3], float (&w)[N][3],
                                  float (&h)[N], float (&rho)[N], float (&inv)[N]) {
  float ww[N];
  bool ok = true;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const float q0 = x[k][0] - S.cf[0], q1 = x[k][1] - S.cf[1], q2 = x[k][2] - S.cf[2];
    h[k] = __builtin_fmaf(q2, S.af[2], __builtin_fmaf(q1, S.af[1], q0 * S.af[0]));
    w[k][0] = __builtin_fmaf(-h[k], S.af[0], q0);
    w[k][1] = __builtin_fmaf(-h[k], S.af[1], q1);
    w[k][2] = __builtin_fmaf(-h[k], S.af[2], q2);
    ww[k] = __builtin_fmaf(w[k][2], w[k][2], __builtin_fmaf(w[k][1], w[k][1], w[k][0] * w[k][0]));
    ok &= sl_sqrt_inv(ww[k], rho[k], inv[k]);
  }
  if (!ok) {
#pragma unroll
    for (int k = 0; k < N; ++k) sl_sqrt_inv_any(ww[k], rho[k], inv[k]);
  }
}

// Adds an inlier's Jacobian terms (15 of J J^T, 5 of J d) to g.
__device__ inline void refit_add(const RefitState& S, const float (&w)[3], float hh, float inv,
                                 float d, float (&g)[kRefitTerms]) {
  const float n1 =
      __builtin_fmaf(w[2], S.e1f[2], __builtin_fmaf(w[1], S.e1f[1], w[0] * S.e1f[0])) * inv;
  const float n2 =
      __builtin_fmaf(w[2], S.e2f[2], __builtin_fmaf(w[1], S.e2f[1], w[0] * S.e2f[0])) * inv;
  const float J[5] = {-hh * n1, -hh * n2, -n1, -n2, -1.0f};
  int t = 0;
#pragma unroll
  for (int a = 0; a < 5; ++a)
#pragma unroll
    for (int b = a; b < 5; ++b) {
      g[t] = __builtin_fmaf(J[a], J[b], g[t]);
      ++t;
    }
#pragma unroll
  for (int a = 0; a < 5; ++a) g[15 + a] = __builtin_fmaf(J[a], d, g[15 + a]);
}

__device__ inline void write_invalid(double* out, double k) {
  for (int i = 0; i < 6; ++i) out[i] = 0.0;
  out[5] = 1.0;
  out[6] = -1.0;
  out[7] = k;
}

// Refit chunk ck = {cluster, first point (cluster-relative), points, chunk
// index within the cluster}; cluster record cl = {first chunk id, chunks,
// first membership word, 0}.  Membership words: two per 64 points of the
// cluster, written by the wave that owns those 64 points (the team form: a
// byte per thread and chunk).

// First membership word of cluster c, `start` points into the batch: 64 words
// per chunk, at most (start / kRefitChunk + c) chunks before it.
__host__ __device__ inline size_t member_word(int64_t start, int c) {
  return (size_t)(kRefitChunk / 32) * (size_t)(start / kRefitChunk + c);
}

// Ors a wave's 64 bits b into the mask from bit `first` on: a lane for each of
// the (up to three) words, which other waves and clusters share.
__device__ inline void or_mask(uint32_t* __restrict__ mask, int first, uint64_t b) {
  const int lane = threadIdx.x & 63;
  if (b == 0 || lane >= 3) return;
  const uint32_t sh = (uint32_t)first & 31u;
  const uint32_t word = lane == 0   ? (uint32_t)b << sh
                        : lane == 1 ? (uint32_t)((b << sh) >> 32)
                                    : (sh ? (uint32_t)(b >> (64u - sh)) : 0u);
  if (word) atomicOr(mask + (first >> 5) + lane, word);
}

// Round 0: best hypothesis, global mask bits, membership bits, initial model.
// A flagged cluster (alt_flags) takes its hypotheses from the alternate set
// (its own counts, hypothesis count and sample stream, no proposal) and
// refits with the alternate round and step counts.
__global__ __launch_bounds__(kRefitBlock) void cyl_refit_init_kernel(
    const float* __restrict__ xyz, const int32_t* __restrict__ offsets,
    const CylFrame* __restrict__ frames, const int32_t* __restrict__ counts,
    const int4* __restrict__ rchunks, const int4* __restrict__ rclus, int n_hyp, float thr,
    float max_radius, uint32_t k0, uint32_t k1, uint32_t tag, int refit_rounds, int refit_iters,
    const float* __restrict__ prop, const int32_t* __restrict__ active,
    const int32_t* __restrict__ alt_flags, const int32_t* __restrict__ alt_counts, int alt_n_hyp,
    uint32_t alt_tag, int alt_rounds, int alt_iters, RefitState* __restrict__ state,
    uint32_t* __restrict__ member, uint32_t* __restrict__ mask,
    int32_t* __restrict__ best_out, double* __restrict__ model) {
  constexpr int W = kRefitBlock / 64;
  __shared__ long long redk[W];
  __shared__ HypOut best_h;
  const int4 ck = rchunks[blockIdx.x];
  const int c = ck.x;
  if (c < 0) return;  // padding of the per-XCD interleave
  if (active && !active[c]) {
    if (ck.w == 0 && threadIdx.x == 0) state[c].status = kRefitInactive;
    return;
  }
  const int off = offsets[c];
  const int n = offsets[c + 1] - off;
  const float* P = xyz + 3 * (size_t)off;
  const CylFrame f = frames[c];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const bool alt = alt_flags && alt_flags[c];
  const int32_t* cnts = alt ? alt_counts : counts;
  const int nh = alt ? alt_n_hyp : n_hyp;
  const uint32_t tg = alt ? alt_tag : tag;
  const float* pc = alt ? nullptr : cluster_prop(prop, c);

  // best hypothesis: key = count * 2^32 + (2^32 - 1 - index), max wins
  long long key = -1;
  for (int h = threadIdx.x; h < nh; h += kRefitBlock) {
    const long long kk = ((long long)cnts[(size_t)c * nh + h] << 32) |
                         (long long)(0xFFFFFFFFu - (uint32_t)h);
    key = kk > key ? kk : key;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const long long other = __shfl_xor(key, o, 64);
    key = other > key ? other : key;
  }
  if (lane == 0) redk[wave] = key;
  __syncthreads();
  key = redk[0];
#pragma unroll
  for (int w = 1; w < W; ++w) key = redk[w] > key ? redk[w] : key;
  const int best = (n >= 3 && nh > 0) ? (int)(0xFFFFFFFFu - (uint32_t)(key & 0xFFFFFFFFll)) : -1;
  if (threadIdx.x == 0) {
    if (best >= 0) {
      int32_t idx[3];
      best_h = hyp_for(P, n, c, best, f, thr, max_radius, k0, k1, tg, idx, pc);
    } else {
      best_h.valid = 0;
      best_h.A = best_h.B = 0.f;
      best_h.L = INFINITY;
      best_h.U = -INFINITY;
      best_h.cu = best_h.cv = best_h.r = 0.f;
    }
  }
  __syncthreads();
  const HypOut h = best_h;

  // membership bits of the chunk (cluster-relative, 64-aligned per wave) and
  // the global mask's
  const int4 cl = rclus[c];
  uint32_t* mem = member + cl.z;
  const int end = ck.y + ck.z;
  float px[kRefitPerThread][3];
#pragma unroll
  for (int j = 0; j < kRefitPerThread; ++j) {
    const int i = ck.y + kRefitBlock * j + (int)threadIdx.x;
    const float* q = P + 3 * (size_t)min(i, end - 1);
#pragma unroll
    for (int k = 0; k < 3; ++k) px[j][k] = q[k];
  }
#pragma unroll
  for (int j = 0; j < kRefitPerThread; ++j) {
    const int gbase = ck.y + kRefitBlock * j + 64 * wave;  // first point of this wave's group
    float u, v, s;
    local_uvs(f, px[j][0], px[j][1], px[j][2], &u, &v, &s);
    const uint64_t b =
        __builtin_amdgcn_ballot_w64(gbase + lane < end && is_inlier(u, v, s, h));
    if (lane == 0 && gbase < end) {
      mem[gbase >> 5] = (uint32_t)b;
      mem[(gbase >> 5) + 1] = (uint32_t)(b >> 32);
    }
    if (mask) or_mask(mask, off + gbase, b);
  }
  if (ck.w != 0 || threadIdx.x != 0) return;
  // the cluster's first chunk: initial model (the inlier count of the best
  // hypothesis is its score)
  if (best_out) best_out[c] = best;
  RefitState S;
  S.status = kRefitActive;
  S.skip_round = -1;
  S.rounds = alt ? alt_rounds : refit_rounds;
  S.iters = alt ? alt_iters : refit_iters;
  const int kin = best >= 0 ? cnts[(size_t)c * nh + best] : 0;
  if (kin < 3 || !h.valid) {
    S.status = kRefitInvalid;
    write_invalid(model + (size_t)c * SLOAM_CYL_MODEL_STRIDE, (double)kin);
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    S.a[i] = f.axis[i];
    S.c[i] = (double)h.cu * (double)f.e1[i] + (double)h.cv * (double)f.e2[i];
  }
  S.r = (double)h.r;
  refit_model_f32(S);
  state[c] = S;
}

// One Gauss-Newton step's partials of the chunk [first, end) of a cluster
// (points P, frame f, model S, membership bits mem), by all threads of the
// workgroup: the chunk's (sum, error) pairs into out[kRefitTerms] and its
// inlier count into *out_count.  In a re-selecting step the membership bits
// of the chunk are rewritten from the model.
__device__ inline void refit_step_chunk(const float* __restrict__ P, const CylFrame& f,
                                        const RefitState& S, uint32_t* __restrict__ mem,
                                        int first, int end, bool reselect, float thr,
                                        RefitRed<kRefitTerms>& red, int* cnt_w, Comp2* out,
                                        int32_t* out_count) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  float g[kRefitTerms];
#pragma unroll
  for (int q = 0; q < kRefitTerms; ++q) g[q] = 0.0f;
  int cnt = 0;
  // every point of the thread loaded before any is used (the loads overlap)
  float px[kRefitPerThread][3];
#pragma unroll
  for (int j = 0; j < kRefitPerThread; ++j) {
    const int i = first + kRefitBlock * j + (int)threadIdx.x;
    if (i < end) {
      const float* q = P + 3 * (size_t)i;
      px[j][0] = q[0];
      px[j][1] = q[1];
      px[j][2] = q[2];
    } else {
      px[j][0] = px[j][1] = px[j][2] = 0.0f;
    }
  }
#pragma unroll
  for (int j = 0; j < kRefitPerThread; j += 2) {
    __builtin_amdgcn_sched_barrier(0);  // a pair at a time (registers)
    float x[2][3], hh[2], rho[2], inv[2], w[2][3];
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int k = 0; k < 3; ++k) x[e][k] = px[j + e][k] - f.m[k];
    refit_dist<2>(S, x, w, hh, rho, inv);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int gbase = first + kRefitBlock * (j + e) + 64 * wave;
      const int i = gbase + lane;
      const float d = rho[e] - S.rf;
      bool in = false;
      if (i < end)
        in = reselect ? (d < thr && d > -thr) : ((mem[i >> 5] >> (i & 31)) & 1u) != 0u;
      if (reselect) {
        const uint64_t b = __builtin_amdgcn_ballot_w64(in);
        if (lane == 0 && gbase < end) {
          mem[gbase >> 5] = (uint32_t)b;
          mem[(gbase >> 5) + 1] = (uint32_t)(b >> 32);
        }
      }
      if (in) {
        ++cnt;
        if (rho[e] > 0.0f) refit_add(S, w[e], hh[e], inv[e], d, g);
      }
    }
  }
  chunk_partial<kRefitTerms>(g, red, out);
  const int bc = block_sum_int(cnt, cnt_w);
  if (threadIdx.x == 0) *out_count = bc;
}

// Term q of a step's sums over a cluster's nck chunks: the chunks' (sum,
// error) pairs of term q added in chunk order, then sum + error in FP64.
__device__ inline double refit_term(const Comp2* __restrict__ partial, int nck, int q) {
  Comp2 t = {0.0f, 0.0f};
  for (int k = 0; k < nck; ++k) comp_add(t, partial[(size_t)k * kRefitTerms + q]);
  return (double)t.s + (double)t.e;
}

// Sum of one int per lane over a wave (every lane gets it).
__device__ inline int wave_sum_int(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// The Gauss-Newton step's solve of one cluster by one wave: lane q <
// kRefitTerms sums term q over the chunks, then the FP64 5x5 normal equations
// and the next model (lane 0 writes S).  Too few inliers stop the cluster; a
// failed factorisation skips the rest of the round.  The operations and their
// order are a scalar Cholesky's, with a row of the factor per lane (the right
// side is row 5, so the forward substitution is part of it): a column's
// divisions run at once, where one lane made the 25 divisions and roots of
// the step one after the other.
__device__ inline void refit_solve_wave(RefitState& S, const Comp2* part, const int32_t* pc, int nck,
                                        int round) {
  const int lane = threadIdx.x & 63;
  const double mine = lane < kRefitTerms ? refit_term(part, nck, lane) : 0.0;
  int cnt = 0;
  if (nck <= 4) {
    for (int k = 0; k < nck; ++k) cnt += pc[k];
  } else {
    for (int k = lane; k < nck; k += 64) cnt += pc[k];
    cnt = wave_sum_int(cnt);
  }
  if (cnt < 5) {
    if (lane == 0) S.status = kRefitStopped;
    return;
  }
  const int r = min(lane, 5);
  double t, Lr[5], row[5], diag[5];
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    const int lo = min(r, c), hi = max(r, c);
    const double v = __shfl(mine, r == 5 ? 15 + c : lo * 5 - lo * (lo - 1) / 2 + (hi - lo), 64);
    row[c] = r == 5 ? -v : v;
  }
  bool ok = true;
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    t = row[j];
#pragma unroll
    for (int k = 0; k < j; ++k) t = t - Lr[k] * sl_lane_value(Lr[k], j);
    const double s = sl_lane_value(t, j);
    ok = ok && (s > 0.0);
    diag[j] = sqrt(s);
    Lr[j] = t / diag[j];
  }
  if (!ok) {
    if (lane == 0) S.skip_round = round;
    return;
  }
  double x[5];
#pragma unroll
  for (int i = 4; i >= 0; --i) {
    double u = sl_lane_value(Lr[i], 5);
#pragma unroll
    for (int k = i + 1; k < 5; ++k) u = u - sl_lane_value(Lr[i], k) * x[k];
    x[i] = u / diag[i];
  }
  RefitState N = S;
  double na[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) na[i] = N.a[i] + x[0] * N.e1[i] + x[1] * N.e2[i];
  const double nl = sqrt(na[0] * na[0] + na[1] * na[1] + na[2] * na[2]);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    N.a[i] = na[i] / nl;
    N.c[i] = N.c[i] + x[2] * N.e1[i] + x[3] * N.e2[i];
  }
  N.r = N.r + x[4];
  if (!(N.r > 0.0)) N.status = kRefitStopped;
  refit_model_f32(N);
  if (lane == 0) S = N;
}

// The final pass over the chunk [first, end): the chunk sums of the final
// inliers' coordinates (frame-relative) into out[3] and their count.
__device__ inline void refit_final_chunk(const float* __restrict__ P, const CylFrame& f,
                                         const RefitState& S, int first, int end, float thr,
                                         RefitRed<3>& red, int* cnt_w, Comp2* out,
                                         int32_t* out_count) {
  const bool pos = S.r > 0.0;
  float g[3] = {0.0f, 0.0f, 0.0f};
  int cnt = 0;
  if (pos) {
    float px[kRefitPerThread][3];
#pragma unroll
    for (int j = 0; j < kRefitPerThread; ++j) {
      const int i = first + kRefitBlock * j + (int)threadIdx.x;
      if (i < end) {
        const float* q = P + 3 * (size_t)i;
        px[j][0] = q[0];
        px[j][1] = q[1];
        px[j][2] = q[2];
      }
    }
#pragma unroll 2
    for (int j = 0; j < kRefitPerThread; ++j) {
      const int i = first + kRefitBlock * j + (int)threadIdx.x;
      if (i < end) {
        const float x[1][3] = {{px[j][0] - f.m[0], px[j][1] - f.m[1], px[j][2] - f.m[2]}};
        float w[1][3], hh[1], rho[1], inv[1];
        refit_dist<1>(S, x, w, hh, rho, inv);
        const float d = rho[0] - S.rf;
        if (d < thr && d > -thr) {
          g[0] = g[0] + x[0][0];
          g[1] = g[1] + x[0][1];
          g[2] = g[2] + x[0][2];
          ++cnt;
        }
      }
    }
  }
  chunk_partial<3>(g, red, out);
  const int bc = block_sum_int(cnt, cnt_w);
  if (threadIdx.x == 0) *out_count = bc;
}

// The output record of one cluster by one wave from its final pass's chunk
// partials: lanes 0..2 sum the coordinates over the chunks, lane 0 writes
// root (the final inliers' centroid projected on the axis), ray, radius,
// inliers; invalid without a positive radius or three inliers.
__device__ inline void refit_finish_wave(const RefitState& S, const CylFrame& f,
                                         const Comp2* __restrict__ partial,
                                         const int32_t* __restrict__ pcount, int nck,
                                         double* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const double mine = lane < 3 ? refit_term(partial, nck, lane) : 0.0;
  int tot_cnt = 0;
  for (int k = lane; k < nck; k += 64) tot_cnt += pcount[k];
  tot_cnt = wave_sum_int(tot_cnt);
  const double sum[3] = {__shfl(mine, 0, 64), __shfl(mine, 1, 64), __shfl(mine, 2, 64)};
  if (lane != 0) return;
  const double k = (double)tot_cnt;
  if (!(S.r > 0.0) || tot_cnt < 3) {
    write_invalid(out, k);
    return;
  }
  double mean[3];
  for (int i = 0; i < 3; ++i) mean[i] = sum[i] / k;
  const double ht =
      (mean[0] - S.c[0]) * S.a[0] + (mean[1] - S.c[1]) * S.a[1] + (mean[2] - S.c[2]) * S.a[2];
  double ray[3] = {S.a[0], S.a[1], S.a[2]};
  sl_sign_normalise(ray);
  for (int i = 0; i < 3; ++i) {
    out[i] = (double)f.m[i] + S.c[i] + ht * S.a[i];
    out[3 + i] = ray[i];
  }
  out[6] = S.r;
  out[7] = k;
}

// One Gauss-Newton step (launch `step` of the refit: round step / iters,
// iteration step % iters of each cluster's own schedule), one workgroup per
// chunk.
__global__ __launch_bounds__(kRefitBlock) void cyl_refit_step_kernel(
    const float* __restrict__ xyz, const int32_t* __restrict__ offsets,
    const CylFrame* __restrict__ frames, const int4* __restrict__ rchunks,
    const int4* __restrict__ rclus, const RefitState* __restrict__ state,
    uint32_t* __restrict__ member, Comp2* __restrict__ partial, int32_t* __restrict__ pcount,
    int step, float thr) {
  __shared__ RefitRed<kRefitTerms> red;
  __shared__ int cnt_w[kRefitBlock / 64];
  const int4 ck = rchunks[blockIdx.x];
  const int c = ck.x;
  if (c < 0) return;
  const RefitState S = state[c];
  if (S.status != kRefitActive) return;
  if (step >= S.rounds * S.iters) return;
  const int round = step / S.iters, it = step % S.iters;
  if (S.skip_round == round) return;
  const int4 cl = rclus[c];
  const int chunk_id = cl.x + ck.w;
  refit_step_chunk(xyz + 3 * (size_t)offsets[c], frames[c], S, member + cl.z, ck.y, ck.y + ck.z,
                   round > 0 && it == 0, thr, red, cnt_w,
                   partial + (size_t)chunk_id * kRefitTerms, pcount + chunk_id);
}

// The Gauss-Newton step's solve after the step's chunk partials, one wave
// per cluster (kRefitWaveClusters per workgroup).
__global__ __launch_bounds__(64 * kRefitWaveClusters) void cyl_refit_solve_kernel(
    int n_big, const int4* __restrict__ big, const int4* __restrict__ rclus,
    RefitState* __restrict__ state, const Comp2* __restrict__ partial,
    const int32_t* __restrict__ pcount, int step) {
  const int b = blockIdx.x * kRefitWaveClusters + (int)(threadIdx.x >> 6);
  if (b >= n_big) return;
  const int c = big[b].x;
  RefitState S = state[c];
  if (S.status != kRefitActive) return;
  if (step >= S.rounds * S.iters) return;
  const int round = step / S.iters;
  if (S.skip_round == round) return;
  const int4 cl = rclus[c];
  refit_solve_wave(S, partial + (size_t)cl.x * kRefitTerms, pcount + cl.x, cl.y, round);
  if ((threadIdx.x & 63) == 0) state[c] = S;
}

// Final inliers under the final model and their centroid's chunk sums.
__global__ __launch_bounds__(kRefitBlock) void cyl_refit_final_kernel(
    const float* __restrict__ xyz, const int32_t* __restrict__ offsets,
    const CylFrame* __restrict__ frames, const int4* __restrict__ rchunks,
    const int4* __restrict__ rclus, const RefitState* __restrict__ state,
    Comp2* __restrict__ partial, int32_t* __restrict__ pcount, float thr) {
  __shared__ RefitRed<3> red;
  __shared__ int cnt_w[kRefitBlock / 64];
  const int4 ck = rchunks[blockIdx.x];
  const int c = ck.x;
  if (c < 0) return;
  const RefitState S = state[c];
  if (S.status == kRefitInvalid || S.status == kRefitInactive) return;
  const int4 cl = rclus[c];
  const int chunk_id = cl.x + ck.w;
  refit_final_chunk(xyz + 3 * (size_t)offsets[c], frames[c], S, ck.y, ck.y + ck.z, thr, red,
                    cnt_w, partial + (size_t)chunk_id * kRefitTerms, pcount + chunk_id);
}

// The output record of each cluster from the final pass's chunk partials,
// one wave per cluster (kRefitWaveClusters per workgroup).
__global__ __launch_bounds__(64 * kRefitWaveClusters) void cyl_refit_finish_kernel(
    int n_big, const int4* __restrict__ big, const CylFrame* __restrict__ frames,
    const int4* __restrict__ rclus, const RefitState* __restrict__ state,
    const Comp2* __restrict__ partial, const int32_t* __restrict__ pcount,
    double* __restrict__ model) {
  const int b = blockIdx.x * kRefitWaveClusters + (int)(threadIdx.x >> 6);
  if (b >= n_big) return;
  const int c = big[b].x;
  const RefitState S = state[c];
  if (S.status == kRefitInvalid || S.status == kRefitInactive) return;
  const int4 cl = rclus[c];
  refit_finish_wave(S, frames[c], partial + (size_t)cl.x * kRefitTerms, pcount + cl.x, cl.y,
                    model + (size_t)c * SLOAM_CYL_MODEL_STRIDE);
}

// ---------------------------------------------------------------------------
// The whole refit of one cluster by one team of NT threads (a wave or a
// workgroup): best hypothesis, mask, every Gauss-Newton step, final pass and
// output record.  The sums are the per-step form's, value for value: a team
// of 64 plays the 256 threads of a chunk in four turns (virtual thread
// 64 b + lane), sums with no points in them are skipped (TwoSum with zero
// changes nothing), and the 5x5 solve is the same operations with a row per
// lane.
// ---------------------------------------------------------------------------
// a wave takes clusters of up to this many points (up to 256 only: 3000
// clusters of 40..700 points take 166 us for 149, up to 128: 178)
constexpr int kWaveRefit = 512;

template <int NT>
struct TeamLds {
  // rows of 36: a chain reads four values at a time, 16 chains distinct banks
  alignas(16) float v[kRefitTerms][NT / kRefitGroup][kRefitGroup + 4];
  Comp2 grp[kRefitTerms][kRefitGroups];
  Comp2 part[(NT == kRefitBlock ? kRefitMaxChunks : 1) * kRefitTerms];
  int pc[NT == kRefitBlock ? kRefitMaxChunks : 1];
  RefitState S;
  HypOut best;
  long long redk[NT / 64];
  int cnt[NT / 64];
};

// Orders LDS traffic within a team.
template <int NT>
__device__ inline void team_sync() {
  if constexpr (NT == 64) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

// The team's points of the chunk [first, end), relative to the frame centre m:
// px[NVB * J] (turn b, point j of virtual
// thread NT b + t at index b J + j).
template <int NT>
__device__ inline void team_load(const float* __restrict__ P, const float (&m)[3], int first,
                                 int end, float (&px)[kRefitPerThread][3]) {
  constexpr int NVB = kRefitBlock / NT, J = kRefitPerThread / NVB;
  const int t = NT == 64 ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
#pragma unroll
  for (int b = 0; b < NVB; ++b)
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int i = first + kRefitBlock * j + NT * b + t;
      if (i < end) {
        const float* q = P + 3 * (size_t)i;
#pragma unroll
        for (int k = 0; k < 3; ++k) px[b * J + j][k] = q[k] - m[k];
      } else {
        px[b * J + j][0] = px[b * J + j][1] = px[b * J + j][2] = 0.0f;
      }
    }
}

// TwoSum chains over the LDS values of turn b (NT threads' worth of groups).
template <int NT, int K>
__device__ inline void team_chains(TeamLds<NT>& L, int b, int used) {
  constexpr int G = NT / kRefitGroup;  // groups of this turn
  const int t = NT == 64 ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
  if (t < K * G) {
    const int k = t / G, q = t % G;
    Comp2 s = {0.0f, 0.0f};
    if ((NT * b + kRefitGroup * q) < used) {
      const float4* row = reinterpret_cast<const float4*>(L.v[k][q]);
#pragma unroll
      for (int j = 0; j < kRefitGroup / 4; ++j) {
        const float4 x = row[j];
        comp_add(s, x.x);
        comp_add(s, x.y);
        comp_add(s, x.z);
        comp_add(s, x.w);
      }
    }
    L.grp[k][G * b + q] = s;
  }
}

// Chunk partials from the group sums; count = inliers of this wave.
template <int NT, int K>
__device__ inline void team_close(TeamLds<NT>& L, int ck, int count) {
  const int t = NT == 64 ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
  if constexpr (NT != 64)
    if ((t & 63) == 0) L.cnt[t >> 6] = count;
  team_sync<NT>();
  if (t < K) {
    Comp2 s = {0.0f, 0.0f};
#pragma unroll
    for (int q = 0; q < kRefitGroups; ++q) comp_add(s, L.grp[t][q]);
    L.part[ck * kRefitTerms + t] = s;
  }
  if (t == 0) {
    if constexpr (NT != 64) {
      count = 0;
#pragma unroll
      for (int w = 0; w < NT / 64; ++w) count += L.cnt[w];
    }
    L.pc[ck] = count;
  }
}

template <int NT>
__device__ inline void refit_team(const float* __restrict__ xyz, int off, int n, int c,
                                  const CylFrame& f, const int32_t* __restrict__ cnts, int nh,
                                  uint32_t tag, const float* pc_prop, int rounds, int iters,
                                  float thr, float max_radius, uint32_t k0, uint32_t k1,
                                  uint8_t* mem, uint32_t* __restrict__ mask,
                                  int32_t* __restrict__ best_out, double* __restrict__ out,
                                  TeamLds<NT>& L) {
  constexpr int NVB = kRefitBlock / NT, J = kRefitPerThread / NVB, G = J < 4 ? J : 4;
  const int t = NT == 64 ? (int)(threadIdx.x & 63) : (int)threadIdx.x;
  const int lane = t & 63, wave = t >> 6;
  const float* P = xyz + 3 * (size_t)off;
  const int nck = NT == 64 ? 1 : max(1, (n + kRefitChunk - 1) / kRefitChunk);
  if (nck > (NT == 64 ? 1 : kRefitMaxChunks)) return;  // excluded by the plans' cluster bound
  float px[kRefitPerThread][3];
  if (nck == 1) team_load<NT>(P, f.m, 0, n, px);

  // best hypothesis: key = count * 2^32 + (2^32 - 1 - index), max wins
  long long key = -1;
  for (int h = t; h < nh; h += NT) {
    const long long kk =
        ((long long)cnts[h] << 32) | (long long)(0xFFFFFFFFu - (uint32_t)h);
    key = kk > key ? kk : key;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const long long other = __shfl_xor(key, o, 64);
    key = other > key ? other : key;
  }
  if constexpr (NT != 64) {
    if (lane == 0) L.redk[wave] = key;
    __syncthreads();
    key = L.redk[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) key = L.redk[w] > key ? L.redk[w] : key;
  }
  const int best = (n >= 3 && nh > 0) ? (int)(0xFFFFFFFFu - (uint32_t)(key & 0xFFFFFFFFll)) : -1;
  if (wave == 0) {
    // every lane of the wave makes the same hypothesis and model
    HypOut h;
    if (best >= 0) {
      int32_t idx[3];
      h = hyp_for(P, n, c, best, f, thr, max_radius, k0, k1, tag, idx, pc_prop);
    } else {
      h.valid = 0;
      h.A = h.B = 0.f;
      h.L = INFINITY;
      h.U = -INFINITY;
      h.cu = h.cv = h.r = 0.f;
    }
    // the inlier count of the best hypothesis is its score
    const int kin = best >= 0 ? cnts[best] : 0;
    RefitState S;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      S.a[i] = f.axis[i];
      S.c[i] = (double)h.cu * (double)f.e1[i] + (double)h.cv * (double)f.e2[i];
    }
    S.r = (double)h.r;
    S.status = kRefitActive;
    S.skip_round = -1;
    if (kin < 3 || !h.valid) {
      S.status = kRefitInvalid;
      if (lane == 0) write_invalid(out, (double)kin);
    }
    refit_model_f32(S);
    if (lane == 0) {
      L.best = h;
      L.S = S;
      if (best_out) *best_out = best;
    }
  }
  // group sums of turns without points stay zero
  for (int q = t; q < kRefitTerms * kRefitGroups; q += NT)
    L.grp[q / kRefitGroups][q % kRefitGroups] = Comp2{0.0f, 0.0f};
  team_sync<NT>();
  const HypOut h = L.best;

  // round-0 membership: the inliers of the best hypothesis.  bit b J + j of a
  // thread's byte of a chunk; mem holds the bytes of a cluster of several
  uint32_t bits = 0;
#pragma unroll 1
  for (int ck = 0; ck < nck; ++ck) {
    const int first = ck * kRefitChunk, end = min(n, first + kRefitChunk);
    if (nck > 1) team_load<NT>(P, f.m, first, end, px);
    bits = 0;
#pragma unroll
    for (int v = 0; v < kRefitPerThread; ++v) {
      const int i = first + kRefitBlock * (v % J) + NT * (v / J) + t;
      float uu, vv, ss;
      rel_uvs(f, px[v], &uu, &vv, &ss);
      const bool in = i < end && is_inlier(uu, vv, ss, h);
      bits |= in ? 1u << v : 0u;
      if (mask) or_mask(mask, off + i - lane, __builtin_amdgcn_ballot_w64(in));
    }
    if (nck > 1) mem[ck * kRefitBlock + t] = (uint8_t)bits;
  }
  if (L.S.status == kRefitInvalid) return;

  // the FP32 model, uniform over the team
  RefitState M;
  auto fetch = [&]() {
    auto uni = [](float v) {
      return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
    };
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      M.af[i] = uni(L.S.af[i]);
      M.cf[i] = uni(L.S.cf[i]);
      M.e1f[i] = uni(L.S.e1f[i]);
      M.e2f[i] = uni(L.S.e2f[i]);
    }
    M.rf = uni(L.S.rf);
  };
  const int steps = rounds * iters;
  for (int step = 0; step < steps && L.S.status == kRefitActive; ++step) {
    const int round = step / iters, it = step % iters;
    if (L.S.skip_round == round) continue;
    fetch();
    const bool reselect = round > 0 && it == 0;
    for (int ck = 0; ck < nck; ++ck) {
      const int first = ck * kRefitChunk, end = min(n, first + kRefitChunk);
      if (nck > 1) team_load<NT>(P, f.m, first, end, px);
      if (nck > 1) bits = mem[ck * kRefitBlock + t];
      int count = 0;
#pragma unroll
      for (int b = 0; b < NVB; ++b) {
        if (first + NT * b >= end) break;
        float g[kRefitTerms];
#pragma unroll
        for (int q = 0; q < kRefitTerms; ++q) g[q] = 0.0f;
#pragma unroll
        for (int j = 0; j < J; j += G) {
          // G points at a time: more of them in flight take too many registers
          __builtin_amdgcn_sched_barrier(0);
          const int i = first + kRefitBlock * j + NT * b + t, v = b * J + j;
          if (i - t >= end) break;  // no point of the team's turn
          float x[G][3], hh[G], rho[G], inv[G], w[G][3], d[G];
#pragma unroll
          for (int e = 0; e < G; ++e)
#pragma unroll
            for (int k = 0; k < 3; ++k) x[e][k] = px[v + e][k];
          refit_dist<G>(M, x, w, hh, rho, inv);
#pragma unroll
          for (int e = 0; e < G; ++e) d[e] = rho[e] - M.rf;
          if (reselect) {
#pragma unroll
            for (int e = 0; e < G; ++e) {
              const bool in = i + kRefitBlock * e < end && d[e] < thr && d[e] > -thr;
              bits = (bits & ~(1u << (v + e))) | (in ? 1u << (v + e) : 0u);
            }
          }
#pragma unroll
          for (int e = 0; e < G; ++e) {
            const bool in = ((bits >> (v + e)) & 1u) != 0u;
            count += __popcll(__builtin_amdgcn_ballot_w64(in));
            if (in && rho[e] > 0.0f) refit_add(M, w[e], hh[e], inv[e], d[e], g);
          }
        }
        const int tg = t / kRefitGroup, tl = t % kRefitGroup;
        team_sync<NT>();
#pragma unroll
        for (int q = 0; q < kRefitTerms; ++q) L.v[q][tg][tl] = g[q];
        team_sync<NT>();
        team_chains<NT, kRefitTerms>(L, b, end - first);
      }
      if (nck > 1 && reselect) mem[ck * kRefitBlock + t] = (uint8_t)bits;
      team_close<NT, kRefitTerms>(L, ck, count);
    }
    team_sync<NT>();
    if (wave == 0) refit_solve_wave(L.S, L.part, L.pc, nck, round);
    team_sync<NT>();
  }

  // final inliers' centroid and the record
  fetch();
  const bool pos = L.S.r > 0.0;
  for (int ck = 0; ck < nck; ++ck) {
    const int first = ck * kRefitChunk, end = min(n, first + kRefitChunk);
    if (nck > 1) team_load<NT>(P, f.m, first, end, px);
    int count = 0;
#pragma unroll
    for (int b = 0; b < NVB; ++b) {
      if (first + NT * b >= end) break;
      float g[3] = {0.0f, 0.0f, 0.0f};
      if (pos)
#pragma unroll
        for (int j = 0; j < J; j += G) {
          const int i = first + kRefitBlock * j + NT * b + t, v = b * J + j;
          if (i - t >= end) break;
          float x[G][3], hh[G], rho[G], inv[G], w[G][3];
#pragma unroll
          for (int e = 0; e < G; ++e)
#pragma unroll
            for (int k = 0; k < 3; ++k) x[e][k] = px[v + e][k];
          refit_dist<G>(M, x, w, hh, rho, inv);
#pragma unroll
          for (int e = 0; e < G; ++e) {
            const float d = rho[e] - M.rf;
            const bool in = i + kRefitBlock * e < end && d < thr && d > -thr;
            count += __popcll(__builtin_amdgcn_ballot_w64(in));
            if (in) {
#pragma unroll
              for (int k = 0; k < 3; ++k) g[k] = g[k] + x[e][k];
            }
          }
        }
      const int tg = t / kRefitGroup, tl = t % kRefitGroup;
      team_sync<NT>();
#pragma unroll
      for (int q = 0; q < 3; ++q) L.v[q][tg][tl] = g[q];
      team_sync<NT>();
      team_chains<NT, 3>(L, b, end - first);
    }
    team_close<NT, 3>(L, ck, count);
  }
  team_sync<NT>();
  if (wave == 0) {
    refit_finish_wave(L.S, f, L.part, L.pc, nck, out);
  }
}

// The whole refit, one team per cluster.  teams (host plans): per workgroup
// either one cluster {c, -2, ..} or up to four of at most kWaveRefit points
// {c0, c1, c2, c3} (-1: none), a wave each.  Without it workgroup b takes
// cluster b.  A flagged cluster (alt_flags) takes its hypotheses from the
// alternate set and refits with the alternate schedule; clusters not in
// `active` are left alone.
//
// Latency-bound: a step of a 2048-point cluster is 3.0k cycles of distances
// and products, 4k of TwoSum sums, 5k of FP64 solve.  Against a launch per step
// and one per solve: 2000 clusters of 50..5000 points 164 -> 107 us, 4096 of
// them 213 -> 176, 12 clusters of 90..1400 points (were one launch, too)
// 53 -> 35.  In a batch the largest cluster is what ends last (90 us for 3
// chunks); two teams of 1024 threads a CU, or more priority for it, were no
// faster.
__global__ __launch_bounds__(kRefitBlock, 4) void cyl_refit_team_kernel(
    const float* __restrict__ xyz, const int32_t* __restrict__ offsets, int n_clusters,
    const CylFrame* __restrict__ frames, const int32_t* __restrict__ counts,
    const int4* __restrict__ teams, int n_hyp, float thr,
    float max_radius, uint32_t k0, uint32_t k1, uint32_t tag, int refit_rounds, int refit_iters,
    const float* __restrict__ prop, const int32_t* __restrict__ active,
    const int32_t* __restrict__ alt_flags, const int32_t* __restrict__ alt_counts, int alt_n_hyp,
    uint32_t alt_tag, int alt_rounds, int alt_iters, const int32_t* __restrict__ bcnt,
    uint32_t* __restrict__ member, uint32_t* __restrict__ mask, int32_t* __restrict__ best_out,
    double* __restrict__ model) {
  constexpr int kW = kRefitBlock / 64;
  union Lds {
    TeamLds<kRefitBlock> block;
    TeamLds<64> wave[kW];
    __device__ Lds() {}
  };
  __shared__ Lds L;
  int c = blockIdx.x;
  bool by_wave = false;
  if (teams) {
    const int4 tm = teams[blockIdx.x];
    by_wave = tm.y != -2;
    const int w = threadIdx.x >> 6;
    c = !by_wave || w == 0 ? tm.x : (w == 1 ? tm.y : (w == 2 ? tm.z : tm.w));
  }
  c = __builtin_amdgcn_readfirstlane(c);
  if (c < 0 || c >= n_clusters || (bcnt && c >= bcnt[0]) || (active && !active[c])) return;
  const int off = offsets[c];
  const int n = offsets[c + 1] - off;
  const CylFrame f = frames[c];
  const bool alt = alt_flags && alt_flags[c];
  const int nh = alt ? alt_n_hyp : n_hyp;
  const int32_t* cnts = (alt ? alt_counts : counts) + (size_t)c * nh;
  const uint32_t tg = alt ? alt_tag : tag;
  const float* pc = alt ? nullptr : cluster_prop(prop, c);
  const int rounds = alt ? alt_rounds : refit_rounds, iters = alt ? alt_iters : refit_iters;
  int32_t* bo = best_out ? best_out + c : nullptr;
  double* out = model + (size_t)c * SLOAM_CYL_MODEL_STRIDE;
  if (by_wave)
    refit_team<64>(xyz, off, n, c, f, cnts, nh, tg, pc, rounds, iters, thr, max_radius, k0, k1,
                   nullptr, mask, bo, out, L.wave[threadIdx.x >> 6]);
  else
    refit_team<kRefitBlock>(xyz, off, n, c, f, cnts, nh, tg, pc, rounds, iters, thr, max_radius,
                            k0, k1,
                            reinterpret_cast<uint8_t*>(member + member_word(off - offsets[0], c)),
                            mask, bo, out, L.block);
}

}  // namespace

// ---------------------------------------------------------------------------
// plans
// ---------------------------------------------------------------------------
struct sloam_cyl_plan {
  sloam_ctx* ctx = nullptr;
  sloam_cyl_fit_cfg cfg{};
  int32_t n_clusters = 0;
  int64_t n_points = 0;
  int hcap = 0;
  int tile = 0;
  int n_work = 0;
  int4* d_work = nullptr;
  // refit: chunks {cluster, first point, points, chunk index} in launch
  // order, and per cluster {first chunk id, chunks, first membership word, 0}
  int n_rchunks = 0;
  int4* d_rchunks = nullptr;
  int4* d_rclus = nullptr;
  int n_seed = 0;                    // seed workgroups (clusters + padding)
  int32_t* d_seed_order = nullptr;   // their clusters (in d_tables)
  CylFrame* d_frames = nullptr;
  int32_t* d_counts = nullptr;  // used when the caller passes no counts buffer
  int32_t* d_rescue = nullptr;  // per cluster: refitted again by the plain method
  RefitState* d_state = nullptr;
  uint32_t* d_member = nullptr;  // membership bits of the current round
  Comp2* d_partial = nullptr;    // per chunk: kRefitTerms (sum, error) pairs
  int32_t* d_pcount = nullptr;   // per chunk: inliers counted
  int n_xcd = 1;
  // counted plans: the layout is made on the device at every exec from the
  // offsets and the cluster count at d_n (at most cap clusters and
  // cap_points points); n_clusters and n_work are then the grid
  // sizes, d_cnt the batch's own {clusters, work items, refit chunks,
  // overflow}
  bool counted = false;
  // refit: the clusters of cyl_refit_team (largest first), and the large ones
  // (big: their number) with one launch per Gauss-Newton step, whose chunks are
  // d_rchunks; d_big lists them, as teams too (for a few of them at a time)
  int n_teams = 0, n_big = 0;
  int4* d_teams = nullptr;
  int4* d_big = nullptr;
  const int32_t* d_n = nullptr;
  int64_t cap_points = 0;
  int cpc = 0;  // work items per cluster
  int32_t* d_cnt = nullptr;
  // d_work, d_rchunks and d_rclus share one allocation, uploaded in one copy;
  // allocated sizes (bytes for the tables, elements otherwise) only grow
  // across sloam_cyl_plan_reset
  void* d_tables = nullptr;
  size_t cap_tables = 0, cap_frames = 0, cap_counts = 0, cap_state = 0, cap_member = 0,
         cap_partial = 0, cap_rescue = 0;
  // pinned staging of the tables (bytes): their uploads are asynchronous on
  // the context stream, ahead of the runs that read them
  void* h_stage = nullptr;
  size_t cap_stage = 0;
};

static int round_up(int x, int m) { return (x + m - 1) / m * m; }

// Launches the axis seeds of plan p.  The sums of a large batch pass through
// the refit states' memory, which the refit writes later.
static void launch_seed(sloam_cyl_plan* p, const float* d_xyz, const int32_t* d_offsets,
                        const int32_t* d_active) {
  hipStream_t stream = p->ctx->stream;
  const bool ord = !p->counted && p->n_seed > 0;
  static_assert(sizeof(RefitState) >= 9 * sizeof(long long), "sums fit the refit states");
  long long* sums = !p->counted && p->n_clusters >= kAxisClusters
                        ? reinterpret_cast<long long*>(p->d_state)
                        : nullptr;
  hipLaunchKernelGGL(cyl_seed_kernel, dim3(ord ? p->n_seed : p->n_clusters), dim3(kBlock), 0,
                     stream, d_xyz, d_offsets, p->n_clusters, d_active,
                     p->counted ? p->d_cnt : nullptr, p->d_frames, sums,
                     ord ? p->d_seed_order : nullptr);
  if (sums)
    hipLaunchKernelGGL(cyl_axis_kernel, dim3((p->n_clusters + 63) / 64), dim3(64), 0, stream,
                       d_offsets, p->n_clusters, d_active, sums, p->d_frames);
}

// Launches the refit of plan p: one team per cluster, and for the large
// clusters the init pass, one launch per Gauss-Newton step (as many as the
// longest schedule among the clusters) and the final pass.
// alt_flags (nullable) marks the clusters that take their best hypothesis
// from alt_counts (alt_n_hyp hypotheses of sample stream alt_tag, no
// proposal) and refit with alt_rounds x alt_iters steps, instead of counts.
// few: only a few clusters are active, the large ones take a team each too.
static int launch_refit(sloam_cyl_plan* p, const float* d_xyz, const int32_t* d_offsets,
                        const int32_t* counts, const float* d_proposal, const int32_t* d_active,
                        const int32_t* alt_flags, const int32_t* alt_counts, int alt_n_hyp,
                        uint32_t alt_tag, int alt_rounds, int alt_iters, uint32_t* d_mask,
                        int32_t* d_best, double* d_model, bool few = false) {
  sloam_ctx* ctx = p->ctx;
  const sloam_cyl_fit_cfg& cfg = p->cfg;
  if (p->n_clusters == 0) return SLOAM_OK;
  const uint32_t k0 = (uint32_t)cfg.seed;
  const uint32_t k1 = (uint32_t)(cfg.seed >> 32);
  const uint32_t tag = (uint32_t)cfg.stream_tag;
  const dim3 block(kRefitBlock);
  const int32_t* cnt = p->counted ? p->d_cnt : nullptr;
  auto team = [&](const int4* teams, int n) -> int {
    if (n == 0) return SLOAM_OK;
    hipLaunchKernelGGL(cyl_refit_team_kernel, dim3(n), block, 0, ctx->stream, d_xyz, d_offsets,
                       p->n_clusters, p->d_frames, counts, teams, cfg.n_hyp, cfg.thr,
                       cfg.max_radius, k0, k1, tag, cfg.refit_rounds, cfg.refit_iters, d_proposal,
                       d_active, alt_flags, alt_counts, alt_n_hyp, alt_tag, alt_rounds, alt_iters,
                       cnt, p->d_member, d_mask, d_best, d_model);
    SLOAM_HIP(ctx, hipGetLastError());
    return SLOAM_OK;
  };
  if (p->counted) return team(nullptr, p->n_clusters);
  int st = team(p->d_teams, p->n_teams);
  if (st || p->n_big == 0) return st;
  if (few) return team(p->d_big, p->n_big);
  const dim3 grid(p->n_rchunks);
  hipLaunchKernelGGL(cyl_refit_init_kernel, grid, block, 0, ctx->stream, d_xyz, d_offsets,
                     p->d_frames, counts, p->d_rchunks, p->d_rclus, cfg.n_hyp, cfg.thr,
                     cfg.max_radius, k0, k1, tag, cfg.refit_rounds, cfg.refit_iters, d_proposal,
                     d_active, alt_flags, alt_counts, alt_n_hyp, alt_tag, alt_rounds, alt_iters,
                     p->d_state, p->d_member, d_mask, d_best, d_model);
  SLOAM_HIP(ctx, hipGetLastError());
  // one wave per cluster
  const dim3 cgrid((p->n_big + kRefitWaveClusters - 1) / kRefitWaveClusters),
      cblock(64 * kRefitWaveClusters);
  int steps = cfg.refit_rounds * cfg.refit_iters;
  if (alt_flags) steps = std::max(steps, alt_rounds * alt_iters);
  for (int s = 0; s < steps; ++s) {
    hipLaunchKernelGGL(cyl_refit_step_kernel, grid, block, 0, ctx->stream, d_xyz, d_offsets,
                       p->d_frames, p->d_rchunks, p->d_rclus, p->d_state, p->d_member,
                       p->d_partial, p->d_pcount, s, cfg.thr);
    SLOAM_HIP(ctx, hipGetLastError());
    hipLaunchKernelGGL(cyl_refit_solve_kernel, cgrid, cblock, 0, ctx->stream, p->n_big, p->d_big,
                       p->d_rclus, p->d_state, p->d_partial, p->d_pcount, s);
    SLOAM_HIP(ctx, hipGetLastError());
  }
  hipLaunchKernelGGL(cyl_refit_final_kernel, grid, block, 0, ctx->stream, d_xyz, d_offsets,
                     p->d_frames, p->d_rchunks, p->d_rclus, p->d_state, p->d_partial,
                     p->d_pcount, cfg.thr);
  SLOAM_HIP(ctx, hipGetLastError());
  hipLaunchKernelGGL(cyl_refit_finish_kernel, cgrid, cblock, 0, ctx->stream, p->n_big, p->d_big,
                     p->d_frames, p->d_rclus, p->d_state, p->d_partial, p->d_pcount, d_model);
  SLOAM_HIP(ctx, hipGetLastError());
  return SLOAM_OK;
}

// Layout of a counted plan, made on the device: the work list (cluster c's
// hypothesis chunks at c * cpc .. c * cpc + cpc - 1, clusters in index order)
// and cnt = {clusters, work items, refit chunks, overflow}.  A batch beyond the
// capacities, or with a cluster beyond the host plans' bound, sets overflow
// and zero counts (nothing runs).  One workgroup of 256 threads.
__global__ __launch_bounds__(256) void cyl_layout_kernel(
    const int32_t* __restrict__ offsets, const int32_t* __restrict__ d_n, int cap,
    long long cap_points, int n_hyp, int hcap, int cpc, int4* __restrict__ work,
    int32_t* __restrict__ cnt) {
  const int nin = *d_n;
  const int n = min(max(nin, 0), cap);
  bool over = nin > cap || nin < 0;
  __shared__ int chunks;
  if (threadIdx.x == 0) chunks = 0;
  __syncthreads();
  int nck = 0;
  for (int c = threadIdx.x; c < n; c += 256) {
    const int len = offsets[c + 1] - offsets[c];
    over = over || len > kRefitMaxPoints || len < 0;
    nck += max(1, (len + kRefitChunk - 1) / kRefitChunk);
    for (int j = 0; j < cpc; ++j)
      work[(size_t)c * cpc + j] = make_int4(c, j * hcap, min(hcap, n_hyp - j * hcap), len);
  }
  if (nck) atomicAdd(&chunks, nck);
  over = __syncthreads_or(over) ||
         (long long)offsets[n] - (long long)offsets[0] > cap_points;
  if (threadIdx.x == 0) {
    cnt[0] = over ? 0 : n;
    cnt[1] = over ? 0 : n * cpc;
    cnt[2] = over ? 0 : chunks;
    cnt[3] = over ? 1 : 0;
  }
}

// Enqueues the device layout of a counted plan (nothing for other plans).
static int layout_counted(sloam_cyl_plan* p, const int32_t* d_offsets) {
  if (!p->counted) return SLOAM_OK;
  sloam_ctx* ctx = p->ctx;
  hipLaunchKernelGGL(cyl_layout_kernel, dim3(1), dim3(256), 0, ctx->stream, d_offsets, p->d_n,
                     p->n_clusters, (long long)p->cap_points, p->cfg.n_hyp, p->hcap, p->cpc,
                     p->d_work, p->d_cnt);
  SLOAM_HIP(ctx, hipGetLastError());
  return SLOAM_OK;
}

// Fallback flags of the learned fit: a cluster (n >= 3) is refitted by the
// plain method when its best verifying hypothesis holds fewer than
// min_ratio * n inliers.
__global__ __launch_bounds__(256) void cyl_decide_kernel(const int32_t* __restrict__ offsets,
                                                         int n_clusters,
                                                         const int32_t* __restrict__ counts,
                                                         int n_hyp, float min_ratio,
                                                         const int32_t* __restrict__ bcnt,
                                                         int32_t* __restrict__ flags,
                                                         int32_t* __restrict__ n_flagged) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  bool a = false;
  if (c < n_clusters && (!bcnt || c < bcnt[0])) {
    const int n = offsets[c + 1] - offsets[c];
    int best = 0;
    for (int h = 0; h < n_hyp; ++h) best = max(best, counts[(size_t)c * n_hyp + h]);
    a = n >= 3 && (double)best < (double)min_ratio * (double)n;
    flags[c] = a ? 1 : 0;
  }
  const uint64_t b = __builtin_amdgcn_ballot_w64(a);
  if ((threadIdx.x & 63) == 0 && b && n_flagged) atomicAdd(n_flagged, __builtin_popcountll(b));
}

__global__ __launch_bounds__(256) void cyl_fallback_kernel(const int32_t* __restrict__ offsets,
                                                           int n_clusters,
                                                           const double* __restrict__ model,
                                                           float min_ratio,
                                                           int32_t* __restrict__ active,
                                                           int32_t* __restrict__ n_active) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  bool a = false;
  if (c < n_clusters) {
    const int n = offsets[c + 1] - offsets[c];
    const double* m = model + (size_t)c * SLOAM_CYL_MODEL_STRIDE;
    a = n >= 3 && !(m[6] > 0.0 && m[7] >= (double)min_ratio * (double)n);
    active[c] = a ? 1 : 0;
  }
  const uint64_t b = __builtin_amdgcn_ballot_w64(a);
  if ((threadIdx.x & 63) == 0 && b && n_active) atomicAdd(n_active, __builtin_popcountll(b));
}

// Rescue flags of the learned fit, after its refit: a cluster (n >= 3) that
// the verify stage kept is fitted again by the plain method when its refitted
// model is invalid or keeps fewer than min_ratio * n inliers; it joins the
// fallback flags (and their count).
__global__ __launch_bounds__(256) void cyl_rescue_kernel(const int32_t* __restrict__ offsets,
                                                         int n_clusters,
                                                         const double* __restrict__ model,
                                                         float min_ratio,
                                                         const int32_t* __restrict__ bcnt,
                                                         int32_t* __restrict__ fallback,
                                                         int32_t* __restrict__ rescue,
                                                         int32_t* __restrict__ n_flagged) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  bool a = false;
  if (c < n_clusters) {
    if (!bcnt || c < bcnt[0]) {
      const int n = offsets[c + 1] - offsets[c];
      const double* m = model + (size_t)c * SLOAM_CYL_MODEL_STRIDE;
      a = fallback[c] == 0 && n >= 3 && !(m[6] > 0.0 && m[7] >= (double)min_ratio * (double)n);
      if (a) fallback[c] = 1;
    }
    rescue[c] = a ? 1 : 0;
  }
  const uint64_t b = __builtin_amdgcn_ballot_w64(a);
  if ((threadIdx.x & 63) == 0 && b && n_flagged) atomicAdd(n_flagged, __builtin_popcountll(b));
}

// Grows the device buffer *ptr (element size elem) to hold n elements;
// contents are not kept.
static int grow(sloam_ctx* ctx, void** ptr, size_t* cap, size_t n, size_t elem) {
  if (n <= *cap) return SLOAM_OK;
  sloam_dev_free(*ptr);
  *ptr = nullptr;
  *cap = 0;
  const int st = sloam_dev_alloc(ctx, ptr, n * elem);
  if (st) return st;
  *cap = n;
  return SLOAM_OK;
}

// Lays the batch h_offsets (n_clusters + 1 entries) out on plan p, whose cfg,
// hcap and tile are set: the scoring work list and the refit chunks,
// uploaded into buffers that only grow.
static int plan_layout(sloam_cyl_plan* p, const int32_t* h_offsets, int32_t n_clusters) {
  sloam_ctx* ctx = p->ctx;
  const sloam_cyl_fit_cfg& cfg = p->cfg;
  if (h_offsets[0] != 0) return SLOAM_ERR_INVALID_ARG;
  for (int i = 0; i < n_clusters; ++i) {
    const int64_t len = (int64_t)h_offsets[i + 1] - h_offsets[i];
    if (len < 0) return SLOAM_ERR_INVALID_ARG;
    if (len > kRefitMaxPoints) return SLOAM_ERR_TOO_LARGE;  // integer-exact covariance bound
  }
  p->n_clusters = n_clusters;
  p->n_points = h_offsets[n_clusters];
  if (cfg.hyp_chunk == 0) {
    // no chunk asked for: 256 hypotheses a workgroup (each workgroup takes the
    // cluster's points into the local frame, for all its hypotheses), fewer
    // where that would leave CUs idle, down to one pass of each wave.  12
    // trees x 1024 hypotheses: 48 workgroups took 34 us, 384 take 8.  (Counted
    // plans, laid out for their capacity, keep 256; a chunk that is asked for
    // stays, as the 128 of the drop-in's tree fits and the autotuner's choices,
    // of which 64 is the smallest.)
    const int least = kWaves * kHB;
    p->hcap = std::min(256, round_up(cfg.n_hyp, least));
    while (p->hcap > least &&
           (int64_t)n_clusters * ((cfg.n_hyp + p->hcap - 1) / p->hcap) < kScoreFill)
      p->hcap = round_up(p->hcap / 2, least);
  }

  // work list: clusters by decreasing size (ties: lower index), each cluster
  // split into hypothesis chunks.  Workgroups go to the XCDs round robin
  // (workgroup b on XCD b mod n_xcd), each XCD with its own L2: clusters are
  // dealt to per-XCD bins by least load (largest first) and the launch order
  // interleaves the bins, so all chunks of a cluster run on one XCD and read
  // its points through one L2.  Bins are padded with empty items (cluster -1).
  std::vector<int> order(n_clusters);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
    return (h_offsets[a + 1] - h_offsets[a]) > (h_offsets[b + 1] - h_offsets[b]);
  });
  const int n_xcd = p->n_xcd;
  const int chunks = (cfg.n_hyp + p->hcap - 1) / p->hcap;
  std::vector<std::vector<int4>> bins(n_xcd);
  std::vector<long long> load(n_xcd, 0);
  for (int c : order) {
    const int len = h_offsets[c + 1] - h_offsets[c];
    const int x = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    for (int h0 = 0; h0 < cfg.n_hyp; h0 += p->hcap) {
      const int hc = std::min(p->hcap, cfg.n_hyp - h0);
      bins[x].push_back(make_int4(c, h0, hc, len));
    }
    load[x] += (long long)std::max(len, 1) * chunks;
  }
  // the seed: one workgroup per cluster, in each bin's order, bins interleaved
  std::vector<std::vector<int32_t>> sbins(n_xcd);
  for (int x = 0; x < n_xcd; ++x)
    for (const int4& w : bins[x])
      if (sbins[x].empty() || sbins[x].back() != w.x) sbins[x].push_back(w.x);
  size_t slongest = 0;
  for (const auto& b : sbins) slongest = std::max(slongest, b.size());
  std::vector<int32_t> seed;
  seed.reserve(slongest * n_xcd);
  for (size_t k = 0; k < slongest; ++k)
    for (int x = 0; x < n_xcd; ++x) seed.push_back(k < sbins[x].size() ? sbins[x][k] : -1);
  p->n_seed = (int)seed.size();
  size_t longest = 0;
  for (const auto& b : bins) longest = std::max(longest, b.size());
  std::vector<int4> work;
  work.reserve(longest * n_xcd);
  for (size_t k = 0; k < longest; ++k)
    for (int x = 0; x < n_xcd; ++x)
      work.push_back(k < bins[x].size() ? bins[x][k] : make_int4(-1, 0, 0, 0));
  p->n_work = (int)work.size();
  // refit chunks: every cluster (even an empty one) has at least one; the
  // clusters are dealt to per-XCD bins as above and the bins interleaved, so
  // all chunks of a cluster run on one XCD
  std::vector<std::vector<int4>> rbins(n_xcd);
  std::vector<long long> rload(n_xcd, 0);
  std::vector<int4> rclus(n_clusters);
  int n_chunk_ids = 0;
  for (int c = 0; c < n_clusters; ++c) {
    const int len = h_offsets[c + 1] - h_offsets[c];
    const int nck = std::max(1, (len + kRefitChunk - 1) / kRefitChunk);
    rclus[c] = make_int4(n_chunk_ids, nck, (int)member_word(h_offsets[c], c), 0);
    n_chunk_ids += nck;
  }
  const size_t n_words = member_word(h_offsets[n_clusters], n_clusters);
  int team_chunks = 0;
  for (int c = 0; c < n_clusters; ++c) team_chunks = std::max(team_chunks, rclus[c].y);
  if (team_chunks > kRefitTeamChunks) team_chunks = 1;
  std::vector<int4> big;
  for (int c : order) {
    const int len = h_offsets[c + 1] - h_offsets[c];
    if (rclus[c].y <= team_chunks) continue;
    big.push_back(make_int4(c, -2, 0, 0));
    const int x = (int)(std::min_element(rload.begin(), rload.end()) - rload.begin());
    for (int k = 0; k < rclus[c].y; ++k) {
      const int first = k * kRefitChunk;
      rbins[x].push_back(make_int4(c, first, std::min(kRefitChunk, len - first), k));
    }
    rload[x] += std::max(len, 1);
  }
  size_t rlongest = 0;
  for (const auto& b : rbins) rlongest = std::max(rlongest, b.size());
  std::vector<int4> rchunks;
  rchunks.reserve(rlongest * n_xcd);
  for (size_t k = 0; k < rlongest; ++k)
    for (int x = 0; x < n_xcd; ++x)
      rchunks.push_back(k < rbins[x].size() ? rbins[x][k] : make_int4(-1, 0, 0, 0));
  p->n_rchunks = (int)rchunks.size();
  // teams, largest clusters first: a workgroup each, and of a batch that has
  // more clusters than the chip holds workgroups the small ones a wave each
  std::vector<int4> teams;
  int4 four = make_int4(-1, -1, -1, -1);
  int in_four = 0;
  for (int c : order) {
    if (rclus[c].y > team_chunks) continue;
    if (n_clusters <= kRefitTeamBlocks || h_offsets[c + 1] - h_offsets[c] > kWaveRefit) {
      teams.push_back(make_int4(c, -2, 0, 0));
      continue;
    }
    (in_four == 0 ? four.x : in_four == 1 ? four.y : in_four == 2 ? four.z : four.w) = c;
    if (++in_four == 4) {
      teams.push_back(four);
      four = make_int4(-1, -1, -1, -1);
      in_four = 0;
    }
  }
  if (in_four) teams.push_back(four);
  p->n_teams = (int)teams.size();
  p->n_big = (int)big.size();
  const size_t wb = sizeof(int4) * work.size(), cb = sizeof(int4) * rchunks.size(),
               lb = sizeof(int4) * rclus.size(), eb = sizeof(int4) * teams.size(),
               bb = sizeof(int4) * big.size(), sb = sizeof(int32_t) * seed.size();
  const size_t tb = wb + cb + lb + eb + bb + sb;
  int st = grow(ctx, &p->d_tables, &p->cap_tables, tb, 1);
  if (!st) st = grow(ctx, (void**)&p->d_frames, &p->cap_frames, n_clusters, sizeof(CylFrame));
  if (!st)
    st = grow(ctx, (void**)&p->d_counts, &p->cap_counts, (size_t)n_clusters * cfg.n_hyp,
              sizeof(int32_t));
  if (!st)
    st = grow(ctx, (void**)&p->d_state, &p->cap_state, n_clusters, sizeof(RefitState));
  if (!st) st = grow(ctx, (void**)&p->d_member, &p->cap_member, std::max<size_t>(n_words, 1),
                     sizeof(uint32_t));
  if (!st) st = grow(ctx, (void**)&p->d_rescue, &p->cap_rescue, n_clusters, sizeof(int32_t));
  if (!st && (size_t)n_chunk_ids > p->cap_partial) {
    sloam_dev_free(p->d_pcount);
    p->d_pcount = nullptr;
    st = grow(ctx, (void**)&p->d_partial, &p->cap_partial, n_chunk_ids,
              sizeof(Comp2) * kRefitTerms);
    if (!st) st = sloam_dev_alloc(ctx, (void**)&p->d_pcount, sizeof(int32_t) * p->cap_partial);
  }
  if (st) return st;
  p->d_work = static_cast<int4*>(p->d_tables);
  p->d_rchunks = reinterpret_cast<int4*>(static_cast<char*>(p->d_tables) + wb);
  p->d_rclus = reinterpret_cast<int4*>(static_cast<char*>(p->d_tables) + wb + cb);
  p->d_teams = reinterpret_cast<int4*>(static_cast<char*>(p->d_tables) + wb + cb + lb);
  p->d_big = p->d_teams + teams.size();
  p->d_seed_order =
      reinterpret_cast<int32_t*>(static_cast<char*>(p->d_tables) + wb + cb + lb + eb + bb);
  // the tables through the pinned staging buffer, in one copy (the caller
  // has made sure that no earlier upload from it is pending)
  if (tb > p->cap_stage) {
    if (p->h_stage) (void)hipHostFree(p->h_stage);
    p->h_stage = nullptr;
    p->cap_stage = 0;
    const size_t sz = tb + tb / 2;
    hipError_t e = hipHostMalloc(&p->h_stage, sz);
    if (e != hipSuccess) return sloam_record_hip_error(ctx, e, "hipHostMalloc(plan staging)");
    p->cap_stage = sz;
  }
  char* stage = static_cast<char*>(p->h_stage);
  if (wb) std::memcpy(stage, work.data(), wb);
  if (cb) std::memcpy(stage + wb, rchunks.data(), cb);
  if (lb) std::memcpy(stage + wb + cb, rclus.data(), lb);
  if (eb) std::memcpy(stage + wb + cb + lb, teams.data(), eb);
  if (bb) std::memcpy(stage + wb + cb + lb + eb, big.data(), bb);
  if (sb) std::memcpy(stage + wb + cb + lb + eb + bb, seed.data(), sb);
  if (tb) SLOAM_HIP(ctx, hipMemcpyAsync(p->d_tables, stage, tb, hipMemcpyHostToDevice, ctx->stream));
  return SLOAM_OK;
}

// A plan with cfg's launch shapes and no batch yet (nullptr when cfg is
// invalid; *st says why).
static sloam_cyl_plan* plan_new(sloam_ctx* ctx, const sloam_cyl_fit_cfg* cfg, int* st) {
  *st = SLOAM_ERR_INVALID_ARG;
  if (cfg->n_hyp < 1 || cfg->n_hyp > (1 << 20) || !(cfg->thr > 0.0f) ||
      !(cfg->max_radius > 0.0f) || cfg->refit_iters < 0 || cfg->refit_rounds < 0 ||
      cfg->hyp_chunk < 0 || cfg->tile_points < 0)
    return nullptr;
  sloam_cyl_plan* p = new (std::nothrow) sloam_cyl_plan();
  if (!p) {
    *st = SLOAM_ERR_ALLOC;
    return nullptr;
  }
  p->ctx = ctx;
  p->cfg = *cfg;
  // hypotheses per workgroup: a multiple of kWaves * kHB
  int chunk = cfg->hyp_chunk > 0 ? cfg->hyp_chunk : 256;
  chunk = std::min(chunk, round_up(cfg->n_hyp, kWaves * kHB));
  p->hcap = round_up(chunk, kWaves * kHB);
  p->tile = cfg->tile_points > 0 ? round_up(cfg->tile_points, 64) : 2048;
  // keep the workgroup's LDS within 64 KiB: shrink the point tile if needed
  const int hyp_bytes = p->hcap * (int)(sizeof(float4) + sizeof(int));
  if (hyp_bytes > kMaxLds - 64 * 12) {
    delete p;
    *st = SLOAM_ERR_TOO_LARGE;
    return nullptr;
  }
  p->tile = std::min(p->tile, ((kMaxLds - hyp_bytes) / 12) / 64 * 64);
  int n_xcd = 1;
  if (hipDeviceGetAttribute(&n_xcd, hipDeviceAttributeNumberOfXccs, ctx->device) != hipSuccess ||
      n_xcd < 1)
    n_xcd = 1;
  (void)hipGetLastError();
  p->n_xcd = n_xcd;
  *st = SLOAM_OK;
  return p;
}

extern "C" {

int sloam_cyl_plan_create(sloam_ctx* ctx, const int32_t* h_offsets, int32_t n_clusters,
                          const sloam_cyl_fit_cfg* cfg, sloam_cyl_plan** out) {
  if (!ctx || !h_offsets || !cfg || !out || n_clusters < 0) return SLOAM_ERR_INVALID_ARG;
  *out = nullptr;
  SLOAM_HIP(ctx, hipSetDevice(ctx->device));
  int st = SLOAM_OK;
  sloam_cyl_plan* p = plan_new(ctx, cfg, &st);
  if (!p) return st;
  st = plan_layout(p, h_offsets, n_clusters);
  if (st) {
    sloam_cyl_plan_destroy(p);
    return st;
  }
  *out = p;
  return SLOAM_OK;
}

int sloam_cyl_plan_create_counted(sloam_ctx* ctx, int32_t cap_clusters, int64_t cap_points,
                                  const int32_t* d_n_clusters, const sloam_cyl_fit_cfg* cfg,
                                  sloam_cyl_plan** out) {
  if (!ctx || !cfg || !out || !d_n_clusters || cap_clusters < 1 || cap_points < 0 ||
      cap_points > ((int64_t)1 << 31) - 1 || cap_clusters > (1 << 20))
    return SLOAM_ERR_INVALID_ARG;
  *out = nullptr;
  SLOAM_HIP(ctx, hipSetDevice(ctx->device));
  int st = SLOAM_OK;
  sloam_cyl_plan* p = plan_new(ctx, cfg, &st);
  if (!p) return st;
  p->counted = true;
  p->d_n = d_n_clusters;
  p->cap_points = cap_points;
  p->cpc = (cfg->n_hyp + p->hcap - 1) / p->hcap;
  p->n_clusters = cap_clusters;
  p->n_points = cap_points;
  p->n_work = cap_clusters * p->cpc;
  const size_t words = member_word(cap_points, cap_clusters);
  const size_t tb = sizeof(int4) * (size_t)p->n_work;
  st = grow(ctx, &p->d_tables, &p->cap_tables, tb, 1);
  if (!st) st = grow(ctx, (void**)&p->d_frames, &p->cap_frames, cap_clusters, sizeof(CylFrame));
  if (!st)
    st = grow(ctx, (void**)&p->d_counts, &p->cap_counts, (size_t)cap_clusters * cfg->n_hyp,
              sizeof(int32_t));
  if (!st) st = grow(ctx, (void**)&p->d_member, &p->cap_member, words, sizeof(uint32_t));
  if (!st) st = grow(ctx, (void**)&p->d_rescue, &p->cap_rescue, cap_clusters, sizeof(int32_t));
  if (!st) st = sloam_dev_alloc(ctx, (void**)&p->d_cnt, sizeof(int32_t) * 4);
  if (st) {
    sloam_cyl_plan_destroy(p);
    return st;
  }
  p->d_work = static_cast<int4*>(p->d_tables);
  *out = p;
  return SLOAM_OK;
}

int sloam_cyl_plan_counts(const sloam_cyl_plan* p, const int32_t** d_counts) {
  if (!p || !d_counts || !p->counted) return SLOAM_ERR_INVALID_ARG;
  *d_counts = p->d_cnt;
  return SLOAM_OK;
}

int sloam_cyl_plan_reset(sloam_cyl_plan* p, const int32_t* h_offsets, int32_t n_clusters) {
  if (!p || !h_offsets || n_clusters < 0 || p->counted) return SLOAM_ERR_INVALID_ARG;
  sloam_ctx* ctx = p->ctx;
  if (ctx->capturing) return SLOAM_ERR_INVALID_ARG;
  SLOAM_HIP(ctx, hipSetDevice(ctx->device));
  // earlier runs of the plan read the buffers about to be rewritten
  SLOAM_HIP(ctx, hipStreamSynchronize(ctx->stream));
  const int st = plan_layout(p, h_offsets, n_clusters);
  if (st) {
    // no half-made layout: the plan holds an empty batch
    p->n_clusters = 0;
    p->n_points = 0;
    p->n_work = 0;
    p->n_rchunks = 0;
    p->n_teams = 0;
    p->n_big = 0;
  }
  return st;
}

int sloam_cyl_fallback(sloam_ctx* ctx, const int32_t* d_offsets, int32_t n_clusters,
                       const double* d_model, float min_inlier_ratio, int32_t* d_active,
                       int32_t* d_n_active) {
  if (!ctx || n_clusters < 0 || (n_clusters > 0 && (!d_offsets || !d_model || !d_active)))
    return SLOAM_ERR_INVALID_ARG;
  SLOAM_HIP(ctx, hipSetDevice(ctx->device));
  if (d_n_active) {
    int st = sloam_fill_u32(ctx, (uint32_t*)d_n_active, 1, 0u);
    if (st) return st;
  }
  if (n_clusters == 0) return SLOAM_OK;
  {
    SloamKernelScope ks(ctx, "cyl_fallback");
    hipLaunchKernelGGL(cyl_fallback_kernel, dim3((n_clusters + 255) / 256), dim3(256), 0,
                       ctx->stream, d_offsets, n_clusters, d_model, min_inlier_ratio, d_active,
                       d_n_active);
  }
  SLOAM_HIP(ctx, hipGetLastError());
  return SLOAM_OK;
}

int sloam_cyl_learned_exec(sloam_cyl_plan* verify, sloam_cyl_plan* plain, const float* d_xyz,
                           const int32_t* d_offsets, const float* d_proposal,
                           float min_inlier_ratio, int32_t* d_counts_verify,
                           int32_t* d_counts_plain, int32_t* d_fallback, int32_t* d_n_fallback,
                           int32_t* d_best, double* d_model) {
  if (!verify || !plain || !d_offsets || !d_model || !d_fallback) return SLOAM_ERR_INVALID_ARG;
  if (verify->ctx != plain->ctx || verify->n_clusters != plain->n_clusters ||
      verify->n_points != plain->n_points)
    return SLOAM_ERR_INVALID_ARG;
  const sloam_cyl_fit_cfg& vc = verify->cfg;
  const sloam_cyl_fit_cfg& pc = plain->cfg;
  if (vc.thr != pc.thr || vc.max_radius != pc.max_radius || vc.seed != pc.seed)
    return SLOAM_ERR_INVALID_ARG;
  if (verify->n_points > 0 && !d_xyz) return SLOAM_ERR_INVALID_ARG;
  sloam_ctx* ctx = verify->ctx;
  if (verify->n_clusters == 0) return SLOAM_OK;
  SLOAM_HIP(ctx, hipSetDevice(ctx->device));
  const uint32_t k0 = (uint32_t)vc.seed;
  const uint32_t k1 = (uint32_t)(vc.seed >> 32);
  int32_t* cv = d_counts_verify ? d_counts_verify : verify->d_counts;
  int32_t* cp = d_counts_plain ? d_counts_plain : plain->d_counts;
  const int S = verify->n_clusters;
  if (verify->counted != plain->counted ||
      (verify->counted && (verify->d_n != plain->d_n || verify->cap_points != plain->cap_points)))
    return SLOAM_ERR_INVALID_ARG;
  int st0 = layout_counted(verify, d_offsets);
  if (!st0) st0 = layout_counted(plain, d_offsets);
  if (st0) return st0;
  const int32_t* vcnt = verify->counted ? verify->d_cnt : nullptr;
  {
    // one axis seed per cluster serves both hypothesis sets
    SloamKernelScope ks(ctx, "cyl_seed");
    launch_seed(verify, d_xyz, d_offsets, nullptr);
  }
  SLOAM_HIP(ctx, hipGetLastError());
  if (verify->n_work > 0) {
    const size_t lds =
        (size_t)verify->hcap * (sizeof(float4) + sizeof(int)) + 3 * sizeof(float) * verify->tile;
    SloamKernelScope ks(ctx, "cyl_score");
    hipLaunchKernelGGL(cyl_score_kernel, dim3(verify->n_work), dim3(kBlock), lds, ctx->stream,
                       d_xyz, d_offsets, verify->d_frames, verify->d_work, vc.n_hyp, verify->hcap,
                       verify->tile, vc.thr, vc.max_radius, k0, k1, (uint32_t)vc.stream_tag,
                       d_proposal, nullptr, vcnt, cv, nullptr);
  }
  SLOAM_HIP(ctx, hipGetLastError());
  {
    SloamKernelScope ks(ctx, "cyl_decide");
    if (d_n_fallback) {
      const int st = sloam_fill_u32(ctx, (uint32_t*)d_n_fallback, 1, 0u);
      if (st) return st;
    }
    hipLaunchKernelGGL(cyl_decide_kernel, dim3((S + 255) / 256), dim3(256), 0, ctx->stream,
                       d_offsets, S, cv, vc.n_hyp, min_inlier_ratio, vcnt, d_fallback,
                       d_n_fallback);
  }
  SLOAM_HIP(ctx, hipGetLastError());
  if (plain->n_work > 0) {
    // the plain hypotheses of the flagged clusters, in the same seed frames
    const size_t lds =
        (size_t)plain->hcap * (sizeof(float4) + sizeof(int)) + 3 * sizeof(float) * plain->tile;
    SloamKernelScope ks(ctx, "cyl_score");
    hipLaunchKernelGGL(cyl_score_kernel, dim3(plain->n_work), dim3(kBlock), lds, ctx->stream,
                       d_xyz, d_offsets, verify->d_frames, plain->d_work, pc.n_hyp, plain->hcap,
                       plain->tile, pc.thr, pc.max_radius, k0, k1, (uint32_t)pc.stream_tag,
                       nullptr, d_fallback, plain->counted ? plain->d_cnt : nullptr, cp, nullptr);
  }
  SLOAM_HIP(ctx, hipGetLastError());
  {
    SloamKernelScope ks(ctx, "cyl_refit");
    const int st = launch_refit(verify, d_xyz, d_offsets, cv, d_proposal, nullptr, d_fallback, cp,
                                pc.n_hyp, (uint32_t)pc.stream_tag, pc.refit_rounds,
                                pc.refit_iters, nullptr, d_best, d_model);
    if (st) return st;
  }
  {
    // rescue: the verified clusters whose refit failed or kept fewer than
    // min_inlier_ratio * n inliers take the plain method's fit after all
    // (scored with the plain hypotheses in the same seed frames, refitted
    // alone)
    SloamKernelScope ks(ctx, "cyl_rescue");
    hipLaunchKernelGGL(cyl_rescue_kernel, dim3((S + 255) / 256), dim3(256), 0, ctx->stream,
                       d_offsets, S, d_model, min_inlier_ratio, vcnt, d_fallback,
                       verify->d_rescue, d_n_fallback);
    SLOAM_HIP(ctx, hipGetLastError());
    if (plain->n_work > 0) {
      const size_t lds =
          (size_t)plain->hcap * (sizeof(float4) + sizeof(int)) + 3 * sizeof(float) * plain->tile;
      hipLaunchKernelGGL(cyl_score_kernel, dim3(plain->n_work), dim3(kBlock), lds, ctx->stream,
                         d_xyz, d_offsets, verify->d_frames, plain->d_work, pc.n_hyp,
                         plain->hcap, plain->tile, pc.thr, pc.max_radius, k0, k1,
                         (uint32_t)pc.stream_tag, nullptr, verify->d_rescue,
                         plain->counted ? plain->d_cnt : nullptr, cp, nullptr);
      SLOAM_HIP(ctx, hipGetLastError());
    }
    const int st = launch_refit(verify, d_xyz, d_offsets, cv, nullptr, verify->d_rescue,
                                verify->d_rescue, cp, pc.n_hyp, (uint32_t)pc.stream_tag,
                                pc.refit_rounds, pc.refit_iters, nullptr, d_best, d_model,
                                /*few=*/true);
    if (st) return st;
  }
  return SLOAM_OK;
}

int sloam_cyl_autotune(sloam_ctx* ctx, const int32_t* h_offsets, int32_t n_clusters,
                       const sloam_cyl_fit_cfg* cfg, const float* d_xyz, const int32_t* d_offsets,
                       sloam_cyl_fit_cfg* out) {
  if (!ctx || !h_offsets || !cfg || !out || n_clusters < 0) return SLOAM_ERR_INVALID_ARG;
  *out = *cfg;
  if (n_clusters == 0) return SLOAM_OK;
  if (!d_xyz || !d_offsets) return SLOAM_ERR_INVALID_ARG;
  // choices are cached per batch shape: every shape gives the same results
  static std::mutex mu;
  static std::map<std::tuple<int, int, int, int>, std::pair<int, int>> cache;
  const auto key = std::make_tuple(ctx->device, n_clusters, (int)h_offsets[n_clusters], cfg->n_hyp);
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(key);
    if (it != cache.end()) {
      out->hyp_chunk = it->second.first;
      out->tile_points = it->second.second;
      return SLOAM_OK;
    }
  }
  SLOAM_HIP(ctx, hipSetDevice(ctx->device));
  double* d_model = nullptr;
  int st = sloam_dev_alloc(ctx, (void**)&d_model,
                           sizeof(double) * SLOAM_CYL_MODEL_STRIDE * (size_t)n_clusters);
  if (st) return st;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  (void)hipEventCreate(&e0);
  (void)hipEventCreate(&e1);
  float best_ms = 1e30f;
  int best_chunk = 0, best_tile = 0;
  const int chunks[] = {64, 128, 256, 512};
  const int tiles[] = {1024, 2048, 4096};
  for (int ch : chunks) {
    if (ch > round_up(cfg->n_hyp, kWaves * kHB) && ch != 64) continue;
    for (int tl : tiles) {
      sloam_cyl_fit_cfg c = *cfg;
      c.hyp_chunk = ch;
      c.tile_points = tl;
      sloam_cyl_plan* p = nullptr;
      if (sloam_cyl_plan_create(ctx, h_offsets, n_clusters, &c, &p) != SLOAM_OK) continue;
      float ms = 0.f;
      bool ok = sloam_cyl_plan_exec(p, d_xyz, d_offsets, nullptr, nullptr, nullptr, nullptr,
                                    d_model) == SLOAM_OK;
      ok = ok && hipEventRecord(e0, ctx->stream) == hipSuccess;
      for (int r = 0; r < 3 && ok; ++r)
        ok = sloam_cyl_plan_exec(p, d_xyz, d_offsets, nullptr, nullptr, nullptr, nullptr,
                                 d_model) == SLOAM_OK;
      ok = ok && hipEventRecord(e1, ctx->stream) == hipSuccess &&
           hipEventSynchronize(e1) == hipSuccess && hipEventElapsedTime(&ms, e0, e1) == hipSuccess;
      sloam_cyl_plan_destroy(p);
      if (ok && ms < best_ms) {
        best_ms = ms;
        best_chunk = ch;
        best_tile = tl;
      }
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  sloam_dev_free(d_model);
  if (best_chunk == 0) return SLOAM_ERR_HIP;
  {
    std::lock_guard<std::mutex> lk(mu);
    cache[key] = std::make_pair(best_chunk, best_tile);
  }
  out->hyp_chunk = best_chunk;
  out->tile_points = best_tile;
  return SLOAM_OK;
}

void sloam_cyl_plan_destroy(sloam_cyl_plan* p) {
  if (!p) return;
  // pending uploads read the staging buffer
  if (p->h_stage) {
    (void)hipStreamSynchronize(p->ctx->stream);
    (void)hipHostFree(p->h_stage);
  }
  sloam_dev_free(p->d_tables);
  sloam_dev_free(p->d_frames);
  sloam_dev_free(p->d_counts);
  sloam_dev_free(p->d_state);
  sloam_dev_free(p->d_member);
  sloam_dev_free(p->d_partial);
  sloam_dev_free(p->d_pcount);
  sloam_dev_free(p->d_rescue);
  sloam_dev_free(p->d_cnt);
  delete p;
}

int sloam_cyl_plan_exec(sloam_cyl_plan* p, const float* d_xyz, const int32_t* d_offsets,
                        int32_t* d_counts, int32_t* d_samples, uint32_t* d_mask, int32_t* d_best,
                        double* d_model) {
  return sloam_cyl_plan_exec_ex(p, d_xyz, d_offsets, nullptr, nullptr, d_counts, d_samples, d_mask,
                                d_best, d_model);
}

int sloam_cyl_plan_exec_ex(sloam_cyl_plan* p, const float* d_xyz, const int32_t* d_offsets,
                           const float* d_proposal, const int32_t* d_active, int32_t* d_counts,
                           int32_t* d_samples, uint32_t* d_mask, int32_t* d_best,
                           double* d_model) {
  if (!p || !d_offsets || !d_model || (p->n_points > 0 && !d_xyz)) return SLOAM_ERR_INVALID_ARG;
  if (d_active && d_mask) return SLOAM_ERR_INVALID_ARG;  // the mask is cleared for all clusters
  sloam_ctx* ctx = p->ctx;
  if (p->n_clusters == 0) return SLOAM_OK;
  SLOAM_HIP(ctx, hipSetDevice(ctx->device));
  const sloam_cyl_fit_cfg& cfg = p->cfg;
  const uint32_t k0 = (uint32_t)cfg.seed;
  const uint32_t k1 = (uint32_t)(cfg.seed >> 32);
  const uint32_t tag = (uint32_t)cfg.stream_tag;
  int32_t* counts = d_counts ? d_counts : p->d_counts;
  if (p->counted && d_mask) return SLOAM_ERR_INVALID_ARG;  // its size is the batch's
  int st0 = layout_counted(p, d_offsets);
  if (st0) return st0;
  const int32_t* cnt = p->counted ? p->d_cnt : nullptr;
  if (d_mask) {
    int st = sloam_fill_u32(ctx, d_mask, (size_t)((p->n_points + 31) / 32), 0u);
    if (st) return st;
  }
  {
    SloamKernelScope ks(ctx, "cyl_seed");
    launch_seed(p, d_xyz, d_offsets, d_active);
  }
  SLOAM_HIP(ctx, hipGetLastError());
  if (p->n_work > 0) {
    const size_t lds = (size_t)p->hcap * (sizeof(float4) + sizeof(int)) + 3 * sizeof(float) * p->tile;
    SloamKernelScope ks(ctx, "cyl_score");
    hipLaunchKernelGGL(cyl_score_kernel, dim3(p->n_work), dim3(kBlock), lds, ctx->stream, d_xyz,
                       d_offsets, p->d_frames, p->d_work, cfg.n_hyp, p->hcap, p->tile, cfg.thr,
                       cfg.max_radius, k0, k1, tag, d_proposal, d_active, cnt, counts, d_samples);
  }
  SLOAM_HIP(ctx, hipGetLastError());
  {
    SloamKernelScope ks(ctx, "cyl_refit");
    const int st = launch_refit(p, d_xyz, d_offsets, counts, d_proposal, d_active, nullptr,
                                nullptr, 0, 0u, cfg.refit_rounds, cfg.refit_iters, d_mask, d_best,
                                d_model);
    if (st) return st;
  }
  SLOAM_HIP(ctx, hipGetLastError());
  return SLOAM_OK;
}

}  // extern "C"
