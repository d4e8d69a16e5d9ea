// Event-blocked Gaussian-kernel sums for the hit-cloud MMD of the fit loss (losses_jax.py:13-39,
// 58-80) and the intensity of nll_loss (:329-361): out[i][k] = sum_j exp(-|x_i - y_j|^2 * inv)
// * c[j][k], k < 4, over the points y_j of x_i's event, in D = 3 or 4 dimensions.  Points of
// different events never form a kernel value (the reference's event offsets make those exactly
// zero).  Distances and the exponential are float32; terms are summed in float32 over runs of
// kRbfRun consecutive terms (at most 32: a relative rounding of ~32 * 2^-24 = 2e-6 of the run's sum
// in the worst case, ~3e-7 typically) and the runs in float64 (a float64 add per term would double
// the work per pair).  Fixed summation order: bitwise reproducible.
//
// The lanes of a wave walk one candidate span together (wave-uniform indices, so y_j and c_j are
// scalar loads shared by the wave): lanes are grouped by their span (range kernel) or by their event
// (grid kernel), and a wave whose lanes straddle two events walks each group in turn.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lsim {

constexpr int kRbfRun = 32;
constexpr float kLog2e = 1.4426950408889634f;

struct RbfAcc {
  double s0, s1, s2, s3;  // closed runs
  float f0, f1, f2, f3;   // the open run
  int run;                // terms in the open run
};

// Terms j = ja .. jb - 1 (wave-uniform bounds) into the open run; full runs close into float64.
template <int D>
__device__ __forceinline__ void rbf_span(const float4& p, const float4* __restrict__ y, const float4* __restrict__ c,
                                         int ja, int jb, float inv_l2, RbfAcc& a) {
  // (constant address space: the loads of a wave-uniform index stay scalar behind a barrier too)
  using Const4 = const __attribute__((address_space(4))) float __attribute__((ext_vector_type(4)));
  const Const4* yq = (const Const4*)(uintptr_t)y;
  const Const4* cq = (const Const4*)(uintptr_t)c;
  // the lanes walking a span share its run position: keep it (and so the loop) wave-uniform
  int run = __builtin_amdgcn_readfirstlane(a.run);
  while (ja < jb) {
    const int n = jb - ja < kRbfRun - run ? jb - ja : kRbfRun - run;
#pragma unroll 4
    for (int u = 0; u < n; ++u) {
      const auto q = yq[ja + u], w = cq[ja + u];
      const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
      float d2 = dx * dx + dy * dy + dz * dz;
      if (D == 4) {
        const float dw = p.w - q.w;
        d2 += dw * dw;
      }
      const float k = __builtin_amdgcn_exp2f(-d2 * inv_l2);  // exp(-d2 inv), inv_l2 = inv log2(e)
      a.f0 += k * w.x;
      a.f1 += k * w.y;
      a.f2 += k * w.z;
      a.f3 += k * w.w;
    }
    ja += n;
    run += n;
    if (run == kRbfRun) {
      a.s0 += (double)a.f0;
      a.s1 += (double)a.f1;
      a.s2 += (double)a.f2;
      a.s3 += (double)a.f3;
      a.f0 = a.f1 = a.f2 = a.f3 = 0.f;
      run = 0;
    }
  }
  a.run = run;
}

__device__ __forceinline__ void rbf_store(const RbfAcc& a, double* o) {
  o[0] = a.s0 + (double)a.f0;
  o[1] = a.s1 + (double)a.f1;
  o[2] = a.s2 + (double)a.f2;
  o[3] = a.s3 + (double)a.f3;
}

// Span form: point i sums over y[lo_i .. hi_i) (the caller's event ranges).
template <int D>
__global__ __launch_bounds__(256) void k_rbf_sums(const float4* __restrict__ x, int64_t nx, const int32_t* __restrict__ lo,
                                                  const int32_t* __restrict__ hi, const float4* __restrict__ y,
                                                  const float4* __restrict__ c, float inv, double* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool valid = i < nx;
  const float4 p = valid ? x[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  const int mlo = valid ? lo[i] : 0, mhi = valid ? hi[i] : 0;
  RbfAcc a = {0.0, 0.0, 0.0, 0.0, 0.f, 0.f, 0.f, 0.f, 0};
  bool pending = valid;
  for (uint64_t pm = __ballot(pending); pm != 0; pm = __ballot(pending)) {
    const int lead = __builtin_ctzll(pm);
    const int ja = __builtin_amdgcn_readlane(mlo, lead), jb = __builtin_amdgcn_readlane(mhi, lead);
    const bool mine = pending && mlo == ja && mhi == jb;
    if (mine) rbf_span<D>(p, y, c, ja, jb, inv * kLog2e, a);
    pending = pending && !mine;
  }
  if (valid) rbf_store(a, out + i * 4);
}

// ---- grid form: only the grid columns that can hold a non-zero kernel value are walked ----
//
// The candidates are sorted by key = ((event * Gx + cx) * Gy + cy) * Gz + cz, the cell of a point
// being clamp(floor((v - lo) / h), 0, G - 1) per axis (grid[] = lo xyz, h xyz, G xyz); the edge
// cells reach to infinity.  For the queries of one event in a wave (bounding box B), a cell column
// (cx, cy) is walked over the z cells within the cull radius rc of B, and skipped when its
// x-y distance from B exceeds rc.  Every skipped pair is at least rc apart in the first three
// coordinates, where exp(-d^2 inv) is exactly 0 in float32 (rc^2 inv > 106: e^-106 < 2^-152, below
// the smallest denormal): the sums are those of all pairs of the event, in another order.

__device__ __forceinline__ int rbf_cell(float v, float lo, float h, int G) {
  const float c = floorf((v - lo) / h);
  return (int)fminf(fmaxf(c, 0.f), (float)(G - 1));
}

// distance along one axis between [b0, b1] and cell c
__device__ __forceinline__ float rbf_gap(int c, float b0, float b1, float lo, float h, int G) {
  const float c0 = c == 0 ? -__builtin_inff() : lo + (float)c * h;
  const float c1 = c == G - 1 ? __builtin_inff() : lo + (float)(c + 1) * h;
  return fmaxf(fmaxf(c0 - b1, b0 - c1), 0.f);
}

__device__ __forceinline__ int rbf_lower_bound(const int64_t* __restrict__ k, int n, int64_t key) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (int)(((unsigned)lo + (unsigned)hi) >> 1);
    if (k[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ float wave_min_f(float v) {
#pragma unroll
  for (int m = kWave / 2; m >= 1; m >>= 1) v = fminf(v, __shfl_xor(v, m, kWave));
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

__device__ __forceinline__ float wave_max_f(float v) {
#pragma unroll
  for (int m = kWave / 2; m >= 1; m >>= 1) v = fmaxf(v, __shfl_xor(v, m, kWave));
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// A workgroup holds 64 queries, the same in each of its kRbfWaves waves, which share their candidates: thread
// t finds the span of column b0 + t, a scan of the spans' lengths joins them into one list, and wave w walks
// the w-th part of it.  One wave to 64 queries left most of the chip idle and waited for the wave with the
// longest list (both sums of a 20k-segment fit step: 1188 -> 188 us); a fixed split keeps the order of the sums.
// A pair costs 11 float32 instructions and an exponential, which now bound it; y and c come by scalar loads.
constexpr int kRbfWaves = 8;
constexpr int kRbfCols = kRbfWaves * kWave;

template <int D>
__global__ __launch_bounds__(kRbfCols) void k_rbf_grid(const float4* __restrict__ x, const int32_t* __restrict__ ev,
                                                       int64_t nx, const float4* __restrict__ y,
                                                       const float4* __restrict__ c, const int64_t* __restrict__ ykey,
                                                       int32_t ny, const float* __restrict__ grid, float inv, float rc,
                                                       const uint32_t* __restrict__ perm, double* __restrict__ out) {
  __shared__ int s_start[kRbfCols], s_end[kRbfCols];  // a column's candidates; their end in the joined list
  __shared__ int s_tot[kRbfWaves];
  __shared__ double s_sum[kRbfWaves][4][kWave];
  const int t = threadIdx.x, lane = t & (kWave - 1), wid = __builtin_amdgcn_readfirstlane(t / kWave);
  const int64_t i = (int64_t)blockIdx.x * kWave + lane;
  const bool valid = i < nx;
  const float4 p = valid ? x[i] : make_float4(0.f, 0.f, 0.f, 0.f);
  const int my_ev = valid ? ev[i] : 0;
  const float lox = grid[0], loy = grid[1], loz = grid[2], hx = grid[3], hy = grid[4], hz = grid[5];
  const int Gx = (int)grid[6], Gy = (int)grid[7], Gz = (int)grid[8];
  const float inf = __builtin_inff();
  RbfAcc a = {0.0, 0.0, 0.0, 0.0, 0.f, 0.f, 0.f, 0.f, 0};
  bool pending = valid;
  for (uint64_t pm = __ballot(pending); pm != 0; pm = __ballot(pending)) {  // (alike in every wave)
    const int e = __builtin_amdgcn_readlane(my_ev, __builtin_ctzll(pm));
    const bool mine = pending && my_ev == e;
    const float bx0 = wave_min_f(mine ? p.x : inf), bx1 = wave_max_f(mine ? p.x : -inf);
    const float by0 = wave_min_f(mine ? p.y : inf), by1 = wave_max_f(mine ? p.y : -inf);
    const float bz0 = wave_min_f(mine ? p.z : inf), bz1 = wave_max_f(mine ? p.z : -inf);
    const int cxa = rbf_cell(bx0 - rc, lox, hx, Gx), cxb = rbf_cell(bx1 + rc, lox, hx, Gx);
    const int cya = rbf_cell(by0 - rc, loy, hy, Gy), cyb = rbf_cell(by1 + rc, loy, hy, Gy);
    const int ncy = cyb - cya + 1, ncol = cxb < cxa || cyb < cya ? 0 : (cxb - cxa + 1) * ncy;
    for (int b0 = 0; b0 < ncol; b0 += kRbfCols) {
      // this thread's column, and where its candidates end in its wave's part of the list
      int j0 = 0, j1 = 0;
      const int col = b0 + t;
      if (col < ncol) {
        const int cx = cxa + col / ncy, cy = cya + col % ncy;
        const float gx = rbf_gap(cx, bx0, bx1, lox, hx, Gx), gy = rbf_gap(cy, by0, by1, loy, hy, Gy);
        const float r2 = rc * rc - gx * gx - gy * gy;
        if (r2 >= 0.f) {
          const float rz = sqrtf(r2);
          const int cza = rbf_cell(bz0 - rz, loz, hz, Gz), czb = rbf_cell(bz1 + rz, loz, hz, Gz);
          const int64_t kb = (((int64_t)e * Gx + cx) * Gy + cy) * Gz;
          j0 = rbf_lower_bound(ykey, ny, kb + cza);
          j1 = rbf_lower_bound(ykey, ny, kb + czb + 1);
        }
      }
      int n = j1 - j0;
#pragma unroll
      for (int m = 1; m < kWave; m <<= 1) {
        const int v = __shfl_up(n, m, kWave);
        if (lane >= m) n += v;
      }
      __syncthreads();  // (the list of the round before has been walked)
      s_start[t] = j0;
      s_end[t] = n;
      if (lane == kWave - 1) s_tot[wid] = n;
      __syncthreads();
      int tot = 0;
      for (int w = 0; w < kRbfWaves; ++w) tot += __builtin_amdgcn_readfirstlane(s_tot[w]);
      // positions la .. lb - 1 of the joined list are this wave's
      const int la = (int)((int64_t)tot * wid / kRbfWaves), lb = (int)((int64_t)tot * (wid + 1) / kRbfWaves);
      for (int w = 0, wa = 0, we = 0; w < kRbfWaves && wa < lb; ++w, wa = we) {
        we = wa + __builtin_amdgcn_readfirstlane(s_tot[w]);
        if (we <= la) continue;  // (none of this wave's among these 64 columns)
        const int q1 = s_end[w * kWave + lane], qs = s_start[w * kWave + lane];
        const int up = __shfl_up(q1, 1, kWave);
        const int q0 = lane == 0 ? 0 : up;
        const int k0 = max(la - wa, q0), k1 = min(lb - wa, q1);  // this column's part of this wave's list
        const int ja = qs + (k0 - q0), jb = qs + (k1 - q0);
        for (uint64_t m = __ballot(k0 < k1); m != 0; m &= m - 1) {
          const int cc = __builtin_ctzll(m);
          const int ua = __builtin_amdgcn_readlane(ja, cc), ub = __builtin_amdgcn_readlane(jb, cc);
          if (mine) rbf_span<D>(p, y, c, ua, ub, inv * kLog2e, a);
        }
      }
    }
    pending = pending && !mine;
  }
  s_sum[wid][0][lane] = a.s0 + (double)a.f0;
  s_sum[wid][1][lane] = a.s1 + (double)a.f1;
  s_sum[wid][2][lane] = a.s2 + (double)a.f2;
  s_sum[wid][3][lane] = a.s3 + (double)a.f3;
  __syncthreads();
  // thread t < 256: column t % 4 of query t / 4
  const int64_t o = (int64_t)blockIdx.x * kWave + t / 4;
  if (t < 4 * kWave && o < nx) {
    double v = 0.0;
#pragma unroll
    for (int w = 0; w < kRbfWaves; ++w) v += s_sum[w][t % 4][t / 4];
    out[(perm ? (int64_t)perm[o] : o) * 4 + t % 4] = v;
  }
}

// ---- two clouds onto one grid (lsim_rbf_mmd_sums) ----
//
// The points x (charges px) and y (py), float64 and in any order, become the grid form's sorted arrays:
// the grid from the bounds of both, one stable sort of both by (cloud, event, cell), one gather.  Formed by
// some 120 tensor operations a step before, of a few microseconds each to launch (20k-segment fit step: 3.76 -> 2.90 ms).

constexpr int kRbfBoundBlocks = 64;
constexpr int kRbfMaxCells = 64;                // per axis
constexpr int kRbfCellBits = 18;                // 64^3 cells

struct RbfClouds {
  const double *x, *px;   // [nx][3], [nx]
  const int64_t* ex;
  int64_t nx;
  const double *y, *py;
  const int64_t* ey;
  int64_t ny;
};

__device__ __forceinline__ float4 rbf_point(const RbfClouds& r, int64_t i) {
  const double* p = i < r.nx ? r.x + i * 3 : r.y + (i - r.nx) * 3;
  return make_float4((float)p[0], (float)p[1], (float)p[2], 0.f);
}

// part [kRbfBoundBlocks][6]: minima and maxima of x, y, z
__global__ __launch_bounds__(256) void k_rbf_bounds(RbfClouds r, float* __restrict__ part) {
  __shared__ float sh[6][256 / kWave];
  const int64_t n = r.nx + r.ny;
  float v[6] = {__builtin_inff(), __builtin_inff(), __builtin_inff(), -__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const float4 p = rbf_point(r, i);
    v[0] = fminf(v[0], p.x), v[1] = fminf(v[1], p.y), v[2] = fminf(v[2], p.z);
    v[3] = fmaxf(v[3], p.x), v[4] = fmaxf(v[4], p.y), v[5] = fmaxf(v[5], p.z);
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const float w = k < 3 ? wave_min_f(v[k]) : wave_max_f(v[k]);
    if (threadIdx.x % kWave == 0) sh[k][threadIdx.x / kWave] = w;
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    float w = sh[threadIdx.x][0];
    for (int k = 1; k < 256 / kWave; ++k)
      w = threadIdx.x < 3 ? fminf(w, sh[threadIdx.x][k]) : fmaxf(w, sh[threadIdx.x][k]);
    part[blockIdx.x * 6 + threadIdx.x] = w;
  }
}

// One wave: grid [9] with cells about a third of the cull radius wide, at most kRbfMaxCells an axis.
__global__ __launch_bounds__(kWave) void k_rbf_grid_of(const float* __restrict__ part, float rc, float* __restrict__ grid) {
  const int t = threadIdx.x;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float lo = wave_min_f(part[t * 6 + k]), ext = wave_max_f(part[t * 6 + 3 + k]) - lo;
    const float G = fminf(fmaxf(ceilf(ext / (rc / 3.f)), 1.f), (float)kRbfMaxCells);
    if (t == 0) {
      grid[k] = lo;
      grid[3 + k] = ext > 0.f ? ext / G : 1.f;
      grid[6 + k] = G;
    }
  }
}

__device__ __forceinline__ int rbf_cell_index(const float4& p, const float* __restrict__ g) {
  const int cx = rbf_cell(p.x, g[0], g[3], (int)g[6]), cy = rbf_cell(p.y, g[1], g[4], (int)g[7]);
  return (cx * (int)g[7] + cy) * (int)g[8] + rbf_cell(p.z, g[2], g[5], (int)g[8]);
}

// Sort keys of the three stages, least significant first (each stable): cell, event, cloud.
__global__ __launch_bounds__(256) void k_rbf_keys(RbfClouds r, const float* __restrict__ grid, int stage,
                                                  const uint32_t* __restrict__ vin, uint32_t* __restrict__ keys,
                                                  uint32_t* __restrict__ vals) {
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (j >= r.nx + r.ny) return;
  const int64_t i = vin ? (int64_t)vin[j] : j;
  if (!vin) vals[j] = (uint32_t)j;
  if (stage == 0) keys[j] = (uint32_t)rbf_cell_index(rbf_point(r, i), grid);
  else if (stage == 1) keys[j] = (uint32_t)(int32_t)(i < r.nx ? r.ex[i] : r.ey[i - r.nx]) ^ 0x80000000u;
  else keys[j] = i < r.nx ? 0u : 1u;
}

// The sorted arrays: point, charge-weighted columns, key, event (its cloud's points first to last).
__global__ __launch_bounds__(256) void k_rbf_gather(RbfClouds r, const float* __restrict__ grid,
                                                    const uint32_t* __restrict__ perm, float4* __restrict__ pts,
                                                    float4* __restrict__ cols, int64_t* __restrict__ key,
                                                    int32_t* __restrict__ ev) {
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (j >= r.nx + r.ny) return;
  const int64_t i = (int64_t)perm[j];
  const bool is_x = i < r.nx;
  const double* p = is_x ? r.x + i * 3 : r.y + (i - r.nx) * 3;
  const double w = is_x ? r.px[i] : r.py[i - r.nx];
  const int32_t e = (int32_t)(is_x ? r.ex[i] : r.ey[i - r.nx]);
  const float4 q = make_float4((float)p[0], (float)p[1], (float)p[2], 0.f);
  pts[j] = q;
  cols[j] = make_float4((float)w, (float)(w * p[0]), (float)(w * p[1]), (float)(w * p[2]));
  key[j] = (int64_t)e * (int)grid[6] * (int)grid[7] * (int)grid[8] + rbf_cell_index(q, grid);
  ev[j] = e;
}

// Event-blocked nearest neighbour for the chamfer loss (losses_jax.py:195-229
// chamfer_distance_3d_og): for query i, the index of the nearest point among y[lo_i .. hi_i) by
// squared distance (dx^2 + dy^2) + dz^2 in float32, the first on ties as argmin takes it, and that
// distance.  The first n_origin queries also see the origin, a zero-weight padding point that
// comes after every real point (it wins only when strictly nearer; index -1).  No candidate:
// index -1, distance +inf.
__global__ __launch_bounds__(256) void k_nearest(const float4* __restrict__ x, int64_t nx, const int32_t* __restrict__ lo,
                                                 const int32_t* __restrict__ hi, const float4* __restrict__ y,
                                                 int64_t n_origin, int32_t* __restrict__ idx, float* __restrict__ dmin) {
#pragma clang fp contract(off)
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nx) return;
  const float4 p = x[i];
  float best = __builtin_inff();
  int32_t bi = -1;
  for (int j = lo[i], j1 = hi[i]; j < j1; ++j) {
    const float4 q = y[j];
    const float dx = p.x - q.x, dy = p.y - q.y, dz = p.z - q.z;
    const float d = (dx * dx + dy * dy) + dz * dz;
    if (d < best) {
      best = d;
      bi = j;
    }
  }
  if (i < n_origin) {
    const float d = (p.x * p.x + p.y * p.y) + p.z * p.z;
    if (d < best) {
      best = d;
      bi = -1;
    }
  }
  idx[i] = bi;
  dmin[i] = best;
}

}  // namespace lsim
