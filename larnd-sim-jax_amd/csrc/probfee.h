// Probabilistic self-trigger readout (fee_jax.py:334-461 _find_one_hit_step and
// get_adc_values_average_noise_vmap): a beam search of V charge-reset paths per pixel row over
// the tick grid, with Gaussian reset noise sigma, giving per hit index s and tick t the log
// probability that hit s starts at t and its expected charge.
//
// Per row, with q_sum the cumulative charge (T ticks), c_v and p_v the reset charge and log
// probability of path v, sh(t) = min(t + interval + 1, T - 1) and z(x) = (x - threshold) / sigma:
//   log_guess[v,t] = logdiffPhi(z(CM[t+1] - c_v), z(CM[t] - c_v)),  CM = cumulative max of q_sum
//                    (cummax(q_sum - c) = cummax(q_sum) - c, so one CM serves every path);
//   log_event[v,t] = min(logdiffPhi(z(q_sum[sh] - c_v), z(q_sum[t] - c_v)), log_guess), then
//                    soft-clamped at -1000 and soft-masked by the expected charge
//                    esp[t] = q_sum[sh] + threshold - (q_sum[t+1] + q_sum[t]) / 2;
//   out_logp[s,t]  = logsumexp_v(log_event + p_v),  out_charge[s,t] = esp[t];
//   total[t]       = logsumexp_v(log_guess + p_v);
//   select[t]      = LF[t] + total[t], LF[t] = log Phi(z(RCM[e(t)] - q_sum[sh(t)+1])), RCM the
//                    reverse cumulative max, e(t) = min(sh(t) + interval + 1, T - 1) (the path
//                    charge cancels in this term, so it is one value per tick);
//   the V ticks of largest select (lower tick first on ties) become the next paths:
//   p'_k = total[t_k], c'_k = q_sum[min(sh(t_k) + 1, T - 1)].
// The reference stops all rows at once when no row has logsumexp(p') > log(stop) any more; the
// step launches read and set that flag in device memory, and stopped steps write -1000 / 0.
// Rows are independent: one workgroup per row and step, ticks in contiguous chunks per thread,
// the row's tables in LDS, the top-V selection by V rounds of a block arg-max.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lsim {

constexpr int kPfThreads = 256;
constexpr int kPfMaxTicks = 2048;
constexpr int kPfMaxPaths = 32;
constexpr int kPfChunk = (kPfMaxTicks + kPfThreads - 1) / kPfThreads;  // ticks per thread

struct PfDev {
  int T;          // ticks per row
  int V;          // paths kept (fee_paths_scaling)
  int S;          // hit indices (MAX_ADC_VALUES)
  int interval;   // ADC hold interval in ticks
  float theta;    // discrimination threshold (e-)
  float zs;       // 1 / reset-noise sigma
  float ts;       // t_sampling
  float log_stop; // log of the stop threshold
  float minus_one = -1.f;  // an argument, so that functions of it are evaluated on the device like the others
};

// log Phi(x) in float32 from one scaled complementary error function, u = |x| / sqrt 2:
// x < 0: -u^2 + log(erfcx(u) / 2) (accurate far into the tail); x >= 0: log1p(-exp(-u^2) erfcx(u) / 2).
// No branch on the sign around the expensive part, so lanes of either sign share one erfcx.
__device__ __forceinline__ float pf_log_ndtr(float x) {
  const float u = fabsf(x) * 0.70710678118654752f;
  const float ex = erfcxf(u);
  const float u2 = u * u;
  return x < 0.f ? -u2 + logf(0.5f * ex) : log1pf(-0.5f * expf(-u2) * ex);
}

// softplus(x) = max(x, 0) + log1p(exp(-|x|)); beyond |x| = 30 the correction is below float32
// resolution (x itself, or exp(x) = log1p(exp(x)) to 1e-13), so the transcendental calls are skipped.
__device__ __forceinline__ float pf_softplus(float x) {
  if (x > 30.f) return x;
  if (x < -30.f) return expf(x);
  return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x)));
}

// lo + softplus((x - lo) s) / s (fee_jax.py:13-20)
__device__ __forceinline__ float pf_soft_max(float x, float lo, float s) { return lo + pf_softplus((x - lo) * s) / s; }

// sigmoid(c s) t + (1 - sigmoid(c s)) f (fee_jax.py:22-30)
__device__ __forceinline__ float pf_soft_where(float c, float t, float f, float s) {
  const float x = c * s;
  // sigmoid(x): 1 in float32 above 30 (1 + exp(-30) rounds to 1); exp(x) below -30 (to 1e-13)
  const float w = x > 30.f ? 1.f : (x < -30.f ? expf(x) : 1.f / (1.f + expf(-x)));
  return w * t + (1.f - w) * f;
}

// The clamped log(1 - exp(sd)) of log(Phi(a) - Phi(b)) = log Phi(a) + log(1 - exp(sd)), sd = log Phi(b) -
// log Phi(a) (fee_jax.py:32-54).
__device__ __forceinline__ float pf_log_one_minus(float sd) {
  float ne = -expm1f(sd);
  ne = pf_soft_max(ne, 1e-30f, 1e10f);
  return pf_soft_max(logf(ne), -100.f, 10.f);
}

// log(Phi(a) - Phi(b)) with the reference's smooth clamps (fee_jax.py:32-54), from la = log Phi(a)
// and lb = log Phi(b).  The reference takes sd = -1 unless a > b; `none` = pf_log_one_minus(-1), so that
// lanes without a rise (most ticks: the charge does not move) skip the functions.
__device__ __forceinline__ float pf_log_diff(float a, float b, float la, float lb, float none) {
  float lt = none;
  if (a > b) lt = pf_log_one_minus(lb - la);
  return pf_soft_where(a - b, la + lt, -1000.f, 1000.f);
}

// Running logsumexp: (m, sum) with sum = sum_i exp(x_i - m).
__device__ __forceinline__ void pf_lse_add(float& m, float& sum, float x) {
  if (x > m) {
    sum = sum * expf(m - x) + 1.f;
    m = x;
  } else {
    sum += expf(x - m);
  }
}

// Block-wide inclusive scan (sum, double) of one value per thread; returns the inclusive prefix.
__device__ __forceinline__ double pf_block_scan(double v, double* sh) {
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  double inc = v;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const double u = __shfl_up(inc, d, kWave);
    if (lane >= d) inc += u;
  }
  if (lane == kWave - 1) sh[wid] = inc;
  __syncthreads();
  double base = 0.0;
  for (int w = 0; w < wid; ++w) base += sh[w];
  __syncthreads();
  return base + inc;
}

// Per row: q_sum, its cumulative max, LF and esp (all independent of the step).
// tab layout per row: [q_sum T][CM T][LF T-1 (+1 pad)][esp T-1 (+1 pad)].
__global__ __launch_bounds__(kPfThreads) void k_pf_prep(PfDev d, const float* __restrict__ wfs, int64_t P,
                                                       float* __restrict__ tab) {
  __shared__ float s_q[kPfMaxTicks];
  __shared__ float s_r[kPfMaxTicks];
  __shared__ double s_w[kPfThreads / kWave];
  __shared__ float s_wm[kPfThreads / kWave];
  const int64_t row = blockIdx.x;
  const int T = d.T;
  const float* w = wfs + row * T;
  const int t0 = threadIdx.x * kPfChunk;
  // cumulative sum of q = wfs * t_sampling (double prefix, rounded once)
  double loc[kPfChunk];
  double run = 0.0;
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k) {
    const int t = t0 + k;
    const double q = t < T ? (double)(w[t] * d.ts) : 0.0;
    run += q;
    loc[k] = run;
  }
  const double base = pf_block_scan(run, s_w) - run;
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k)
    if (t0 + k < T) s_q[t0 + k] = (float)(base + loc[k]);
  __syncthreads();
  float* qs = tab + row * 4 * (int64_t)T;
  float* cm = qs + T;
  float* lf = cm + T;
  float* esp = lf + T;
  // forward and reverse cumulative max: chunk maxima, exclusive prefix / suffix maxima over
  // threads (wave shuffles, then the wave totals in LDS), then a walk over the chunk
  const float ninf = -__builtin_inff();
  float m = ninf;
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k)
    if (t0 + k < T) m = fmaxf(m, s_q[t0 + k]);
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  float inc = m;
#pragma unroll
  for (int dd = 1; dd < kWave; dd <<= 1) {
    const float u = __shfl_up(inc, dd, kWave);
    if (lane >= dd) inc = fmaxf(inc, u);
  }
  const float up1 = __shfl_up(inc, 1, kWave);
  if (lane == kWave - 1) s_wm[wid] = inc;
  __syncthreads();
  float excl_f = lane > 0 ? up1 : ninf;
  for (int ww = 0; ww < wid; ++ww) excl_f = fmaxf(excl_f, s_wm[ww]);
  __syncthreads();
  float incr = m;
#pragma unroll
  for (int dd = 1; dd < kWave; dd <<= 1) {
    const float u = __shfl_down(incr, dd, kWave);
    if (lane + dd < kWave) incr = fmaxf(incr, u);
  }
  const float dn1 = __shfl_down(incr, 1, kWave);
  if (lane == 0) s_wm[wid] = incr;
  __syncthreads();
  float excl_r = lane + 1 < kWave ? dn1 : ninf;
  for (int ww = wid + 1; ww < kPfThreads / kWave; ++ww) excl_r = fmaxf(excl_r, s_wm[ww]);
  float cf = excl_f;
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k) {
    const int t = t0 + k;
    if (t < T) {
      cf = fmaxf(cf, s_q[t]);
      cm[t] = cf;
    }
  }
  float cr = excl_r;
#pragma unroll
  for (int k = kPfChunk - 1; k >= 0; --k) {
    const int t = t0 + k;
    if (t < T) {
      cr = fmaxf(cr, s_q[t]);
      s_r[t] = cr;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k) {
    const int t = t0 + k;
    if (t < T) qs[t] = s_q[t];
    if (t < T - 1) {
      const int sh = min(t + d.interval + 1, T - 1);
      const int nx = min(sh + 1, T - 1);
      const int e = min(sh + d.interval + 1, T - 1);
      lf[t] = pf_log_ndtr((s_r[e] - s_q[nx] - d.theta) * d.zs);
      esp[t] = s_q[sh] + d.theta - 0.5f * (s_q[t + 1] + s_q[t]);
    }
  }
}

// ---- what the ticks of a row share ----
//
// Away from its pulses a waveform is zero, so q_sum and CM repeat from tick to tick, and with them
// everything a path computes there.  Per row:
//   run    a maximal stretch of ticks with one value of q_sum: log Phi is evaluated once per run and path
//          (CM's values are values of q_sum, so they share the runs; entry `nrun` stands for -inf, which
//          CM is only while q_sum has been NaN from the first tick);
//   group  a maximal stretch of ticks t with the same CM[t], CM[t+1], q_sum[t], q_sum[t+1] and q_sum[sh(t)]:
//          log_event, log_guess and their sums over the paths are evaluated once per group.
// The values are those of evaluating every tick, bit for bit.
struct PfShare {
  short rid[kPfMaxTicks];     // tick -> run of q_sum
  short cid[kPfMaxTicks];     // tick -> run with the value of CM
  float rv[kPfMaxTicks + 1];  // run -> value of q_sum
};

// Block-wide inclusive scan (sum or max) of one non-negative int per thread.
template <bool MAX>
__device__ __forceinline__ int pf_block_scan_i(int v, int* sh) {
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  int inc = v;
#pragma unroll
  for (int dd = 1; dd < kWave; dd <<= 1) {
    const int u = __shfl_up(inc, dd, kWave);
    if (lane >= dd) inc = MAX ? max(inc, u) : inc + u;
  }
  if (lane == kWave - 1) sh[wid] = inc;
  __syncthreads();
  int base = 0;
  for (int w = 0; w < wid; ++w) base = MAX ? max(base, sh[w]) : base + sh[w];
  __syncthreads();
  return MAX ? max(base, inc) : base + inc;
}

// Fills S from the row's q_sum and CM (global); nrun: number of runs.  Ends with a barrier.  sh: one int
// per wave; tot: one int.
__device__ __forceinline__ void pf_runs(const PfDev& d, const float* __restrict__ qs, const float* __restrict__ cm, PfShare& S,
                                        int* sh, int* tot, int& nrun) {
  const int T = d.T, t0 = threadIdx.x * kPfChunk;
  bool nw[kPfChunk];
  int cnt = 0, rec = 0;  // rec: 1 + the last tick of the chunk at which CM takes a new value
  float q[kPfChunk];
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k) {
    const int t = t0 + k;
    nw[k] = false;
    q[k] = 0.f;
    if (t < T) {
      q[k] = qs[t];
      nw[k] = t == 0 || !(q[k] == qs[t - 1]);
      if ((t == 0 || !(cm[t] == cm[t - 1])) && q[k] == cm[t]) rec = t + 1;
    }
    cnt += nw[k] ? 1 : 0;
  }
  int id = pf_block_scan_i<false>(cnt, sh) - cnt;
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k) {
    const int t = t0 + k;
    if (t < T) {
      if (nw[k]) S.rv[id++] = q[k];
      S.rid[t] = (short)(id - 1);
    }
  }
  if (threadIdx.x == kPfThreads - 1) {
    *tot = id;
    S.rv[id] = -__builtin_inff();
  }
  // the last record before this chunk, then along it
  const int inc = pf_block_scan_i<true>(rec, sh);  // (its barriers complete rid, rv and tot)
  int before = __shfl_up(inc, 1, kWave);
  if ((threadIdx.x & (kWave - 1)) == 0) before = 0;
  sh[threadIdx.x / kWave] = 0;
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) == kWave - 1) sh[threadIdx.x / kWave] = inc;
  __syncthreads();
  if ((threadIdx.x & (kWave - 1)) == 0 && threadIdx.x > 0) before = sh[threadIdx.x / kWave - 1];
  nrun = *tot;
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k) {
    const int t = t0 + k;
    if (t < T) {
      if ((t == 0 || !(cm[t] == cm[t - 1])) && q[k] == cm[t]) before = t + 1;
      S.cid[t] = before > 0 ? S.rid[before - 1] : (short)nrun;
    }
  }
  __syncthreads();
}

// Groups of ticks: did[t] = group of tick t < T - 1, first[g] = its first tick.  As pf_runs otherwise.
__device__ __forceinline__ void pf_groups(const PfDev& d, const PfShare& S, short* did, short* first, int* sh, int* tot,
                                          int& ngroup) {
  const int T = d.T, n = T - 1, t0 = threadIdx.x * kPfChunk;
  bool nw[kPfChunk];
  int cnt = 0;
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k) {
    const int t = t0 + k;
    nw[k] = false;
    if (t < n) {
      const int sh0 = min(t + d.interval + 1, T - 1);
      nw[k] = t == 0 || S.cid[t] != S.cid[t - 1] || S.cid[t + 1] != S.cid[t] || S.rid[t] != S.rid[t - 1] ||
              S.rid[t + 1] != S.rid[t] || S.rid[sh0] != S.rid[min(t + d.interval, T - 1)];
    }
    cnt += nw[k] ? 1 : 0;
  }
  int id = pf_block_scan_i<false>(cnt, sh) - cnt;
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k) {
    const int t = t0 + k;
    if (t < n) {
      if (nw[k]) first[id++] = (short)t;
      did[t] = (short)(id - 1);
    }
  }
  if (threadIdx.x == kPfThreads - 1) *tot = id;
  __syncthreads();
  ngroup = *tot;
}

// Paths with the same reset charge have the same log_event and log_guess at every tick, so their
// terms differ only by p_v: merge them into one path with p = logsumexp of theirs (in path order).
// At step 0 all V start paths share charge 0 and collapse into one.  One wave, lane v < V with (c, p) of
// path v: the number of merged paths; lane v's path belongs to merged path `group`, and lane u of the
// first path of a merged one has `lead` set and its p.
__device__ __forceinline__ int pf_merge_paths(int V, int lane, float c, float& p, int& group, bool& lead) {
  int first = lane;
  for (int u = V - 1; u >= 0; --u) {
    const float cu = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c), u));
    if (u < lane && cu == c) first = u;
  }
  lead = lane < V && first == lane;
  const uint64_t lm = __ballot(lead);
  for (uint64_t m = __ballot(lane < V && !lead); m != 0; m &= m - 1) {
    const int v = __builtin_ctzll(m);
    const int f = __builtin_amdgcn_readlane(first, v);
    const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), f));
    const float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p), v)), mx = fmaxf(a, b);
    const float r = mx + log1pf(expf(fminf(a, b) - mx));
    if (lane == f) p = r;
  }
  group = __popcll(lm & ((1ull << first) - 1));
  return __popcll(lm);
}

// One beam-search step for every row.  The paths are kept per step (the tape of the adjoint):
// tc[s][row][v], tp[s][row][v] = reset charge and log probability of path v entering step s
// (s = 0 .. S; slot 0 holds the start paths), tk[s][row][k] = the tick of the k-th selected path of
// step s.  flags[s] != 0: step s runs; a row whose new paths keep probability sets flags[s + 1].
//
// Bound by the transcendental functions of (path, group) pairs, about 400 instructions each; a
// thread holds the sums of its groups over the paths.  (Every tick evaluated, the paths merged by one
// thread and the top V ticks by V block-wide rounds of two barriers and 64 lanes of re-reads took
// 5.4 ms for 1024 rows of 2000 ticks with pulses on a fifth of them.)
__global__ __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_pf_step(PfDev d, int s, const float* __restrict__ tab, int64_t P,
                                                       float* __restrict__ tc, float* __restrict__ tp,
                                                       int* __restrict__ tk, int* __restrict__ flags,
                                                       float* __restrict__ out_logp, float* __restrict__ out_q) {
  __shared__ PfShare S;
  __shared__ short s_did[kPfMaxTicks];       // tick -> group
  __shared__ float s_tab[kPfMaxTicks + 1];   // run -> log Phi(z(q - c)) of the path; after the paths: group -> out_logp
  __shared__ float s_tot[kPfMaxTicks];       // group -> total; before the paths: group -> its first tick
  short* const s_first = (short*)s_tot;
  __shared__ float s_c[kPfMaxPaths], s_p[kPfMaxPaths];
  __shared__ uint64_t s_key[2][kPfThreads / kWave];
  __shared__ int s_top[kPfMaxPaths];
  __shared__ int s_sh[kPfThreads / kWave], s_nrun, s_ngroup, s_nv;
  const int64_t row = blockIdx.x;
  const int T = d.T, V = d.V, n = T - 1;
  float* ol = out_logp + (row * d.S + s) * (int64_t)n;
  float* oq = out_q + (row * d.S + s) * (int64_t)n;
  if (!flags[s]) {  // every row has stopped: the reference's inactive branch
    for (int t = threadIdx.x; t < n; t += kPfThreads) {
      ol[t] = -1000.f;
      oq[t] = 0.f;
    }
    return;
  }
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  const float* qs = tab + row * 4 * (int64_t)T;
  const float* cm = qs + T;
  const float* lf = cm + T;
  const float* esp = lf + T;
  float* in_c = tc + ((int64_t)s * P + row) * V;
  float* in_p = tp + ((int64_t)s * P + row) * V;
  float* st_c = tc + ((int64_t)(s + 1) * P + row) * V;
  float* st_p = tp + ((int64_t)(s + 1) * P + row) * V;
  if (wid == 0) {
    const bool on = lane < V;
    const float c = on && s > 0 ? in_c[lane] : 0.f;
    float p = !on ? 0.f : (s == 0 ? (lane == 0 ? 0.f : -1000.f) : in_p[lane]);
    if (on && s == 0) {  // the start paths, for the adjoint
      in_c[lane] = c;
      in_p[lane] = p;
    }
    int group;
    bool lead;
    const int nv = pf_merge_paths(V, lane, c, p, group, lead);
    if (lead) {
      s_c[group] = c;
      s_p[group] = p;
    }
    if (lane == 0) s_nv = nv;
  }
  int nrun, ngroup;
  pf_runs(d, qs, cm, S, s_sh, &s_nrun, nrun);  // (its barriers complete the merged paths)
  pf_groups(d, S, s_did, s_first, s_sh, &s_ngroup, ngroup);
  const int NV = s_nv;
  float hmax[kPfChunk], hsum[kPfChunk], gmax[kPfChunk], gsum[kPfChunk];
  float we[kPfChunk];         // weight of the expected-charge mask, one per tick for every path
  int ca[kPfChunk], qa[kPfChunk];  // runs of CM[t + 1] << 16 | CM[t], and of q_sum[sh] << 16 | q_sum[t]
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k) {
    hmax[k] = -__builtin_inff();
    gmax[k] = -__builtin_inff();
    hsum[k] = 0.f;
    gsum[k] = 0.f;
    we[k] = 0.f;
    ca[k] = qa[k] = 0;
    const int g = k * kPfThreads + threadIdx.x;
    if (g < ngroup) {
      const int t = s_first[g];
      const float x = (esp[t] - d.theta) * 10.f;
      we[k] = x > 30.f ? 1.f : (x < -30.f ? expf(x) : 1.f / (1.f + expf(-x)));
      ca[k] = S.cid[t + 1] << 16 | S.cid[t];
      qa[k] = S.rid[min(t + d.interval + 1, T - 1)] << 16 | S.rid[t];
    }
  }
  const float none = pf_log_one_minus(d.minus_one);
  // one pass over the (merged) paths with running logsumexp accumulators (max and shifted sum)
  for (int v = 0; v < NV; ++v) {
    const float c = s_c[v], pv = s_p[v];
    for (int r = threadIdx.x; r <= nrun; r += kPfThreads) s_tab[r] = pf_log_ndtr((S.rv[r] - c - d.theta) * d.zs);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPfChunk; ++k) {
      if (k * kPfThreads + (int)threadIdx.x < ngroup) {
        const int c1 = ca[k] >> 16, c0 = ca[k] & 0xffff, q1 = qa[k] >> 16, q0 = qa[k] & 0xffff;
        const float a1 = (S.rv[c1] - c - d.theta) * d.zs, b1 = (S.rv[c0] - c - d.theta) * d.zs;
        const float lg = pf_log_diff(a1, b1, s_tab[c1], s_tab[c0], none);
        const float a2 = (S.rv[q1] - c - d.theta) * d.zs, b2 = (S.rv[q0] - c - d.theta) * d.zs;
        float le = pf_log_diff(a2, b2, s_tab[q1], s_tab[q0], none);
        le = fminf(le, lg);
        le = pf_soft_max(le, -1000.f, 1.f);
        le = we[k] * le + (1.f - we[k]) * -1000.f;
        pf_lse_add(hmax[k], hsum[k], le + pv);
        pf_lse_add(gmax[k], gsum[k], lg + pv);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k) {
    const int g = k * kPfThreads + threadIdx.x;
    if (g < ngroup) {
      s_tab[g] = hmax[k] + logf(hsum[k]);
      s_tot[g] = gmax[k] + logf(gsum[k]);
    }
  }
  __syncthreads();
  // outputs, and the selection scores as ordered keys: score, then the lower tick (NaN: 0, never taken
  // before a number)
  uint64_t key[kPfChunk];
  auto score_key = [&](float v, int t) {
    const uint32_t b = __float_as_uint(v + 0.f);
    const uint32_t u = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    return v == v ? (uint64_t)u << 32 | (uint32_t)(0x7fffffff - t) : 0ull;
  };
  uint64_t best = 0;
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k) {
    const int t = k * kPfThreads + threadIdx.x;
    key[k] = 0;
    if (t < n) {
      const int g = s_did[t];
      ol[t] = s_tab[g];
      oq[t] = esp[t];
      key[k] = score_key(lf[t] + s_tot[g], t);
    }
    best = key[k] > best ? key[k] : best;
  }
  // top V ticks of select, lower tick first on ties: V rounds of one barrier; the thread that held the
  // round's tick (its score becomes -inf) finds its next best
  for (int r = 0; r < V; ++r) {
    uint64_t m = best;
#pragma unroll
    for (int dd = kWave / 2; dd > 0; dd >>= 1) {
      const uint64_t o = __shfl_xor(m, dd, kWave);
      m = o > m ? o : m;
    }
    if (lane == 0) s_key[r & 1][wid] = m;
    __syncthreads();  // (round r + 1 writes the other row)
    for (int w = 0; w < kPfThreads / kWave; ++w) m = s_key[r & 1][w] > m ? s_key[r & 1][w] : m;
    int i0 = 0x7fffffff - (int)(uint32_t)m;
    if (m == 0 || i0 >= n) i0 = 0;  // no number left (cannot happen for finite inputs)
    if (threadIdx.x == 0) s_top[r] = i0;
    if (i0 % kPfThreads == (int)threadIdx.x) {
      best = 0;
#pragma unroll
      for (int k = 0; k < kPfChunk; ++k) {
        if (k == i0 / kPfThreads) key[k] = score_key(-__builtin_inff(), i0);
        best = key[k] > best ? key[k] : best;
      }
    }
  }
  __syncthreads();
  if (wid != 0) return;
  float tot = -__builtin_inff();
  if (lane < V) {
    const int t = s_top[lane];
    const int nx = min(min(t + d.interval + 1, T - 1) + 1, T - 1);
    tot = s_tot[s_did[t]];
    st_c[lane] = S.rv[S.rid[nx]];
    st_p[lane] = tot;
    tk[((int64_t)s * P + row) * V + lane] = t;
  }
  float m = -__builtin_inff();
  for (int v = 0; v < V; ++v) m = fmaxf(m, __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tot), v)));
  const float ex = lane < V ? expf(tot - m) : 0.f;
  float sum = 0.f;
  for (int v = 0; v < V; ++v) sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ex), v));
  if (lane == 0 && m + logf(sum) > d.log_stop) atomicOr(flags + s + 1, 1);
}

// ------------------------------------------------------------------------------------------
// Adjoint of the beam search
// ------------------------------------------------------------------------------------------
//
// Reverse-mode derivative of (out_logp, out_q) with respect to the waveforms, with the path
// selections held fixed (top_k is under stop_gradient in the reference, fee_jax.py:377), as
// jax.grad takes it.  Per executed step s, in reverse, with G and Gq the cotangents of out_logp[s]
// and out_q[s] and (dc', dp') those of the paths the step selected:
//   p'_k = total[t_k]  -> d total[t_k] += dp'_k;  c'_k = q_sum[nx(t_k)] -> d q_sum[nx(t_k)] += dc'_k
//   total[t] = lse_v(lg[v,t] + p_v), out_logp[t] = lse_v(le[v,t] + p_v): softmax weights to lg, le, p
//   le = soft_where(esp - theta, soft_max(min(ld, lg), -1000, 1), -1000, 10)   (ties of min: half each)
//   ld = logdiffPhi(z(q_sum[sh] - c), z(q_sum[t] - c)), lg = logdiffPhi(z(CM[t+1] - c), z(CM[t] - c))
//   esp[t] = q_sum[sh] + theta - (q_sum[t+1] + q_sum[t]) / 2
// which gives d q_sum, d CM and, per path, d c and d p; paths merged in the forward (equal charge)
// share their group's derivative in proportion exp(p_v - p_group).  Then CM = cummax(q_sum): each
// d CM[t] goes to the last tick <= t where q_sum attains the running maximum (torch.cummax's
// choice; jax splits ties, a corner no fixture reaches).  Finally q_sum = cumsum(wfs t_sampling):
// d wfs[t] = t_sampling * sum_{u >= t} d q_sum[u].  Sums over paths and steps are float64, in a
// fixed order.

// d log(Phi(a) - Phi(b)) with the smooth clamps of pf_log_diff (fee_jax.py:32-54): returns the value
// and, for a cotangent g on it, the cotangents of a and b.
__device__ __forceinline__ float pf_sigmoid(float x) {
  return x > 30.f ? 1.f : (x < -30.f ? expf(x) : 1.f / (1.f + expf(-x)));
}

// d log Phi(x) / dx = phi(x) / Phi(x), from lx = log Phi(x)
__device__ __forceinline__ float pf_dlog_ndtr(float x, float lx) {
  return expf(-0.5f * x * x - lx) * 0.3989422804014327f;
}

// The cotangents of a and b for a cotangent g on pf_log_diff(a, b, la, lb, none); da, db = d log Phi / dx
// at a and b (pf_dlog_ndtr).
__device__ __forceinline__ void pf_log_diff_adj(float a, float b, float la, float lb, float da, float db, float none, float g,
                                                float& ga, float& gb) {
  float lt2 = none, g_sd = 0.f;
  const float w = a == b ? 0.5f : pf_sigmoid((a - b) * 1000.f);
  const float g_lp = w * g;
  if (a > b) {
    const float sd = lb - la;
    const float ne = -expm1f(sd);
    const float ne2 = pf_soft_max(ne, 1e-30f, 1e10f);
    const float lt = logf(ne2);
    lt2 = pf_soft_max(lt, -100.f, 10.f);
    const float g_lt = g_lp * pf_sigmoid((lt + 100.f) * 10.f);
    const float g_ne = g_lt / ne2 * pf_sigmoid((ne - 1e-30f) * 1e10f);
    g_sd = -expf(sd) * g_ne;
  }
  const float lp = la + lt2;
  const float g_amb = 1000.f * w * (1.f - w) * (lp + 1000.f) * g;
  const float g_la = g_lp - g_sd;
  const float g_lb = g_sd;
  ga = g_la * da + g_amb;
  gb = g_lb * db - g_amb;
}

template <typename T>
__device__ __forceinline__ T pf_block_sum(T v, T* sh) {
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
#pragma unroll
  for (int m = kWave / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m, kWave);
  if (lane == 0) sh[wid] = v;
  __syncthreads();
  T tot = 0;
  for (int w = 0; w < kPfThreads / kWave; ++w) tot += sh[w];
  __syncthreads();
  return tot;
}

// Two block sums at once (each wave's by shuffles, the waves in order); sh: two rows of the waves' values,
// which the next call may overwrite only after another barrier.
__device__ __forceinline__ void pf_block_sum2(double& u, double& v, double (*sh)[kPfThreads / kWave]) {
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
#pragma unroll
  for (int m = kWave / 2; m >= 1; m >>= 1) {
    u += __shfl_xor(u, m, kWave);
    v += __shfl_xor(v, m, kWave);
  }
  if (lane == 0) {
    sh[0][wid] = u;
    sh[1][wid] = v;
  }
  __syncthreads();
  u = v = 0.0;
  for (int w = 0; w < kPfThreads / kWave; ++w) {
    u += sh[0][w];
    v += sh[1][w];
  }
}

// One workgroup per row: every executed step in reverse, then the cumulative max and sum.
//
// log Phi and its derivative are evaluated once per run of q_sum and path.  The ticks are laid on the
// threads by kind (does CM rise at t + 1; does the held charge differ): where neither does, log_guess and
// log_event have no transcendental function of their own, and the waves that hold only such ticks (four
// fifths of a row with a few pulses) skip them.  The sums are per tick in float64, as before.
__global__ __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(2))) void k_pf_adj(PfDev d, const float* __restrict__ tab, int64_t P,
                                                      const float* __restrict__ tc, const float* __restrict__ tp,
                                                      const int* __restrict__ tk, const int* __restrict__ flags,
                                                      const float* __restrict__ out_logp,
                                                      const float* __restrict__ g_logp, const float* __restrict__ g_q,
                                                      float* __restrict__ d_wfs) {
  __shared__ PfShare S;
  __shared__ double s_buf[kPfMaxTicks + 1];  // per-path tables by run: log Phi, then its derivative; at the end d q_sum
  float* const s_lq = (float*)s_buf;
  float* const s_dl = s_lq + kPfMaxTicks + 1;
  __shared__ short s_perm[kPfMaxTicks];  // position -> tick, by kind
  __shared__ short s_kof[kPfMaxTicks];   // selected tick -> its path slot k, -1 elsewhere
  __shared__ double s_dqx[kPfMaxTicks];  // d q_sum at the selected paths' reset ticks; at the end d CM
  __shared__ float s_mc[kPfMaxPaths], s_mp[kPfMaxPaths], s_tot[kPfMaxPaths];
  __shared__ float s_dtk[kPfMaxPaths];   // d total at the selected ticks, by path slot
  __shared__ double s_dcm[kPfMaxPaths], s_dpm[kPfMaxPaths];
  __shared__ double s_red[kPfThreads / kWave], s_red2[2][2][kPfThreads / kWave];
  __shared__ int s_sh[kPfThreads / kWave], s_nrun, s_nv;
  const int64_t row = blockIdx.x;
  const int T = d.T, V = d.V, n = T - 1;
  const int t0 = threadIdx.x * kPfChunk;
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
  const float* qs = tab + row * 4 * (int64_t)T;
  const float* cm = qs + T;
  const float* espg = cm + 2 * T;
  int nrun;
  pf_runs(d, qs, cm, S, s_sh, &s_nrun, nrun);
  for (int t = threadIdx.x; t < T; t += kPfThreads) {
    s_dqx[t] = 0.0;
    s_kof[t] = -1;
  }
  // positions: ticks by kind (2 bits), in tick order within a kind
  {
    int kind[kPfChunk], lo = 0, hi = 0;  // counts of kinds 0 and 1, of 2 and 3 (16 bits each)
#pragma unroll
    for (int k = 0; k < kPfChunk; ++k) {
      const int t = t0 + k;
      kind[k] = -1;
      if (t < n) {
        kind[k] = (S.cid[t + 1] != S.cid[t] ? 2 : 0) + (S.rid[min(t + d.interval + 1, T - 1)] != S.rid[t] ? 1 : 0);
        (kind[k] < 2 ? lo : hi) += 1 << (16 * (kind[k] & 1));
      }
    }
    const int ilo = pf_block_scan_i<false>(lo, s_sh), ihi = pf_block_scan_i<false>(hi, s_sh);
    if (threadIdx.x == kPfThreads - 1) {
      s_sh[0] = ilo;
      s_sh[1] = ihi;
    }
    __syncthreads();
    const int tl = s_sh[0];
    const int th = s_sh[1];
    int at[4] = {(ilo - lo) & 0xffff, (tl & 0xffff) + ((ilo - lo) >> 16), (tl & 0xffff) + (tl >> 16) + ((ihi - hi) & 0xffff),
                 (tl & 0xffff) + (tl >> 16) + (th & 0xffff) + ((ihi - hi) >> 16)};
#pragma unroll
    for (int k = 0; k < kPfChunk; ++k)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (kind[k] == c) s_perm[at[c]++] = (short)(t0 + k);
  }
  __syncthreads();
  // per position (own slots): d q_sum[t], d q_sum[t+1], d q_sum[sh(t)], d CM[t], d CM[t+1]
  double aq[kPfChunk], bq[kPfChunk], cq[kPfChunk], dc0[kPfChunk], dc1[kPfChunk];
  int ca[kPfChunk], qa[kPfChunk];  // runs of CM[t + 1] << 16 | CM[t], and of q_sum[sh] << 16 | q_sum[t]
  auto tick_of = [&](int k) {  // of slot k of this thread, -1: none
    const int i = k * kPfThreads + (int)threadIdx.x;
    return i < n ? (int)s_perm[i] : -1;
  };
  float we[kPfChunk];
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k) {
    aq[k] = bq[k] = cq[k] = dc0[k] = dc1[k] = 0.0;
    const int i = k * kPfThreads + threadIdx.x;
    ca[k] = qa[k] = 0;
    we[k] = 0.f;
    if (i < n) {
      const int t = s_perm[i];
      ca[k] = S.cid[t + 1] << 16 | S.cid[t];
      qa[k] = S.rid[min(t + d.interval + 1, T - 1)] << 16 | S.rid[t];
      we[k] = pf_sigmoid((espg[t] - d.theta) * 10.f);
    }
  }
  int n_run = 0;
  while (n_run < d.S && flags[n_run]) ++n_run;
  const float none = pf_log_one_minus(d.minus_one);
  double dcN = 0.0, dpN = 0.0;  // wave 0, lane v < V: cotangents of the paths that the step selected
  for (int s = n_run - 1; s >= 0; --s) {
    const float* ol = out_logp + (row * d.S + s) * (int64_t)n;
    const float* gl = g_logp + (row * d.S + s) * (int64_t)n;
    const float* gq = g_q + (row * d.S + s) * (int64_t)n;
    float c_v = 0.f, p_v = 0.f, mp_v = 0.f;
    int grp = 0, t_v = 0;
    if (wid == 0) {
      int nx = -1;
      if (lane < V) {
        c_v = tc[((int64_t)s * P + row) * V + lane];
        p_v = tp[((int64_t)s * P + row) * V + lane];
        s_tot[lane] = tp[((int64_t)(s + 1) * P + row) * V + lane];  // total[t_k] of this step's selections
        t_v = tk[((int64_t)s * P + row) * V + lane];
        s_dtk[lane] = (float)dpN;
        s_kof[t_v] = (short)lane;
        nx = min(min(t_v + d.interval + 1, T - 1) + 1, T - 1);
      }
      // c'_k = q_sum[nx(t_k)]: in slot order (several k can share a reset tick), by the first lane of a tick
      bool lead_nx = lane < V;
      double acc = lead_nx ? s_dqx[nx] : 0.0;
      for (int u = 0; u < V; ++u) {
        const int nu = __builtin_amdgcn_readlane(nx, u);
        const double du = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(dcN), u),
                                           __builtin_amdgcn_readlane(__double2loint(dcN), u));
        if (nu == nx) {
          acc += du;
          if (u < lane) lead_nx = false;
        }
      }
      if (lead_nx) s_dqx[nx] = acc;
      // the forward's merge of equal-charge paths
      mp_v = p_v;
      bool lead;
      const int nv = pf_merge_paths(V, lane, c_v, mp_v, grp, lead);
      if (lead) {
        s_mc[grp] = c_v;
        s_mp[grp] = mp_v;
      }
      if (lane == 0) s_nv = nv;
    }
    __syncthreads();
    const int NV = s_nv;
    float gk[kPfChunk], olk[kPfChunk], desp[kPfChunk];
#pragma unroll
    for (int k = 0; k < kPfChunk; ++k) {
      const int t = tick_of(k);
      gk[k] = t >= 0 ? gl[t] : 0.f;
      olk[k] = t >= 0 ? ol[t] : 0.f;
      desp[k] = 0.f;
    }
    for (int u = 0; u < NV; ++u) {
      const float c = s_mc[u], pv = s_mp[u];
      for (int r = threadIdx.x; r <= nrun; r += kPfThreads) {
        const float x = (S.rv[r] - c - d.theta) * d.zs;
        const float l = pf_log_ndtr(x);
        s_lq[r] = l;
        s_dl[r] = pf_dlog_ndtr(x, l);
      }
      __syncthreads();
      double dcu = 0.0, dpu = 0.0;
#pragma unroll
      for (int k = 0; k < kPfChunk; ++k) {
        if (k * kPfThreads + (int)threadIdx.x < n) {
          const int c1 = ca[k] >> 16, c0 = ca[k] & 0xffff, q1 = qa[k] >> 16, q0 = qa[k] & 0xffff;
          const float a1 = (S.rv[c1] - c - d.theta) * d.zs, b1 = (S.rv[c0] - c - d.theta) * d.zs;
          const float a2 = (S.rv[q1] - c - d.theta) * d.zs, b2 = (S.rv[q0] - c - d.theta) * d.zs;
          // values first (the cotangents of ld and lg depend on them)
          float ga1, gb1, ga2, gb2;
          const float lg = pf_log_diff(a1, b1, s_lq[c1], s_lq[c0], none);
          const float ld = pf_log_diff(a2, b2, s_lq[q1], s_lq[q0], none);
          const float mn = fminf(ld, lg);
          const float sm = pf_soft_max(mn, -1000.f, 1.f);
          const float le = we[k] * sm + (1.f - we[k]) * (-1000.f);
          // out_logp = lse(le + p): softmax weight of this path
          const float wh = expf(le + pv - olk[k]);
          const float g_le = gk[k] * wh;
          dpu += (double)g_le;
          float g_lg = 0.f;
          const int kk = s_kof[tick_of(k)];
          if (kk >= 0) {  // total[t] = lse(lg + p) feeds a selected path
            const float wt = expf(lg + pv - s_tot[kk]);
            const float g = s_dtk[kk] * wt;
            g_lg += g;
            dpu += (double)g;
          }
          desp[k] += g_le * (sm + 1000.f) * 10.f * we[k] * (1.f - we[k]);
          const float g_mn = g_le * we[k] * pf_sigmoid(mn + 1000.f);
          float g_ld = 0.f;
          if (ld < lg) g_ld = g_mn;
          else if (lg < ld) g_lg += g_mn;
          else {
            g_ld = 0.5f * g_mn;
            g_lg += 0.5f * g_mn;
          }
          pf_log_diff_adj(a2, b2, s_lq[q1], s_lq[q0], s_dl[q1], s_dl[q0], none, g_ld, ga2, gb2);
          pf_log_diff_adj(a1, b1, s_lq[c1], s_lq[c0], s_dl[c1], s_dl[c0], none, g_lg, ga1, gb1);
          cq[k] += (double)(d.zs * ga2);
          aq[k] += (double)(d.zs * gb2);
          dc1[k] += (double)(d.zs * ga1);
          dc0[k] += (double)(d.zs * gb1);
          dcu -= (double)(d.zs * (ga1 + gb1 + ga2 + gb2));
        }
      }
      pf_block_sum2(dcu, dpu, s_red2[u & 1]);  // (its barrier: the tables have been read)
      if (threadIdx.x == 0) {
        s_dcm[u] = dcu;
        s_dpm[u] = dpu;
      }
    }
    __syncthreads();
    // esp[t] = q_sum[sh] + theta - (q_sum[t+1] + q_sum[t]) / 2
#pragma unroll
    for (int k = 0; k < kPfChunk; ++k) {
      if (const int t = tick_of(k); t >= 0) {
        const double ge = (double)desp[k] + (double)gq[t];
        cq[k] += ge;
        bq[k] -= 0.5 * ge;
        aq[k] -= 0.5 * ge;
      }
    }
    // cotangents of the paths entering this step (the previous step's selections)
    if (wid == 0 && lane < V) {
      const double share = (double)expf(p_v - s_mp[grp]);
      dcN = s_dcm[grp] * share;
      dpN = s_dpm[grp] * share;
      s_kof[t_v] = -1;
    }
    __syncthreads();
  }
  // d q_sum: own ticks, then t + 1, then sh(t) (injective below the clamp), the clamped ticks sh(t) = T - 1
  // together
  double* dqs = s_buf;
  double* dcmv = s_dqx;
  for (int t = threadIdx.x; t < T; t += kPfThreads) dqs[t] = s_dqx[t];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k)
    if (const int t = tick_of(k); t >= 0) {
      dqs[t] += aq[k];
      dcmv[t] = dc0[k];
    }
  if (threadIdx.x == 0) dcmv[n] = 0.0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k)
    if (const int t = tick_of(k); t >= 0) {
      dqs[t + 1] += bq[k];
      dcmv[t + 1] += dc1[k];
    }
  __syncthreads();
  const int t_clamp = T - 1 - d.interval - 1;  // ticks t >= t_clamp have sh(t) = T - 1
  double cl = 0.0;
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k)
    if (const int t = tick_of(k); t >= 0) {
      if (t < t_clamp) dqs[t + d.interval + 1] += cq[k];
      else cl += cq[k];
    }
  cl = pf_block_sum<double>(cl, s_red);
  if (threadIdx.x == 0) dqs[T - 1] += cl;
  __syncthreads();
  // CM = cummax(q_sum): d CM[t] to the last tick <= t where q_sum reaches the running maximum (tick 0 before
  // any).  Chunk by chunk: a run of d CM that began in an earlier chunk is carried over the threads by a
  // segmented scan of (sum since the last such tick, is there one).
  {
    double since = 0.0;
    bool any = false;
    int last = 0;
#pragma unroll
    for (int k = 0; k < kPfChunk; ++k) {
      const int t = t0 + k;
      if (t < T) {
        if (t == 0 || S.rv[S.rid[t]] == S.rv[S.cid[t]]) {
          since = 0.0;
          any = true;
          last = t;
        }
        since += dcmv[t];
      }
    }
    // inclusive over the wave's threads: sum since the last attaining tick, and whether there was one
    double sum = since;
    int has = any ? 1 : 0, at = last;
#pragma unroll
    for (int dd = 1; dd < kWave; dd <<= 1) {
      const double us = __shfl_up(sum, dd, kWave);
      const int uh = __shfl_up(has, dd, kWave), ua = __shfl_up(at, dd, kWave);
      if (lane >= dd && !has) {
        sum += us;
        has = uh;
        at = ua;
      }
    }
    __shared__ int s_has[kPfThreads / kWave], s_at[kPfThreads / kWave];
    if (lane == kWave - 1) {
      s_red[wid] = sum;
      s_has[wid] = has;
      s_at[wid] = at;
    }
    __syncthreads();
    // what reaches this thread's chunk from before it
    double in_s = __shfl_up(sum, 1, kWave);
    int in_h = __shfl_up(has, 1, kWave), in_a = __shfl_up(at, 1, kWave);
    if (lane == 0) {
      in_s = 0.0;
      in_h = 0;
      in_a = 0;
    }
    for (int w = wid - 1; w >= 0 && !in_h; --w) {
      in_s += s_red[w];
      in_h = s_has[w];
      in_a = s_at[w];
    }
    // each attaining tick receives its run's sum when the run ends: at the next one, or at the row's end
    double acc = in_s;
    int cur = in_a;
#pragma unroll
    for (int k = 0; k < kPfChunk; ++k) {
      const int t = t0 + k;
      if (t < T) {
        if (t == 0 || S.rv[S.rid[t]] == S.rv[S.cid[t]]) {
          if (t > 0) dqs[cur] += acc;
          acc = 0.0;
          cur = t;
        }
        acc += dcmv[t];
        if (t == T - 1) dqs[cur] += acc;
      }
    }
  }
  __syncthreads();
  // d wfs[t] = t_sampling * sum_{u >= t} d q_sum[u]: chunk sums, an exclusive suffix scan over
  // threads, then the walk down the chunk
  double loc = 0.0;
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k)
    if (t0 + k < T) loc += dqs[t0 + k];
  const double incl = pf_block_scan(loc, s_red);  // inclusive prefix over threads
  const double total = pf_block_sum<double>(loc, s_red);
  double suffix = total - incl + loc;  // sum over u >= t0
  float* dw = d_wfs + row * (int64_t)T;
#pragma unroll
  for (int k = 0; k < kPfChunk; ++k) {
    const int t = t0 + k;
    if (t < T) {
      dw[t] = (float)(suffix * d.ts);
      suffix -= dqs[t];
    }
  }
}

}  // namespace lsim
