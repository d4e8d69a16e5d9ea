// Adjoint of the LUT chain for the 7 physics parameters (Ab, kb, eField, lifetime, vdrift,
// long_diff, tran_diff).  Integer decisions are held at their forward values, as reverse-mode
// AD through the reference does (floor/astype/searchsorted/argmax carry no gradient).
//
// Stage 1 (one thread per pixel row): the self-trigger adjoint.  The ADC value of pass k is
// Q^(k)[e_k]; pass k then sets Q^(k+1) = max(Q^(k) - Q^(k)[g_k], 0).  Reverse mode over the 2H
// tracked points gives the adjoint of Q^(0), and because Q^(0) is the cumulative sum of
// t_sampling * wfs, d loss / d wfs is piecewise constant with at most 2H steps.
// Stage 2 (one workgroup per pixel row, like the forward's waveform kernel): for every segment
// whose stripes reach the row, inner products of the row's step function with the segment's
// template windows come from window prefix sums; they give d loss / d (charge, transverse width,
// fractional tick, longitudinal width) of the pair, which the per-segment chain factors
// (k_adj_records) turn into the 7 gradients; a fixed-order block reduction writes per-row
// partial gradients.
// Stage 3: fixed-order reduction of the partials (and of the hit-z term) to 7 values.
#pragma once
#include "forward.h"

namespace lsim {

constexpr int kNGrad = 7;
// waves per pixel-row workgroup of the adjoint; the bins' pass has few pairs a row (2 waves 414, 4 476, 1 556 us
// for 200k segments, where the stripes' takes 403, 352 and 490)
constexpr int kAdjWaves = 4, kAdjNearWaves = 2;

__device__ __forceinline__ double readlane_d(double v, int j) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), j);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), j);
  return __hiloint2double(hi, lo);
}

// One wave per row (kFeeRows rows per workgroup).  Lane j < 2H follows tracked point j: the reverse
// pass over the H self-trigger passes keeps A[j] = d loss / d Q at point j in lane j, each pass's
// masked sum taken in point order; the points are then merged by tick (lane-parallel: the first
// lane of a tick owns it and sums the lanes of that tick in lane order), and lane 0 turns the
// per-tick jumps into the step function (suffix sums, equal neighbours merged, zero tail dropped).
constexpr int kFeeRows = 4;

__global__ __launch_bounds__(kFeeRows * kWave) void k_fee_adjoint(Dev d, const FeeTape* __restrict__ tape,
                                                                  const float* __restrict__ d_adc,
                                                                  const float* __restrict__ d_z,
                                                                  const int64_t* __restrict__ n_rows_dev, int64_t max_rows,
                                                                  Pieces* __restrict__ pieces, double* __restrict__ dz_part) {
  __shared__ int spos[kFeeRows][2 * kMaxH];
  __shared__ double sval[kFeeRows][2 * kMaxH];
  __shared__ int sx[kFeeRows][2 * kMaxH];
  __shared__ float sc[kFeeRows][2 * kMaxH];
  __shared__ int sn[kFeeRows];
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const int64_t r = (int64_t)blockIdx.x * kFeeRows + wv;
  int64_t P = *n_rows_dev;
  if (P > max_rows) P = max_rows;
  if (r >= max_rows) return;
  if (r >= P) {
    if (lane == 0) dz_part[r] = 0.0;
    return;
  }
  const FeeTape* tp = tape + r;
  const int H = d.H, np2 = 2 * H;
  const bool act = lane < np2;
  // everything the passes read, loaded at once: lane k < H holds pass k's mask and ADC term
  const int p = act ? (int)tp->pt[lane] : 0x7fffffff;
  const int mk = lane < H ? (int)tp->mask[lane] : 0;
  const double gk = lane < H ? (double)d_adc[r * H + lane] * (double)tp->slope[lane] : 0.0;
  double zk = 0.0;
  if (d_z && lane < H) {
    const int pl = tp->plane;
    const double za = d.tpc[pl][2][0], zc = d.tpc[pl][2][1];
    const double sgn = (zc - za) > 0 ? 1.0 : ((zc - za) < 0 ? -1.0 : 0.0);
    zk = (double)d_z[r * H + lane] * (double)tp->tick[lane] * d.ts * sgn;
  }
  double A = 0.0;
  for (int k = H - 1; k >= 0; --k) {
    const uint32_t m = (uint32_t)__builtin_amdgcn_readlane(mk, k);
    double s = 0.0;
    for (int j = 0; j < np2; ++j) {
      const double aj = readlane_d(A, j);
      if ((m >> j) & 1u) s += aj;
    }
    if (act && !((m >> lane) & 1u)) A = 0.0;
    if (lane == H + k) A -= s;
    if (lane == k) A += gk;
  }
  double dz = 0.0;  // d loss / d vdrift_eff through the hit z positions, summed in pass order
  for (int k = 0; k < H; ++k) dz += readlane_d(zk, k);
  // merge the points by tick
  bool owner = act;
  double val = 0.0;
  for (int j = 0; j < np2; ++j) {
    const int pj = __builtin_amdgcn_readlane(p, j);
    const double aj = readlane_d(A, j);
    if (act && pj == p) {
      val += aj;
      if (j < lane) owner = false;
    }
  }
  int rank = 0;
  for (int j = 0; j < np2; ++j) {
    const int pj = __builtin_amdgcn_readlane(p, j);
    const int oj = __builtin_amdgcn_readlane(owner ? 1 : 0, j);
    if (oj && pj < p) ++rank;
  }
  if (owner) {
    spos[wv][rank] = p;
    sval[wv][rank] = val;
  }
  const int n = __popcll(__ballot(owner));
  // wave-local LDS: stores and loads of one wave complete in program order; the wave barriers
  // keep the compiler from moving them across
  __builtin_amdgcn_wave_barrier();
  if (lane == 0) {
    // step values G on (pos[q-1], pos[q]]: suffix sums of the jumps
    double suf = 0.0;
    for (int q = n - 1; q >= 0; --q) {
      suf += sval[wv][q];
      sc[wv][q] = (float)(suf * d.ts);
    }
    // keep only the steps where G changes, then drop a zero tail
    int m = 0;
    float last = 0.f;
    for (int q = 0; q < n; ++q) {
      const float cq = sc[wv][q];
      if (m > 0 && cq == last) {
        sx[wv][m - 1] = spos[wv][q];  // same value: extend the previous piece
      } else {
        sx[wv][m] = spos[wv][q];
        sc[wv][m] = cq;
        last = cq;
        ++m;
      }
    }
    while (m > 0 && sc[wv][m - 1] == 0.f) --m;
    sn[wv] = m;
    dz_part[r] = dz;
  }
  __builtin_amdgcn_wave_barrier();
  const int mm = __builtin_amdgcn_readfirstlane(sn[wv]);
  Pieces* pc = pieces + r;
  if (lane == 0) {
    pc->n = mm;
    pc->pad[0] = pc->pad[1] = pc->pad[2] = 0;
  }
  if (lane < 2 * kMaxH) {
    pc->x[lane] = lane < mm ? sx[wv][lane] : 0x7fffffff;
    pc->c[lane] = lane < mm ? sc[wv][lane] : 0.f;
  }
}

// Per-segment factors of the chain rule, in the same (sorted) order as the SegRec records.
struct __align__(16) AdjRec {
  double fN[4];          // d n_e / d (Ab, kb, eField, lifetime)
  double fS[2];          // d sigma_T / d (eField, tran_diff)
  double fL[2];          // d lambda / d (eField, long_diff)
  double fF;             // d f / d eField
  double dl[3];          // d (a, b, c) / d lambda of the Lagrange weights
  float dwx[5], dwy[5];  // d w / d sigma_T of the transverse weights
  float pad[2];
};
static_assert(sizeof(AdjRec) == 144, "AdjRec layout");

// One thread per record: recompute the segment's physics (float64) and store the chain factors.
__global__ __launch_bounds__(256) void k_adj_records(Dev d, SegIn in, const uint32_t* __restrict__ keys,
                                                     const uint32_t* __restrict__ vals, int64_t n,
                                                     AdjRec* __restrict__ adj) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n || keys[s] >= (uint32_t)d.n_cells) return;
  Phys ph;
  seg_physics(d, in, vals[s], ph);
  double wx[kMaxNb], wy[kMaxNb], dwx[kMaxNb], dwy[kMaxNb];
  tran_weights(d, ph.x0, ph.st, wx, dwx);
  tran_weights(d, ph.y0, ph.st, wy, dwy);
  const double v = d.v, dv = d.dv;
  const double att = exp(-ph.td / d.lifetime) * (double)ph.mask;
  AdjRec A;
  A.fN[0] = ph.dq_dAb * att;
  A.fN[1] = ph.dq_dkb * att;
  A.fN[2] = ph.dq_dE_rec * att + ph.ne * ph.td * dv / (v * d.lifetime);
  A.fN[3] = ph.ne * ph.td / (d.lifetime * d.lifetime);
  A.fS[0] = -ph.st * dv / (2 * v);
  A.fS[1] = d.tran_diff > 0 ? ph.st / (2 * d.tran_diff) : 0.0;
  A.fL[0] = -1.5 * ph.lam * dv / v;
  A.fL[1] = d.long_diff > 0 ? ph.lam / (2 * d.long_diff) : 0.0;
  A.fF = -ph.tau * dv / v;
  const double s0 = d.sig[ph.idx - 1], s1 = d.sig[ph.idx], s2 = d.sig[ph.idx + 1];
  const double l = ph.lam;
  A.dl[0] = (2 * l - s1 - s2) / ((s0 - s1) * (s0 - s2));
  A.dl[1] = (2 * l - s0 - s2) / ((s1 - s0) * (s1 - s2));
  A.dl[2] = (2 * l - s0 - s1) / ((s2 - s0) * (s2 - s1));
#pragma unroll
  for (int k = 0; k < kMaxNb; ++k) {
    A.dwx[k] = k < d.nb ? (float)dwx[k] : 0.f;
    A.dwy[k] = k < d.nb ? (float)dwy[k] : 0.f;
  }
  A.pad[0] = A.pad[1] = 0.f;
  adj[s] = A;
}

// The row's step function G in LDS: breakpoints x[q] (ascending) and values c[q], G(o) = c[q] on
// (x[q-1], x[q]] and 0 past x[np-1]; jumps dc[q] = c[q] - c[q+1] (c[np] = 0); and qlut[o] = the first
// q with x[q] >= o, for 0 <= o < nout (np when none).
struct RowG {
  const int* x;
  const float* c;
  const float* dc;
  const uint16_t* qlut;
  int np;
  __device__ __forceinline__ double at(int o) const {  // G(o), 0 <= o < nout
    const int q = qlut[o];
    return q < np ? (double)c[q] : 0.0;
  }
};

// Window placement of one (segment, row) pair (sim_jax.py:170-261): (1-f) V at o = S + j, f V at
// o = S - 1 + j, (1-f) Delta at S - 1 and f Delta at S - 2, S = nt - L - k0; G's values at the two
// correction ticks and the tick ranges of the two windows kept in the row.
struct PairCtx {
  int S, lo1, hi1, lo0, hi0;
  bool interior;  // both windows whole: lo1 = S, hi1 = S + L - 1, lo0 = S - 1, hi0 = S + L - 2
  double f, ne, gc0, gc1, gc;
};

// Window dot products of one (segment, row) pair, telescoped over G's breakpoints.  With
// CX[k] = sum_{j<k} X[j] and F(o) = CX[o - S + sh + 1],
//   sum_{o=lo}^{hi} G(o) X[o - S + sh] = G(hi) F(hi) - G(lo) F(lo - 1) + sum_{lo <= x_q < hi} dc_q F(x_q),
// so each breakpoint inside the window costs one prefix-sum load per table.  y1: the (1-f) window
// (sh = 0, o in [lo1, hi1]); y0: the f window (sh = 1, o in [lo0, hi0]).  NT tables at stride ts.
// Whole windows take fewer loads: F(lo - 1) = CX[0] = 0, both F(hi) are CX[L], and a breakpoint
// needs the adjacent CX[x_q - S + 1] (y1) and CX[x_q - S + 2] (y0).
template <int NT>
__device__ __forceinline__ void g_dots(const RowG& G, const double* __restrict__ CX, int64_t ts, const PairCtx& c, int L,
                                       double* y1, double* y0) {
  const int S = c.S, lo1 = c.lo1, hi1 = c.hi1, lo0 = c.lo0, hi0 = c.hi0;
  if (c.interior) {
    const double gh1 = G.at(hi1), gh0 = G.at(hi0);
#pragma unroll
    for (int k = 0; k < NT; ++k) {
      const double cl = CX[k * ts + L];
      y1[k] = gh1 * cl;
      y0[k] = gh0 * cl;
    }
    const int q1 = G.qlut[hi1];  // breakpoints x_q < hi1
    for (int q = G.qlut[lo0]; q < q1; ++q) {
      const int xq = G.x[q];
      const double dq = (double)G.dc[q];
      const int i = xq - S + 1;  // 0 <= i <= L - 1
#pragma unroll
      for (int k = 0; k < NT; ++k) {
        const double v1 = CX[k * ts + i], v0 = CX[k * ts + i + 1];
        if (xq >= lo1) y1[k] += dq * v1;
        if (xq < hi0) y0[k] += dq * v0;
      }
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < NT; ++k) y1[k] = y0[k] = 0.0;
  const bool w1 = lo1 <= hi1, w0 = lo0 <= hi0;
  if (w1) {
    const double gh = G.at(hi1), gl = G.at(lo1);
#pragma unroll
    for (int k = 0; k < NT; ++k) y1[k] = gh * CX[k * ts + hi1 - S + 1] - gl * CX[k * ts + lo1 - S];
  }
  if (w0) {
    const double gh = G.at(hi0), gl = G.at(lo0);
#pragma unroll
    for (int k = 0; k < NT; ++k) y0[k] = gh * CX[k * ts + hi0 - S + 2] - gl * CX[k * ts + lo0 - S + 1];
  }
  if (!w1 && !w0) return;
  const int lo = lo0 < lo1 ? lo0 : lo1;
  const int q1 = G.qlut[hi1 > 0 ? hi1 : 0];  // breakpoints x_q < hi1 (hi0 <= hi1)
  for (int q = G.qlut[lo]; q < q1; ++q) {
    const int xq = G.x[q];
    const double dq = (double)G.dc[q];
    if (w1 && xq >= lo1) {
#pragma unroll
      for (int k = 0; k < NT; ++k) y1[k] += dq * CX[k * ts + xq - S + 1];
    }
    if (w0 && xq >= lo0 && xq < hi0) {
#pragma unroll
      for (int k = 0; k < NT; ++k) y0[k] += dq * CX[k * ts + xq - S + 2];
    }
  }
}

// Distinct LUT cells of the diffusion bins that land on the row along one axis (pixel offset a):
// bins with the same cell have their weights summed (the bin weights factorise, w = wx wy, and
// every other factor depends on the cell only), so each distinct (cx, cy) is visited once.
template <int NB>
__device__ __forceinline__ void axis_cells(int u, int a, int nsb, const float* w, const float* dw, bool* ok, int* cell,
                                           float* W, float* DW) {
  constexpr int SYM = (NB - 1) / 2;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    ok[i] = false;
    cell[i] = 0;
    W[i] = 0.f;
    DW[i] = 0.f;
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int v = u + i - SYM;
    const int dv = v < 0 ? -1 : (v >= nsb ? 1 : 0);
    if (dv != a) continue;
    const int cc = offset_bin(v - dv * nsb, 0, nsb);
    bool merged = false;
#pragma unroll
    for (int j = 0; j < i; ++j) {
      if (!merged && ok[j] && cell[j] == cc) {
        W[j] += w[i];
        DW[j] += dw[i];
        merged = true;
      }
    }
    if (!merged) {
      ok[i] = true;
      cell[i] = cc;
      W[i] = w[i];
      DW[i] = dw[i];
    }
  }
}

// G vanishes from tick S - 2 on: the pair has no gradient
__device__ __forceinline__ bool pair_dead(int S, const RowG& G) { return G.qlut[S - 2 > 0 ? S - 2 : 0] >= G.np; }

// (window start S, charge, fractional tick) -> the pair's placement; G must not vanish at S - 2
__device__ __forceinline__ void pair_ctx(const Dev& d, int S, float ne, float f, const RowG& G, PairCtx& c) {
  const int L = d.L, nout = d.nout;
  c.S = S;
  c.f = (double)f;
  c.ne = (double)ne;
  c.gc1 = (S - 2 >= 0 && S - 2 <= nout - 2) ? G.at(S - 2) : 0.0;
  c.gc0 = (S - 1 >= 0 && S - 1 <= nout - 2) ? G.at(S - 1) : 0.0;
  c.gc = (1.0 - c.f) * c.gc0 + c.f * c.gc1;
  c.lo1 = S > 1 ? S : 1;
  c.hi1 = (S + L - 1) < (nout - 1) ? (S + L - 1) : (nout - 1);
  c.lo0 = (S - 1) > 1 ? (S - 1) : 1;
  c.hi0 = (S + L - 2) < (nout - 1) ? (S + L - 2) : (nout - 1);
  c.interior = c.lo1 == S && c.hi1 == S + L - 1 && c.lo0 == S - 1 && c.hi0 == S + L - 2;
}

// The neighbour stripe of pixel offset (a, b) != (0, 0) of a segment at sub-bins (ux, uy):
// d loss / d n_e (gN) and / d f (gF).
__device__ __forceinline__ void stripe_adjoint(const Dev& d, const Tables& tb, int ux, int uy, const PairCtx& c, int a,
                                               int b, const RowG& G, double& gN, double& gF) {
  const int L = d.L, nsb = d.nsb;
  const int64_t sidx = (int64_t)offset_bin(ux, a, nsb) * d.ly + offset_bin(uy, b, nsb);
  double y1, y0;
  g_dots<1>(G, tb.CTN + sidx * (L + 1), 0, c, L, &y1, &y0);
  const float2 D = tb.DN[(int64_t)(d.nt - L - c.S) * d.lx * d.ly + sidx];  // tick-major, k0 = nt - L - S
  const double corr = (double)D.x - c.f * (double)D.y, dy = (double)D.y;
  gN += (1.0 - c.f) * y1 + c.f * y0 + c.gc * corr;
  gF += c.ne * (y0 - y1 + (c.gc1 - c.gc0) * corr - c.gc * dy);
}

// The diffusion bins of x-bin i (and every later x-bin with the same LUT cell, merged into it)
// landing on pixel offset (a, b), |a|, |b| <= 1: d loss / d (n_e, f, sigma_T, lambda) summed over
// the y bins.  false (nothing added) when bin i misses column a
// or an earlier x-bin has its cell.
template <int NB>
__device__ __forceinline__ bool xbin_adjoint(const Dev& d, const Tables& tb, const SegRec& R, const AdjRec* __restrict__ Ap,
                                             const PairCtx& c, int a, int b, int i, const RowG& G, double& gN,
                                             double& gF, double& gS, double& gL) {
  constexpr int SYM = (NB - 1) / 2;
  const int L = d.L, nsb = d.nsb, cm = d.cm;
  const int ux = R.uxy & 0xffff, uy = R.uxy >> 16;
  const int vi = ux + i - SYM;
  const int di = vi < 0 ? -1 : (vi >= nsb ? 1 : 0);
  if (di != a) return false;
  const int cx = offset_bin(vi - di * nsb, 0, nsb);
  float WXi = 0.f, DWXi = 0.f;
#pragma unroll
  for (int k = 0; k < NB; ++k) {
    const int v = ux + k - SYM;
    const int dv = v < 0 ? -1 : (v >= nsb ? 1 : 0);
    if (dv != a || offset_bin(v - dv * nsb, 0, nsb) != cx) continue;
    if (k < i) return false;  // merged into x-bin k
    WXi += R.wx[k];
    DWXi += Ap->dwx[k];
  }
  bool oky[NB];
  int cyv[NB];
  float WY[NB], DWY[NB];
  axis_cells<NB>(uy, b, nsb, R.wy, Ap->dwy, oky, cyv, WY, DWY);
  const int64_t tstride = (int64_t)cm * cm * (L + 1);
  const double la = (double)R.la, lb = (double)R.lb, lc = (double)R.lc;
  const double da = Ap->dl[0], db = Ap->dl[1], dc = Ap->dl[2];
  const double f = c.f, ne = c.ne;
#pragma unroll
  for (int jj = 0; jj < NB; ++jj) {
    if (!oky[jj]) continue;
    const int64_t cell = ((int64_t)R.idx * cm + cx) * cm + cyv[jj];
    double y1[3], y0[3];
    g_dots<3>(G, tb.CTM + (cell - (int64_t)cm * cm) * (L + 1), tstride, c, L, y1, y0);
    const float2 D = tb.DM[(int64_t)R.k0 * d.nm * cm * cm + cell];  // tick-major
    const double corr = (double)D.x - f * (double)D.y, dy = (double)D.y;
    const double wxy = (double)WXi * (double)WY[jj];
    const double dwxy = (double)DWXi * (double)WY[jj] + (double)WXi * (double)DWY[jj];
    const double Y1 = la * y1[0] + lb * y1[1] + lc * y1[2];
    const double Y0 = la * y0[0] + lb * y0[1] + lc * y0[2];
    const double gn = (1.0 - f) * Y1 + f * Y0 + c.gc * corr;  // d loss / d n_bin per unit weight
    gN += gn * wxy;
    gS += gn * ne * dwxy;
    gF += ne * wxy * (Y0 - Y1 + (c.gc1 - c.gc0) * corr - c.gc * dy);
    gL += ne * wxy * ((1.0 - f) * (da * y1[0] + db * y1[1] + dc * y1[2]) + f * (da * y0[0] + db * y0[1] + dc * y0[2]));
  }
  return true;
}

// Chain rule to the 7 parameters from the pair's d loss / d (n_e, f, sigma_T, lambda).
__device__ __forceinline__ void add_chain(const AdjRec* __restrict__ Ap, double gN, double gF, double gS, double gL,
                                          bool near, double* g) {
  g[0] += gN * Ap->fN[0];
  g[1] += gN * Ap->fN[1];
  g[2] += gN * Ap->fN[2] + gF * Ap->fF;
  g[3] += gN * Ap->fN[3];
  if (near) {
    g[2] += gS * Ap->fS[0] + gL * Ap->fL[0];
    g[5] += gL * Ap->fL[1];
    g[6] += gS * Ap->fS[1];
  }
}


// Stage 2, row-owned: one workgroup per pixel row holds the row's step function in LDS and walks
// the segments of its neighbourhood cells (the same pairs the forward's waveform kernel visits),
// every thread taking pairs from the flattened list; fixed-order block reduction to the row's 7
// partial gradients.  Two passes (separate launches, separate partials): NEAR = false takes the
// stripes of every offset but the centre (little register state, high occupancy), NEAR = true the
// diffusion bins of the 3x3 cells.  The stripes of the 8 cells around the centre, when they were items of the
// second pass beside the bins that mostly miss those cells, kept few lanes of a wave busy (near and far
// 575 + 319 -> 414 + 352 us for 200k segments; a side pair's bins as one item: 878).  Rows without
// gradient (no valid hit) exit at once.  (A waveform cotangent takes k_rows_adj_dense instead.)
template <int NB, int WAVES, bool NEAR>
__global__ __launch_bounds__(WAVES * kWave) __attribute__((amdgpu_waves_per_eu(4))) void k_rows_adj(Dev d, Tables tb, const SegRec* __restrict__ rec,
                                                            const PairRec* __restrict__ prs,
                                                            const AdjRec* __restrict__ adj, const int2* __restrict__ rng,
                                                            const int* __restrict__ row_cell,
                                                            const int* __restrict__ n_rows_dev, int64_t max_rows,
                                                            const Pieces* __restrict__ pieces,
                                                            double* __restrict__ partial) {
  constexpr int NT = WAVES * kWave;
  constexpr int kNP = 2 * kMaxH;  // breakpoints held in LDS
  __shared__ int c_beg[kMaxCells], c_cum[kMaxCells + 1], c_ab[kMaxCells];
  __shared__ int ncls[3];
  __shared__ int cell_scratch[3 * kMaxCells];
  __shared__ int spx[kNP];
  __shared__ float spc[kNP], sdc[kNP];
  __shared__ uint16_t qlut[kMaxOut];
  __shared__ double red[kNGrad][NT / kWave];
  const int t = threadIdx.x;
  const int P0 = *n_rows_dev;
  const int P = P0 < max_rows ? P0 : (int)max_rows;
  const int64_t row = run_row();
  if (row >= P) {
    if (row < max_rows && t < kNGrad) partial[row * kNGrad + t] = 0.0;
    return;
  }
  const int r = (int)row;
  const Pieces* pr = pieces + r;
  const int np = pr->n;
  {
    if (np == 0) {
      if (t < kNGrad) partial[(int64_t)r * kNGrad + t] = 0.0;
      return;
    }
    if (t < np) {
      spx[t] = pr->x[t];
      spc[t] = pr->c[t];
      sdc[t] = pr->c[t] - (t + 1 < np ? pr->c[t + 1] : 0.f);
    }
    __syncthreads();
    // qlut[o] = number of breakpoints below o = first q with x[q] >= o (np from nout on: G = 0 there)
    for (int o = t; o < kMaxOut; o += NT) {
      int q = 0;
      for (int k = 0; k < np; ++k) q += spx[k] < o ? 1 : 0;
      qlut[o] = (uint16_t)q;
    }
  }
  __syncthreads();  // qlut complete
  // this pass's cells in (a, b) order, each with its live pairs only: window starts ascend within a
  // cell and a pair is dead from the first start at which G has vanished, so the live pairs lead
  const RowG G{spx, spc, sdc, qlut, np};
  list_cells<NT>(
      d, rng, row_cell[r],
      [&](int a, int b) {
        const bool centre = a == 0 && b == 0;
        if (NEAR) return centre ? 0 : (a >= -1 && a <= 1 && b >= -1 && b <= 1 ? 1 : -1);
        return !centre && a >= -d.nn && a <= d.nn && b >= -d.nn && b <= d.nn ? 0 : -1;
      },
      [&](int b, int e) {
        int lo = b, hi = e;  // the first dead pair of [b, e)
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if (pair_dead(prs[mid].S, G)) hi = mid;
          else lo = mid + 1;
        }
        return lo - b;
      },
      cell_scratch, c_beg, c_cum, c_ab, ncls);
  double g[kNGrad];
#pragma unroll
  for (int k = 0; k < kNGrad; ++k) g[k] = 0.0;
  const int nct = ncls[2];
  const int tot = c_cum[nct];
  int cur = 0;
  const int lane = t & (kWave - 1), wid = t / kWave;
  if (!NEAR) {
    // stripes, one item a pair.  Each thread fetches its next pair's record (the first 16 bytes
    // of the pair record) and chain factors while the current pair's table loads are in flight.
    struct FarItem {
      int4 P;  // S, ne, f, uv
      double fN0, fN1, fN2, fN3, fF;
      int ab;
    };
    auto fetch = [&](int i, FarItem& x) {
      while (i >= c_cum[cur + 1]) ++cur;
      const int sg = c_beg[cur] + (i - c_cum[cur]);
      x.ab = c_ab[cur];
      x.P = *reinterpret_cast<const int4*>(prs + sg);
      const AdjRec* A = adj + sg;
      x.fN0 = A->fN[0];
      x.fN1 = A->fN[1];
      x.fN2 = A->fN[2];
      x.fN3 = A->fN[3];
      x.fF = A->fF;
    };
    FarItem x, y;
    if (t < tot) fetch(t, x);
    for (int it = t; it < tot; it += NT) {
      if (it + NT < tot) fetch(it + NT, y);
      const float ne = __int_as_float(x.P.y);
      if (ne != 0.f) {  // every listed pair is live (G does not vanish before its window)
        PairCtx pc;
        pair_ctx(d, x.P.x, ne, __int_as_float(x.P.z), G, pc);
        double gN = 0.0, gF = 0.0;
        stripe_adjoint(d, tb, x.P.w & 0xffff, (int)((uint32_t)x.P.w >> 16), pc, (x.ab >> 8) - 64, (x.ab & 255) - 64, G, gN,
                       gF);
        g[0] += gN * x.fN0;
        g[1] += gN * x.fN1;
        g[2] += gN * x.fN2 + gF * x.fF;
        g[3] += gN * x.fN3;
      }
      x = y;
    }
  }
  // diffusion bins: a pair is NB items on consecutive threads, by x-bin row; few side pairs are reached by any
  for (int it = t; NEAR && it < tot * NB; it += NT) {
    const int i = it / NB, part = it - i * NB;
    while (i >= c_cum[cur + 1]) ++cur;
    const int s = c_beg[cur] + (i - c_cum[cur]);
    const int a = (c_ab[cur] >> 8) - 64, b = (c_ab[cur] & 255) - 64;
    const int uv = prs[s].uv;
    if (!bins_reach<NB>(uv & 0xffff, a, d.nsb) || !bins_reach<NB>((int)((uint32_t)uv >> 16), b, d.nsb)) continue;
    const SegRec R = rec[s];
    if (R.ne == 0.f) continue;
    const int S = d.nt - d.L - R.k0;
    if (pair_dead(S, G)) continue;
    PairCtx pc;
    pair_ctx(d, S, R.ne, R.f, G, pc);
    double gN = 0.0, gF = 0.0, gS = 0.0, gL = 0.0;
    if (xbin_adjoint<NB>(d, tb, R, adj + s, pc, a, b, part, G, gN, gF, gS, gL)) add_chain(adj + s, gN, gF, gS, gL, true, g);
  }
#pragma unroll
  for (int k = 0; k < kNGrad; ++k) {
    const double v = wave_sum(g[k]);
    if (lane == 0) red[k][wid] = v;
  }
  __syncthreads();
  if (t < kNGrad) {
    double v = 0.0;
    for (int w = 0; w < NT / kWave; ++w) v += red[t][w];
    partial[(int64_t)r * kNGrad + t] = v;
  }
}

// ------------------------------------------------------------------------------------------
// Stage 2 with a waveform cotangent (lsim_backward_wfs)
// ------------------------------------------------------------------------------------------
//
// G(o) = gw[r][o] + the self-trigger's step function: one value per output tick, so the window
// sums are plain dot products, and they take the forward's access pattern with reads in place of
// stores.  A wave works on four windows at once, 16 lanes each: lane l of a group holds the padded window
// samples p = 64 c + 4 l .. + 3 (c < 3; output tick o = S - 2 + p) by three 16-byte loads, G(o) comes from
// LDS, and the f window's sum takes G(o - 1) instead of the next sample, so no lane needs another's.
// The window sums of a pair enter the gradients linearly, so every lane scales its own share by
// the pair's chain factors and adds it to its 7 partial gradients: no reduction per pair, one
// per row at the end (fixed order: deterministic).
//   Stripes (the raw-window stripe of every pixel offset but the centre, |a|, |b| <= nn): blocks
//     of 64 pairs whose factors the lanes compute in parallel and stage in LDS; each group of lanes then
//     reads its pair's.  The boundary-correction terms (no window) are added by the lane that set the pair up.
//   Diffusion bins landing on the row (the 3x3 cells; side rows only for segments near the pixel
//     edge): one (segment, row) item per wave at a time.  A lane per bin merges the bins of one LUT cell,
//     adds the cell's terms without a window and leaves weight and cell in LDS; four cells at a time take
//     the sums of G with T_m and with the differences dm = T_{m-1} - T_m, dp = T_{m+1} - T_m from the
//     interleaved template windows of TM3: V = (la + lb + lc) T_m + la dm + lc dp for n_e, f, sigma_T, and
//     dV/dlambda = da dm + dc dp for lambda (the three Lagrange derivatives sum to zero).
// A window's products are formed and added in float64; only those with the templates' differences, which enter with
// small weights (and alone in lambda's derivative), three at a time in float32 first.  Sums of twelve products in
// float32 were less exact than a lane's three of a whole wave per window, and 436 us where these take 506 (50k-segment
// step with a waveform loss; by threes throughout 480).
// A whole wave per window spent its time on what it did once a window or cell in every lane (25 float64
// instructions a cell, 7 a stripe, 16-byte reads of the stage) and on 4-byte loads: 796 us; several groups of four
// windows in flight did not help.

constexpr int kGOff = 192;                       // LDS index of output tick 0
constexpr int kGLen = kMaxOut + 2 * kGOff + 64;  // ticks -kGOff .. kMaxOut + kGOff + 63

// One stripe pair as staged for the wave (64 bytes).
struct __align__(16) DenseStripe {
  int S;             // window start, clamped to 2 when the window misses the row (factors 0 then)
  int off;           // byte offset of the pair's padded raw-window row in TNP
  float c1, c0, ne;  // 1 - f, f, charge (0 for padding and for windows that miss the row)
  int pad;
  double fN[4], fF;
};
static_assert(sizeof(DenseStripe) == 64, "DenseStripe layout");

// One merged LUT cell of a bins item: its weight and the weight's derivative in sigma_T.
struct DenseCell {
  double w, dw;
  int cell, pad;
};
typedef float f32x4 __attribute__((ext_vector_type(4)));

// G at a correction tick (those are kept for 0 <= o <= nout - 2); Gw holds 0 at tick 0 (a window
// tick is kept from 1 on), G0 holds G(0).
__device__ __forceinline__ double g_corr(const float* Gw, float G0, int o, int nout) {
  return (o >= 0 && o <= nout - 2) ? (double)(o == 0 ? G0 : Gw[kGOff + o]) : 0.0;
}

// The window of a pair meets the output ticks 1 .. nout - 1 (window ticks S - 1 .. S + L - 1)
__device__ __forceinline__ bool window_live(int S, int L, int nout) { return S >= 2 - L && S <= nout; }

template <int NB, int WAVES>
__global__ __launch_bounds__(WAVES * kWave) __attribute__((amdgpu_waves_per_eu(4))) void k_rows_adj_dense(Dev d, Tables tb, const SegRec* __restrict__ rec,
                                                                  const PairRec* __restrict__ prs,
                                                                  const AdjRec* __restrict__ adj,
                                                                  const int2* __restrict__ rng,
                                                                  const int* __restrict__ row_cell,
                                                                  const int* __restrict__ n_rows_dev, int64_t max_rows,
                                                                  const Pieces* __restrict__ pieces,
                                                                  const float* __restrict__ gw,
                                                                  double* __restrict__ partial) {
  constexpr int NT = WAVES * kWave;
  constexpr int SYM = (NB - 1) / 2;
  __shared__ float Gw[kGLen];
  __shared__ DenseStripe stage[WAVES][kWave];
  __shared__ DenseCell s_cells[WAVES][NB * NB + 3];
  __shared__ int c_beg[kMaxCells], c_cum[kMaxCells + 1], c_ab[kMaxCells];
  __shared__ int ncls[3];
  __shared__ int cell_scratch[3 * kMaxCells];
  __shared__ double red[kNGrad][WAVES];
  __shared__ float sG0;
  __shared__ int s_any;
  const int t = threadIdx.x;
  const int lane = t & (kWave - 1), wid = t / kWave;
  const int P0 = *n_rows_dev;
  const int P = P0 < max_rows ? P0 : (int)max_rows;
  double* out_near = partial + max_rows * kNGrad;  // the second half of the partials: zero here
  const int64_t row = run_row();
  if (row >= P) {
    if (row < max_rows && t < kNGrad) partial[row * kNGrad + t] = out_near[row * kNGrad + t] = 0.0;
    return;
  }
  const int r = (int)row;
  const int nout = d.nout, L = d.L;
  // G over the padded tick range: window ticks 1 .. nout - 1, zero elsewhere
  if (t == 0) s_any = 0;
  __syncthreads();
  {
    const Pieces* pr = pieces + r;
    const float* gr = gw + (int64_t)r * nout;
    const int nf = pr->n;
    bool any = false;
    for (int i = t; i < kGLen; i += NT) {
      const int o = i - kGOff;
      float v = 0.f;
      if (o >= 0 && o < nout) {
        float cf = 0.f;
        for (int k = nf - 1; k >= 0; --k)
          if (pr->x[k] >= o) cf = pr->c[k];
        v = gr[o] + cf;
        any = any || v != 0.f;
        if (o == 0) sG0 = v;
      }
      Gw[i] = (o >= 1 && o < nout) ? v : 0.f;
    }
    if (any) s_any = 1;
  }
  __syncthreads();
  if (!s_any) {  // no cotangent on this row
    if (t < kNGrad) {
      partial[(int64_t)r * kNGrad + t] = 0.0;
      out_near[(int64_t)r * kNGrad + t] = 0.0;
    }
    return;
  }
  const float G0 = sG0;
  // cells: far (stripes), side (stripes and bins), centre (bins)
  list_cells<NT>(
      d, rng, row_cell[r],
      [](int a, int b) {
        const bool near = a >= -1 && a <= 1 && b >= -1 && b <= 1;
        return !near ? 0 : ((a == 0 && b == 0) ? 2 : 1);
      },
      [](int b, int e) { return e - b; }, cell_scratch, c_beg, c_cum, c_ab, ncls);
  double g[kNGrad];
#pragma unroll
  for (int k = 0; k < kNGrad; ++k) g[k] = 0.0;
  const int nsb = d.nsb, lxly = d.lx * d.ly;
  const int n_stripe_cells = d.nn >= 1 ? ncls[1] : ncls[0];
  const int nstripe = c_cum[n_stripe_cells];
  const __amdgpu_buffer_rsrc_t tnp =
      __builtin_amdgcn_make_buffer_rsrc((void*)tb.TNP, 0, d.lx * d.ly * kWinPad * 4, kBufDesc3);
  const int sub = lane & 15, grp = lane >> 4;
  // ---- stripes ----
  for (int b0 = wid * kWave; b0 < nstripe; b0 += WAVES * kWave) {
    const int p = b0 + lane;
    DenseStripe z;
    z.S = 2;
    z.off = 0;
    z.c1 = z.c0 = z.ne = 0.f;
    z.pad = 0;
    z.fN[0] = z.fN[1] = z.fN[2] = z.fN[3] = z.fF = 0.0;
    if (p < nstripe) {
      int lo = 0, hi = n_stripe_cells - 1;  // the cell holding p: last c with c_cum[c] <= p
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (c_cum[mid] <= p) lo = mid;
        else hi = mid - 1;
      }
      const int sg = c_beg[lo] + (p - c_cum[lo]);
      const int ab = c_ab[lo];
      const int a = (ab >> 8) - 64, b = (ab & 255) - 64;
      const PairRec R = prs[sg];
      if (R.ne != 0.f) {
        const int S = R.S;
        const double f = (double)R.f, ne = (double)R.ne;
        const int ux = R.u(), uy = R.v();
        const int sidx = offset_bin(ux, a, nsb) * d.ly + offset_bin(uy, b, nsb);
        const float2 D = tb.DN[(int64_t)(d.nt - L - S) * lxly + sidx];  // tick-major, k0 = nt - L - S
        const double corr = (double)D.x - f * (double)D.y, dy = (double)D.y;
        const double gc0 = g_corr(Gw, G0, S - 1, nout), gc1 = g_corr(Gw, G0, S - 2, nout);
        const double gc = (1.0 - f) * gc0 + f * gc1;
        const AdjRec* A = adj + sg;
        const double fN0 = A->fN[0], fN1 = A->fN[1], fN2 = A->fN[2], fN3 = A->fN[3], fF = A->fF;
        // the correction terms of the pair (no window)
        const double gNc = gc * corr, gFc = ne * ((gc1 - gc0) * corr - gc * dy);
        g[0] += gNc * fN0;
        g[1] += gNc * fN1;
        g[2] += gNc * fN2 + gFc * fF;
        g[3] += gNc * fN3;
        if (window_live(S, L, nout)) {
          z.S = S;
          z.off = sidx * kWinPad * 4;
          z.c1 = (float)(1.0 - f);
          z.c0 = R.f;
          z.ne = R.ne;
          z.fN[0] = fN0;
          z.fN[1] = fN1;
          z.fN[2] = fN2;
          z.fN[3] = fN3;
          z.fF = fF;
        }
      }
    }
    stage[wid][lane] = z;
    __builtin_amdgcn_wave_barrier();
    const int n = __builtin_amdgcn_readfirstlane(nstripe - b0 < kWave ? nstripe - b0 : kWave);
    for (int i = 0; i < n; i += 4) {
      // four pairs at a time, 16 lanes each (entries past n are padding: factors 0, a window at S = 2)
      const DenseStripe& q = stage[wid][i + grp];
      f32x4 x[3];
#pragma unroll
      for (int c = 0; c < 3; ++c)
        x[c] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(tnp, q.off + sub * 16, c * 4 * kWave, 0));
      double u1 = 0.0, u0 = 0.0;
      const float* gp = Gw + kGOff + q.S - 2 + 4 * sub;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        double g0 = (double)gp[kWave * c - 1];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const double g1 = (double)gp[kWave * c + k], xk = (double)x[c][k];
          u1 = __builtin_fma(g1, xk, u1);
          u0 = __builtin_fma(g0, xk, u0);
          g0 = g1;
        }
      }
      const double aa = (double)q.c1 * u1 + (double)q.c0 * u0, bb = (double)q.ne * (u0 - u1);
      g[0] += q.fN[0] * aa;
      g[1] += q.fN[1] * aa;
      g[2] += q.fN[2] * aa + q.fF * bb;
      g[3] += q.fN[3] * aa;
    }
    __builtin_amdgcn_wave_barrier();  // the stage is rewritten by the next block
  }
  // ---- diffusion bins of the 3x3 cells ----
  const int kb0 = c_cum[ncls[0]], kb1 = c_cum[ncls[2]];
  int cur = ncls[0];
  for (int k = kb0 + wid; k < kb1; k += WAVES) {
    while (k >= c_cum[cur + 1]) ++cur;
    const int s = __builtin_amdgcn_readfirstlane(c_beg[cur] + (k - c_cum[cur]));
    const int ab = __builtin_amdgcn_readfirstlane(c_ab[cur]);
    const int a = (ab >> 8) - 64, b = (ab & 255) - 64;
    const SegRec R = rec[s];
    if (R.ne == 0.f) continue;
    const int ux = R.uxy & 0xffff, uy = R.uxy >> 16;
    if (!bins_reach<NB>(ux, a, nsb) || !bins_reach<NB>(uy, b, nsb)) continue;
    const AdjRec* A = adj + s;
    const int S = d.nt - L - R.k0;
    const double f = (double)R.f, ne = (double)R.ne;
    const double gc0 = g_corr(Gw, G0, S - 1, nout), gc1 = g_corr(Gw, G0, S - 2, nout);
    const double gc = (1.0 - f) * gc0 + f * gc1;
    const bool live = window_live(S, L, nout);
    // lane i NB + j: x-bin i, y-bin j.  Bins on one LUT cell are merged into the first of them, axis by axis.
    const int cm = d.cm;
    const int bi = lane / NB, bj = lane - bi * NB;
    int cx = 0, cy = 0;
    float WX = 0.f, WY = 0.f, DWX = 0.f, DWY = 0.f;
    bool mine = lane < NB * NB;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int vx = ux + k - SYM, vy = uy + k - SYM;
      const int dx = vx < 0 ? -1 : (vx >= nsb ? 1 : 0), dy = vy < 0 ? -1 : (vy >= nsb ? 1 : 0);
      const int cxk = dx == a ? offset_bin(vx - dx * nsb, 0, nsb) : -1, cyk = dy == b ? offset_bin(vy - dy * nsb, 0, nsb) : -1;
      cx = k == bi ? cxk : cx;
      cy = k == bj ? cyk : cy;
    }
    mine = mine && cx >= 0 && cy >= 0;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int vx = ux + k - SYM, vy = uy + k - SYM;
      const int dx = vx < 0 ? -1 : (vx >= nsb ? 1 : 0), dy = vy < 0 ? -1 : (vy >= nsb ? 1 : 0);
      const int cxk = dx == a ? offset_bin(vx - dx * nsb, 0, nsb) : -1, cyk = dy == b ? offset_bin(vy - dy * nsb, 0, nsb) : -1;
      WX += cxk == cx ? R.wx[k] : 0.f;
      DWX += cxk == cx ? A->dwx[k] : 0.f;
      WY += cyk == cy ? R.wy[k] : 0.f;
      DWY += cyk == cy ? A->dwy[k] : 0.f;
      mine = mine && !(k < bi && cxk == cx) && !(k < bj && cyk == cy);
    }
    const double w = (double)WX * (double)WY, dw = (double)DWX * (double)WY + (double)WX * (double)DWY;
    const int cell = mine ? (R.idx * cm + cx) * cm + cy : 0;
    double gN = 0.0, gF = 0.0, gS = 0.0, gL = 0.0;
    // every cell's terms without a window, by its lane
    if (mine) {
      const float2 D = tb.DM[(int64_t)R.k0 * d.nm * cm * cm + cell];  // tick-major
      const double corr = (double)D.x - f * (double)D.y, dy = (double)D.y;
      gN = gc * corr * w;
      gS = gc * corr * ne * dw;
      gF = ne * w * ((gc1 - gc0) * corr - gc * dy);
    }
    const uint64_t m = __ballot(mine);
    const int nc = __popcll(m);
    if (live && nc > 0) {
      // the cells in slots 0 .. nc - 1, up to a multiple of 4 filled with the first one at no weight
      DenseCell* cells = s_cells[wid];
      const int rank = __popcll(m & ((1ull << lane) - 1));
      if (mine) cells[rank] = DenseCell{w, dw, cell, 0};
      const int cell0 = __builtin_amdgcn_readlane(cell, __builtin_ctzll(m));
      if (lane < 3) cells[nc + lane] = DenseCell{0.0, 0.0, cell0, 0};
      __builtin_amdgcn_wave_barrier();
      float gv[3][5];
#pragma unroll
      for (int c = 0; c < 3; ++c)
#pragma unroll
        for (int k = 0; k < 5; ++k) gv[c][k] = Gw[kGOff + S - 3 + 4 * sub + kWave * c + k];
      const double la = (double)R.la, lc = (double)R.lc, ls = la + (double)R.lb + lc;
      const double da = A->dl[0], dc = A->dl[2];
      double U1 = 0.0, U0 = 0.0, D1 = 0.0, D0 = 0.0, L1 = 0.0, L0 = 0.0;
      for (int k4 = 0; k4 < nc; k4 += 4) {
        const DenseCell q = cells[k4 + grp];
        const f32x4* T = (const f32x4*)(tb.TM3 + (int64_t)q.cell * kWinPad) + 3 * sub;
        f32x4 v[3][3];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int k = 0; k < 3; ++k) v[c][k] = T[c * (3 * kWave / 4) + k];
        // sums of G and of G one tick on with T_m and its differences from T_{m-1}, T_{m+1}
        double y1 = 0.0, y0 = 0.0, p1 = 0.0, p0 = 0.0, n1 = 0.0, n0 = 0.0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          float a1 = 0.f, a0 = 0.f, b1 = 0.f, b0 = 0.f;
#pragma unroll
          for (int c = 0; c < 3; ++c) {
            const float tm = v[c][(3 * k) / 4][(3 * k) % 4], tc = v[c][(3 * k + 1) / 4][(3 * k + 1) % 4],
                        tp = v[c][(3 * k + 2) / 4][(3 * k + 2) % 4];
            const float dm = tm - tc, dp = tp - tc;
            float g1 = gv[c][k + 1], g0 = gv[c][k];
            asm volatile("" : "+v"(g1), "+v"(g0));  // converted here: kept in float64 over the loop they take 30 registers
            y1 = __builtin_fma((double)g1, (double)tc, y1);
            y0 = __builtin_fma((double)g0, (double)tc, y0);
            a1 = __builtin_fmaf(g1, dm, a1);
            a0 = __builtin_fmaf(g0, dm, a0);
            b1 = __builtin_fmaf(g1, dp, b1);
            b0 = __builtin_fmaf(g0, dp, b0);
          }
          p1 += (double)a1;
          p0 += (double)a0;
          n1 += (double)b1;
          n0 += (double)b0;
        }
        const double u1 = ls * y1 + la * p1 + lc * n1, u0 = ls * y0 + la * p0 + lc * n0;
        U1 += q.w * u1;
        U0 += q.w * u0;
        D1 += q.dw * u1;
        D0 += q.dw * u0;
        L1 += q.w * (da * p1 + dc * n1);
        L0 += q.w * (da * p0 + dc * n0);
      }
      __builtin_amdgcn_wave_barrier();  // the slots are rewritten by the next item
      gN += (1.0 - f) * U1 + f * U0;
      gS += ne * ((1.0 - f) * D1 + f * D0);
      gF += ne * (U0 - U1);
      gL += ne * ((1.0 - f) * L1 + f * L0);
    }
    add_chain(A, gN, gF, gS, gL, true, g);
  }
  // fixed-order block reduction of the lanes' partial gradients
#pragma unroll
  for (int k = 0; k < kNGrad; ++k) {
    const double v = wave_sum(g[k]);
    if (lane == 0) red[k][wid] = v;
  }
  __syncthreads();
  if (t < kNGrad) {
    double v = 0.0;
    for (int w = 0; w < WAVES; ++w) v += red[t][w];
    partial[(int64_t)r * kNGrad + t] = v;
    out_near[(int64_t)r * kNGrad + t] = 0.0;
  }
}

// One pass over the per-row partials (all 7 gradients and the hit-z term per thread), then a
// fixed-order combine: butterfly within each wave, waves in index order.  Deterministic.
constexpr int kReduceThreads = 1024;

__global__ __launch_bounds__(kReduceThreads) void k_grad_reduce(Dev d, const double* __restrict__ partial, int64_t nblocks,
                                                                const double* __restrict__ dz_part,
                                                                const int64_t* __restrict__ n_rows_dev, int64_t max_rows,
                                                                double* __restrict__ out) {
  __shared__ double sh[kNGrad + 1][kReduceThreads / kWave];
  int64_t P = *n_rows_dev;
  if (P > max_rows) P = max_rows;
  double acc[kNGrad + 1];
#pragma unroll
  for (int k = 0; k <= kNGrad; ++k) acc[k] = 0.0;
  for (int64_t b = threadIdx.x; b < nblocks; b += blockDim.x) {
#pragma unroll
    for (int k = 0; k < kNGrad; ++k) acc[k] += partial[b * kNGrad + k];
  }
  for (int64_t r = threadIdx.x; r < P; r += blockDim.x) acc[kNGrad] += dz_part[r];
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x / kWave;
#pragma unroll
  for (int k = 0; k <= kNGrad; ++k) {
    const double v = wave_sum(acc[k]);
    if (lane == 0) sh[k][wid] = v;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot[kNGrad + 1];
    for (int k = 0; k <= kNGrad; ++k) {
      tot[k] = 0.0;
      for (int w = 0; w < (int)(blockDim.x / kWave); ++w) tot[k] += sh[k][w];
    }
    for (int k = 0; k < kNGrad; ++k) out[k] = tot[k];
    out[2] += tot[kNGrad] * d.dv;  // hit z depends on eField through the drift velocity
  }
}

}  // namespace lsim
