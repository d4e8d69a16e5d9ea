// Forward kernels: segment keys and records, cell / pixel-row enumeration, the row-owned
// waveform kernel with the fused self-trigger, hit compaction, and the response tables.
#pragma once
#include "device.h"
#include "scan_sort.h"

namespace lsim {

// Window tables of the raw response are zero padded: P[p] = W[p - 2] for 2 <= p < L + 2 and 0
// elsewhere, kWinPad entries per series, read without bounds tests (windows up to kMaxWindow samples).
constexpr int kWinPad = 3 * kWave;
constexpr int kMaxWindow = kWinPad - 5;
constexpr int kXcd = 8;  // XCDs of an MI355X (workgroup i runs on XCD i % 8)

// Per-segment record of the window paths (sorted order): window start, charge, fractional tick and
// sub-bin position.
struct __align__(16) PairRec {
  int S;          // first output tick of the (1-f) window: nt - L - k0
  float ne, f;
  int uv;         // u | v << 16, sixteen bits each as in SegRec
  __device__ __forceinline__ int u() const { return uv & 0xffff; }
  __device__ __forceinline__ int v() const { return (int)((uint32_t)uv >> 16); }
};
static_assert(sizeof(PairRec) == 16, "PairRec layout");

// ------------------------------------------------------------------------------------------
// small utility kernels
// ------------------------------------------------------------------------------------------

template <typename T>
__global__ void k_fill(T* __restrict__ p, int64_t n, T v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}

template <typename T>
inline void fill(T* p, int64_t n, T v, hipStream_t st) {
  if (n <= 0) return;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL((k_fill<T>), dim3((unsigned)blocks), dim3(256), 0, st, p, n, v);
}

// ------------------------------------------------------------------------------------------
// 1. cell key per segment (input order)
// ------------------------------------------------------------------------------------------

// Sort keys of a segment.  Cell key = main-pixel cell of the segment in the halo-extended grid,
// or n_cells (sorts last) for segments that neither create a pixel row nor carry charge: padding
// rows (eventID < 0), events out of range, and zero-charge segments whose main pixel is off the
// pixel plane.  Window key = the first output tick S = nt - L - k0 of the segment's windows,
// clamped to [0, nout + 2]: segments are ordered by cell, then by S (an adjoint row's live pairs,
// those whose windows start before its gradient vanishes, then lead each cell).
__device__ __forceinline__ void seg_keys(const Dev& d, const SegIn& in, int64_t i, uint32_t& cell_key, uint32_t& s_key,
                                         int* status) {
  Phys ph;
  seg_physics(d, in, i, ph);
  int64_t c = cell_of(d, ph.ev, ph.plane, ph.mpx, ph.mpy);
  const bool on_plane = ph.mpx >= 0 && ph.mpx < d.nx && ph.mpy >= 0 && ph.mpy < d.ny;
  bool keep = c >= 0 && (ph.mask ? true : on_plane);
  if (status && ph.ev >= d.n_events) atomicOr(status, LSIM_STATUS_BAD_EVENT);
  cell_key = keep ? (uint32_t)c : (uint32_t)d.n_cells;
  const int S = d.nt - d.L - ph.k0;
  s_key = (uint32_t)(S < 0 ? 0 : (S > d.nout + 2 ? d.nout + 2 : S));
}

// First sort stage: window keys (input order).
__global__ void k_keys(Dev d, SegIn in, uint32_t* __restrict__ keys, uint32_t* __restrict__ vals, int* __restrict__ status) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= in.n) return;
  uint32_t ck, sk;
  seg_keys(d, in, i, ck, sk, status);
  keys[i] = sk;
  vals[i] = (uint32_t)i;
}

// Second stage: the cell keys of the window-sorted order (a stable sort by cell follows).
__global__ void k_cell_keys(Dev d, SegIn in, const uint32_t* __restrict__ vals, int64_t n, uint32_t* __restrict__ keys) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  uint32_t ck, sk;
  seg_keys(d, in, vals[j], ck, sk, nullptr);
  keys[j] = ck;
}

// ------------------------------------------------------------------------------------------
// 2. records in cell order, cell ranges, pixel rows
// ------------------------------------------------------------------------------------------

// Boundary corrections of every (row offset, segment) pair of record R, written where the record
// is built: dtot[ab][i] = n_e (D.x - f D.y) of the neighbour stripe (raw response, unless the offset
// is (0, 0)) plus, for |a|, |b| <= 1, the sum over the diffusion bins landing on that row of
// n_bin (D.x - f D.y) of the idx template (sim_jax.py:227-261), D = (C[nt-L] - C[k0],
// C[k0+1] - C[k0]), ab = (a + n)(2n + 1) + (b + n).  The D tables are tick-major, so all of one
// segment's entries lie in the tick-k0 plane; the waveform kernels then read dtot[ab][cell range]
// contiguously.
//
// The stripe entries come from DNS, the raw response's D of every (tick, sub-bin x, sub-bin y)
// regrouped so that one segment's WW entries are contiguous (k_lut_dns).  A wave stages each batch
// of kCorrBatch entries of its 64 segments through LDS: lane e of load m fetches element
// e + 64 m of the batch (segment (e + 64 m) / kCorrBatch, entry (e + 64 m) % kCorrBatch), so one
// load instruction reads about seven segments' runs of kCorrBatch contiguous entries instead of 64
// scattered ones; each lane then takes its own segment's entries from LDS.  The diffusion-bin loads
// are issued one x-bin row at a time so that each thread has several in flight; each entry still
// receives its terms in the same order (its stripe term, then its diffusion bins by x-bin, y-bin).
constexpr int kCorrBatch = 9;
constexpr int kRecThreads = 256;

//
// part < 0: all of a segment's corrections.  Otherwise a share of them: part p < parts - 1 batch p without
// the entries of |a|, |b| <= 1, part parts - 1 those and the diffusion bins.
template <int NB>
__device__ __forceinline__ void seg_corrections(const Dev& d, const float2* __restrict__ DNS, const float2* __restrict__ DM,
                                                const SegRec& R, bool live, int ux, int uy, int64_t i, int64_t n,
                                                float2* __restrict__ stage, int* __restrict__ base,
                                                float* __restrict__ dtot, int part, int parts) {
  constexpr int SYM = (NB - 1) / 2;
  const int W = 2 * d.ne + 1, WW = W * W, nsb = d.nsb, cm = d.cm;
  const int lane = threadIdx.x & (kWave - 1);
  const float f = R.f;
  // the WW entries of (k0, ux, uy) start here (fits an int: nt nsb^2 WW < 2^31 for every valid LUT)
  base[lane] = live ? (int)((((int64_t)R.k0 * nsb + ux) * nsb + uy) * WW) : -1;
  __builtin_amdgcn_wave_barrier();
  float dn[9];  // entries (a, b) in [-1, 1]^2, index (a + 1) * 3 + (b + 1)
  // stripe terms of every entry
  const bool near = part < 0 || part == parts - 1, far = part < 0 || !near;
  // (the near entries lie between (-1, -1) and (1, 1))
  const int first = part < 0 ? 0 : (near ? (d.ne - 1) * W + d.ne - 1 : part * kCorrBatch);
  const int last = part < 0 ? WW : (near ? (d.ne + 1) * W + d.ne + 2 : first + 1);
  for (int ab0 = first; ab0 < last; ab0 += kCorrBatch) {
#pragma unroll
    for (int m = 0; m < kCorrBatch; ++m) {
      const int e = lane + kWave * m;
      const int sg = e / kCorrBatch, u = e - sg * kCorrBatch;
      const int b = base[sg];
      stage[e] = (b >= 0 && ab0 + u < WW) ? DNS[b + ab0 + u] : make_float2(0.f, 0.f);
    }
    // wave-local LDS: the stores and loads of one wave complete in program order; the wave
    // barriers keep the compiler from moving them across
    __builtin_amdgcn_wave_barrier();
    float2 D[kCorrBatch];
#pragma unroll
    for (int u = 0; u < kCorrBatch; ++u) {
      const int ab = ab0 + u;
      const int a = ab / W - d.ne, b = ab % W - d.ne;
      const bool on = ab < WW && (a != 0 || b != 0) && a >= -d.nn && a <= d.nn && b >= -d.nn && b <= d.nn;
      D[u] = on ? stage[lane * kCorrBatch + u] : make_float2(0.f, 0.f);
    }
    __builtin_amdgcn_wave_barrier();  // every lane has its entries before the next batch is staged
    if (!live) continue;
    float dl[kCorrBatch];  // all of the batch's values before its stores: no store between two uses
#pragma unroll
    for (int u = 0; u < kCorrBatch; ++u) {
      const int ab = ab0 + u;
      const int a = ab / W - d.ne, b = ab % W - d.ne;
      const bool on = ab < WW && (a != 0 || b != 0) && a >= -d.nn && a <= d.nn && b >= -d.nn && b <= d.nn;
      dl[u] = on ? R.ne * (D[u].x - f * D[u].y) : 0.f;
    }
#pragma unroll
    for (int u = 0; u < kCorrBatch; ++u) {
      const int ab = ab0 + u;
      if (ab >= WW) break;
      const int a = ab / W - d.ne, b = ab % W - d.ne;
      const float delta = dl[u];
      if (a >= -1 && a <= 1 && b >= -1 && b <= 1) {
#pragma unroll
        for (int e = 0; e < 9; ++e)
          if (e == (a + 1) * 3 + (b + 1)) dn[e] = delta;
      } else if (far) {
        dtot[(int64_t)ab * n + i] = delta;
      }
    }
  }
  if (!live || !near) return;
  const float2* DMk = DM + ((int64_t)R.k0 * d.nm + R.idx) * cm * cm;
  // diffusion bins of the idx template, one x-bin row of loads at a time
#pragma unroll
  for (int k = 0; k < NB; ++k) {
    const int vx = ux + k - SYM;
    const int dx = vx < 0 ? -1 : (vx >= nsb ? 1 : 0);
    const float wxs = R.ne * R.wx[k];
    const int cx = offset_bin(vx - dx * nsb, 0, nsb);
    float2 D[NB];
    float c[NB];
    int e[NB];
#pragma unroll
    for (int jj = 0; jj < NB; ++jj) {
      const int vy = uy + jj - SYM;
      const int dy = vy < 0 ? -1 : (vy >= nsb ? 1 : 0);
      c[jj] = wxs * R.wy[jj];
      e[jj] = (dx + 1) * 3 + (dy + 1);
      D[jj] = c[jj] != 0.f ? DMk[cx * cm + offset_bin(vy - dy * nsb, 0, nsb)] : make_float2(0.f, 0.f);
    }
#pragma unroll
    for (int jj = 0; jj < NB; ++jj) {
      if (c[jj] == 0.f) continue;
      const float v = c[jj] * (D[jj].x - f * D[jj].y);
#pragma unroll
      for (int q = 0; q < 9; ++q)
        if (q == e[jj]) dn[q] += v;
    }
  }
#pragma unroll
  for (int q = 0; q < 9; ++q) {
    const int a = q / 3 - 1, b = q % 3 - 1;
    dtot[(int64_t)((a + d.ne) * W + (b + d.ne)) * n + i] = dn[q];
  }
}

// The record of the segment with input index src at sorted position i, and its pair record; whole = false
// leaves out what only the diffusion bins need (their weights) and writes neither.
__device__ __forceinline__ void record(const Dev& d, const SegIn& in, int64_t src, int64_t i, SegRec& r, int& ux, int& uy,
                                       SegRec* __restrict__ rec, PairRec* __restrict__ prs, bool whole) {
  Phys ph;
  seg_physics(d, in, src, ph);
  r.bx = ph.bx;
  r.by = ph.by;
  r.k0 = ph.k0;
  r.idx = ph.idx;
  r.ne = (float)ph.ne;
  r.f = (float)ph.f;
  r.la = (float)ph.la;
  r.lb = (float)ph.lb;
  r.lc = (float)ph.lc;
  ux = pymod_i(ph.bx, d.nsb);
  uy = pymod_i(ph.by, d.nsb);
  r.uxy = ux | (uy << 16);
  if (!whole) return;
  double wx[kMaxNb], wy[kMaxNb];
  tran_weights(d, ph.x0, ph.st, wx, nullptr);
  tran_weights(d, ph.y0, ph.st, wy, nullptr);
#pragma unroll
  for (int k = 0; k < kMaxNb; ++k) {
    r.wx[k] = k < d.nb ? (float)wx[k] : 0.f;
    r.wy[k] = k < d.nb ? (float)wy[k] : 0.f;
  }
  rec[i] = r;
  PairRec P;
  P.S = d.nt - d.L - ph.k0;
  P.ne = r.ne;
  P.f = r.f;
  P.uv = r.uxy;
  prs[i] = P;
}

// One thread per segment in sorted order (kRecThreads per workgroup): the records and the boundary
// corrections.  Threads past the end or of dropped segments stay to stage their wave's loads.
template <int NB>
__global__ __launch_bounds__(kRecThreads) void k_records(Dev d, SegIn in, const uint32_t* __restrict__ keys,
                                                         const uint32_t* __restrict__ vals, int64_t n,
                                                         const float2* __restrict__ DNS, const float2* __restrict__ DM,
                                                         SegRec* __restrict__ rec, PairRec* __restrict__ prs,
                                                         float* __restrict__ dtot) {
  __shared__ float2 stage[kRecThreads / kWave][kWave * kCorrBatch];
  __shared__ int sbase[kRecThreads / kWave][kWave];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int wid = threadIdx.x / kWave;
  const bool live = i < n && keys[i] < (uint32_t)d.n_cells;
  SegRec r = {};
  int ux = 0, uy = 0;
  const int parts = gridDim.y, part = parts == 1 ? -1 : (int)blockIdx.y;
  if (live) record(d, in, vals[i], i, r, ux, uy, rec, prs, part < 0 || part == parts - 1);
  seg_corrections<NB>(d, DNS, DM, r, live, ux, uy, i, n, stage[wid], sbase[wid], dtot, part, parts);
}

// Parts of k_records for n segments.  A segment's batches are a chain of loads of 3 to 5 us each; with few
// segments waves of their own take it apart, at the price of the segment's physics in each (whole / parts:
// 1k segments 48 / 30 us, 30k 65 / 47, 50k 82 / 61, 200k 103 / 153).
constexpr int64_t kRecSplitMax = 65536;
inline int rec_parts(const Dev& d, int64_t n) {
  const int W = 2 * d.ne + 1;
  return n <= kRecSplitMax ? (W * W + kCorrBatch - 1) / kCorrBatch + 1 : 1;
}

// Cell ranges [begin, end) in the sorted order and the "first segment of an on-plane cell" flag
// whose prefix sum numbers the pixel rows (ascending pixel id = ascending cell key).
__global__ void k_cells(Dev d, const uint32_t* __restrict__ keys, int64_t n, int2* __restrict__ rng, int* __restrict__ flag) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t k = keys[i];
  int fl = 0;
  if (k < (uint32_t)d.n_cells) {
    const bool first = (i == 0) || keys[i - 1] != k;
    const bool last = (i == n - 1) || keys[i + 1] != k;
    if (first) rng[k].x = (int)i;
    if (last) rng[k].y = (int)(i + 1);
    if (first) {
      const int cx = (int)(k % d.gx) - d.halo;
      const int cy = (int)((k / d.gx) % d.gy) - d.halo;
      fl = (cx >= 0 && cx < d.nx && cy >= 0 && cy < d.ny) ? 1 : 0;
    }
  }
  flag[i] = fl;
}

__global__ void k_rows_map(Dev d, const uint32_t* __restrict__ keys, const int* __restrict__ flag, const int* __restrict__ ridx,
                           int64_t n, int* __restrict__ row_cell, const int* __restrict__ n_rows,
                           int64_t* __restrict__ n_rows_out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0 && n_rows_out) *n_rows_out = (int64_t)*n_rows;
  if (i >= n || !flag[i]) return;
  row_cell[ridx[i]] = (int)keys[i];
}

// A count for the caller (dst and status may be NULL), with the row overflow flag if it exceeds max_rows >= 0.
__device__ __forceinline__ void copy_count(const int* __restrict__ src, int64_t* __restrict__ dst, int64_t max_rows,
                                           int* __restrict__ status) {
  const int64_t v = (int64_t)*src;
  if (dst) *dst = v;
  if (status && max_rows >= 0 && v > max_rows) atomicOr(status, LSIM_STATUS_ROWS_OVERFLOW);
}

__global__ void k_copy_count(const int* __restrict__ src, int64_t* __restrict__ dst, int64_t max_rows, int* __restrict__ status) {
  copy_count(src, dst, max_rows, status);
}

// ------------------------------------------------------------------------------------------
// 3. the waveform kernel: one workgroup owns one pixel row
// ------------------------------------------------------------------------------------------


struct Tables {
  const float3* TM3;  // [nm][cm][cm][kWinPad] padded (T_{m-1}, T_m, T_{m+1}) windows of the diffusion bins
  const float* TM;    // [nm][cm][cm][L]   main-bin template windows
  const float* TMW;   // [cm][cm][nm][bin_stride(L)] the same, two zeros before each window (and after the last)
  const float* TN;    // [lx][ly][L]       raw response window (neighbours)
  const float* TNP;   // [lx][ly][kWinPad] the same, padded
  const float2* DM;   // [nt][nm][cm][cm]  (C[nt-L]-C[k], C[min(k+1,nt-1)]-C[k]) of template m (tick-major)
  const float2* DN;   // [nt][lx][ly]      same for the raw response
  const double* CTM;  // [nm][cm][cm][L+1] window prefix sums (adjoint)
  const double* CTN;  // [lx][ly][L+1]
};

struct RowOut {
  float* wfs;          // [max_rows][nout] or null
  float* adc;          // [max_rows][H]
  int* ticks;          // [max_rows][H]
  FeeTape* tape;       // [max_rows] or null
  int* hit_cnt;        // [max_rows]
  int64_t* pixel_ids;  // [max_rows]
  int64_t* n_rows = nullptr;  // the row count and overflow flag for the caller (row kernel only)
  int* status = nullptr;
};

// NaN passes through both clamps, as through jnp.maximum / jnp.minimum (a waveform poisoned by an
// overflowing current keeps its NaN charge, as in the reference).
__device__ __forceinline__ double digitize(const Dev& d, double q) {
  double x = q * d.gain + d.vped - d.vcm;
  x = (x > 0 || x != x) ? x : 0.0;
  double y = x * d.adcc / (d.vref - d.vcm);
  return (y < d.adcc || y != y) ? y : d.adcc;
}

// JAX's derivative of digitize (ties of max/min split the gradient evenly).
__device__ __forceinline__ double digitize_slope(const Dev& d, double q) {
  const double x = q * d.gain + d.vped - d.vcm;
  const double fx = x > 0 ? 1.0 : (x == 0 ? 0.5 : 0.0);
  const double y = (x > 0 ? x : 0.0) * d.adcc / (d.vref - d.vcm);
  const double fy = y < d.adcc ? 1.0 : (y == d.adcc ? 0.5 : 0.0);
  return fx * fy * d.gain * d.adcc / (d.vref - d.vcm);
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int m = kWave / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m, kWave);
  return v;
}

// Self-trigger of one row (fee_jax.py:168-279, noise off), then digitisation (fee_jax.py:55-71).
// The float64 cumulative charge Q stays in registers: thread t holds ticks t * TPER + u in q[u]
// (as finish_row leaves them) and takes the tick after its last one from the next lane (DPP, or
// LDS across waves once, then updated by the same resets).  Q0 (LDS) is the unreset copy: what pass k
// needs of a single tick (the window's end, the reset point) every thread takes from there and
// puts through the k resets itself, so a pass has one barrier, for its crossing, and none for its
// charges (two barriers, and 64-bit maxima by lane shuffles where ballots do, took 4.0 of the 30 ms of
// a 160k-row launch; 2.1 with ballots).  Wave 0 then writes the outputs and the tape with one lane per
// pass (and one lane per tape point for the clamp masks).
template <int NT>
__device__ void fee_row(const Dev& d, double (&q)[kMaxOut / NT], const double* Q0, int r, int plane,
                        const RowOut& out, int (*sh_int)[NT / kWave]) {
  constexpr int TPER = kMaxOut / NT;
  constexpr int NW = NT / kWave;
  __shared__ int s_pe[kMaxH], s_pg[kMaxH], s_pi[kMaxH];
  __shared__ double s_pa[kMaxH];
  __shared__ double s_reset[kMaxH];  // Q[g] of each pass (written before the next pass's barrier)
  __shared__ double s_first[NW];
  const int t = threadIdx.x;
  const int nout = d.nout;
  const int lane = t & (kWave - 1), wid = t / kWave;
  const int H = d.H;
  const int o0 = t * TPER;
  // reset index of a pass without a crossing (i* = nout - 2), and its window end
  int g_none = nout - 2 + 1 + d.interval + 1;
  if (g_none >= nout) g_none = nout - 1;
  int e_none = nout - 2 + 1 + d.interval;
  if (e_none >= nout) e_none = nout - 1;
  if (lane == 0) s_first[wid] = q[0];
  __syncthreads();  // also: Q0 is complete
  double nx = __shfl_down(q[0], 1, kWave);  // Q[o0 + TPER]
  if (lane == kWave - 1) nx = wid + 1 < NW ? s_first[wid + 1] : 0.0;
  const double q_gnone = Q0[g_none];
  auto reset_by = [](double v, double c) {
    const double x = v - c;
    return x < 0 ? 0.0 : x;
  };
  // A wave's first crossing: lanes hold ticks in order, so the first lane with one has it.  kAbove: no
  // crossing, but some Q[1 .. nout-1] at or above thr; kBelow: none (what a crossing needs).
  constexpr int kBelow = 0x7fffffff, kAbove = kBelow - 1;
  for (int k = 0; k < H; ++k) {
    int cand = kBelow;
    bool above = false;
#pragma unroll
    for (int u = TPER - 1; u >= 0; --u) {
      const int o = o0 + u;
      const double q1 = u + 1 < TPER ? q[u + 1] : nx;
      const bool up = o <= nout - 2 && q1 >= d.thr;
      above = above || up;
      if (up && q[u] <= d.thr) cand = o;
    }
    const uint64_t mc = __ballot(cand != kBelow), ma = __ballot(above);
    const int first = __builtin_amdgcn_readlane(cand, mc ? __builtin_ctzll(mc) : 0);
    if (lane == 0) sh_int[k & 1][wid] = mc ? first : (ma ? kAbove : kBelow);
    __syncthreads();  // (pass k + 1 writes the other row, pass k + 2 after the next barrier)
    int istar = kBelow;
    for (int w = 0; w < NW; ++w) istar = sh_int[k & 1][w] < istar ? sh_int[k & 1][w] : istar;
    if (istar == kBelow && (k > 0 || q_gnone >= 0.0)) {
      // Nothing reaches the threshold: no crossing in this pass, and none later either.  A reset
      // Q <- max(Q - Q[g], 0) with Q[g] >= 0 never raises a value above max(Q, 0) < thr.  After
      // the first pass Q >= 0 everywhere, so Q[g] >= 0; in the first pass (the raw cumulative
      // charge may be negative) it is checked.  Every remaining pass ends at i* = nout-2 (no hit)
      // with e and g at their clamps, exactly as running it would; Q is not read again (the tape
      // follows Q0).
      if (t == 0) {
        double v = Q0[e_none];
        for (int p = 0; p < k; ++p) v = reset_by(v, s_reset[p]);
        for (int kk = k; kk < H; ++kk) {
          s_pe[kk] = e_none;
          s_pg[kk] = g_none;
          s_pi[kk] = nout - 2;
          s_pa[kk] = v;
        }
      }
      break;
    }
    if (istar >= kAbove) istar = nout - 2;
    int e = istar + 1 + d.interval;
    if (e >= nout) e = nout - 1;
    int g = istar + 1 + d.interval + 1;
    if (g >= nout) g = nout - 1;
    double Qg = Q0[g], Qe = Q0[e];
    for (int p = 0; p < k; ++p) {
      const double c = s_reset[p];
      Qg = reset_by(Qg, c);
      Qe = reset_by(Qe, c);
    }
    if (t == 0) {
      s_pe[k] = e;
      s_pg[k] = g;
      s_pi[k] = istar;
      s_pa[k] = Qe;
      s_reset[k] = Qg;
    }
#pragma unroll
    for (int u = 0; u < TPER; ++u)
      if (o0 + u < nout) q[u] = reset_by(q[u], Qg);
    nx = reset_by(nx, Qg);  // the next thread's first tick, reset as its owner resets it
  }
  __syncthreads();
  if (t >= kWave) return;
  // lane k < H: pass k's hit
  bool hit = false;
  float slope = 0.f;
  int tick = nout - 2;
  if (t < H) {
    const double a = s_pa[t];
    const int i = s_pi[t];
    const bool invalid = (a < d.thr) || (i == nout - 2);
    tick = invalid ? nout - 2 : i;
    out.adc[(int64_t)r * H + t] = (float)digitize(d, invalid ? 0.0 : a);
    out.ticks[(int64_t)r * H + t] = tick;
    hit = tick < nout - 3;
    slope = invalid ? 0.f : (float)digitize_slope(d, a);
  }
  const int hits = __popcll(__ballot(hit));
  if (t == 0) out.hit_cnt[r] = hits;
  if (!out.tape) return;
  // the clamp masks: lane j < 2H follows Q at point j (e_j, then g_{j-H}) through the passes
  FeeTape* tp = out.tape + r;
  double v = 0.0;
  if (t < 2 * H) {
    const int p = t < H ? s_pe[t] : s_pg[t - H];
    tp->pt[t] = (int16_t)p;
    v = Q0[p];
  }
  uint32_t mine = 0;
  for (int k = 0; k < H; ++k) {
    const double qg = __shfl(v, H + k, kWave);
    const double x = v - qg;
    const uint32_t m = (uint32_t)(__ballot(t < 2 * H && x >= 0) & 0xffffffffull);
    if (t == k) mine = m;
    v = x < 0 ? 0.0 : x;
  }
  if (t < H) {
    tp->mask[t] = mine;
    tp->slope[t] = slope;
    tp->tick[t] = tick;
  }
  if (t == 0) tp->plane = plane;
}

// Sum of the per-wave partial rows, waveform store, float64 cumulative charge: thread t holds
// Q[t * TPER + u] in q[u] (consecutive ticks per thread); Q0 receives a copy in LDS.
template <int NT>
__device__ void finish_row(const Dev& d, const float* acc, int nwaves, int rstride, double (&q)[kMaxOut / NT],
                           double* Q0, int r, const RowOut& out, double* shd) {
  constexpr int TPER = kMaxOut / NT;
  const int t = threadIdx.x;
  float row[TPER];
  double loc[TPER];
  double run = 0.0;
#pragma unroll
  for (int u = 0; u < TPER; ++u) {
    const int o = t * TPER + u;
    float v = 0.f;
    if (o < d.nout)
      for (int w = 0; w < nwaves; ++w) v += acc[w * rstride + o];
    row[u] = v;
    if (o < d.nout) run += (double)v * d.ts;
    loc[u] = run;
  }
  if (out.wfs) {
#pragma unroll
    for (int u = 0; u < TPER; ++u) {
      const int o = t * TPER + u;
      if (o < d.nout) out.wfs[(int64_t)r * d.nout + o] = row[u];
    }
  }
  double tot;
  const double ex = block_exclusive_scan<double>(run, shd, tot);
#pragma unroll
  for (int u = 0; u < TPER; ++u) q[u] = ex + loc[u];
  // the scan's barriers follow every read of the partial rows, which Q0 may now overwrite
#pragma unroll
  for (int u = 0; u < TPER; ++u) {
    const int o = t * TPER + u;
    if (o < d.nout) Q0[o] = q[u];
  }
}

// Contributions of one segment to one pixel row.  The segment's stripes landing on the row share
// one time window: V[j] = sum over stripes n_st * X_st[j], j < L, placed as (1-f) V at output
// tick S+j and f V at S-1+j (S = nt - L - k0), plus the cumsum boundary correction Delta at
// output ticks S-1 ((1-f) Delta) and S-2 (f Delta) (sim_jax.py:170-261).  Window ticks are kept for
// 1 <= o <= nout-1, corrections for 0 <= o <= nout-2 (the reference's garbage column takes the
// rest).
//
// Slack after each wave's partial row: an interior window (2 <= S, S + L <= nout) is stored three ticks
// per lane from S - 2 while 3 lane < L + 2, so it writes up to S + L + 1.
__host__ __device__ inline int row_pad(int) { return 4; }

// lane i receives lane i+1's value, lane 63 receives 0 (DPP wave shift; bound_ctrl supplies the
// zero, so no register needs clearing first)
__device__ __forceinline__ float lane_next0(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x130 /* wave_shl:1 */, 0xf, 0xf, true));
}

// Store of a whole window V held three samples per lane: lane l holds V[3 l - 2 + k] in vk, zero outside
// 0 <= m < L, for 3 l < L + 2 (the lanes that call it).  Output m receives so V[m] + sf V[m+1], and outputs -1 and -2
// their boundary corrections d1 and d2.  INSIDE windows (2 <= S and S + L <= nout) need no tick checks.
//
// The rounding is fixed: fma(so, V[m], sf V[m+1]), then the correction, then the row's tick.  d1 and d2 come rounded
// except that in windows that reach the row's ends a FUSED one is the multiply-add of its factors (so, sf) and delta.
template <bool INSIDE, bool FUSED>
__device__ __forceinline__ void store_window(float* accw, int lane, float v0, float v1, float v2, float so, float sf,
                                             float d1, float d2, float delta, int S, int L, int nout) {
#pragma clang fp contract(off)
  const float nx = lane_next0(v0);
  const int m = 3 * lane - 2;
  float c0 = __builtin_fmaf(so, v0, sf * v1), c1 = __builtin_fmaf(so, v1, sf * v2), c2 = __builtin_fmaf(so, v2, sf * nx);
  float* p = accw + S + m;
  if (INSIDE) {
    const float first = lane == 0 ? 1.f : 0.f;
    const float a0 = p[0], a1 = p[1], a2 = p[2];
    c0 = __builtin_fmaf(d2, first, c0);
    c1 = __builtin_fmaf(d1, first, c1);
    p[0] = a0 + c0;
    p[1] = a1 + c1;
    p[2] = a2 + c2;
  } else {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int o = S + m + k;
      if (m + k < L && o >= 0 && o < nout) {
        float val = o >= 1 ? (k == 0 ? c0 : (k == 1 ? c1 : c2)) : 0.f;
        if (o <= nout - 2 && m + k == -1) val = FUSED ? __builtin_fmaf(so, delta, val) : val + d1;
        if (o <= nout - 2 && m + k == -2) val = FUSED ? __builtin_fmaf(sf, delta, val) : val + d2;
        p[k] += val;
      }
    }
  }
}

// 0x00020000: word 3 of a raw (stride 0) buffer descriptor on gfx9-family GPUs.
constexpr int kBufDesc3 = 0x00020000;

// pairs whose windows a wave has in flight (128 events of 72k segments: 4 56.9, 8 55.3, 16 54.6 ms; 200k segments 8
// and 16 alike, and a row's last block is padded to a whole group)
constexpr int kFarGroup = 8;

// A pair with a non-finite factor (window T) at output tick o: what storing its whole padded window leaves there
// (a non-finite charge times the padding's zeros is NaN from S - 2 to S + 186 of an interior window).
__device__ __forceinline__ float odd_pair(const float* __restrict__ T, float so, float sf, int S, int o, int L, int nout) {
  const int m = o - S;
  const bool interior = S >= 2 && S + L <= nout;
  if (m < -2 || m > (interior ? 3 * (kWave - 1) - 3 : L - 1)) return 0.f;
  const float v = m >= 0 && m < L ? T[m] : 0.f, vn = m + 1 >= 0 && m + 1 < L ? T[m + 1] : 0.f;
  float val = interior || o >= 1 ? so * v + sf * vn : 0.f;
  if (interior ? m <= kWave - 4 : (m < 0 && o <= nout - 2)) val += 0.f * (so + sf);
  return val;
}

// Distinct LUT cells of a segment's diffusion bins that land on pixel offset a along one axis, with
// the bins' weights summed per cell: bins on the same cell read the same template window and the
// bin weights factorise (n_bin = n_e wx wy), so each distinct (cx, cy) is visited once with weight
// W[i] W[j].  ok[i] marks the distinct entries (slot of the first bin of each cell).  Later bins' weights are
// rounded and added, those of slot 0's cell by multiply-adds.
template <int NB>
__device__ __forceinline__ void axis_merge(int u, int a, int nsb, const float* w, float scale, bool* ok, int* cell,
                                           float* W) {
#pragma clang fp contract(off)
  constexpr int SYM = (NB - 1) / 2;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    ok[i] = false;
    cell[i] = 0;
    W[i] = 0.f;
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int v = u + i - SYM;
    const int dv = v < 0 ? -1 : (v >= nsb ? 1 : 0);
    if (dv != a) continue;
    const int cc = offset_bin(v - dv * nsb, 0, nsb);
    const float wi = scale * w[i];
    bool merged = false;
#pragma unroll
    for (int j = 0; j < i; ++j) {
      if (!merged && ok[j] && cell[j] == cc) {
        W[j] = j == 0 ? __builtin_fmaf(scale, w[i], W[j]) : W[j] + wi;
        merged = true;
      }
    }
    if (!merged) {
      ok[i] = true;
      cell[i] = cc;
      W[i] = wi;
    }
  }
}

// A segment's diffusion bins along one axis reach pixel offset a (|a| <= 1) when some bin
// position u + i - SYM, i < NB, lies in pixel a: always for a = 0, else only near the edge.
template <int NB>
__device__ __forceinline__ bool bins_reach(int u, int a, int nsb) {
  constexpr int SYM = (NB - 1) / 2;
  return a == 0 ? true : (a > 0 ? u + (NB - 1 - SYM) >= nsb : u - SYM < 0);
}

// Window of one segment's diffusion bins that land on one pixel: V[m] = sum_bins n_bin * (la T_{idx-1} +
// lb T_idx + lc T_{idx+1})[cx][cy][m] (sim_jax.py:186-194), three samples per lane as store_window takes
// them, each distinct LUT cell once.  `st` holds the merged bins of the two axes, NB each: weights along
// x (charge included) and y, byte offsets of the cells in TMW along x and y.  Lane i NB + j forms the
// product of bin i along x and bin j along y; the wave then walks the non-zero ones in order, four at a time:
// weight and offset by a lane read, the three templates' rows (neighbours in TMW) by one 12-byte load per lane
// each, per sample their interpolation and one multiply-add.  TMW (1.5 MB for 100 templates of 150 samples) stays
// in each XCD's L2.
// lane12: 12 * lane for the lanes that hold samples, past the table for the others (they read 0).
__host__ __device__ inline int bin_stride(int L) { return L + 2; }
__host__ __device__ inline int64_t bin_floats(int nm, int cm, int L) { return (int64_t)nm * cm * cm * bin_stride(L) + 4; }
constexpr int kBinItems = 16;  // items whose merged bins a wave stages at a time

template <int NB>
__device__ __forceinline__ void bins_window(__amdgpu_buffer_rsrc_t tmw, const int* st, int base, int ws4, int lane,
                                            int lane12, float la, float lb, float lc, float& v0, float& v1, float& v2) {
  float c = 0.f;
  int off = 0;
  if (lane < NB * NB) {
    const int i = lane / NB, j = lane - i * NB;
    c = __int_as_float(st[i]) * __int_as_float(st[NB + j]);
    off = base + st[2 * NB + i] + st[3 * NB + j];
  }
  float V[3] = {0.f, 0.f, 0.f};
  for (uint64_t m = __ballot(c != 0.f); m != 0;) {
    constexpr int G = 4;
    float w[G];
    typedef float f32x3 __attribute__((ext_vector_type(3)));
    f32x3 qa[G], qb[G], qc[G];
    int bit = 0;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const bool on = m != 0;  // past the last one: its row again with no weight
      bit = on ? __builtin_ctzll(m) : bit;
      m &= m - 1;
      const float wg = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c), bit));
      w[g] = on ? wg : 0.f;
      const int o = __builtin_amdgcn_readlane(off, bit);
      qa[g] = __builtin_bit_cast(f32x3, __builtin_amdgcn_raw_buffer_load_b96(tmw, lane12, o, 0));
      qb[g] = __builtin_bit_cast(f32x3, __builtin_amdgcn_raw_buffer_load_b96(tmw, lane12, o + ws4, 0));
      qc[g] = __builtin_bit_cast(f32x3, __builtin_amdgcn_raw_buffer_load_b96(tmw, lane12, o + 2 * ws4, 0));
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const float T = __builtin_fmaf(lc, qc[g][k], __builtin_fmaf(la, qa[g][k], lb * qb[g][k]));
        V[k] = __builtin_fmaf(w[g], T, V[k]);
      }
    }
  }
  v0 = V[0];
  v1 = V[1];
  v2 = V[2];
}

// Dynamic LDS of the waveform kernel: the per-wave partial rows (reused afterwards for the unreset
// float64 cumulative charge of the tape), then the neighbourhood's cell lists (ncell begins, ncell + 1
// cumulative counts, ncell offsets).
__host__ __device__ inline size_t rows_acc_bytes(int waves, int nout, int L) {
  const size_t acc = (size_t)waves * (nout + row_pad(L)) * 4, q = (size_t)nout * 8;
  return ((acc > q ? acc : q) + 15) & ~(size_t)15;
}
inline size_t rows_lds_bytes(int waves, int nout, int L, int ncell) {
  return rows_acc_bytes(waves, nout, L) + (size_t)(3 * ncell + 1) * 4;
}

constexpr int kMaxCells = 17 * 17;  // (2n+1)^2 for number_pix_neighbors <= 8

// The non-empty cells of a row's neighbourhood.  Cell i = (a, b), a, b in [-nn, nn] in row-major
// order, is the segment cell of the pixel (px - a, py - b); it is listed when cls(a, b) >= 0 and
// it holds segments, ordered by (cls, i); cnt(begin, end) gives how many of the cell's leading
// segments to list (a cell with none is left out).  One thread per cell loads the cell's segment range;
// then wave 0 ranks the listed cells, 64 at a time per class, with a ballot (the place) and a wave
// scan of the counts (the segments before each).  Writes c_beg, c_ab (a + 64 << 8 | b + 64), c_cum[0..k] (exclusive sums of the
// cells' segment counts) and ncls[c] = number of listed cells of class <= c, c < 3.  scratch
// holds 3 * kMaxCells ints; the call begins and ends with every thread of the block in it.
template <int NT, class Cls, class Cnt>
__device__ __forceinline__ void list_cells(const Dev& d, const int2* __restrict__ rng, int cell, Cls cls, Cnt cnt,
                                           int* scratch, int* c_beg, int* c_cum, int* c_ab, int* ncls) {
  const int t = threadIdx.x;
  const int side = 2 * d.ne + 1, ncell = side * side;
  const int px = cell % d.gx - d.halo;
  const int py = (cell / d.gx) % d.gy - d.halo;
  const int evp = cell / (d.gx * d.gy);
  int* s_key = scratch;
  int* s_cnt = scratch + kMaxCells;
  int* s_beg = scratch + 2 * kMaxCells;
  for (int i = t; i < ncell; i += NT) {
    const int a = i / side - d.ne, b = i % side - d.ne;
    const int c = cls(a, b);
    const int qx = px - a, qy = py - b;
    int key = -1, n = 0, beg = 0;
    if (c >= 0 && qx >= -d.halo && qx < d.nx + d.halo && qy >= -d.halo && qy < d.ny + d.halo) {
      const int2 rg = rng[((int64_t)evp * d.gy + (qy + d.halo)) * d.gx + (qx + d.halo)];
      const int m = rg.y > rg.x ? cnt(rg.x, rg.y) : 0;
      if (m > 0) {
        key = c * ncell + i;
        n = m;
        beg = rg.x;
      }
    }
    s_key[i] = key;
    s_cnt[i] = n;
    s_beg[i] = beg;
  }
  __syncthreads();
  // ranks in (class, i) order: wave 0 walks the cells class by class, 64 at a time; a ballot gives
  // each listed cell its rank and a wave scan of the counts the segments before it
  if (t < kWave) {
    const int lane = t;
    int rank0 = 0, before0 = 0;
    for (int c = 0; c < 3; ++c) {
      for (int i0 = 0; i0 < ncell; i0 += kWave) {
        const int i = i0 + lane;
        const int key = i < ncell ? s_key[i] : -1;
        const bool on = key >= 0 && key / ncell == c;
        const uint64_t m = __ballot(on);
        if (m == 0) continue;
        const int n = on ? s_cnt[i] : 0;
        int inc = n;
#pragma unroll
        for (int dd = 1; dd < kWave; dd <<= 1) {
          const int u = __shfl_up(inc, dd, kWave);
          if (lane >= dd) inc += u;
        }
        if (on) {
          const int rk = rank0 + __popcll(m & ((1ull << lane) - 1));
          const int a = i / side - d.ne, b = i % side - d.ne;
          c_beg[rk] = s_beg[i];
          c_cum[rk] = before0 + (inc - n);
          c_ab[rk] = ((a + 64) << 8) | (b + 64);
        }
        rank0 += __popcll(m);
        before0 += __shfl(inc, kWave - 1, kWave);
      }
      if (lane == 0) ncls[c] = rank0;
    }
    if (lane == 0) c_cum[rank0] = before0;
  }
  __syncthreads();
}

// The same lists for the forward, by one wave (lane l of `lane`, which alone calls it): classes 0 (far), 1
// (side) and 2 (centre), no condition on the segments.  The cells are walked in (class, i) order, lane l
// taking cells 2 l and 2 l + 1 of each 128, so one wave scan of the counts numbers 128 cells; no scratch.
// The block's other waves go on meanwhile; a barrier must follow.
__device__ __forceinline__ void list_cells_fwd(const Dev& d, const int2* __restrict__ rng, int cell, int lane, int* c_beg,
                                               int* c_cum, int* c_ab, int* ncls) {
  const int n = d.ne, side = 2 * n + 1, ncell = side * side, nfar = ncell - 9;
  const int px = cell % d.gx - d.halo;
  const int py = (cell / d.gx) % d.gy - d.halo;
  const int evp = cell / (d.gx * d.gy);
  const int top = (n - 1) * side, mid = top + 3 * (side - 3);  // far cells before the rows a = -1 .. 1, and through them
  int rank0 = 0, before0 = 0;
  for (int i0 = 0; i0 < ncell; i0 += 2 * kWave) {
    int cnt[2], beg[2], ab[2], cls[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int i = i0 + 2 * lane + h;
      int a = 0, b = 0;
      cls[h] = i < nfar ? 0 : (i < ncell - 1 ? 1 : 2);
      if (i < top) {
        a = i / side - n;
        b = i % side - n;
      } else if (i < mid) {
        const int j = i - top, w = side - 3;
        a = j / w - 1;
        b = j % w - n;
        if (b >= -1) b += 3;
      } else if (i < nfar) {
        const int j = i - mid;
        a = j / side + 2;
        b = j % side - n;
      } else if (i < ncell - 1) {
        const int j = i - nfar, k = j < 4 ? j : j + 1;  // 3 x 3 without its centre
        a = k / 3 - 1;
        b = k % 3 - 1;
      }
      const int qx = px - a, qy = py - b;
      cnt[h] = beg[h] = 0;
      ab[h] = ((a + 64) << 8) | (b + 64);
      if (i < ncell && qx >= -d.halo && qx < d.nx + d.halo && qy >= -d.halo && qy < d.ny + d.halo) {
        const int2 rg = rng[((int64_t)evp * d.gy + (qy + d.halo)) * d.gx + (qx + d.halo)];
        beg[h] = rg.x;
        cnt[h] = rg.y > rg.x ? rg.y - rg.x : 0;
      }
    }
    // listed cells before this lane's, and their segments
    const uint64_t m0 = __ballot(cnt[0] > 0), m1 = __ballot(cnt[1] > 0);
    const uint64_t lt = (1ull << lane) - 1;
    int inc = cnt[0] + cnt[1];
#pragma unroll
    for (int dd = 1; dd < kWave; dd <<= 1) {
      const int u = __shfl_up(inc, dd, kWave);
      if (lane >= dd) inc += u;
    }
    int rk = rank0 + __popcll(m0 & lt) + __popcll(m1 & lt), before = before0 + inc - cnt[0] - cnt[1];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (cnt[h] == 0) continue;
      c_beg[rk] = beg[h];
      c_cum[rk] = before;
      c_ab[rk] = ab[h];
      ++rk;
      before += cnt[h];
    }
    // listed cells of class <= c, c < 3
    const uint64_t f0 = __ballot(cnt[0] > 0 && cls[0] == 0), f1 = __ballot(cnt[1] > 0 && cls[1] == 0);
    const uint64_t s0 = __ballot(cnt[0] > 0 && cls[0] <= 1), s1 = __ballot(cnt[1] > 0 && cls[1] <= 1);
    if (lane == 0) {
      ncls[0] = (i0 ? ncls[0] : 0) + __popcll(f0) + __popcll(f1);
      ncls[1] = (i0 ? ncls[1] : 0) + __popcll(s0) + __popcll(s1);
    }
    rank0 += __popcll(m0) + __popcll(m1);
    before0 += __builtin_amdgcn_readlane(inc, kWave - 1);
  }
  if (lane == 0) {
    ncls[2] = rank0;
    c_cum[rank0] = before0;
  }
}

// ------------------------------------------------------------------------------------------
// rows on the XCDs
// ------------------------------------------------------------------------------------------
//
// Workgroups are dispatched round-robin over the XCDs (workgroup i runs on XCD i % kXcd) and, within one, as
// its CUs come free.  The row kernels hand the rows out in row order by runs of kRowRun: neighbours along a
// pixel row, which share most of their segments, land in one L2, and every XCD gets its share of the dense
// and of the empty parts of an event.  One contiguous band an XCD, cut at equal shares of the estimated work
// in an order by cell tiles, with the last quarter of the rows handed out by counters, balanced worse: 200k
// segments 1.52 -> 1.21 ms, 128 events of 72k segments 52.5 -> 50.5 ms, and the adjoint's equal row counts an
// XCD 720 -> 575 us (near), 420 -> 319 (far), 570 -> 430 (waveforms).  Runs of 4 to 64 are within 3 %.  (Each
// pair of figures on the row kernels of the time; they take 1.32 and 55.3 ms, 414, 352 and 506 us as they are now.)
constexpr int kRowRun = 16;

__device__ __forceinline__ int64_t run_row() {  // of this workgroup; at or past the number of rows: none
  const int64_t x = blockIdx.x % kXcd, j = blockIdx.x / kXcd;
  return (j / kRowRun * kXcd + x) * kRowRun + j % kRowRun;
}

inline int64_t run_grid(int64_t max_rows) {
  return (max_rows + kXcd * kRowRun - 1) / (kXcd * kRowRun) * (kXcd * kRowRun);
}

// One workgroup per pixel row.  Whether a charge within rounding of the threshold crosses it, and so a hit's tick,
// hangs on the order in which the row's float32 terms are added, so the order is part of the result: wave w sums the
// pairs of blocks w, w + WAVES, .. of 64 pairs of the far and side cells in pair order (cells in list order, a
// cell's segments by window and input order), each block's stripes and then its diffusion bins; then the centre
// cell's segments w, w + WAVES, .. ; then the waves' partial rows are added in order.  (Pairs sorted by time and
// summed by 64-tick chunks, two multiply-adds a pair and chunk, took 1.20 ms for 200k segments and 50.6 for 128
// events of 72k, where this order takes 1.32 and 55.3, but moved about one hit in 3 million to another tick.)
//
// What bounds it: the issue of vector instructions, 20 a stripe pair (six lane reads of the pair's values, a
// lane shift, nine for its three samples a lane, two corrections, two addresses), and the bins' 12 multiply-adds a
// cell; occupancy is 4 workgroups a CU by LDS (38 KB).  The same order with three 4-byte loads and as many lane
// shifts a pair, a branch on each pair's window and the bins as unrolled scalar code took 1.60 and 67.9 ms.
template <int NB, int WAVES>
__global__ __launch_bounds__(WAVES * kWave) __attribute__((amdgpu_waves_per_eu(4))) void k_rows_fwd(Dev d, Tables tb, const SegRec* __restrict__ rec,
                                                            const int2* __restrict__ rng, const int* __restrict__ row_cell,
                                                            const int* __restrict__ n_rows_dev, int64_t max_rows,
                                                            const float* __restrict__ dtot,
                                                            const PairRec* __restrict__ prs, int64_t nseg, RowOut out) {
  constexpr int NT = WAVES * kWave;
  extern __shared__ __align__(16) char smem[];
  __shared__ double shd[NT / kWave];
  __shared__ int shi[2][NT / kWave];
  __shared__ int ncls[3];  // far cells, + the 8 side cells, + the centre cell

  const int P0 = *n_rows_dev;
  const int P = P0 < max_rows ? P0 : (int)max_rows;
  const int64_t row = run_row();
  if (row == 0 && threadIdx.x == 0) copy_count(n_rows_dev, out.n_rows, max_rows, out.status);
  if (row >= P) {
    if (row < max_rows && threadIdx.x == 0) out.hit_cnt[row] = 0;  // (the hit scan runs over max_rows)
    return;
  }
  const int r = (int)row;
  const int nout = d.nout;
  float* acc = (float*)smem;
  // this row's neighbourhood cells: far, then the 8 side cells, then the centre, each in (a, b) order
  const int ncell = (2 * d.ne + 1) * (2 * d.ne + 1);
  int* const c_beg = (int*)(smem + rows_acc_bytes(WAVES, nout, d.L));
  int* const c_cum = c_beg + ncell;
  int* const c_ab = c_cum + ncell + 1;
  const int t = threadIdx.x;
  const int lane = t & (kWave - 1);
  const int wid = __builtin_amdgcn_readfirstlane(t / kWave);
  const int rstride = nout + row_pad(d.L);
  const int cell = row_cell[r];
  const int evp = cell / (d.gx * d.gy);  // ev * ntpc + plane
  const int plane = evp % d.ntpc;
  if (t == 0) {
    const int px = cell % d.gx - d.halo;
    const int py = (cell / d.gx) % d.gy - d.halo;
    out.pixel_ids[r] = ((int64_t)evp * d.ny + py) * d.nx + px;
  }
  if (wid == 0) list_cells_fwd(d, rng, cell, lane, c_beg, c_cum, c_ab, ncls);
  __shared__ int s_bins[WAVES][kBinItems][4 * NB];
  {
    const int nz = WAVES * rstride, n4 = nz / 4;
    for (int o = t; o < n4; o += NT) reinterpret_cast<float4*>(acc)[o] = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int o = 4 * n4 + t; o < nz; o += NT) acc[o] = 0.f;
  }
  __syncthreads();

  float* accw = acc + wid * rstride;
  const int nsc = ncls[1], nct = ncls[2];  // far + side cells, all cells
  const int nsb = d.nsb, L = d.L, cm = d.cm, side = 2 * d.ne + 1, ws4 = 4 * bin_stride(L);
  const bool holds = 3 * lane < L + 2;  // does the lane hold samples of a window
  const int lane12 = holds ? 12 * lane : 0x7ffffff0;
  const __amdgpu_buffer_rsrc_t tnp =
      __builtin_amdgcn_make_buffer_rsrc((void*)tb.TNP, 0, d.lx * d.ly * kWinPad * 4, kBufDesc3);
  const __amdgpu_buffer_rsrc_t tmw = __builtin_amdgcn_make_buffer_rsrc(
      (void*)tb.TMW, 0, (int)(uint32_t)(bin_floats(d.nm, cm, L) * 4), kBufDesc3);
  // The wave's blocks of 64 pairs: of the far and side cells' pairs, flattened, blocks wid, wid + WAVES, ..;
  // then of the centre cell's segments wid, wid + WAVES, .. .
  const int nfar = c_cum[nsc], nall = c_cum[nct];
  const int nfb = (nfar - wid * kWave + WAVES * kWave - 1) / (WAVES * kWave);
  const int ncb = (nall - nfar - wid + WAVES * kWave - 1) / (WAVES * kWave);
  struct Pair {
    PairRec P;
    float D;      // boundary correction
    int sg, ab;   // segment (-1: none), row offset
  };
  auto fetch = [&](int i, Pair& B) {
    B = Pair{PairRec{0, 0.f, 0.f, 0}, 0.f, -1, 0};
    int lo = nsc;
    const int p = i < nfb ? (i * WAVES + wid) * kWave + lane : nfar + wid + WAVES * (kWave * (i - nfb) + lane);
    if (i >= nfb + ncb || p >= (i < nfb ? nfar : nall)) return;
    if (i < nfb) {
      int hi = nsc - 1;  // the cell holding p: last c with c_cum[c] <= p
      lo = 0;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (c_cum[mid] <= p) lo = mid;
        else hi = mid - 1;
      }
    }
    B.sg = c_beg[lo] + (p - c_cum[lo]);
    B.ab = c_ab[lo];
    B.P = prs[B.sg];
    B.D = dtot[(int64_t)(((B.ab >> 8) - 64 + d.ne) * side + ((B.ab & 255) - 64 + d.ne)) * nseg + B.sg];
  };
  Pair nxt;
  fetch(0, nxt);
  for (int i = 0; i < nfb + ncb; ++i) {
    const Pair B = nxt;
    fetch(i + 1, nxt);  // (its loads arrive while this block is worked on)
    const PairRec P = B.P;
    const int a = (B.ab >> 8) - 64, b = (B.ab & 255) - 64;
    const int ux = P.u(), uy = P.v();
    const float omf = 1.f - P.f;
    const float d1 = omf * B.D, d2 = P.f * B.D;
    if (i < nfb) {
      // stripes (with none, nn = 0, a side pixel gets the correction and its diffusion bins only)
      const bool on = a >= -d.nn && a <= d.nn && b >= -d.nn && b <= d.nn;
      const float st = on ? 1.f : 0.f;
      float so = st * (P.ne * omf), sf = st * (P.ne * P.f);
      const int row = on ? offset_bin(ux, a, nsb) * d.ly + offset_bin(uy, b, nsb) : 0;
      const bool odd = B.sg >= 0 && !(fabsf(so) + fabsf(sf) < __builtin_inff());
      int S = P.S, off = row * (kWinPad * 4);
      float e1 = d1, e2 = d2;
      if (B.sg < 0 || odd || P.ne == 0.f) {  // no pair: a window inside the row that adds nothing
        S = 2;
        off = 0;
        so = sf = e1 = e2 = 0.f;
      }
      const int n = min(nfar - (i * WAVES + wid) * kWave, kWave);
      const uint64_t edge = __ballot(S < 2 || S + L > nout);
      if (holds) {
        auto from = [](float v, int j) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j)); };
        for (int j = 0; j < n; j += kFarGroup) {
          typedef float f32x3 __attribute__((ext_vector_type(3)));
          f32x3 v[kFarGroup];
#pragma unroll
          for (int g = 0; g < kFarGroup; ++g)
            v[g] = __builtin_bit_cast(
                f32x3, __builtin_amdgcn_raw_buffer_load_b96(tnp, lane12, __builtin_amdgcn_readlane(off, j + g), 0));
          if (((edge >> j) & ((1 << kFarGroup) - 1)) == 0) {
#pragma unroll
            for (int g = 0; g < kFarGroup; ++g)
              store_window<true, false>(accw, lane, v[g][0], v[g][1], v[g][2], from(so, j + g), from(sf, j + g),
                                        from(e1, j + g), from(e2, j + g), 0.f, __builtin_amdgcn_readlane(S, j + g), L, nout);
            continue;
          }
#pragma unroll
          for (int g = 0; g < kFarGroup; ++g) {
            const float p = from(so, j + g), q = from(sf, j + g), c1 = from(e1, j + g), c2 = from(e2, j + g);
            const int at = __builtin_amdgcn_readlane(S, j + g);
            if ((edge >> (j + g)) & 1) store_window<false, false>(accw, lane, v[g][0], v[g][1], v[g][2], p, q, c1, c2, 0.f, at, L, nout);
            else store_window<true, false>(accw, lane, v[g][0], v[g][1], v[g][2], p, q, c1, c2, 0.f, at, L, nout);
          }
        }
      }
      for (uint64_t m = __ballot(odd); m != 0; m &= m - 1) {
        const int j = __builtin_ctzll(m);
        const float* T = tb.TNP + (int64_t)__builtin_amdgcn_readlane(row, j) * kWinPad + 2;
        const float q = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(st * (P.ne * omf)), j));
        const float r = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(st * (P.ne * P.f)), j));
        for (int o = lane; o < nout; o += kWave)
          accw[o] += odd_pair(T, q, r, __builtin_amdgcn_readlane(P.S, j), o, L, nout);
      }
    }
    // Diffusion bins that land on this pixel: of every segment of the centre cell, and of those of the side
    // cells near their pixel's edge.  Lane by lane: does any bin land here, and the bins merged per LUT cell
    // along each axis, staged in LDS for the wave, which then computes and stores one pair's window after
    // the other.
    const bool bins = B.sg >= 0 && a >= -1 && a <= 1 && b >= -1 && b <= 1 && P.ne != 0.f && bins_reach<NB>(ux, a, nsb) &&
                      bins_reach<NB>(uy, b, nsb);
    uint64_t m = __ballot(bins);
    if (m == 0) continue;
    bool ok[NB];
    int base = 0, cxs[NB], cys[NB];
    float la = 0.f, lb = 0.f, lc = 0.f, WX[NB], WY[NB];
    if (bins) {
      const SegRec& R = rec[B.sg];
      la = R.la;
      lb = R.lb;
      lc = R.lc;
      base = (R.idx - 1) * ws4;
      axis_merge<NB>(ux, a, nsb, R.wx, P.ne, ok, cxs, WX);
      axis_merge<NB>(uy, b, nsb, R.wy, 1.f, ok, cys, WY);
    }
    const float delta = i < nfb ? 0.f : B.D;  // (a side pair's correction went with its stripe)
    while (m != 0) {
      const int rank = __popcll(m & ((1ull << lane) - 1));
      if (((m >> lane) & 1) && rank < kBinItems) {
        int* stg = s_bins[wid][rank];
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          stg[k] = __float_as_int(WX[k]);
          stg[NB + k] = __float_as_int(WY[k]);
          stg[2 * NB + k] = cxs[k] * cm * d.nm * ws4;
          stg[3 * NB + k] = cys[k] * d.nm * ws4;
        }
      }
      __builtin_amdgcn_wave_barrier();  // wave-local LDS: program order
      for (int k = 0; k < kBinItems && m != 0; ++k) {
        const int j = __builtin_ctzll(m);
        m &= m - 1;
        auto get = [&](float v) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j)); };
        float v0, v1, v2;
        bins_window<NB>(tmw, s_bins[wid][k], __builtin_amdgcn_readlane(base, j), ws4, lane, lane12, get(la), get(lb),
                        get(lc), v0, v1, v2);
        const float dl = get(delta), f = get(P.f);
        const int S = __builtin_amdgcn_readlane(P.S, j);
        if (holds) {
          if (S >= 2 && S + L <= nout) store_window<true, true>(accw, lane, v0, v1, v2, 1.f - f, f, (1.f - f) * dl, f * dl, dl, S, L, nout);
          else store_window<false, true>(accw, lane, v0, v1, v2, 1.f - f, f, (1.f - f) * dl, f * dl, dl, S, L, nout);
        }
      }
      __builtin_amdgcn_wave_barrier();  // the stage is rewritten
    }
  }
  __syncthreads();
  double q[kMaxOut / NT];
  double* Q0 = (double*)smem;
  finish_row<NT>(d, acc, WAVES, rstride, q, Q0, r, out, shd);
  fee_row<NT>(d, q, Q0, r, plane, out, shi);
}

// Self-trigger on caller waveforms (simulate_stochastic on an arbitrary wfs): one workgroup per
// row, the same finish/fee code as the fused path.
template <int NT>
__global__ __launch_bounds__(NT) void k_fee_rows(Dev d, const float* __restrict__ wfs, const int64_t* __restrict__ pids,
                                                 int64_t n_rows, RowOut out) {
  __shared__ __align__(16) char smem[kMaxOut * 8];
  __shared__ float accs[kMaxOut];
  __shared__ double shd[NT / kWave];
  __shared__ int shi[2][NT / kWave];
  const int64_t r = blockIdx.x;
  if (r >= n_rows) return;
  for (int o = threadIdx.x; o < kMaxOut; o += NT) accs[o] = o < d.nout ? wfs[r * d.nout + o] : 0.f;
  __syncthreads();
  const int64_t pid = pids[r];
  const int npl = d.nx * d.ny;
  const int plane = pid >= 0 ? (int)((pid / npl) % d.ntpc) : 0;
  double q[kMaxOut / NT];
  double* Q0 = (double*)smem;
  RowOut o2 = out;
  o2.wfs = nullptr;
  finish_row<NT>(d, accs, 1, d.nout, q, Q0, (int)r, o2, shd);
  fee_row<NT>(d, q, Q0, (int)r, plane, o2, shi);
  if (threadIdx.x == 0 && pid < 0) out.hit_cnt[r] = 0;
}

// ------------------------------------------------------------------------------------------
// 4. hit compaction (sim_jax.py:619-647) with coordinates (detsim_jax.py:296-319)
// ------------------------------------------------------------------------------------------

struct HitOut {
  float *adc, *x, *y, *z, *tick, *prob;
  int64_t *event, *pixel;
  int32_t* index;
};

__global__ void k_hits(Dev d, const int64_t* __restrict__ pids, const float* __restrict__ adc, const int* __restrict__ ticks,
                       const int* __restrict__ hit_off, const int64_t* __restrict__ n_rows_dev, int64_t max_rows,
                       int64_t n_rows_static, HitOut h) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t P = n_rows_dev ? *n_rows_dev : n_rows_static;
  if (P > max_rows) P = max_rows;
  const int H = d.H;
  if (i >= P * H) return;
  const int64_t r = i / H;
  const int k = (int)(i % H);
  const int tick = ticks[i];
  if (!(tick < d.nout - 3)) return;
  const int64_t pid = pids[r];
  if (pid < 0) return;
  int before = 0;
  for (int kk = 0; kk < k; ++kk) before += (ticks[r * H + kk] < d.nout - 3) ? 1 : 0;
  const int64_t pos = (int64_t)hit_off[r] + before;
  if (pos < 0 || pos >= P * H) return;  // offsets come from a scan of per-row counts <= H
  const int npl = d.nx * d.ny;
  const int px = (int)(pid % d.nx), py = (int)((pid / d.nx) % d.ny);
  const int plane = (int)((pid / npl) % d.ntpc);
  const int64_t ev = pid / ((int64_t)npl * d.ntpc);
  const double za = d.tpc[plane][2][0], zc = d.tpc[plane][2][1];
  const double sgn = (zc - za) > 0 ? 1.0 : ((zc - za) < 0 ? -1.0 : 0.0);
  h.adc[pos] = adc[i];
  h.x[pos] = (float)((double)px * d.pitch + d.tpc[plane][0][0] + d.pitch / 2);
  h.y[pos] = (float)((double)py * d.pitch + d.tpc[plane][1][0] + d.pitch / 2);
  h.z[pos] = (float)(za + (double)tick * d.ts * d.v * sgn);
  h.tick[pos] = (float)tick;
  h.prob[pos] = 1.0f;
  h.event[pos] = ev;
  h.pixel[pos] = pid;
  h.index[pos] = (int32_t)i;
}

// ------------------------------------------------------------------------------------------
// 4b. negative pixel ids of the reference's pixel set
// ------------------------------------------------------------------------------------------

// The reference's pixel set is the sorted unique main-pixel ids plus an appended -1
// (sim_jax.py:716-721).  Besides the ids >= 0 (the rows built here) it holds negative ids:
// a padding segment (eventID -1, optimize/dataio.py:347-359) on the pixel plane gets the id
// pixel2id packs for event -1 (detsim_jax.py:230-244), and a segment whose main pixel is off the
// plane gets -1.  Those rows carry no charge and no hits, so only their ids are produced here.
// Every such id lies in [-ntpc ny nx, -1]; bit (id + ntpc ny nx) of `bits` marks it (integer
// atomics: the bit set does not depend on the order).  eventID < -1 is invalid input and skipped.
__global__ void k_neg_mark(Dev d, SegIn in, uint32_t* __restrict__ bits) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= in.n) return;
  const int ev = to_int_clamped((double)ldcol(in.ev, i, in.stride));
  if (ev < -1) return;
  Phys ph;
  seg_physics(d, in, i, ph);
  const bool on_plane = ph.mpx >= 0 && ph.mpx < d.nx && ph.mpy >= 0 && ph.mpy < d.ny;
  if (ev >= 0 && on_plane) return;
  const int64_t span = (int64_t)d.ntpc * d.ny * d.nx;
  const int64_t b = on_plane ? pixel_id(d, -1, ph.plane, ph.mpx, ph.mpy) + span : span - 1;
  if (b < 0 || b >= span) return;
  atomicOr(&bits[b >> 5], 1u << (b & 31));
}

// The marked ids in ascending order (one workgroup of kPadThreads threads: each takes a
// contiguous run of bitmap words, counts its bits, and writes its ids after a block scan).
constexpr int kPadThreads = 1024;

__global__ __launch_bounds__(kPadThreads) void k_pad_list(const uint32_t* __restrict__ bits, int64_t span,
                                                         int64_t* __restrict__ ids, int64_t max_ids,
                                                         int64_t* __restrict__ n_out) {
  __shared__ int64_t part[kPadThreads];
  const int t = threadIdx.x;
  const int64_t words = (span + 31) >> 5;
  const int64_t per = (words + kPadThreads - 1) / kPadThreads;
  const int64_t w0 = (int64_t)t * per, w1 = w0 + per < words ? w0 + per : words;
  int64_t cnt = 0;
  for (int64_t w = w0; w < w1; ++w) cnt += __popc(bits[w]);
  part[t] = cnt;
  __syncthreads();
  for (int off = 1; off < kPadThreads; off <<= 1) {  // inclusive Hillis-Steele scan
    const int64_t v = t >= off ? part[t - off] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  int64_t pos = part[t] - cnt;
  for (int64_t w = w0; w < w1; ++w) {
    uint32_t m = bits[w];
    while (m) {
      const int k = __ffs(m) - 1;
      m &= m - 1;
      if (pos < max_ids) ids[pos] = w * 32 + k - span;
      ++pos;
    }
  }
  if (t == kPadThreads - 1) *n_out = part[t];
}

// ------------------------------------------------------------------------------------------
// 5. response tables (consts_jax.py:427-447), float64 arithmetic
// ------------------------------------------------------------------------------------------

// One workgroup per (template m, cx, cy) series: template values over the full time range,
// prefix sums, then the window, boundary-difference and window-prefix tables.
// main != 0: m in [0, nm), (cx, cy) in [0, cm)^2 -> TM, DM, CTM; else the raw response over all
// (cx, cy) -> TN, DN, CTN.
__global__ __launch_bounds__(256) void k_lut_tables(Dev d, const float* __restrict__ raw, int main_tables, float* __restrict__ Tw,
                                                    float* __restrict__ Twp, float2* __restrict__ Dt,
                                                    double* __restrict__ CT) {
  __shared__ double T[kMaxOut];
  __shared__ double g[128];
  __shared__ double shd[4];
  const int series = blockIdx.x;
  int m, cx, cy;
  if (main_tables) {
    m = series / (d.cm * d.cm);
    cx = (series / d.cm) % d.cm;
    cy = series % d.cm;
  } else {
    m = 0;
    cx = series / d.ly;
    cy = series % d.ly;
  }
  const int nt = d.nt, ext = d.ext;
  const float* R = raw + ((int64_t)cx * d.ly + cy) * nt;
  // normalised Gaussian kernel of template m (norm.pdf(k, scale=sigma), consts_jax.py:427-428)
  if (threadIdx.x == 0) {
    const double s = d.sig[m];
    double sum = 0.0;
    for (int k = -ext; k <= ext; ++k) {
      const double z = (double)k / s;
      const double v = exp(-0.5 * z * z) / (sqrt(2.0 * M_PI) * s);
      g[k + ext] = v;
      sum += v;
    }
    for (int k = 0; k <= 2 * ext; ++k) g[k] /= sum;
  }
  __syncthreads();
  for (int t = threadIdx.x; t < nt; t += blockDim.x) {
    double v;
    if (m == 0) {
      v = (double)R[t];
    } else {
      v = 0.0;
      for (int k = -ext; k <= ext; ++k) {
        const int tt = t + k;
        if (tt >= 0 && tt < nt) v += (double)R[tt] * g[k + ext];
      }
    }
    T[t] = v;
  }
  __syncthreads();
  // inclusive prefix sum C[t] (blocked: each thread 8 consecutive entries)
  constexpr int PER = kMaxOut / 256;
  double loc[PER];
  double run = 0.0;
  for (int u = 0; u < PER; ++u) {
    const int t = threadIdx.x * PER + u;
    if (t < nt) run += T[t];
    loc[u] = run;
  }
  double tot;
  const double ex = block_exclusive_scan<double>(run, shd, tot);
  __syncthreads();
  const int L = d.L;
  // keep the window values (float32, as used by the forward) before T is overwritten
  __shared__ float win[kMaxOut];
  for (int j = threadIdx.x; j < L; j += blockDim.x) win[j] = (float)T[nt - L + j];
  __syncthreads();
  for (int u = 0; u < PER; ++u) {
    const int t = threadIdx.x * PER + u;
    if (t < nt) T[t] = ex + loc[u];  // T now holds C
  }
  __syncthreads();
  const int64_t sbase = (int64_t)series;
  for (int j = threadIdx.x; j < L; j += blockDim.x) Tw[sbase * L + j] = win[j];
  if (Twp)
    for (int p = threadIdx.x; p < kWinPad; p += blockDim.x)
      Twp[sbase * kWinPad + p] = (p >= 2 && p < L + 2) ? win[p - 2] : 0.f;
  const double cref = T[nt - L];
  for (int k = threadIdx.x; k < nt; k += blockDim.x) {
    const double c0 = T[k];
    const double c1 = T[k + 1 < nt ? k + 1 : nt - 1];
    Dt[(int64_t)k * gridDim.x + sbase] = make_float2((float)(cref - c0), (float)(c1 - c0));  // tick-major
  }
  if (threadIdx.x == 0) {
    double c = 0.0;
    CT[sbase * (L + 1)] = 0.0;
    for (int j = 0; j < L; ++j) {
      c += (double)win[j];
      CT[sbase * (L + 1) + j + 1] = c;
    }
  }
}

// The template windows TM regrouped as TMW, with the leading zeros of each row (and two values past the
// last row).
__global__ void k_lut_tmw(Dev d, const float* __restrict__ TM, float* __restrict__ TMW, int64_t total) {
  const int ws = bin_stride(d.L);
  const int64_t cc = (int64_t)d.cm * d.cm, rows = cc * d.nm;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = i / ws;
    const int j = (int)(i - row * ws) - 2;
    const int64_t m = row % d.nm, cell = row / d.nm;
    TMW[i] = row < rows && j >= 0 ? TM[(m * cc + cell) * d.L + j] : 0.f;
  }
}

// Padded (T_{m-1}, T_m, T_{m+1}) windows for m in [1, nm-2]; other slabs are zero.
// DNS[k][ux][uy][ab] = DN[k][offset_bin(ux, a)][offset_bin(uy, b)] for the (2 ne + 1)^2 row offsets
// (a, b) = (ab / W - ne, ab % W - ne) of a segment in sub-bin (ux, uy): the raw response's D entries
// of one segment's neighbour stripes, contiguous.
__global__ void k_lut_dns(Dev d, const float2* __restrict__ DN, float2* __restrict__ DNS) {
  const int W = 2 * d.ne + 1, WW = W * W, nsb = d.nsb;
  const int64_t total = (int64_t)d.nt * nsb * nsb * WW;
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < total; j += (int64_t)gridDim.x * blockDim.x) {
    const int ab = (int)(j % WW);
    const int64_t q = j / WW;
    const int uy = (int)(q % nsb), ux = (int)((q / nsb) % nsb);
    const int64_t k = q / ((int64_t)nsb * nsb);
    const int a = ab / W - d.ne, b = ab % W - d.ne;
    DNS[j] = DN[(k * d.lx + offset_bin(ux, a, nsb)) * d.ly + offset_bin(uy, b, nsb)];
  }
}

__global__ void k_lut_tm3(Dev d, const float* __restrict__ TM, float3* __restrict__ TM3) {
  const int64_t cc = (int64_t)d.cm * d.cm;
  const int64_t n = cc * d.nm * kWinPad;
  const int64_t per = cc * d.L;  // one template slab of TM
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const int p = (int)(i % kWinPad);
    const int64_t series = i / kWinPad;  // m * cm * cm + cx * cm + cy
    const int64_t m = series / cc;
    float3 v = make_float3(0.f, 0.f, 0.f);
    if (m >= 1 && m <= d.nm - 2 && p >= 2 && p < d.L + 2) {
      const int64_t t = series * d.L + (p - 2);
      v = make_float3(TM[t - per], TM[t], TM[t + per]);
    }
    TM3[i] = v;
  }
}

}  // namespace lsim
