// gfx950 kernels of the differentiable path (no counterpart in the reference).
//
// Model (log-uniform grid): disk cell c with bin k, limb L = 1 - u1(1-mu) -
// u2(1-mu)^2 and rigid-rotation velocity delta = vsini y has the integer shift m
// and weight t of the forward engine; phi_pc is the bilinear sample of phase p's
// M x M filling-factor map over [-1, 1]^2 (psi_pc likewise from the facula map,
// when there is one); the phase spectrum is
//   I_p = sum_k sum_d HQ_pk[d] Q_k[j - d] + HS_pk[d] S_k[j - d] + HF_pk[d] Fa_k[j - d],
//   HQ_pk = sum_c L (1 - phi - psi) {(1-t) at d = m, t at d = m-1},  HS_pk likewise with
//   kappa phi, HF_pk with kappa_f (1 + LB(mu)) psi (the reference's facula intensity
//   factor, SOAP_integration.cu:317-323),
// F_p = conv(I_p) with the resolution taps, CCF_p = raw mask CCF of F_p, and the
// Gaussian fit of CCF_p polished to the least-squares optimum gives RV_p, FWHM_p.
// The adjoint runs the same structures backwards: the implicit derivative of
// the fit (H^-1 J^T), the transposed mask and convolution, lag correlations of
// the adjoint spectrum with the seed rows (from which every per-cell derivative
// follows), and the transposed FIR for the seed gradients.  Shifted spectra are
// never stored: the backward recomputes from taps and correlations.
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>

#include "soap_internal.h"

namespace soap {

constexpr int kDT = 256;

// ------------------------------------------------------------ the disk
// Under rigid rotation every cell of a disk row has the same shift (m, t), and a row
// crosses each mu bin in one or two runs, so a phase's taps, scalar gradients and map
// gradients need the cells only through sums over runs ("pieces"): with a = 1 - mu and
// b = 1 + LB(mu), the limb L = 1 - u1 a - u2 a^2 is a combination of 1, a, a^2, and
//   sum_c L phi = M0 - u1 M1 - u2 M2,  M_q = sum_c a^q phi,
// likewise for psi and b psi.  The kernels below form those sums once per (piece,
// phase), lanes over phases and cells in turn (no reduction across lanes and no
// atomics: every sum has a fixed order), and everything after works on pieces: 7,300 of
// them instead of 283,000 cells at grid 600 with 10 bins.

// per-cell tables of the plan
__global__ void k_diff_cells(DiffArgs a, const double *mu_bounds, int32_t *ck, double2 *cell) {
#pragma clang fp contract(off)
  long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long ncell = (long)a.grid * a.grid;
  if (idx >= ncell) return;
  int iy = (int)(idx / a.grid), iz = (int)(idx % a.grid);
  double y = -1. + iy * (2. / a.grid), z = -1. + iz * (2. / a.grid);
  if (!(y * y + z * z <= 1.)) {
    ck[idx] = -1;
    cell[idx] = make_double2(0.0, 0.0);
    return;
  }
  double mu = sqrt(1. - (y * y + z * z));
  int k = a.n_mu - 1;
  for (int b = 0; b < a.n_mu - 1; b++)
    if (mu > mu_bounds[b]) {
      k = b;
      break;
    }
  ck[idx] = k;
  // facula intensity factor 1 + LB(mu) (SOAP_initialize.cu:367, SOAP_integration.cu:317-323)
  cell[idx] = make_double2(1. - mu, 1. + (a.lb[0] + a.lb[1] * mu + a.lb[2] * mu * mu + a.lb[3] * mu * mu * mu));
}

__global__ void k_diff_psum(DiffArgs a, double2 *psum) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= a.n_piece) return;
  const DiffPiece pc = a.piece[i];
  double s1 = 0.0, s2 = 0.0;
  for (int c = 0; c < pc.len; c++) {
    const double ca = a.cell[(long)pc.iy * a.grid + a.col[(long)pc.group * kDiffGroup + c]].x;
    s1 += ca;
    s2 = fma(ca, ca, s2);
  }
  psum[i] = make_double2(s1, s2);
}

// Shift of every disk row, and what follows from it: the rows of each tap index and the
// lags of each bin (over all rows between the bin's first and last, one wave per bin).
// One block (a grid has at most 8192 rows).
constexpr int kDiffRowT = 1024;
__global__ __launch_bounds__(kDiffRowT) void k_diff_rows(DiffArgs a) {
  extern __shared__ int s_rows[];  // [nd][2] first / last row, then [G] tap indices
  int *s_d = s_rows, *s_m = s_rows + 2 * a.nd;
  for (int e = threadIdx.x; e < a.nd; e += blockDim.x) {
    s_d[2 * e] = a.grid;
    s_d[2 * e + 1] = -1;
  }
  __syncthreads();
  const double vsini = a.prm ? a.prm[0] : a.vsini;
  for (int iy = threadIdx.x; iy < a.grid; iy += blockDim.x) {
#pragma clang fp contract(off)
    const double y = -1. + iy * (2. / a.grid);
    const double delta = vsini * y;
    const double beta = delta * 1000. / kC;
    const double g = sqrt((1 + beta) / (1 - beta));
    const double fbeta = -1 * (1 - g);
    const double sh = log1p(fbeta) / a.h;
    const double mc = ceil(sh);
    a.row_m[iy] = (int32_t)mc;
    // dt/d(delta) = -exp((m-s)h)/expm1(h) / (g^2 (1-beta)^2) * 1000/c (m piecewise constant)
    a.row_t[iy] = make_double2(expm1((mc - sh) * a.h) / a.expm1_h,
                               -exp((mc - sh) * a.h) / a.expm1_h / (g * g * (1 - beta) * (1 - beta)) * (1000. / kC) * y);
    const int d0 = (int32_t)mc - a.dmin;  // tap index of offset m; m-1 at d0-1
    const bool in = d0 >= 1 && d0 < a.nd;  // the host bounds every shift
    s_m[iy] = in ? d0 : -1;
    if (in) {
      atomicMin(s_d + 2 * d0, iy);
      atomicMax(s_d + 2 * d0 + 1, iy);
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 2 * a.nd; e += blockDim.x) a.drow[e] = s_d[e];
  const int lane = threadIdx.x & 63;
  for (int k = threadIdx.x >> 6; k < a.n_mu; k += kDiffRowT / 64) {
    int lo = a.nd, hi = -1;
    for (int iy = a.brow[2 * k] + lane; iy <= a.brow[2 * k + 1]; iy += 64) {
      const int d0 = s_m[iy];
      if (d0 < 0) continue;
      lo = min(lo, d0 - 1);
      hi = max(hi, d0);
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      lo = min(lo, __shfl_xor(lo, off));
      hi = max(hi, __shfl_xor(hi, off));
    }
    if (lane == 0) {
      a.blag[2 * k] = lo;
      a.blag[2 * k + 1] = hi;
    }
  }
}

// LDS written by some lanes of a wave and read by others: the LDS serves a wave's
// accesses in order, so only the compiler has to be held
__device__ __forceinline__ void wave_lds_order() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}

// Moments of one piece for up to 64 phases: one wave per (piece, 64 phases).  Group by
// group the wave samples its cells' filling factors bilinearly (two phases x 32 cells per step, loads
// of neighbouring cells from neighbouring nodes) into LDS and then sums them with lanes
// over phases, the cell's own factors read from the lane that holds them.  Blocks are in
// contiguous runs per XCD: neighbouring pieces read the same map rows.  Outputs: mom rows
// 0-2 sum a^q phi, 3-5 sum a^q psi, 6-8 sum a^q b psi, and the sets' tap weights
// sum L (1 - phi - psi), kappa sum L phi, kappa_f sum L b psi.
constexpr int kMomW = 4;       // waves (pieces) per block
constexpr int kMomU = 4;       // sampling steps in flight
constexpr int kMomStride = kDiffGroup + 1;
template <int NS>
__global__ __launch_bounds__(64 * kMomW) void k_diff_moments(DiffArgs a, int blocks_per_xcd) {
  extern __shared__ double s_mom[];  // per wave [phases][kMomStride]
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int blk = (blockIdx.x & 7) * blocks_per_xcd + (blockIdx.x >> 3);
  const int ip = __builtin_amdgcn_readfirstlane(blk * kMomW + w);
  const int p0 = blockIdx.y * 64, np = min(64, a.n_phase - p0), P = a.n_phase;
  if (ip >= a.n_piece) return;  // no barriers below
  double *sp = s_mom + (size_t)w * min(64, P) * kMomStride;
  const CONSTANT int32_t *pi = gc((const int32_t *)(a.piece + ip));
  const int iy = pi[0], group = pi[2], len = pi[3];
  const int M = a.map_res;
  const long MM = (long)M * M;
  const int c = lane & 31, ph = lane >> 5;
  const int i0 = gc(a.map_j)[iy];
  const double fy = gc(a.map_f)[iy];
  double m[9];
#pragma unroll
  for (int q = 0; q < 9; q++) m[q] = 0.0;
  for (int c0 = 0; c0 < len; c0 += kDiffGroup) {
    // this lane's cell and its stencil (the same for every phase)
    const int n_cell = min(kDiffGroup, len - c0), iz = a.col[(long)group * kDiffGroup + c0 + c];
    const double2 me = a.cell[(long)iy * a.grid + iz];
    const double fz = a.map_f[iz];
    const double w00 = (1 - fy) * (1 - fz), w10 = fy * (1 - fz), w01 = (1 - fy) * fz, w11 = fy * fz;
    const long off = (long)i0 * M + a.map_j[iz];
#pragma unroll
    for (int set = 0; set < NS - 1; set++) {
      const double *mp = (set ? a.fmaps : a.maps) + (long)p0 * MM + off;
      for (int s = 0; s < np; s += 2 * kMomU) {
        double x[kMomU][4];
#pragma unroll
        for (int u = 0; u < kMomU; u++) {
          const double *q = mp + (long)min(s + 2 * u + ph, np - 1) * MM;
          x[u][0] = q[0];
          x[u][1] = q[M];
          x[u][2] = q[1];
          x[u][3] = q[M + 1];
        }
#pragma unroll
        for (int u = 0; u < kMomU; u++) {
          const int p = s + 2 * u + ph;
          if (p < np) sp[p * kMomStride + c] = w00 * x[u][0] + w10 * x[u][1] + w01 * x[u][2] + w11 * x[u][3];
        }
      }
      wave_lds_order();
      const double *mine = sp + min(lane, np - 1) * kMomStride;
#pragma unroll 4
      for (int i = 0; i < n_cell; i++) {
        const double f = mine[i], ca = lane_f64(me.x, i);
        const double fa = f * ca;
        m[3 * set] += f;
        m[3 * set + 1] += fa;
        m[3 * set + 2] = fma(fa, ca, m[3 * set + 2]);
        if (set) {
          const double g = f * lane_f64(me.y, i), ga = g * ca;
          m[6] += g;
          m[7] += ga;
          m[8] = fma(ga, ca, m[8]);
        }
      }
      wave_lds_order();
    }
  }
  if (lane >= np) return;
  constexpr int NM = diff_moments(NS);
  double *o = a.mom + (long)ip * NM * P + p0 + lane;
#pragma unroll
  for (int q = 0; q < NM; q++) o[(long)q * P] = m[q];
  const double u1 = a.prm ? a.prm[1] : a.u1, u2 = a.prm ? a.prm[2] : a.u2;
  const double kappa = a.prm ? a.prm[3] : a.kappa, kappa_f = a.prm ? a.prm[4] : a.kappa_f;
  const double s1 = gc((const double *)(a.psum + ip))[0], s2 = gc((const double *)(a.psum + ip))[1];
  double *wt = a.wts + (long)ip * NS * P + p0 + lane;
  const double Lphi = m[0] - u1 * m[1] - u2 * m[2];
  wt[0] = ((double)len - m[0] - m[3]) - u1 * (s1 - m[1] - m[4]) - u2 * (s2 - m[2] - m[5]);
  wt[P] = kappa * Lphi;
  if (NS == 3) wt[2L * P] = kappa_f * (m[6] - u1 * m[7] - u2 * m[8]);
}

// taps (phase, bin k, offset d, set q) = sum over the pieces of bin k whose row has tap index d of w (1 - t),
// and of those with index d + 1 of w t.  Block = (d, k), lanes over phases, the piece
// range split over kTapW waves whose sums are added in wave order; the lanes first load
// the factors of 64 pieces, which are then read from them one by one, so the weight
// loads do not wait on a chain of look-ups.
constexpr int kTapW = 8;
template <int NS>
__global__ __launch_bounds__(64 * kTapW) void k_diff_taps(DiffArgs a) {
  __shared__ double s_t[kTapW][NS][64];
  const int d = blockIdx.x, k = blockIdx.y, P = a.n_phase;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int p = blockIdx.z * 64 + lane, pl = min(p, P - 1);
  const CONSTANT int32_t *ps = gc(a.pstart) + (long)k * (a.grid + 1);
  double acc[NS];
#pragma unroll
  for (int q = 0; q < NS; q++) acc[q] = 0.0;
  for (int side = 0; side < 2; side++) {
    const int dd = d + side;
    if (dd < 1 || dd >= a.nd) continue;
    const int r0 = gc(a.drow)[2 * dd], r1 = gc(a.drow)[2 * dd + 1];
    if (r0 > r1) continue;
    const int i0 = ps[r0], cnt = ps[r1 + 1] - i0;
    const int q0 = i0 + (int)((long)cnt * w / kTapW), q1 = i0 + (int)((long)cnt * (w + 1) / kTapW);
    for (int b = q0; b < q1; b += 64) {
      const int iy = a.piece[min(b + lane, q1 - 1)].iy;
      const double t = a.row_t[iy].x;
      const double f = a.row_m[iy] - a.dmin == dd ? (side ? t : 1.0 - t) : 0.0;
      const double *wt = a.wts + (long)b * NS * P + pl;
      const int m = min(64, q1 - b);
#pragma unroll 8
      for (int i = 0; i < m; i++) {
        const double fi = lane_f64(f, i);
#pragma unroll
        for (int q = 0; q < NS; q++) acc[q] = fma(wt[((long)i * NS + q) * P], fi, acc[q]);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < NS; q++) s_t[w][q][lane] = acc[q];
  __syncthreads();
  if (w == 0 && p < P) {
    const int gp = p / a.grp_p, ngr = (a.n_mu * NS + a.grp_r - 1) / a.grp_r;
    double *op = a.taps_p + ((((long)gp * a.n_mu + k) * a.nd + d) * NS) * 16 + p % a.grp_p;
#pragma unroll
    for (int q = 0; q < NS; q++) {
      double x = s_t[0][q][lane];
#pragma unroll
      for (int i = 1; i < kTapW; i++) x += s_t[i][q][lane];
      op[q * 16] = x;
      const int row = k * NS + q;
      a.taps_r[(((long)p * ngr + row / a.grp_r) * a.nd + d) * 16 + row % a.grp_r] = x;
    }
  }
}

// ------------------------------------------------------------ contractions
// The forward FIR, the seed gradients and the lag correlations are dense products in
// FP64.  Probes that do nothing else sustain 32-47 TFLOP/s with the matrix unit's 16x16x4
// form, which would also pad 50 phases to 64, and 62-66 with the vector unit, so they run
// as outer products on the vector unit: R accumulators per lane and pixel, the R coefficients of a step in one register (lane
// r of each row of 16 lanes holds coefficient r) and broadcast by the multiply-add itself
// (DPP row_newbcast), so that a step costs one coefficient read and one pixel read for R
// multiply-adds.  On the full adjoint (grid 600, 100,000 pixels, 50 phases), 4.0 GFLOP
// each: FIR 104 us (39 TFLOP/s), seed gradients 144 (28), correlations 147 (27), the rest
// of the time being staging and waves too few to hide it; 311, 311 and 324 us with one
// coefficient per LDS word and multiply-add.
#define SOAP_FMB(I) "v_fmac_f64_dpp %" #I ", %[t], %[x] row_newbcast:" #I " row_mask:0xf bank_mask:0xf\n\t"
#define SOAP_FMB4 SOAP_FMB(0) SOAP_FMB(1) SOAP_FMB(2) SOAP_FMB(3)
#define SOAP_FMB8 SOAP_FMB4 SOAP_FMB(4) SOAP_FMB(5) SOAP_FMB(6) SOAP_FMB(7)
#define SOAP_FMB10 SOAP_FMB8 SOAP_FMB(8) SOAP_FMB(9)
#define SOAP_FMB12 SOAP_FMB10 SOAP_FMB(10) SOAP_FMB(11)
#define SOAP_FMB16 SOAP_FMB12 SOAP_FMB(12) SOAP_FMB(13) SOAP_FMB(14) SOAP_FMB(15)
#define SOAP_O4(F) "+v"(F[0]), "+v"(F[1]), "+v"(F[2]), "+v"(F[3])
#define SOAP_O8(F) SOAP_O4(F), "+v"(F[4]), "+v"(F[5]), "+v"(F[6]), "+v"(F[7])
#define SOAP_O10(F) SOAP_O8(F), "+v"(F[8]), "+v"(F[9])
#define SOAP_O12(F) SOAP_O10(F), "+v"(F[10]), "+v"(F[11])
#define SOAP_O16(F) SOAP_O12(F), "+v"(F[12]), "+v"(F[13]), "+v"(F[14]), "+v"(F[15])
// F[r] += t(lane r of this lane's row) x, one rounding each.  Two wait states lie between
// a vector write of t and its broadcast read.
template <int R>
__device__ __forceinline__ void row_fma(double (&F)[R], double t, double x) {
  static_assert(R == 4 || R == 8 || R == 10 || R == 12 || R == 16, "group sizes");
  if constexpr (R == 4)
    asm("s_nop 1\n\t" SOAP_FMB4 : SOAP_O4(F) : [t] "v"(t), [x] "v"(x));
  else if constexpr (R == 8)
    asm("s_nop 1\n\t" SOAP_FMB8 : SOAP_O8(F) : [t] "v"(t), [x] "v"(x));
  else if constexpr (R == 10)
    asm("s_nop 1\n\t" SOAP_FMB10 : SOAP_O10(F) : [t] "v"(t), [x] "v"(x));
  else if constexpr (R == 12)
    asm("s_nop 1\n\t" SOAP_FMB12 : SOAP_O12(F) : [t] "v"(t), [x] "v"(x));
  else
    asm("s_nop 1\n\t" SOAP_FMB16 : SOAP_O16(F) : [t] "v"(t), [x] "v"(x));
}

// I_p[j] = sum_k sum_d HQ[d] Q_k[j - dmin - d] + HS[d] S_k[j - dmin - d] (+ HF[d] Fa_k[j - dmin - d]);
// block = (tile of kDT * XB pixels, group of R phases).  Per bin the NS rows and the
// taps of up to kFirD offsets are staged, the next bin's loads in flight during this
// bin's sums where a block is small (XB = 1: few blocks, nothing else hides them; with
// XB = 2 the registers cost more waves than they save, 104 -> 116 us); the reads of an
// offset are issued before the multiply-adds of the one before it (left to the compiler
// each read waits right before its use).
constexpr int kFirD = 32;
template <int NS, int R, int XB>
__global__ __launch_bounds__(kDT) void k_diff_fir(DiffArgs a) {
  extern __shared__ double s_fir[];  // [NS][row_len], then [kFirD][NS][16]
  constexpr int kRow = XB + 1, kTap = kFirD * NS * 16 / kDT;  // values per thread of a bin's staging
  constexpr bool kAhead = XB == 1;
  const int g = blockIdx.y, lane16 = threadIdx.x & 15, tid = threadIdx.x;
  const long j0 = (long)blockIdx.x * (kDT * XB), n = a.n;
  const int nd = a.nd, n_mu = a.n_mu, row_len = kDT * XB + nd - 1;
  const long src0 = j0 - a.dmin - nd + 1;
  double *s_t = s_fir + NS * row_len;
  double F[XB][R];
#pragma unroll
  for (int b = 0; b < XB; b++)
#pragma unroll
    for (int r = 0; r < R; r++) F[b][r] = 0.0;
  auto row_at = [&](int k, int q, int e) {  // element e of the staged row, 0 outside the spectrum
    const long i = src0 + e;
    const bool in = i >= 0 && i < n;
    const double *X = q == 0 ? a.q : q == 1 ? a.s : a.f;
    const double v = X[(long)k * n + (in ? i : 0)];
    return in ? v : 0.0;
  };
  auto taps_at = [&](int k, int d) { return a.taps_p + ((((long)g * n_mu + k) * nd + d) * NS) * 16; };
  double rv[NS][kRow], tv[kTap];
  auto fetch = [&](int k) {
    const int lo = a.blag[2 * k], hi = a.blag[2 * k + 1];
    if (lo > hi) return;  // uniform
#pragma unroll
    for (int q = 0; q < NS; q++)
#pragma unroll
      for (int u = 0; u < kRow; u++) rv[q][u] = row_at(k, q, min(tid + u * kDT, row_len - 1));
    const double *T = taps_at(k, lo);
    const int nt = min(kFirD, hi + 1 - lo) * NS * 16;
#pragma unroll
    for (int u = 0; u < kTap; u++) tv[u] = T[min(tid + u * kDT, nt - 1)];
  };
  if (kAhead) fetch(0);
  for (int k = 0; k < n_mu; k++) {
    const int lo = a.blag[2 * k], hi = a.blag[2 * k + 1];
    if (!kAhead) fetch(k);
    for (int dc = lo; dc <= hi; dc += kFirD) {
      const int nc = min(kFirD, hi + 1 - dc);
      __syncthreads();
      if (dc == lo) {
#pragma unroll
        for (int q = 0; q < NS; q++) {
#pragma unroll
          for (int u = 0; u < kRow; u++)
            if (tid + u * kDT < row_len) s_fir[q * row_len + tid + u * kDT] = rv[q][u];
          for (int e = tid + kRow * kDT; e < row_len; e += kDT) s_fir[q * row_len + e] = row_at(k, q, e);  // nd > kDT
        }
#pragma unroll
        for (int u = 0; u < kTap; u++)
          if (tid + u * kDT < nc * NS * 16) s_t[tid + u * kDT] = tv[u];
      } else {
        const double *T = taps_at(k, dc);
        for (int e = tid; e < nc * NS * 16; e += kDT) s_t[e] = T[e];
      }
      __syncthreads();
      if (kAhead && dc == lo && k + 1 < n_mu) fetch(k + 1);
      const double *x = s_fir + tid + nd - 1 - dc, *tp = s_t + lane16;
      double t[2][NS], xv[2][NS][XB];
      auto read = [&](int s, int d) {
#pragma unroll
        for (int q = 0; q < NS; q++) {
          t[s][q] = tp[(d * NS + q) * 16];
#pragma unroll
          for (int b = 0; b < XB; b++) xv[s][q][b] = x[q * row_len + b * kDT - d];
        }
      };
      auto sums = [&](int s) {
#pragma unroll
        for (int q = 0; q < NS; q++)
#pragma unroll
          for (int b = 0; b < XB; b++) row_fma<R>(F[b], t[s][q], xv[s][q][b]);
      };
      read(0, 0);
      for (int d = 0; d < nc; d += 2) {
        read(1, min(d + 1, nc - 1));
        __builtin_amdgcn_sched_barrier(0);
        sums(0);
        read(0, min(d + 2, nc - 1));
        __builtin_amdgcn_sched_barrier(0);
        if (d + 1 < nc) sums(1);
      }
    }
    if (kAhead && lo > hi && k + 1 < n_mu) fetch(k + 1);  // a bin without cells: nothing was staged
  }
#pragma unroll
  for (int b = 0; b < XB; b++) {
    const long j = j0 + tid + b * kDT;
    if (j >= n) continue;
#pragma unroll
    for (int r = 0; r < R; r++)
      if (g * R + r < a.n_phase) a.I[(long)(g * R + r) * n + j] = F[b][r];
  }
}

// F_p = conv(I_p) (zero outside wid < i < n-1-wid); residual partials of the
// trimmed range per block: part[p][block]
__global__ __launch_bounds__(kDT) void k_diff_conv(DiffArgs a, ConvArgs c, const double *target, int trim,
                                                   double *part) {
  extern __shared__ double xs[];  // I over [i0 + dlo, i0 + 4*kDT + ntp - 1), taps after
  int p = blockIdx.y;
  long i0 = (long)blockIdx.x * (4 * kDT);
  int span = 4 * kDT + c.ntp - 1;
  double *ct = xs + span;
  const double *X = a.I + (long)p * a.n;
  for (int e = threadIdx.x; e < c.ntp; e += blockDim.x) ct[e] = c.ctap[e];
  for (int e = threadIdx.x; e < span; e += blockDim.x) {
    long m = i0 + c.dlo + e;
    xs[e] = (m >= 0 && m < a.n) ? X[m] : 0.0;
  }
  __syncthreads();
  double acc[4] = {0, 0, 0, 0};
  for (int k = 0; k < c.ntp; k++) {
    double cv = ct[k];
#pragma unroll
    for (int b = 0; b < 4; b++) acc[b] = fma(cv, xs[threadIdx.x + b * kDT + k], acc[b]);
  }
  double r2 = 0.0;
#pragma unroll
  for (int b = 0; b < 4; b++) {
    long i = i0 + threadIdx.x + b * kDT;
    if (i >= a.n) continue;
    double o = ((i > c.wid) && (i + c.wid < a.n - 1)) ? acc[b] : 0.0;
    a.F[(long)p * a.n + i] = o;
    if (i >= trim && i < a.n - trim) {
      double r = o - target[(long)p * a.n + i];
      r2 += r * r;
    }
  }
  __shared__ double s_r[kDT / 64];
  for (int off = 32; off > 0; off >>= 1) r2 += __shfl_xor(r2, off);
  if ((threadIdx.x & 63) == 0) s_r[threadIdx.x >> 6] = r2;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0;
    for (int w = 0; w < kDT / 64; w++) s += s_r[w];
    part[(long)p * gridDim.x + blockIdx.x] = s;
  }
}

// ------------------------------------------------------------ Gaussian fit: polish and adjoint
// gradient (4) and Hessian (10, upper) of 0.5 sum r^2 (BIS_FIT2 model, exact second
// derivatives), summed over the wave's lanes; every lane receives the totals.  Three
// points of a lane are in flight together; points past n add zeros.
__device__ __forceinline__ void gauss_gh(const double *x, const double *y, int n, const double (&th)[4], double (&g)[4],
                                         double (&H)[4][4], double *r2out) {
  const double rs = 2 * sqrt(2 * log(2.0)) / th[3], rf = 1.0 / th[3];
  double v[16];
#pragma unroll
  for (int q = 0; q < 16; q++) v[q] = 0.0;
  const int lane = threadIdx.x & 63;
  for (int i0 = lane; i0 - lane < n; i0 += 192) {
#pragma unroll
    for (int w = 0; w < 3; w++) {
      const bool in = i0 + 64 * w < n;
      const int i = in ? i0 + 64 * w : n - 1;
      const double u = (x[i] - th[2]) * rs, ex = exp(-0.5 * u * u);
      const double e = in ? ex : 0.0, r = in ? th[0] + th[1] * e - y[i] : 0.0;
      const double eu = e * u, ku = th[1] * eu;
      const double j4[4] = {in ? 1.0 : 0.0, e, ku * rs, ku * u * rf};
      const double hh[4][4] = {{0, 0, 0, 0},
                               {0, 0, eu * rs, eu * u * rf},
                               {0, 0, th[1] * e * (u * u - 1) * rs * rs, ku * (u * u - 2) * rs * rf},
                               {0, 0, 0, ku * u * (u * u - 3) * rf * rf}};
      int q = 4;
#pragma unroll
      for (int a = 0; a < 4; a++) {
        v[a] = fma(j4[a], r, v[a]);
#pragma unroll
        for (int b = a; b < 4; b++, q++) v[q] += j4[a] * j4[b] + r * hh[a][b];
      }
      v[14] = fma(r, r, v[14]);
    }
  }
  wave_sums16(v);
  int q = 4;
#pragma unroll
  for (int a = 0; a < 4; a++) {
    g[a] = v[a];
#pragma unroll
    for (int b = a; b < 4; b++) H[a][b] = H[b][a] = v[q++];
  }
  *r2out = v[14];
}

// Gaussian elimination with row pivoting.  Each column's largest entry is brought up by
// exchanges with constant indices (selects), so that the system stays in registers.
__device__ __forceinline__ int solve4(const double (&A_in)[4][4], const double (&b)[4], double (&x)[4]) {
  double A[4][5];
#pragma unroll
  for (int i = 0; i < 4; i++) {
#pragma unroll
    for (int j = 0; j < 4; j++) A[i][j] = A_in[i][j];
    A[i][4] = b[i];
  }
  double inv[4];
#pragma unroll
  for (int col = 0; col < 4; col++) {
#pragma unroll
    for (int r = col + 1; r < 4; r++) {
      const bool up = fabs(A[r][col]) > fabs(A[col][col]);
#pragma unroll
      for (int j = col; j < 5; j++) {
        const double t = A[col][j];
        A[col][j] = up ? A[r][j] : t;
        A[r][j] = up ? t : A[r][j];
      }
    }
    if (A[col][col] == 0.0) return -1;
    inv[col] = 1.0 / A[col][col];
#pragma unroll
    for (int r = col + 1; r < 4; r++) {
      const double f = A[r][col] * inv[col];
#pragma unroll
      for (int j = col + 1; j < 5; j++) A[r][j] -= f * A[col][j];
    }
  }
#pragma unroll
  for (int i = 3; i >= 0; i--) {
    double s = A[i][4];
#pragma unroll
    for (int j = i + 1; j < 4; j++) s -= A[i][j] * x[j];
    x[i] = s * inv[i];
  }
  return 0;
}

// one wave per CCF: theta from the fit parameters (signed amplitude), then
// damped Newton steps on the exact Hessian to the least-squares optimum.
// A full Newton step below kPolishStep of the amplitude and the width is the end of the search: it
// changes the residual by less than its rounding ((1e-7)^2 of it), so comparing
// residuals there decides nothing and used to try up to thirty damped steps (461 us for
// the 50 CCFs of the full adjoint, a chain of about 150 evaluations).  The two undamped
// steps that follow take 1e-7 to rounding.
constexpr double kPolishStep = 1e-7;
__global__ __launch_bounds__(64) void k_fit_polish(const double *v, int n_v, const double *ccf, const double *par,
                                                   double *theta) {
  extern __shared__ double s_fit[];  // velocities, CCF
  const int sp = blockIdx.x, lane = threadIdx.x;
  double *s_v = s_fit, *s_y = s_fit + n_v;
  const double *pp = par + (long)sp * 5;
  const double c0 = pp[0], k0 = pp[1], x0 = pp[3], f0 = pp[4];
  double best = -HUGE_VAL;
  int inear = n_v;
  for (int i = lane; i < n_v; i += 64) {
    const double x = v[i], d = -fabs(x - x0);
    s_v[i] = x;
    s_y[i] = ccf[(long)sp * n_v + i];
    if (d > best) {
      best = d;
      inear = i;
    }
  }
  wave_argmax(best, inear);
  if (inear >= n_v) inear = 0;  // NaN centre
  __syncthreads();
  double th[4] = {c0, s_y[inear] < c0 ? -k0 : k0, x0, f0};
  double g[4], H[4][4], r2;
  gauss_gh(s_v, s_y, n_v, th, g, H, &r2);
  for (int it = 0; it < 60; it++) {
    double mu = 0.0, dx[4] = {0, 0, 0, 0}, tn[4], gn[4], Hn[4][4], r2n = r2;
    bool ok = false, small = false;
    for (int tries = 0; tries < 30; tries++) {
      double Hd[4][4], mg[4];
#pragma unroll
      for (int a = 0; a < 4; a++) {
        mg[a] = -g[a];
#pragma unroll
        for (int b = 0; b < 4; b++) Hd[a][b] = H[a][b] + (a == b ? mu * (fabs(H[a][a]) + 1e-300) : 0.0);
      }
      if (solve4(Hd, mg, dx) == 0) {
#pragma unroll
        for (int a = 0; a < 4; a++) tn[a] = th[a] + dx[a];
        const double sk = kPolishStep * fabs(th[1]), sf = kPolishStep * fabs(th[3]);
        const bool tiny = mu == 0.0 && fabs(dx[0]) <= sk && fabs(dx[1]) <= sk && fabs(dx[2]) <= sf && fabs(dx[3]) <= sf;
        if (tiny) {
          ok = small = true;
          break;
        }
        gauss_gh(s_v, s_y, n_v, tn, gn, Hn, &r2n);
        if (r2n <= r2 * (1 + 1e-15)) {
          ok = true;
          break;
        }
      }
      mu = mu == 0.0 ? 1e-6 : mu * 10;
    }
    if (!ok) break;
    if (!small) {
      small = true;
#pragma unroll
      for (int a = 0; a < 4; a++)
        if (fabs(dx[a]) > 1e-12 * fabs(th[a]) + 1e-300) small = false;
      r2 = r2n;
#pragma unroll
      for (int a = 0; a < 4; a++) {
        g[a] = gn[a];
#pragma unroll
        for (int b = 0; b < 4; b++) H[a][b] = Hn[a][b];
      }
    }
#pragma unroll
    for (int a = 0; a < 4; a++) th[a] = tn[a];
    if (small) break;
  }
  // two undamped Newton steps on the gradient fix the optimum to rounding
  for (int it = 0; it < 2; it++) {
    double mg[4], dx[4];
    gauss_gh(s_v, s_y, n_v, th, g, H, &r2);
#pragma unroll
    for (int a = 0; a < 4; a++) mg[a] = -g[a];
    if (solve4(H, mg, dx) != 0) break;
#pragma unroll
    for (int a = 0; a < 4; a++) th[a] += dx[a];
  }
  if (lane == 0)
#pragma unroll
    for (int a = 0; a < 4; a++) theta[(long)sp * 4 + a] = th[a];
}

// dl/dy_v = J_v . z with H z = dl/dtheta (implicit derivative of the optimum), plus
// the bisector span's direct term coef_p dspan_p/dy_v when bisd holds one
__global__ void k_fit_adjoint(const double *v, int n_v, const double *ccf, const double *theta, const double *dth,
                              const double *bisd, double *gy) {
  int sp = blockIdx.x;
  const double *y = ccf + (long)sp * n_v;
  double th[4], g[4], H[4][4], r2, z[4] = {0, 0, 0, 0};
  for (int a = 0; a < 4; a++) th[a] = theta[(long)sp * 4 + a];
  gauss_gh(v, y, n_v, th, g, H, &r2);
  double b[4];
  for (int a = 0; a < 4; a++) b[a] = dth[(long)sp * 4 + a];
  solve4(H, b, z);
  double s = th[3] / (2 * sqrt(2 * log(2.0)));
  const double *bp = bisd ? bisd + (long)sp * (n_v + kBisHead) : nullptr;
  const double coef = bp ? bp[1] : 0.0;
  for (int i = threadIdx.x; i < n_v; i += blockDim.x) {
    double u = (v[i] - th[2]) / s, e = exp(-u * u / 2);
    double g = z[0] + z[1] * e + z[2] * th[1] * e * u / s + z[3] * th[1] * e * u * u / th[3];
    if (coef != 0.0) g += coef * bp[kBisHead + i];
    gy[(long)sp * n_v + i] = g;
  }
}

// ------------------------------------------------------------ bisector span
// p2 of the interval centred at vr (BIS_FIT2.cpp:233-236: half the inverse
// curvature of the Gaussian at vr) and its derivatives in the centre v0 and in
// s2 = sigma^2.  With u = vr - v0, E = exp(-u^2 / 2 s2): dccf = -u E / s2,
// d2ccf = (u^2 / s2 - 1) E / s2, p2 = -d2ccf / (2 dccf^3); d dccf / du = d2ccf,
// d d2ccf / du = E u (3 - u^2 / s2) / s2^2, d dccf / ds2 = u E (1 - u^2 / 2 s2) / s2^2,
// d d2ccf / ds2 = E [(s2 - 2 u^2) / s2^3 + (u^2 - s2) u^2 / (2 s2^4)].
__device__ void bis_p2(double vr, double v0, double s2, double *p2, double *dp2_dv0, double *dp2_ds2) {
  double dd = (vr - v0) * (vr - v0);
  double dccf = -(vr - v0) / s2 * exp(-dd / 2. / s2);
  double d2ccf = (dd / s2 - 1) / s2 * exp(-dd / 2. / s2);
  double d2rv = -d2ccf / (dccf * dccf * dccf);
  *p2 = d2rv / 2.;
  double u = vr - v0, E = exp(-dd / 2. / s2);
  double d2ccf_u = E * u * (3 - dd / s2) / (s2 * s2);
  double dccf_s = u * E / (s2 * s2) * (1 - dd / (2 * s2));
  double d2ccf_s = E * ((s2 - 2 * dd) / (s2 * s2 * s2) + (dd - s2) * dd / (2 * s2 * s2 * s2 * s2));
  double i3 = 1.0 / (dccf * dccf * dccf);
  double dp2_u = -d2ccf_u * i3 / 2 + 1.5 * d2ccf * d2ccf * i3 / dccf;
  *dp2_dv0 = -dp2_u;
  *dp2_ds2 = -d2ccf_s * i3 / 2 + 1.5 * d2ccf * dccf_s * i3 / dccf;
}

// One 64-lane block per CCF: the span of BIS_FIT2.cpp:214-268 at the polished
// Gaussian theta = (c, k, v0, fwhm) (the forward of the plain fit's bisector,
// with the same per-interval quadratic inverse and walk), and its partial
// derivatives at fixed theta: dspan/dy_v and dspan/dtheta.  Per interval s with
// a = norm_s, b = norm_{s+1}, the quadratic inverse at depth d is
// v_s + dv (d - a) / (b - a) + p2 (d - a) (d - b), so
//   dterm/da = (d - b) (dv / (b - a)^2 - p2), dterm/db = -(d - a) (dv / (b - a)^2 + p2),
//   dterm/dp2 = (d - a) (d - b);  norm_j = (y_j - c) / k.
// Output per CCF (stride n_v + kBisHead): [0] span, [1] loss coefficient (written
// by k_diff_loss), [2..5] dspan/dtheta, [kBisHead + v] dspan/dy_v.
constexpr int kBisLevels = 91;
__global__ __launch_bounds__(64) void k_diff_bis(const double *v, int n_v, const double *ccf, const double *theta,
                                                 double *bisd) {
  extern __shared__ double s_bis[];  // norm, p0, p1, p2
  double *s_nc = s_bis, *s_p0 = s_bis + n_v, *s_p1 = s_bis + 2 * n_v, *s_p2 = s_bis + 3 * n_v;
  __shared__ double s_dA[kBisLevels][2], s_dB[kBisLevels][2];
  __shared__ int s_side[kBisLevels][2];
  const int sp = blockIdx.x;
  const double *y = ccf + (long)sp * n_v;
  double *out = bisd + (long)sp * (n_v + kBisHead);
  const double c = theta[sp * 4 + 0], k = theta[sp * 4 + 1], v0 = theta[sp * 4 + 2], fwhm = theta[sp * 4 + 3];
  const double sigma = fwhm / 2. / sqrt(2. * log(2.));
  const double s2 = sigma * sigma;
  for (int i = threadIdx.x; i < n_v; i += 64) s_nc[i] = -c / k * (1. - y[i] / c);
  __syncthreads();
  for (int i = threadIdx.x; i < n_v - 1; i += 64) {
    double p2, d0, d1;
    bis_p2((v[i] + v[i + 1]) / 2., v0, s2, &p2, &d0, &d1);
    double p1 = (v[i + 1] - v[i] - p2 * (s_nc[i + 1] * s_nc[i + 1] - s_nc[i] * s_nc[i])) / (s_nc[i + 1] - s_nc[i]);
    s_p2[i] = p2;
    s_p1[i] = p1;
    s_p0[i] = v[i] - p1 * s_nc[i] - p2 * (s_nc[i] * s_nc[i]);
  }
  if (threadIdx.x == 0) s_p0[n_v - 1] = s_p1[n_v - 1] = s_p2[n_v - 1] = 0.0;
  int ind_max = 0;
  {
    double best = s_nc[0];
    if (best == best) {  // a NaN first value keeps index 0, as the scan's comparisons do
      for (int i = threadIdx.x; i < n_v; i += 64)
        if (s_nc[i] > best) {
          best = s_nc[i];
          ind_max = i;
        }
      wave_argmax(best, ind_max);
    }
  }
  __syncthreads();
  double top = 0., bot = 0., th4[4] = {0, 0, 0, 0};
  for (int i = threadIdx.x; i < kBisLevels; i += 64) {
    double dep = (double)(i + 5) / 100;
    int i_b, i_r;
    bisector_walk(s_nc, n_v, ind_max, dep, i_b, i_r);
    double b = (s_p0[i_b] + s_p0[i_r]) + (s_p1[i_b] + s_p1[i_r]) * dep + (s_p2[i_b] + s_p2[i_r]) * (dep * dep);
    b /= 2.;
    if (dep >= 0.1 && dep <= 0.4) top += b;
    if (dep >= 0.6 && dep <= 0.9) bot += b;
    // weight of this level in the span, halved for the mean of the two sides
    double w = ((dep >= 0.1) && (dep <= 0.4)) ? 0.5 / 31 : ((dep >= 0.6) && (dep <= 0.9)) ? -0.5 / 31 : 0.0;
    for (int side = 0; side < 2; side++) {
      int sx = side ? i_r : i_b;
      s_side[i][side] = sx;
      if (w == 0.0 || sx + 1 >= n_v) {
        s_dA[i][side] = 0.0;
        s_dB[i][side] = 0.0;
        continue;
      }
      double a = s_nc[sx], bb = s_nc[sx + 1], dv = v[sx + 1] - v[sx];
      double p2, dp2_v0, dp2_s2;
      bis_p2((v[sx] + v[sx + 1]) / 2., v0, s2, &p2, &dp2_v0, &dp2_s2);
      double q = dv / ((bb - a) * (bb - a));
      double dA = w * (dep - bb) * (q - p2), dB = -w * (dep - a) * (q + p2), dP = w * (dep - a) * (dep - bb);
      s_dA[i][side] = dA / k;
      s_dB[i][side] = dB / k;
      th4[0] += -(dA + dB) / k;
      th4[1] += -(dA * a + dB * bb) / k;
      th4[2] += dP * dp2_v0;
      th4[3] += dP * dp2_s2 * 2 * s2 / fwhm;
    }
  }
  __syncthreads();
  // dspan/dy_j: the levels' sides in order, kBisU reads ahead of their adds
  constexpr int kBisU = 7;
  static_assert(kBisLevels % kBisU == 0, "levels per pass");
  for (int j = threadIdx.x; j < n_v; j += 64) {
    double g = 0.0;
    for (int i = 0; i < kBisLevels; i += kBisU) {
      int sx[kBisU][2];
      double dA[kBisU][2], dB[kBisU][2];
#pragma unroll
      for (int u = 0; u < kBisU; u++)
#pragma unroll
        for (int side = 0; side < 2; side++) {
          sx[u][side] = s_side[i + u][side];
          dA[u][side] = s_dA[i + u][side];
          dB[u][side] = s_dB[i + u][side];
        }
#pragma unroll
      for (int u = 0; u < kBisU; u++)
#pragma unroll
        for (int side = 0; side < 2; side++) {
          g += sx[u][side] == j ? dA[u][side] : 0.0;
          g += sx[u][side] + 1 == j ? dB[u][side] : 0.0;
        }
    }
    out[kBisHead + j] = g;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    top += __shfl_xor(top, off);
    bot += __shfl_xor(bot, off);
#pragma unroll
    for (int q4 = 0; q4 < 4; q4++) th4[q4] += __shfl_xor(th4[q4], off);
  }
  if (threadIdx.x == 0) {
    out[0] = top / 31 - bot / 31;  // 31 levels in each range
    out[1] = 0.0;
#pragma unroll
    for (int q4 = 0; q4 < 4; q4++) out[2 + q4] = th4[q4];
  }
}

hipError_t launch_diff_bis(const double *v, int n_v, const double *ccf, const double *theta, int n_ccf, double *bisd,
                           hipStream_t s) {
  if (n_ccf == 0) return hipSuccess;
  if (n_v < 3 || n_v > kMaxVDiff) return hipErrorInvalidValue;
  k_diff_bis<<<n_ccf, 64, (size_t)4 * n_v * sizeof(double), s>>>(v, n_v, ccf, theta, bisd);
  return hipGetLastError();
}

// ------------------------------------------------------------ backward spectra
// G_F = 2 w_spec (F - T) on [trim, n - trim), 0 elsewhere
__global__ void k_diff_gradF(DiffArgs a, const double *target, int trim, double w_spec, double *GF) {
  long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long)a.n_phase * a.n) return;
  long i = e % a.n;
  GF[e] = (i >= trim && i < a.n - trim) ? 2 * w_spec * (a.F[e] - target[e]) : 0.0;
}

// transposed mask as a gather: G_F[p][trim + t] += sum_e gy[p][col_e] val_e over the
// entries e of row t of the pixel-major table (the (velocity, weight) pairs of
// every live mask pixel of the CCF, merged per pixel).  The table is sliced by 64
// rows (one wave): entry k of row t sits at slice_ptr[t / 64] + 64 k + t % 64,
// rows padded with zero weights to their slice's width, so every load is
// coalesced.  Block = (kDT pixels, chunk of kMtP phases), the chunk's gy rows in
// LDS, one owner per output: no atomics.
constexpr int kMtP = 8;
__global__ __launch_bounds__(kDT) void k_mask_transpose(int64_t n_t, int trim, int64_t n, int n_phase, int n_v,
                                                        const int64_t *slice_ptr, const int32_t *slice_w,
                                                        const int32_t *col, const double *val, const double *gy,
                                                        double *GF) {
  extern __shared__ double sg[];  // [kMtP][n_v]
  const int p0 = blockIdx.y * kMtP;
  const int np = min(kMtP, n_phase - p0);
  for (int e = threadIdx.x; e < kMtP * n_v; e += blockDim.x) {
    int c = e / n_v;
    sg[e] = c < np ? gy[(long)(p0 + c) * n_v + e % n_v] : 0.0;
  }
  __syncthreads();
  const long t = (long)blockIdx.x * kDT + threadIdx.x;
  const long sl = t >> 6;
  if (sl * 64 >= n_t) return;  // whole wave past the end (n_t rounds up to slices)
  const int W = slice_w[sl];
  const int64_t base = slice_ptr[sl] + (t & 63);
  double acc[kMtP];
#pragma unroll
  for (int c = 0; c < kMtP; c++) acc[c] = 0.0;
  for (int k = 0; k < W; k++) {
    const int v = col[base + 64L * k];
    const double w = val[base + 64L * k];
#pragma unroll
    for (int c = 0; c < kMtP; c++) acc[c] = fma(sg[c * n_v + v], w, acc[c]);
  }
  if (t >= n_t) return;
#pragma unroll
  for (int c = 0; c < kMtP; c++)
    if (c < np) GF[(long)(p0 + c) * n + trim + t] += acc[c];
}

// G_I[m] = sum_k c_k G_F[m - dlo - k] over the valid outputs (G_F is zero elsewhere)
__global__ __launch_bounds__(kDT) void k_diff_convT(DiffArgs a, ConvArgs c, const double *GF, double *GI) {
  extern __shared__ double xs[];  // G_F over [m0 - dlo - ntp + 1, m0 + 4 kDT - dlo)
  int p = blockIdx.y;
  long m0 = (long)blockIdx.x * (4 * kDT);
  int span = 4 * kDT + c.ntp - 1;
  double *ct = xs + span;
  const double *X = GF + (long)p * a.n;
  long base = m0 - c.dlo - c.ntp + 1;
  for (int e = threadIdx.x; e < c.ntp; e += blockDim.x) ct[e] = c.ctap[e];
  for (int e = threadIdx.x; e < span; e += blockDim.x) {
    long i = base + e;
    xs[e] = (i >= 0 && i < a.n && i > c.wid && i + c.wid < a.n - 1) ? X[i] : 0.0;
  }
  __syncthreads();
  double acc[4] = {0, 0, 0, 0};
  for (int k = 0; k < c.ntp; k++) {
    double cv = ct[k];
    // output m = m0 + tid + b kDT reads G_F[m - dlo - k] at xs[tid + b kDT + ntp - 1 - k]
#pragma unroll
    for (int b = 0; b < 4; b++) acc[b] = fma(cv, xs[threadIdx.x + b * kDT + c.ntp - 1 - k], acc[b]);
  }
#pragma unroll
  for (int b = 0; b < 4; b++) {
    long m = m0 + threadIdx.x + b * kDT;
    if (m < a.n) GI[(long)p * a.n + m] = acc[b];
  }
}

// lag correlations C[k][d][set][p] = sum_j G_I[p][j] X_k[j - dmin - d], in two passes.
// Pass 1: block = (chunk of kCorrT pixels or of kCorrG times that, group of kCorrRB (bin, set) rows, lag tile of
// 16 and group of PB phases); the rows' segments are staged once and each of four waves
// takes a quarter of the pixels.  Lane l of a row of 16 lanes is lag l, the four rows of
// lanes take 16 pixels each of every 64: a step loads G_I of 64 pixels per phase, and
// multiply-add n takes G_I of the row's pixel n from lane n (DPP row_newbcast) and the
// rows' pixel at the lane's lag from LDS, which then serves PB phases.  The lane rows'
// sums are added by swaps between them and the waves' through LDS.  PB kCorrRB = 50
// accumulators keep three waves per SIMD.  Lags are those the group's bins use.  Pass 2
// sums the chunk partials (no atomics).  The order of a sum is the same for every launch:
// kCorrT pixels, kCorrG of those in turn, the groups in turn.  A block takes a whole group
// where that leaves blocks for all CUs (corr_whole): a fourth of the partials to hold.
constexpr int kCorrRB = 5;
constexpr int kCorrT = 1024;
constexpr int kCorrG = 4;
constexpr int kCorrWin = kCorrT + 16;  // staged pixels of a row
// F[p] += g[p](lane N of this lane's row) x
template <int N, int PB>
__device__ __forceinline__ void lag_fma(double (&F)[PB], const double (&g)[PB], double x) {
  static_assert(PB == 8 || PB == 10, "phases per wave");
#define SOAP_LAG(I, J) "v_fmac_f64_dpp %" #I ", %" #J ", %[x] row_newbcast:%c[n] row_mask:0xf bank_mask:0xf\n\t"
  if constexpr (PB == 8)
    asm("s_nop 1\n\t" SOAP_LAG(0, 8) SOAP_LAG(1, 9) SOAP_LAG(2, 10) SOAP_LAG(3, 11) SOAP_LAG(4, 12) SOAP_LAG(5, 13)
            SOAP_LAG(6, 14) SOAP_LAG(7, 15)
        : SOAP_O8(F)
        : "v"(g[0]), "v"(g[1]), "v"(g[2]), "v"(g[3]), "v"(g[4]), "v"(g[5]), "v"(g[6]), "v"(g[7]), [x] "v"(x),
          [n] "i"(N));
  else
    asm("s_nop 1\n\t" SOAP_LAG(0, 10) SOAP_LAG(1, 11) SOAP_LAG(2, 12) SOAP_LAG(3, 13) SOAP_LAG(4, 14) SOAP_LAG(5, 15)
            SOAP_LAG(6, 16) SOAP_LAG(7, 17) SOAP_LAG(8, 18) SOAP_LAG(9, 19)
        : SOAP_O10(F)
        : "v"(g[0]), "v"(g[1]), "v"(g[2]), "v"(g[3]), "v"(g[4]), "v"(g[5]), "v"(g[6]), "v"(g[7]), "v"(g[8]),
          "v"(g[9]), [x] "v"(x), [n] "i"(N));
#undef SOAP_LAG
}
// the 16 pixels of each lane row from pixel N on; xc: the rows' values at pixel N.  The
// next pixel's are read before this one's multiply-adds (left to the compiler each read
// waits right before its use), after the last those of the next step's first pixel.
template <int N, int PB, int RB>
__device__ __forceinline__ void lag_steps(double (&F)[RB][PB], const double (&g)[PB], double (&xc)[RB],
                                          const double *x) {
  if constexpr (N < 16) {
    double xn[RB];
#pragma unroll
    for (int r = 0; r < RB; r++) xn[r] = x[r * kCorrWin + (N < 15 ? N + 1 : 64)];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < RB; r++) lag_fma<N>(F[r], g, xc[r]);
    lag_steps<N + 1>(F, g, xn, x);
#pragma unroll
    for (int r = 0; r < RB; r++) xc[r] = xn[r];
  }
}

// first lag of a row group: the least its bins use
__device__ __forceinline__ int corr_lag0(const DiffArgs &a, int k0, int k1, int &hi) {
  int lo = a.nd;
  hi = -1;
  for (int k = k0; k <= k1; k++) {
    lo = min(lo, a.blag[2 * k]);
    hi = max(hi, a.blag[2 * k + 1]);
  }
  return lo;
}

// a + b with the halves (HALF 32) or the neighbouring rows of 16 lanes (HALF 16) of the
// wave folded: the lower half or even row of the result holds a's, the other b's
template <int HALF>
__device__ __forceinline__ double swap_fold(double a, double b) {
  const long long va = __double_as_longlong(a), vb = __double_as_longlong(b);
  const unsigned al = (unsigned)va, ah = (unsigned)(va >> 32), bl = (unsigned)vb, bh = (unsigned)(vb >> 32);
  unsigned l0, l1, h0, h1;
  if constexpr (HALF == 32) {
    const auto l = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
    l0 = l[0], l1 = l[1], h0 = h[0], h1 = h[1];
  } else {
    const auto l = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
    l0 = l[0], l1 = l[1], h0 = h[0], h1 = h[1];
  }
  return __longlong_as_double(((long long)h0 << 32) | l0) + __longlong_as_double(((long long)h1 << 32) | l1);
}

constexpr int corr_sums(int pb) { return (kCorrRB * pb + 3) / 4 * 4 * 16; }  // of a wave
constexpr int corr_lds(int pb) {  // doubles: the staged rows with room for the last step's read ahead, or the waves' sums
  return kCorrRB * kCorrWin + 64 > 4 * corr_sums(pb) ? kCorrRB * kCorrWin + 64 : 4 * corr_sums(pb);
}
// Cpart [chunk][row][lag tile][P][16]; per: stretches of kCorrT pixels to a chunk
template <int PB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_diff_corr(DiffArgs a, const double *GI,
                                                                                        double *Cpart, int n_z, int per) {
  extern __shared__ double s_x[];  // [kCorrRB][kCorrWin], then the waves' sums; behind them the chunk's sums
  constexpr int RB = kCorrRB, NF = corr_sums(PB) / 64;  // sums per wave, four in a register
  double *s_run = s_x + corr_lds(PB);
  const int rows = a.n_mu * a.ns, r0 = blockIdx.y * RB, ns = a.ns;
  const int chunk = blockIdx.x, z = blockIdx.z % n_z, p0 = blockIdx.z / n_z * PB;
  int hi;
  const int lag0 = corr_lag0(a, r0 / ns, min(rows - 1, r0 + RB - 1) / ns, hi) + 16 * z;
  if (lag0 > hi) return;  // uniform over the block
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, l = lane & 15;
  const long n = a.n;
#pragma unroll 1
  for (int c = 0; c < per; c++) {
    const long j0 = ((long)chunk * per + c) * kCorrT;
    if (j0 >= n) break;  // uniform
    // lag d = lag0 + l reads X[j - dmin - d]: window index (j - j0) + 15 - l
    const long src0 = j0 - a.dmin - lag0 - 15;
    if (c) __syncthreads();  // the last stretch's sums have been read
#pragma unroll
    for (int r = 0; r < RB; r++) {
      const int row = min(r0 + r, rows - 1), set = row % ns;
      const double *X = (set == 0 ? a.q : set == 1 ? a.s : a.f) + (long)(row / ns) * n;
      for (int e = threadIdx.x; e < kCorrWin; e += 256) {
        const long i = src0 + e;
        const bool in = i >= 0 && i < n;
        const double v = X[in ? i : 0];
        s_x[r * kCorrWin + e] = in ? v : 0.0;
      }
    }
    __syncthreads();
    double F[RB][PB], g[PB], gn[PB], xc[RB];
#pragma unroll
    for (int r = 0; r < RB; r++)
#pragma unroll
      for (int p = 0; p < PB; p++) F[r][p] = 0.0;
    const int j1 = (int)min((long)kCorrT, n - j0);  // pixels of the stretch
    auto load = [&](double (&v)[PB], int s) {
      const bool in = s + lane < j1;
      const double *G = GI + j0 + (in ? s + lane : j1 - 1);
#pragma unroll
      for (int p = 0; p < PB; p++) {
        const double xv = G[(long)min(p0 + p, a.n_phase - 1) * n];
        v[p] = in ? xv : 0.0;
      }
    };
    const int s0 = w * (kCorrT / 4), s1 = min(j1, s0 + kCorrT / 4);
    const double *x = s_x + (lane & 48) + 15 - l;
#pragma unroll
    for (int r = 0; r < RB; r++) xc[r] = x[r * kCorrWin + s0];
    if (s0 < s1) load(g, s0);
    for (int s = s0; s < s1; s += 64) {
      load(gn, s + 64);
      lag_steps<0>(F, g, xc, x + s);
#pragma unroll
      for (int p = 0; p < PB; p++) g[p] = gn[p];
    }
    __syncthreads();  // the staged rows become the waves' sums
    const int which = (0x3120 >> (4 * (lane >> 4))) & 15;  // rows 0..3 of a folded register hold sums 0, 2, 1, 3
#pragma unroll
    for (int f = 0; f < NF; f++) {
      double v[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int i = 4 * f + u;
        v[u] = i < RB * PB ? F[i / PB][i % PB] : 0.0;
      }
      s_x[((long)w * NF * 4 + 4 * f + which) * 16 + l] =
          swap_fold<16>(swap_fold<32>(v[0], v[1]), swap_fold<32>(v[2], v[3]));
    }
    __syncthreads();
    for (int e = threadIdx.x; e < RB * PB * 16; e += 256) {  // a thread's own sums: no wait in between
      double t = s_x[e];
#pragma unroll
      for (int i = 1; i < 4; i++) t += s_x[i * NF * 64 + e];
      s_run[e] = c ? s_run[e] + t : t;
    }
  }
  for (int e = threadIdx.x; e < RB * PB * 16; e += 256) {
    const int r = e / (PB * 16), p = e / 16 % PB;
    if (r0 + r < rows && p0 + p < a.n_phase)
      Cpart[((((long)chunk * rows + r0 + r) * n_z + z) * a.n_phase + p0 + p) * 16 + (e & 15)] = s_run[e];
  }
}

static int corr_pb(int n_phase) { return (n_phase + 9) / 10 * 10 <= (n_phase + 7) / 8 * 8 ? 10 : 8; }
// stretches of kCorrT pixels to a block: a whole group where blocks for three to a CU are left
static int corr_per(int64_t n, int n_phase, int rows, int nd) {
  const int64_t groups = (n + (int64_t)kCorrG * kCorrT - 1) / (kCorrG * kCorrT);
  const int pb = corr_pb(n_phase);
  return groups * ((rows + kCorrRB - 1) / kCorrRB) * ((n_phase + pb - 1) / pb) * ((nd + 15) / 16) >= 768 ? kCorrG : 1;
}
static int corr_chunks(int64_t n, int per) { return (int)((n + (int64_t)per * kCorrT - 1) / (per * kCorrT)); }
size_t diff_corr_part(int64_t n, int n_phase, int rows, int nd) {
  return (size_t)corr_chunks(n, corr_per(n, n_phase, rows, nd)) * rows * ((nd + 15) / 16) * n_phase * 16;
}

// one thread per (row, phase, lag of a tile of 16)
__global__ void k_diff_corr_reduce(DiffArgs a, int nchunk, int per, int n_z, const double *Cpart, double *C) {
  const int ns = a.ns, rows = a.n_mu * ns, P = a.n_phase;
  const long tot = (long)n_z * P * 16, e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= rows * tot) return;
  const int row = (int)(e / tot), z = (int)(e % tot / (P * 16)), p = (int)(e % (P * 16) / 16), l = (int)(e % 16);
  const int k = row / ns, r0 = row / kCorrRB * kCorrRB;
  int hi;
  const int d = corr_lag0(a, r0 / ns, min(rows - 1, r0 + kCorrRB - 1) / ns, hi) + 16 * z + l;
  if (d < a.blag[2 * k] || d > a.blag[2 * k + 1]) return;  // no cell of the bin uses it
  constexpr int kU = 16;
  static_assert(kU % kCorrG == 0, "whole groups");
  const double *in = Cpart + e;
  const long cs = rows * tot;
  const int g = kCorrG / per;  // partials of a group: 1 or kCorrG
  double x = 0.0;
  for (int c = 0; c < nchunk; c += kU) {
    double t[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) t[u] = in[min(c + u, nchunk - 1) * cs];
#pragma unroll
    for (int u = 0; u < kU; u += kCorrG) {
      double s = t[u];
#pragma unroll
      for (int v = 1; v < kCorrG; v++) {
        if (c + u + v >= nchunk) break;
        if (g == 1) {
          x += s;
          s = t[u + v];
        } else {
          s += t[u + v];
        }
      }
      if (c + u < nchunk) x += s;
    }
  }
  C[(((long)k * a.nd + d) * ns + row % ns) * P + p] = x;
}

// a_X = (1 - t) C[d0] + t C[d0 - 1] of the bin and phase (C [k][d][set][P])
__device__ __forceinline__ double corr_at(const double *Cd, int ns, int P, int set, double t, double &diff) {
  const double c0 = Cd[(long)set * P], c1 = Cd[(long)(set - ns) * P];
  diff = c1 - c0;
  return (1 - t) * c0 + t * c1;
}

// scalar gradients from the correlations and the moments: one wave per piece, lanes over
// phases; partials per block: [gvsini, gu1, gu2, gkappa, gkappa_f]
__global__ __launch_bounds__(256) void k_diff_piecegrad(DiffArgs a, const double *C, double *part) {
  __shared__ double s_p[4][kDiffScalars];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, P = a.n_phase, ns = a.ns;
  const int ip = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + w);
  double v[16];
#pragma unroll
  for (int q = 0; q < 16; q++) v[q] = 0.0;
  if (ip < a.n_piece) {
    const CONSTANT int32_t *pc = gc((const int32_t *)(a.piece + ip));
    const int iy = pc[0], k = pc[1], len = pc[3];
    const double kappa = a.prm ? a.prm[3] : a.kappa, kappa_f = a.prm ? a.prm[4] : a.kappa_f;
    const double u1 = a.prm ? a.prm[1] : a.u1, u2 = a.prm ? a.prm[2] : a.u2;
    const double t = gc((const double *)(a.row_t + iy))[0], dt = gc((const double *)(a.row_t + iy))[1];
    const int d0 = gc(a.row_m)[iy] - a.dmin, nm = diff_moments(ns);
    const double s[3] = {(double)len, gc((const double *)(a.psum + ip))[0], gc((const double *)(a.psum + ip))[1]};
    if (d0 >= 1 && d0 < a.nd)
      for (int p = lane; p < P; p += 64) {
        const double *Cd = C + ((long)k * a.nd + d0) * ns * P + p;
        const double *mo = a.mom + (long)ip * nm * P + p;
        double bq, bs, bf = 0.0;
        const double aq = corr_at(Cd, ns, P, 0, t, bq), as = corr_at(Cd, ns, P, 1, t, bs);
        const double af = ns == 3 ? corr_at(Cd, ns, P, 2, t, bf) : 0.0;
        double quiet[3], spot[3], fac[3];  // sums of a^q (1 - phi - psi), a^q phi, a^q b psi
#pragma unroll
        for (int q = 0; q < 3; q++) {
          spot[q] = mo[(long)q * P];
          quiet[q] = s[q] - spot[q] - (ns == 3 ? mo[(long)(q + 3) * P] : 0.0);
          fac[q] = ns == 3 ? mo[(long)(q + 6) * P] : 0.0;
        }
        auto limb = [&](const double (&x)[3]) { return x[0] - u1 * x[1] - u2 * x[2]; };
        v[0] += dt * (limb(quiet) * bq + kappa * limb(spot) * bs + kappa_f * limb(fac) * bf);
        v[1] -= quiet[1] * aq + kappa * spot[1] * as + kappa_f * fac[1] * af;
        v[2] -= quiet[2] * aq + kappa * spot[2] * as + kappa_f * fac[2] * af;
        v[3] += limb(spot) * as;
        v[4] += limb(fac) * af;
      }
  }
  wave_sums16(v);
  if (lane == 0)
#pragma unroll
    for (int q = 0; q < kDiffScalars; q++) s_p[w][q] = v[q];
  __syncthreads();
  if (threadIdx.x < kDiffScalars) {
    double x = 0;
    for (int i = 0; i < 4; i++) x += s_p[i][threadIdx.x];
    part[(long)blockIdx.x * kDiffScalars + threadIdx.x] = x;
  }
}

// map-pixel gradients: node (i, j) of phase p sums, over the cells whose bilinear stencil
// holds it, weight x L (kappa a_S - a_Q) for the spot map and weight x L (kappa_f (1 + LB)
// a_F - a_Q) for the facula map.  One wave per (node row, 16 nodes, 64 phases), lanes over
// phases: the wave walks the cells of the disk rows that touch its node row, the
// correlation factors change only with the bin, and a cell costs a few multiply-adds on
// uniform weights; a node's two running sums go to LDS when the walk passes it, and the
// 16-node rows of all phases are written from there.
constexpr int kMgN = 16;
constexpr int kMgStride = kMgN + 1;
template <int NS>
__global__ __launch_bounds__(256) void k_diff_mapgrad(DiffArgs a, const double *C, double *gmaps, double *gfmaps) {
  extern __shared__ double s_mg[];  // per wave [NS - 1][phases][kMgStride]
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int M = a.map_res, G = a.grid, P = a.n_phase;
  const int jb = (blockIdx.x * 4 + w) * kMgN, i = blockIdx.y;
  const int p0 = blockIdx.z * 64, np = min(64, P - p0), ps = min(64, P);
  if (jb >= M) return;  // no barriers below
  double *tile = s_mg + (size_t)w * (NS - 1) * ps * kMgStride;
  for (int e = lane; e < (NS - 1) * ps * kMgStride; e += 64) tile[e] = 0.0;
  wave_lds_order();
  const double kappa = a.prm ? a.prm[3] : a.kappa, kappa_f = a.prm ? a.prm[4] : a.kappa_f;
  const double u1 = a.prm ? a.prm[1] : a.u1, u2 = a.prm ? a.prm[2] : a.u2;
  const int pl = min(lane, np - 1);
  double *mine = tile + pl * kMgStride;
  auto put = [&](int j, double s, double f) {
    if (j < jb || j >= jb + kMgN || lane >= np) return;
    __hip_atomic_fetch_add(mine + (j - jb), s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    if (NS == 3)
      __hip_atomic_fetch_add(mine + ps * kMgStride + (j - jb), f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
  };
  // cells whose stencil can reach the nodes: a superset, filtered by the plan's own nodes
  const double sc = (double)G / (M - 1);
  const int y_lo = max(0, (int)floor((i - 1) * sc) - 1), y_hi = min(G - 1, (int)ceil((i + 1) * sc) + 1);
  const int z_lo = max(0, (int)floor((jb - 1) * sc) - 1), z_hi = min(G - 1, (int)ceil((jb + kMgN) * sc) + 1);
  for (int iy = y_lo; iy <= y_hi; iy++) {
    const int i0 = gc(a.map_j)[iy];
    if (i0 != i && i0 + 1 != i) continue;
    const int d0 = gc(a.row_m)[iy] - a.dmin;
    if (d0 < 1 || d0 >= a.nd) continue;
    const double fy = gc(a.map_f)[iy], wy = i0 == i ? 1 - fy : fy, t = gc((const double *)(a.row_t + iy))[0];
    int kcur = -1, cur = -2;
    double e1 = 0.0, eq = 0.0, ef = 0.0, s0 = 0.0, s1 = 0.0, f0 = 0.0, f1 = 0.0;
    for (int zb = z_lo; zb <= z_hi; zb += 64) {
      // 64 cells of the row, one per lane: bin, first node, weights on its two nodes
      const int iz = min(zb + lane, G - 1), jz = a.map_j[iz];
      const long idx = (long)iy * G + iz;
      const bool in = zb + lane <= z_hi && jz + 1 >= jb && jz < jb + kMgN;
      const int kz = in ? a.ck[idx] : -1;
      const double2 ce = a.cell[idx];
      const double fz = a.map_f[iz], L = 1. - u1 * ce.x - u2 * ce.x * ce.x, wz0 = L * (1 - fz), wz1 = L * fz;
      unsigned long long todo = __ballot(kz >= 0);
      while (todo) {
        const int l = __builtin_ctzll(todo);
        todo &= todo - 1;
        const int k = __builtin_amdgcn_readlane(kz, l), j0 = __builtin_amdgcn_readlane(jz, l);
        if (k != kcur) {
          kcur = k;
          const double *Cd = C + ((long)k * a.nd + d0) * NS * P + p0 + pl;
          double unused;
          eq = wy * corr_at(Cd, NS, P, 0, t, unused);
          e1 = wy * kappa * corr_at(Cd, NS, P, 1, t, unused) - eq;
          if (NS == 3) ef = wy * kappa_f * corr_at(Cd, NS, P, NS - 1, t, unused);
        }
        if (j0 != cur) {
          put(cur, s0, f0);
          const bool next = j0 == cur + 1;
          if (!next) put(cur + 1, s1, f1);
          s0 = next ? s1 : 0.0;
          f0 = next ? f1 : 0.0;
          s1 = f1 = 0.0;
          cur = j0;
        }
        const double w0 = lane_f64(wz0, l), w1 = lane_f64(wz1, l);
        s0 = fma(w0, e1, s0);
        s1 = fma(w1, e1, s1);
        if (NS == 3) {
          const double x = fma(lane_f64(ce.y, l), ef, -eq);
          f0 = fma(w0, x, f0);
          f1 = fma(w1, x, f1);
        }
      }
    }
    put(cur, s0, f0);
    put(cur + 1, s1, f1);
  }
  wave_lds_order();
  const int nj = min(kMgN, M - jb);
  for (int e = lane; e < np * kMgN; e += 64) {
    const int p = e / kMgN, j = e % kMgN;
    if (j >= nj) continue;
    const long o = ((long)(p0 + p) * M + i) * M + jb + j;
    gmaps[o] = tile[p * kMgStride + j];
    if (NS == 3) gfmaps[o] = tile[(ps + p) * kMgStride + j];
  }
}

// seed gradients gX_k[i] = sum_p sum_d HX_pk[d] G_I,p[i + dmin + d]; block = (tile of
// kDT * XB pixels, group of R (bin, set) rows), kSeedP phases staged at a time with the
// taps of up to kSeedD of the offsets the group's bins use; the next phases' loads and
// the next offset's reads are in flight as in k_diff_fir
constexpr int kSeedP = 4;
constexpr int kSeedD = 32;
template <int R, int XB>
__global__ __launch_bounds__(kDT) void k_diff_seedgrad(DiffArgs a, const double *GI, double *gq, double *gs,
                                                       double *gf) {
  extern __shared__ double s_sg[];  // [kSeedP][len], then [kSeedP][kSeedD][16]
  constexpr int kRow = XB + 1, kTap = kSeedD * 16 / kDT;
  constexpr bool kAhead = XB == 1;
  const int g = blockIdx.y, ng = gridDim.y, ns = a.ns, rows = a.n_mu * ns, tid = threadIdx.x, lane16 = tid & 15;
  const long i0 = (long)blockIdx.x * (kDT * XB), n = a.n;
  const int nd = a.nd, len = kDT * XB + nd - 1, P = a.n_phase;
  double *s_t = s_sg + kSeedP * len;
  double F[XB][R];
#pragma unroll
  for (int b = 0; b < XB; b++)
#pragma unroll
    for (int r = 0; r < R; r++) F[b][r] = 0.0;
  int lo = nd, hi = -1;
  for (int k = g * R / ns; k <= min(rows - 1, g * R + R - 1) / ns; k++) {
    lo = min(lo, a.blag[2 * k]);
    hi = max(hi, a.blag[2 * k + 1]);
  }
  auto gi_at = [&](int p, int e) {
    const long j = i0 + a.dmin + e;
    const bool in = j >= 0 && j < n;
    const double v = GI[(long)min(p, P - 1) * n + (in ? j : 0)];
    return in ? v : 0.0;
  };
  auto taps_at = [&](int p, int d) { return a.taps_r + (((long)min(p, P - 1) * ng + g) * nd + d) * 16; };
  double rv[kSeedP][kRow], tv[kSeedP][kTap];
  const int nt = min(kSeedD, hi + 1 - lo) * 16;
  auto fetch = [&](int p0) {
#pragma unroll
    for (int u = 0; u < kSeedP; u++) {
#pragma unroll
      for (int w = 0; w < kRow; w++) rv[u][w] = gi_at(p0 + u, min(tid + w * kDT, len - 1));
      const double *T = taps_at(p0 + u, lo);
#pragma unroll
      for (int w = 0; w < kTap; w++) tv[u][w] = T[min(tid + w * kDT, nt - 1)];
    }
  };
  if (kAhead && lo <= hi) fetch(0);
  for (int p0 = 0; p0 < P && lo <= hi; p0 += kSeedP) {
    const int np = min(kSeedP, P - p0);
    if (!kAhead) fetch(p0);
    for (int dc = lo; dc <= hi; dc += kSeedD) {
      const int nc = min(kSeedD, hi + 1 - dc);
      __syncthreads();
#pragma unroll
      for (int u = 0; u < kSeedP; u++) {
        if (dc == lo) {
#pragma unroll
          for (int w = 0; w < kRow; w++)
            if (tid + w * kDT < len) s_sg[u * len + tid + w * kDT] = rv[u][w];
          for (int e = tid + kRow * kDT; e < len; e += kDT) s_sg[u * len + e] = gi_at(p0 + u, e);  // nd > kDT
#pragma unroll
          for (int w = 0; w < kTap; w++)
            if (tid + w * kDT < nt) s_t[u * kSeedD * 16 + tid + w * kDT] = tv[u][w];
        } else {
          const double *T = taps_at(p0 + u, dc);
          for (int e = tid; e < nc * 16; e += kDT) s_t[u * kSeedD * 16 + e] = T[e];
        }
      }
      __syncthreads();
      if (kAhead && dc == lo && p0 + kSeedP < P) fetch(p0 + kSeedP);
      for (int u = 0; u < np; u++) {
        const double *x = s_sg + u * len + tid + dc, *tp = s_t + u * kSeedD * 16 + lane16;
        constexpr int D = 2;  // offsets per step
        double t[2][D], xv[2][D][XB];
        auto read = [&](int s, int d) {
#pragma unroll
          for (int w = 0; w < D; w++) {
            const int dw = min(d + w, nc - 1);
            t[s][w] = tp[dw * 16];
#pragma unroll
            for (int b = 0; b < XB; b++) xv[s][w][b] = x[b * kDT + dw];
          }
        };
        auto sums = [&](int s, int d) {
#pragma unroll
          for (int w = 0; w < D; w++)
            if (d + w < nc)
#pragma unroll
              for (int b = 0; b < XB; b++) row_fma<R>(F[b], t[s][w], xv[s][w][b]);
        };
        read(0, 0);
        for (int d = 0; d < nc; d += 2 * D) {
          read(1, d + D);
          __builtin_amdgcn_sched_barrier(0);
          sums(0, d);
          read(0, d + 2 * D);
          __builtin_amdgcn_sched_barrier(0);
          sums(1, d + D);
        }
      }
    }
  }
#pragma unroll
  for (int b = 0; b < XB; b++) {
    const long i = i0 + tid + b * kDT;
    if (i >= n) continue;
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int row = g * R + r, k = row / ns, set = row - k * ns;
      if (row < rows) (set == 0 ? gq : set == 1 ? gs : gf)[(long)k * n + i] = F[b][r];
    }
  }
}

// ------------------------------------------------------------ launchers
// The widest shift range that the adjoint accepts (forwards take 2048 offsets).  No kernel here needs it: at this bound the seed gradients hold 57 KB of LDS.
constexpr int kAdjointLags = 761;

// Two pixels per thread serve a coefficient read twice, where that still leaves two
// blocks per CU; one otherwise.
static bool two_pixels(int64_t n, int groups) { return (n + 2 * kDT - 1) / (2 * kDT) * groups >= 512; }

template <int NS, int R>
static hipError_t launch_fir_r(const DiffArgs &a, hipStream_t s) {
  const int groups = (a.n_phase + R - 1) / R;
  const bool two = two_pixels(a.n, groups);
  const int px = two ? 2 * kDT : kDT;
  const size_t lds = (size_t)(NS * (px + a.nd - 1) + kFirD * NS * 16) * sizeof(double);  // at most 74 KB (2048 offsets)
  dim3 gr((unsigned)((a.n + px - 1) / px), groups);
  if (two)
    k_diff_fir<NS, R, 2><<<gr, kDT, lds, s>>>(a);
  else
    k_diff_fir<NS, R, 1><<<gr, kDT, lds, s>>>(a);
  return hipGetLastError();
}

template <int NS>
static hipError_t launch_fir_ns(const DiffArgs &a, hipStream_t s) {
  switch (a.grp_p) {
    case 4: return launch_fir_r<NS, 4>(a, s);
    case 8: return launch_fir_r<NS, 8>(a, s);
    case 10: return launch_fir_r<NS, 10>(a, s);
    case 12: return launch_fir_r<NS, 12>(a, s);
    case 16: return launch_fir_r<NS, 16>(a, s);
    default: return hipErrorInvalidValue;
  }
}

template <int R>
static hipError_t launch_seed_r(const DiffArgs &a, const double *GI, double *gq, double *gs, double *gf,
                                hipStream_t s) {
  const int groups = (a.n_mu * a.ns + R - 1) / R;
  const bool two = two_pixels(a.n, groups);
  const int px = two ? 2 * kDT : kDT;
  const size_t lds = (size_t)kSeedP * (px + a.nd - 1 + kSeedD * 16) * sizeof(double);  // at most 57 KB (kAdjointLags)
  dim3 gr((unsigned)((a.n + px - 1) / px), groups);
  if (two)
    k_diff_seedgrad<R, 2><<<gr, kDT, lds, s>>>(a, GI, gq, gs, gf);
  else
    k_diff_seedgrad<R, 1><<<gr, kDT, lds, s>>>(a, GI, gq, gs, gf);
  return hipGetLastError();
}

template <int PB>
static hipError_t launch_corr_p(const DiffArgs &a, const double *GI, double *Cpart, double *C, hipStream_t s) {
  const int rows = a.n_mu * a.ns, n_tile = (a.n_phase + PB - 1) / PB, n_z = (a.nd + 15) / 16;
  const int per = corr_per(a.n, a.n_phase, rows, a.nd), nch = corr_chunks(a.n, per);
  if ((long)n_tile * n_z > 65535) return hipErrorInvalidValue;
  dim3 gr(nch, (rows + kCorrRB - 1) / kCorrRB, n_tile * n_z);
  const size_t lds = (size_t)(corr_lds(PB) + kCorrRB * PB * 16) * sizeof(double);
  k_diff_corr<PB><<<gr, 256, lds, s>>>(a, GI, Cpart, n_z, per);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const long tot = (long)rows * n_z * a.n_phase * 16;
  k_diff_corr_reduce<<<(unsigned)((tot + kDT - 1) / kDT), kDT, 0, s>>>(a, nch, per, n_z, Cpart, C);
  return hipGetLastError();
}

hipError_t launch_diff_forward_spectra(const DiffArgs &a, const ConvArgs &c, const double *target, int trim,
                                       double *res_part, int *res_blocks, hipStream_t s) {
  hipError_t e;
  if (a.ns != 2 && a.ns != 3) return hipErrorInvalidValue;
  if (a.ns == 3 && (!a.f || !a.fmaps)) return hipErrorInvalidValue;
  k_diff_rows<<<1, kDiffRowT, (size_t)(2 * a.nd + a.grid) * sizeof(int), s>>>(a);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  const unsigned pg = (a.n_phase + 63) / 64;
  const int pw = a.n_phase < 64 ? a.n_phase : 64;
  const unsigned mbx = (a.n_piece + 8 * kMomW - 1) / (8 * kMomW);  // blocks per XCD
  dim3 gm(8 * mbx, pg), gt(a.nd, a.n_mu, pg);
  const size_t lds_mom = (size_t)kMomW * pw * kMomStride * sizeof(double);  // at most 68 KB
  if (a.ns == 3) {
    k_diff_moments<3><<<gm, 64 * kMomW, lds_mom, s>>>(a, (int)mbx);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    k_diff_taps<3><<<gt, 64 * kTapW, 0, s>>>(a);
  } else {
    k_diff_moments<2><<<gm, 64 * kMomW, lds_mom, s>>>(a, (int)mbx);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    k_diff_taps<2><<<gt, 64 * kTapW, 0, s>>>(a);
  }
  if ((e = hipGetLastError()) != hipSuccess) return e;
  e = a.ns == 3 ? launch_fir_ns<3>(a, s) : launch_fir_ns<2>(a, s);
  if (e != hipSuccess) return e;
  size_t lds_conv = (size_t)(4 * kDT + 2 * c.ntp) * sizeof(double);
  if (lds_conv > 65536) return hipErrorInvalidValue;
  int nb = (int)((a.n + 4 * kDT - 1) / (4 * kDT));
  *res_blocks = nb;
  dim3 gc((unsigned)nb, a.n_phase);
  k_diff_conv<<<gc, kDT, lds_conv, s>>>(a, c, target, trim, res_part);
  return hipGetLastError();
}

int diff_conv_blocks(int64_t n) { return (int)((n + 4 * kDT - 1) / (4 * kDT)); }

// loss = sum_p [w_spec r2_p + w_rv (RV_p - rv_t)^2 + w_fw (FWHM_p - fw_t)^2], r2_p the
// residual partials of phase p summed in order; the same order as the host sum
// With device parameters (graph replays) the loss is NaN when vsini leaves the
// bound tap range or when the cell weights leave the accepted range, which is that of
// the series' fixed-point taps: n_cells max|L| max(3, |kappa|, |kappa_f| lbmax) >= 2^30,
// lbmax = max |1 + LB(mu)| (maps are filling factors in [0, 1]).
__global__ __launch_bounds__(kDT) void k_diff_loss(int n_phase, int res_blocks, const double *res_part,
                                                   const double *theta, const double *rv_t, const double *fw_t,
                                                   const double *bis_t, double w_spec, double w_rv, double w_fw,
                                                   double w_bis, double *bisd, int n_v, const double *prm,
                                                   double vsini_max, double n_cells, double lbmax, double *loss,
                                                   double *dth, double *series) {
  extern __shared__ double term[];  // [n_phase]
  for (int p = threadIdx.x; p < n_phase; p += blockDim.x) {
    // the residual partials in order, kResU loads ahead of their adds
    constexpr int kResU = 16;
    const double *rp = res_part + (long)p * res_blocks;
    double r2 = 0;
    int b = 0;
    for (; b + kResU <= res_blocks; b += kResU) {
      double x[kResU];
#pragma unroll
      for (int u = 0; u < kResU; u++) x[u] = rp[b + u];
#pragma unroll
      for (int u = 0; u < kResU; u++) r2 += x[u];
    }
    for (; b < res_blocks; b++) r2 += rp[b];
    double drv = theta[p * 4 + 2] - rv_t[p], dfw = theta[p * 4 + 3] - fw_t[p];
    double t = w_spec * r2 + w_rv * drv * drv + w_fw * dfw * dfw;
    double d4[4] = {0.0, 0.0, 2 * w_rv * drv, 2 * w_fw * dfw};
    if (w_bis != 0.0) {  // span term; its coefficient feeds k_fit_adjoint's direct term
      double *bp = bisd + (long)p * (n_v + kBisHead);
      double db = bp[0] - bis_t[p];
      t += w_bis * db * db;
      double coef = 2 * w_bis * db;
      for (int q = 0; q < 4; q++) d4[q] += coef * bp[2 + q];
      bp[1] = coef;
    }
    term[p] = t;
    for (int q = 0; q < 4; q++) dth[p * 4 + q] = d4[q];
    if (series) {  // RV, FWHM and span of every phase in one piece, for the host
      series[p] = theta[p * 4 + 2];
      series[n_phase + p] = theta[p * 4 + 3];
      series[2 * n_phase + p] = bisd[(long)p * (n_v + kBisHead)];
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double l = 0;
    for (int p = 0; p < n_phase; p++) l += term[p];
    double vs = prm ? prm[0] : 0.0;
    if (prm && !(vs > 0 && vs <= vsini_max)) l = __longlong_as_double(0x7ff8000000000000LL);  // outside the tap range
    if (prm) {
      // max |L| over mu in [0, 1]: the ends and the vertex of the quadratic in (1 - mu)
      const double u1 = prm[1], u2 = prm[2];
      double lmax = fmax(1.0, fabs(1 - u1 - u2));
      if (u2 != 0.0) {
        double x = -u1 / (2 * u2);
        if (x > 0 && x < 1) lmax = fmax(lmax, fabs(1 - u1 * x - u2 * x * x));
      }
      double w = lmax * fmax(3.0, fmax(fabs(prm[3]), fabs(prm[4]) * lbmax));
      if (!(n_cells * w < 1073741824.0)) l = __longlong_as_double(0x7ff8000000000000LL);
    }
    loss[0] = l;
  }
}

// g[q] = sum over blocks of cell_part[b][q]: thread t sums blocks t, t + kDT, ...
// (independent loads), then a fixed-order tree over the threads
__global__ __launch_bounds__(kDT) void k_diff_grad(int n_blocks, const double *cell_part, double *g) {
  __shared__ double red[kDiffScalars][kDT];
  double sq[kDiffScalars];
#pragma unroll
  for (int q = 0; q < kDiffScalars; q++) sq[q] = 0.0;
  for (int b = threadIdx.x; b < n_blocks; b += kDT)
#pragma unroll
    for (int q = 0; q < kDiffScalars; q++) sq[q] += cell_part[(long)b * kDiffScalars + q];
#pragma unroll
  for (int q = 0; q < kDiffScalars; q++) red[q][threadIdx.x] = sq[q];
  __syncthreads();
  for (int off = kDT / 2; off > 0; off >>= 1) {
    if (threadIdx.x < off)
#pragma unroll
      for (int q = 0; q < kDiffScalars; q++) red[q][threadIdx.x] += red[q][threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x < kDiffScalars) g[threadIdx.x] = red[threadIdx.x][0];
}

hipError_t launch_diff_loss(int n_phase, int res_blocks, const double *res_part, const double *theta,
                            const double *rv_t, const double *fw_t, const double *bis_t, double w_spec, double w_rv,
                            double w_fw, double w_bis, double *bisd, int n_v, const double *prm, double vsini_max,
                            double n_cells, double lbmax, double *loss, double *dth, double *series,
                            hipStream_t s) {
  if (n_phase < 1 || (size_t)n_phase * 8 > 65536) return hipErrorInvalidValue;
  if ((w_bis != 0.0 && (!bisd || !bis_t)) || (series && !bisd)) return hipErrorInvalidValue;
  k_diff_loss<<<1, kDT, (size_t)n_phase * 8, s>>>(n_phase, res_blocks, res_part, theta, rv_t, fw_t, bis_t, w_spec,
                                                  w_rv, w_fw, w_bis, bisd, n_v, prm, vsini_max, n_cells, lbmax, loss,
                                                  dth, series);
  return hipGetLastError();
}

hipError_t launch_diff_grad(int n_blocks, const double *cell_part, double *g, hipStream_t s) {
  k_diff_grad<<<1, kDT, 0, s>>>(n_blocks, cell_part, g);
  return hipGetLastError();
}
int diff_piece_blocks(int n_piece) { return (n_piece + 3) / 4; }

hipError_t launch_diff_psum(const DiffArgs &a, double2 *psum, hipStream_t s) {
  k_diff_psum<<<(a.n_piece + kDT - 1) / kDT, kDT, 0, s>>>(a, psum);
  return hipGetLastError();
}

hipError_t launch_diff_cells(const DiffArgs &a, const double *mu_bounds, int32_t *ck, double2 *cell, hipStream_t s) {
  const long ncell = (long)a.grid * a.grid;
  k_diff_cells<<<(unsigned)((ncell + kDT - 1) / kDT), kDT, 0, s>>>(a, mu_bounds, ck, cell);
  return hipGetLastError();
}

hipError_t launch_fit_polish(const double *v, int n_v, const double *ccf, const double *par, int n_ccf, double *theta,
                             hipStream_t s) {
  if (n_ccf == 0) return hipSuccess;
  if (n_v < 1 || n_v > kMaxVDiff) return hipErrorInvalidValue;
  k_fit_polish<<<n_ccf, 64, (size_t)2 * n_v * sizeof(double), s>>>(v, n_v, ccf, par, theta);
  return hipGetLastError();
}

hipError_t launch_diff_backward(const DiffArgs &a, const ConvArgs &c, const double *target, int trim, double w_spec,
                                const double *v, int n_v, const double *ccf, const double *theta, const double *dth,
                                double *gy, int64_t n_t, const int64_t *mt_ptr, const int32_t *mt_w,
                                const int32_t *mt_col, const double *mt_val, double *GF, double *GI, double *Cpart,
                                double *C, double *gmaps, double *gfmaps, double *cell_part, double *gq, double *gs,
                                double *gf, const double *bisd, hipStream_t s) {
  hipError_t e;
  if (a.ns == 3 && (!gf || !gfmaps)) return hipErrorInvalidValue;
  k_fit_adjoint<<<a.n_phase, 64, 0, s>>>(v, n_v, ccf, theta, dth, bisd, gy);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  long tot = (long)a.n_phase * a.n;
  k_diff_gradF<<<(unsigned)((tot + kDT - 1) / kDT), kDT, 0, s>>>(a, target, trim, w_spec, GF);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (n_t > 0) {
    size_t lds_mt = (size_t)kMtP * n_v * sizeof(double);
    if (lds_mt > 65536) return hipErrorInvalidValue;
    dim3 gm((unsigned)((n_t + kDT - 1) / kDT), (a.n_phase + kMtP - 1) / kMtP);
    k_mask_transpose<<<gm, kDT, lds_mt, s>>>(n_t, trim, a.n, a.n_phase, n_v, mt_ptr, mt_w, mt_col, mt_val, gy, GF);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  size_t lds_conv = (size_t)(4 * kDT + 2 * c.ntp) * sizeof(double);
  if (lds_conv > 65536) return hipErrorInvalidValue;
  dim3 gc((unsigned)((a.n + 4 * kDT - 1) / (4 * kDT)), a.n_phase);
  k_diff_convT<<<gc, kDT, lds_conv, s>>>(a, c, GF, GI);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (a.nd > kAdjointLags) return hipErrorInvalidValue;
  e = corr_pb(a.n_phase) == 10 ? launch_corr_p<10>(a, GI, Cpart, C, s) : launch_corr_p<8>(a, GI, Cpart, C, s);
  if (e != hipSuccess) return e;
  k_diff_piecegrad<<<diff_piece_blocks(a.n_piece), 256, 0, s>>>(a, C, cell_part);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  const int pw = a.n_phase < 64 ? a.n_phase : 64;
  dim3 gmg((a.map_res + 4 * kMgN - 1) / (4 * kMgN), a.map_res, (a.n_phase + 63) / 64);
  const size_t lds_mg = (size_t)4 * (a.ns - 1) * pw * kMgStride * sizeof(double);  // at most 70 KB
  if (a.ns == 3)
    k_diff_mapgrad<3><<<gmg, 256, lds_mg, s>>>(a, C, gmaps, gfmaps);
  else
    k_diff_mapgrad<2><<<gmg, 256, lds_mg, s>>>(a, C, gmaps, gfmaps);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  switch (a.grp_r) {
    case 4: return launch_seed_r<4>(a, GI, gq, gs, gf, s);
    case 8: return launch_seed_r<8>(a, GI, gq, gs, gf, s);
    case 10: return launch_seed_r<10>(a, GI, gq, gs, gf, s);
    case 12: return launch_seed_r<12>(a, GI, gq, gs, gf, s);
    case 16: return launch_seed_r<16>(a, GI, gq, gs, gf, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace soap
