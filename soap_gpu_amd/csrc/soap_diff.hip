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
// atomics: every sum has a fixed order), and everything after works on pieces: 12,500 of
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
    const double ca = a.cell[(long)pc.iy * a.grid + pc.iz0 + c].x;
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

// Moments of one piece for up to 64 phases: one wave per (piece, 64 phases).  The wave
// samples its cells' filling factors bilinearly (two phases x 32 cells per step, loads
// of neighbouring cells from neighbouring nodes) into LDS and then sums them with lanes
// over phases, the cell's own factors read from the lane that holds them.  Blocks are in
// contiguous runs per XCD: neighbouring pieces read the same map rows.  Outputs: mom rows
// 0-2 sum a^q phi, 3-5 sum a^q psi, 6-8 sum a^q b psi, and the sets' tap weights
// sum L (1 - phi - psi), kappa sum L phi, kappa_f sum L b psi.
constexpr int kMomW = 4;       // waves (pieces) per block
constexpr int kMomU = 4;       // sampling steps in flight
constexpr int kMomStride = kDiffPiece + 1;
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
  const DiffPiece pc = {pi[0], pi[1], pi[2], pi[3]};
  const int M = a.map_res;
  const long MM = (long)M * M;
  // this lane's cell and its stencil (the same for every phase)
  const int c = lane & 31, ph = lane >> 5;
  const int cc = min(c, pc.len - 1);
  const double2 me = a.cell[(long)pc.iy * a.grid + pc.iz0 + cc];
  const int j0 = a.map_j[pc.iz0 + cc], i0 = gc(a.map_j)[pc.iy];
  const double fz = a.map_f[pc.iz0 + cc], fy = gc(a.map_f)[pc.iy];
  const double w00 = (1 - fy) * (1 - fz), w10 = fy * (1 - fz), w01 = (1 - fy) * fz, w11 = fy * fz;
  const long off = (long)i0 * M + j0;
  double m[9];
#pragma unroll
  for (int q = 0; q < 9; q++) m[q] = 0.0;
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
    for (int i = 0; i < pc.len; i++) {
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
  wt[0] = ((double)pc.len - m[0] - m[3]) - u1 * (s1 - m[1] - m[4]) - u2 * (s2 - m[2] - m[5]);
  wt[P] = kappa * Lphi;
  if (NS == 3) wt[2L * P] = kappa_f * (m[6] - u1 * m[7] - u2 * m[8]);
}

// taps[p][k][d][q] = sum over the pieces of bin k whose row has tap index d of w (1 - t),
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
    double *o = a.taps + (((long)p * a.n_mu + k) * a.nd + d) * NS;
#pragma unroll
    for (int q = 0; q < NS; q++) {
      double x = s_t[0][q][lane];
#pragma unroll
      for (int i = 1; i < kTapW; i++) x += s_t[i][q][lane];
      o[q] = x;
    }
  }
}

// I_p[j] = sum_k sum_d HQ[d] Q_k[j - dmin - d] + HS[d] S_k[j - dmin - d] (+ HF[d] Fa_k[j - dmin - d]);
// block = (tile, p)
template <int NS>
__global__ __launch_bounds__(kDT) void k_diff_fir(DiffArgs a) {
  extern __shared__ double rows[];  // [NS][row_len]
  int p = blockIdx.y;
  long j0 = (long)blockIdx.x * kDT;
  int nd = a.nd, row_len = kDT + nd - 1;
  long src0 = j0 - a.dmin - nd + 1;
  double acc = 0.0;
  for (int k = 0; k < a.n_mu; k++) {
    int lo = a.blag[2 * k], hi = a.blag[2 * k + 1];
    if (lo > hi) continue;  // uniform
    __syncthreads();
    for (int e = threadIdx.x; e < row_len; e += blockDim.x) {
      long i = src0 + e;
      bool in = i >= 0 && i < a.n;
      rows[e] = in ? a.q[(long)k * a.n + i] : 0.0;
      rows[row_len + e] = in ? a.s[(long)k * a.n + i] : 0.0;
      if (NS == 3) rows[2 * row_len + e] = in ? a.f[(long)k * a.n + i] : 0.0;
    }
    __syncthreads();
    const double *T = a.taps + ((long)p * a.n_mu + k) * nd * NS;
    for (int di = lo; di <= hi; di++) {
      int e = threadIdx.x + nd - 1 - di;
#pragma unroll
      for (int q = 0; q < NS; q++) acc = fma(T[di * NS + q], rows[q * row_len + e], acc);
    }
  }
  long j = j0 + threadIdx.x;
  if (j < a.n) a.I[(long)p * a.n + j] = acc;
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

// lag correlations C[k][d][set][p] = sum_j G_I[p][j] X_k[j - dmin - d], in two
// passes.  Pass 1: block = (chunk of kCorrT pixels, bin k, group of kCorrPG
// phases); the bin's two seed-row segments are staged once for the group.  Each
// thread owns kCorrPer consecutive pixels (G_I of the phase in registers) and,
// per group of kCorrL lags, reads one register window of the staged row and
// forms kCorrL partial sums; the block adds them up through LDS ([lag][thread]
// then 32-lane shuffles) into the chunk's partial.  Pass 2 sums the chunk
// partials in chunk order (deterministic, no atomics).
constexpr int kCorrPer = 9;  // odd: a thread stride of kCorrPer doubles is free of LDS bank conflicts
constexpr int kCorrT = kDT * kCorrPer;
constexpr int kCorrL = 8;
constexpr int kCorrPG = 10;
// One pass covers nsp <= 2 seed cubes (x0, x1), written to sets soff, soff + 1 of
// the ns-set tables; the facula set, when present, is a second pass (three staged
// rows would not fit the LDS budget).
__global__ __launch_bounds__(kDT) void k_diff_corr(DiffArgs a, const double *GI, double *Cpart, const double *x0,
                                                   const double *x1, int nsp, int soff) {
  extern __shared__ double lds[];  // row(s) [kCorrT + nd - 1 + kCorrL] each, then [kCorrL][kDT] partials
  const int k = blockIdx.y, chunk = blockIdx.x, nchunk = gridDim.x;
  const long j0 = (long)chunk * kCorrT;
  const int nd = a.nd, rl = kCorrT + nd - 1 + kCorrL, ns = a.ns;
  double *rq = lds, *rs = rq + rl, *red = rq + nsp * rl;
  const long src0 = j0 - a.dmin - nd + 1;
  for (int e = threadIdx.x; e < rl; e += blockDim.x) {
    long i = src0 + e;
    bool in = i >= 0 && i < a.n && e < kCorrT + nd - 1;
    rq[e] = in ? x0[(long)k * a.n + i] : 0.0;
    if (nsp == 2) rs[e] = in ? x1[(long)k * a.n + i] : 0.0;
  }
  __syncthreads();
  const int p1 = min(a.n_phase, (int)(blockIdx.z + 1) * kCorrPG);
  for (int p = blockIdx.z * kCorrPG; p < p1; p++) {
    double g[kCorrPer];
#pragma unroll
    for (int u = 0; u < kCorrPer; u++) {
      long j = j0 + threadIdx.x * kCorrPer + u;
      g[u] = j < a.n ? GI[(long)p * a.n + j] : 0.0;
    }
    double *out = Cpart + (((long)p * a.n_mu + k) * nchunk + chunk) * nd * ns;
    const int dlo = a.blag[2 * k], dhi = a.blag[2 * k + 1];  // the lags this bin's cells use
    for (int set = 0; set < nsp; set++) {
      const double *row = (set ? rs : rq) + threadIdx.x * kCorrPer;
      for (int d0 = dlo; d0 <= dhi; d0 += kCorrL) {
        // lag d = d0 + l reads X[j - dmin - d] = row[u + nd - 1 - d]; window base nd - d0 - kCorrL
        const int wb = nd - d0 - kCorrL;
        double w[kCorrPer + kCorrL - 1];
#pragma unroll
        for (int e = 0; e < kCorrPer + kCorrL - 1; e++) {
          int x = wb + e;
          w[e] = x >= 0 ? row[x] : 0.0;  // x < 0 only for lags d >= nd (discarded)
        }
        double acc[kCorrL];
#pragma unroll
        for (int l = 0; l < kCorrL; l++) {
          acc[l] = 0.0;
#pragma unroll
          for (int u = 0; u < kCorrPer; u++) acc[l] = fma(g[u], w[u + kCorrL - 1 - l], acc[l]);
        }
        __syncthreads();  // red is free
#pragma unroll
        for (int l = 0; l < kCorrL; l++) red[l * kDT + threadIdx.x] = acc[l];
        __syncthreads();
        // kDT threads = kCorrL lags x 32 lanes: each lane sums kDT / 32 partials
        const int l = threadIdx.x >> 5, part = threadIdx.x & 31;
        double x = 0.0;
#pragma unroll
        for (int r = 0; r < kDT / 32; r++) x += red[l * kDT + r * 32 + part];
        for (int off = 16; off > 0; off >>= 1) x += __shfl_xor(x, off);
        if (part == 0 && d0 + l < nd) out[(d0 + l) * ns + soff + set] = x;
      }
    }
  }
}

__global__ void k_diff_corr_reduce(DiffArgs a, int n_pk, int nd, int nchunk, const double *Cpart, double *C) {
  const int ns = a.ns;
  long e = (long)blockIdx.x * blockDim.x + threadIdx.x;  // (p, k) x (d, set)
  if (e >= (long)n_pk * nd * ns) return;
  long pk = e / (nd * ns), r = e % (nd * ns);
  const int d = (int)(r / ns), p = (int)(pk / a.n_mu), k = (int)(pk % a.n_mu);
  double x = 0.0;
  if (d >= a.blag[2 * k] && d <= a.blag[2 * k + 1])  // k_diff_corr computes only these lags
    for (int c = 0; c < nchunk; c++) x += Cpart[(pk * nchunk + c) * nd * ns + r];
  C[((long)k * nd * ns + r) * a.n_phase + p] = x;
}

int diff_corr_chunks(int64_t n) { return (int)((n + kCorrT - 1) / kCorrT); }

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
    const int iy = pc[0], len = pc[2], k = pc[3];
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

// seed gradients gX_k[i] = sum_p sum_d HX_pk[d] G_I,p[i + dmin + d]; block = (tile, bin)
template <int NS>
__global__ __launch_bounds__(kDT) void k_diff_seedgrad(DiffArgs a, const double *GI, double *gq, double *gs,
                                                       double *gf) {
  extern __shared__ double gl[];  // G_I,p over [i0 + dmin, i0 + kDT + dmin + nd - 1)
  int k = blockIdx.y;
  long i0 = (long)blockIdx.x * kDT;
  int nd = a.nd, len = kDT + nd - 1;
  double ax[NS];
#pragma unroll
  for (int q = 0; q < NS; q++) ax[q] = 0.0;
  for (int p = 0; p < a.n_phase; p++) {
    int lo = a.blag[2 * k], hi = a.blag[2 * k + 1];
    if (lo > hi) continue;  // uniform
    __syncthreads();
    for (int e = threadIdx.x; e < len; e += blockDim.x) {
      long j = i0 + a.dmin + e;
      gl[e] = (j >= 0 && j < a.n) ? GI[(long)p * a.n + j] : 0.0;
    }
    __syncthreads();
    const double *T = a.taps + ((long)p * a.n_mu + k) * nd * NS;
    for (int d = lo; d <= hi; d++) {
      double g = gl[threadIdx.x + d];
#pragma unroll
      for (int q = 0; q < NS; q++) ax[q] = fma(T[d * NS + q], g, ax[q]);
    }
  }
  long i = i0 + threadIdx.x;
  if (i < a.n) {
    gq[(long)k * a.n + i] = ax[0];
    gs[(long)k * a.n + i] = ax[1];
    if (NS == 3) gf[(long)k * a.n + i] = ax[NS - 1];
  }
}

// ------------------------------------------------------------ launchers
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
  size_t lds_fir = (size_t)a.ns * (kDT + a.nd - 1) * sizeof(double);
  if (lds_fir > 65536) return hipErrorInvalidValue;
  dim3 gf((unsigned)((a.n + kDT - 1) / kDT), a.n_phase);
  if (a.ns == 3)
    k_diff_fir<3><<<gf, kDT, lds_fir, s>>>(a);
  else
    k_diff_fir<2><<<gf, kDT, lds_fir, s>>>(a);
  if ((e = hipGetLastError()) != hipSuccess) return e;
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
// bound tap range or when the cell weights could exceed the fixed-point tap
// capacity: n_cells max|L| max(3, |kappa|, |kappa_f| lbmax) >= 2^30, lbmax =
// max |1 + LB(mu)| (maps are filling factors in [0, 1]).
__global__ __launch_bounds__(kDT) void k_diff_loss(int n_phase, int res_blocks, const double *res_part,
                                                   const double *theta, const double *rv_t, const double *fw_t,
                                                   const double *bis_t, double w_spec, double w_rv, double w_fw,
                                                   double w_bis, double *bisd, int n_v, const double *prm,
                                                   double vsini_max, double n_cells, double lbmax, double *loss,
                                                   double *dth) {
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
                            double n_cells, double lbmax, double *loss, double *dth, hipStream_t s) {
  if (n_phase < 1 || (size_t)n_phase * 8 > 65536) return hipErrorInvalidValue;
  if (w_bis != 0.0 && (!bisd || !bis_t)) return hipErrorInvalidValue;
  k_diff_loss<<<1, kDT, (size_t)n_phase * 8, s>>>(n_phase, res_blocks, res_part, theta, rv_t, fw_t, bis_t, w_spec,
                                                  w_rv, w_fw, w_bis, bisd, n_v, prm, vsini_max, n_cells, lbmax, loss,
                                                  dth);
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
  size_t lds_corr = (size_t)(2 * (kCorrT + a.nd - 1 + kCorrL) + kCorrL * kDT) * sizeof(double);
  if (lds_corr > 65536) return hipErrorInvalidValue;
  const int nchunk = diff_corr_chunks(a.n);
  dim3 gr((unsigned)nchunk, a.n_mu, (a.n_phase + kCorrPG - 1) / kCorrPG);
  k_diff_corr<<<gr, kDT, lds_corr, s>>>(a, GI, Cpart, a.q, a.s, 2, 0);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  if (a.ns == 3) {
    k_diff_corr<<<gr, kDT, lds_corr, s>>>(a, GI, Cpart, a.f, nullptr, 1, 2);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  long nc = (long)a.n_phase * a.n_mu * a.nd * a.ns;
  k_diff_corr_reduce<<<(unsigned)((nc + kDT - 1) / kDT), kDT, 0, s>>>(a, a.n_phase * a.n_mu, a.nd, nchunk, Cpart, C);
  if ((e = hipGetLastError()) != hipSuccess) return e;
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
  size_t lds_seed = (size_t)(kDT + a.nd - 1) * sizeof(double);
  dim3 gsd((unsigned)((a.n + kDT - 1) / kDT), a.n_mu);
  if (a.ns == 3)
    k_diff_seedgrad<3><<<gsd, kDT, lds_seed, s>>>(a, GI, gq, gs, gf);
  else
    k_diff_seedgrad<2><<<gsd, kDT, lds_seed, s>>>(a, GI, gq, gs, gf);
  return hipGetLastError();
}

}  // namespace soap
