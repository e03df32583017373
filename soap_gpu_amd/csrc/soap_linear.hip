// gfx950 kernels of the linear-wavelength-grid path (the reference's native
// 0.005 A seed format).  On a linear grid a Doppler shift is not a constant
// pixel offset, so the per-cell shift + linear interpolation
// (fast_shift / fast_interp_new, SOAP_integration.cu:232-281) is evaluated in
// gather form for every (cell, pixel): pixel j takes the source index
// i(j) = max{i : ceil(i (1 + fbeta) + fbeta lambda_0 / step) <= j} and the
// reference's interpolation expression at i.  Cells are processed per mu bin
// from bin-sorted cell lists, with the bin's seed-row segments and the
// wavelengths of the tile staged in LDS.  The gathered value depends on a cell
// only through its shift, so each run of cells with bitwise-equal shifts in a
// bin's list (a disk column under solid-body rotation) is gathered once with the
// run's summed weights.  The convolution (conv_inst,
// SOAP_resolution.cu:76-95) has per-pixel Gaussian widths; the mask CCF uses
// the reference's literal index arithmetic (CCF_func.py:45-91).
#include <hip/hip_runtime.h>
#include <math.h>

#include "soap_internal.h"

namespace soap {

constexpr int kLTPB = 256;
constexpr int kQuietSets = 16;  // bin sets of the quiet-star gather (blocks per tile)

// ------------------------------------------------------------ cell lists
// Stable compaction of the block's predicate over 256 candidates: returns this
// thread's slot among the block's selected candidates, *total the count.
__device__ __forceinline__ int block_compact(bool pred, int *s_wave, int *total) {
  unsigned long long m = __ballot(pred);
  int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int before = __popcll(m & ((1ull << lane) - 1ull));
  if (lane == 0) s_wave[wv] = __popcll(m);
  __syncthreads();
  int off = 0, tot = 0;
  for (int w = 0; w < (int)(blockDim.x >> 6); w++) {
    if (w < wv) off += s_wave[w];
    tot += s_wave[w];
  }
  __syncthreads();
  *total = tot;
  return off + before;
}

// Exclusive block-wide prefix sum of v (in thread order); *total = the block's sum.
__device__ __forceinline__ int block_scan_excl(int v, int *s_wave, int *total) {
  int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  int x = v;
  for (int o = 1; o < 64; o <<= 1) {
    int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) s_wave[wv] = x;
  __syncthreads();
  int off = 0, tot = 0;
  for (int w = 0; w < (int)(blockDim.x >> 6); w++) {
    if (w < wv) off += s_wave[w];
    tot += s_wave[w];
  }
  __syncthreads();
  *total = tot;
  return off + x - v;
}

// Cell lists by (phase, mu bin), each in map order: the quiet disk (one phase whose
// box is the whole map; disk cells of bin k, entry = index) and the active regions
// (phase p's scan box; cells of bin k that classify as spot or facula, entry =
// index | type << 30).  Three passes over blocks (p, k, ch), ch = chunk of kChunk
// box cells in map order: count, per-phase offsets, write.
constexpr int kChunk = 4096;

// Box cells c, c + kLTPB, ... of phase p: the position is carried along (a 64-bit division per
// cell and bin before: count 51 -> 45 us, write 78 -> 68 us over 25 phases of
// the production disk).
struct CellWalk {
  int iy, iz, z0, nz, dy, dz;
  __device__ __forceinline__ CellWalk(const CellSrc &s, int p, long c) {
    int y0 = 0;
    z0 = 0;
    nz = s.grid;
    if (s.box) {
      y0 = s.box[p * 4];
      z0 = s.box[p * 4 + 2];
      nz = s.box[p * 4 + 3] - z0;
    }
    const int n = nz > 0 ? nz : 1;  // an empty box has no cells
    iy = y0 + (int)(c / n);
    iz = z0 + (int)(c % n);
    dy = kLTPB / n;
    dz = kLTPB % n;
  }
  __device__ __forceinline__ void next() {
    iy += dy;
    iz += dz;
    if (iz >= z0 + nz) {
      iz -= nz;
      iy++;
    }
  }
};

// entry of the cell for bin k, or -1
__device__ __forceinline__ int cell_entry(const CellSrc &s, int p, int k, const CellWalk &w) {
  int idx = w.iy * s.grid + w.iz;
  if (s.region[idx] != k) return -1;
  if (!s.box) return (s.limb[idx] == -999.0 && s.delta[idx] == -999.0) ? -1 : idx;
  double rc;
  int ty = classify_cell(w.iy, w.iz, 2. / s.grid, s.geo, s.geo_off[p], s.geo_off[p + 1], &rc);
  return ty >= 0 ? (idx | (ty << 30)) : -1;
}

__device__ __forceinline__ long cell_box_size(const CellSrc &s, int p) {
  if (!s.box) return (long)s.grid * s.grid;
  const int32_t *bx = s.box + p * 4;
  return (long)(bx[1] - bx[0]) * (bx[3] - bx[2]);
}

__global__ __launch_bounds__(kLTPB) void k_cells_count(CellSrc s, int32_t *cnt) {
  __shared__ int s_n;
  long b = blockIdx.x;
  int ch = (int)(b % s.nch);
  long pk = b / s.nch;
  int k = (int)(pk % s.n_mu), p = (int)(pk / s.n_mu);
  long lo = (long)ch * kChunk, nbox = cell_box_size(s, p);
  long hi = lo + kChunk < nbox ? lo + kChunk : nbox;
  if (threadIdx.x == 0) s_n = 0;
  __syncthreads();
  int n = 0;
  CellWalk w(s, p, lo + threadIdx.x);
  for (long c = lo + threadIdx.x; c < hi; c += kLTPB, w.next()) n += cell_entry(s, p, k, w) >= 0;
  if (n) atomicAdd(&s_n, n);
  __syncthreads();
  if (threadIdx.x == 0) cnt[b] = s_n;
}

// Phase p = blockIdx.x: exclusive offsets over (k, ch) within the phase, in place;
// bin_off[p][k] = offset of (k, 0), bin_off[p][n_mu] = the phase's total.
__global__ __launch_bounds__(kLTPB) void k_cells_offsets(int n_mu, int nch, int32_t *cnt, int32_t *bin_off) {
  __shared__ int s_wave[kLTPB / 64];
  int p = blockIdx.x;
  long ne = (long)n_mu * nch;
  int32_t *c = cnt + (long)p * ne;
  long per = (ne + kLTPB - 1) / kLTPB;
  long e0 = threadIdx.x * per, e1 = e0 + per < ne ? e0 + per : ne;
  int sum = 0;
  for (long e = e0; e < e1; e++) sum += c[e];
  int tot;
  int run = block_scan_excl(sum, s_wave, &tot);
  for (long e = e0; e < e1; e++) {
    int v = c[e];
    c[e] = run;
    if (e % nch == 0) bin_off[(long)p * (n_mu + 1) + e / nch] = run;
    run += v;
  }
  if (threadIdx.x == 0) bin_off[(long)p * (n_mu + 1) + n_mu] = tot;
}

__global__ __launch_bounds__(kLTPB) void k_cells_write(CellSrc s, const int32_t *off, const int64_t *list_off,
                                                       int32_t *cells) {
  __shared__ int s_wave[kLTPB / 64];
  long b = blockIdx.x;
  int ch = (int)(b % s.nch);
  long pk = b / s.nch;
  int k = (int)(pk % s.n_mu), p = (int)(pk / s.n_mu);
  long lo = (long)ch * kChunk, nbox = cell_box_size(s, p);
  if (lo >= nbox) return;  // uniform over the block
  long hi = lo + kChunk < nbox ? lo + kChunk : nbox;
  int32_t *out = cells + (list_off ? list_off[p] : 0) + off[b];
  int run = 0;
  CellWalk w(s, p, lo + threadIdx.x);
  for (long c0 = lo; c0 < hi; c0 += kLTPB, w.next()) {
    long c = c0 + threadIdx.x;
    int e = c < hi ? cell_entry(s, p, k, w) : -1;
    int tot;
    int slot = block_compact(e >= 0, s_wave, &tot);
    if (e >= 0) out[run + slot] = e;
    run += tot;
  }
}

hipError_t launch_cell_lists(const CellSrc &src, const int64_t *list_off, int32_t *cnt, int32_t *cells,
                             int32_t *bin_off, hipStream_t st) {
  long blocks = (long)src.n_phase * src.n_mu * src.nch;
  if (blocks == 0) return hipSuccess;
  if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
  k_cells_count<<<(unsigned)blocks, kLTPB, 0, st>>>(src, cnt);
  k_cells_offsets<<<src.n_phase, kLTPB, 0, st>>>(src.n_mu, src.nch, cnt, bin_off);
  k_cells_write<<<(unsigned)blocks, kLTPB, 0, st>>>(src, cnt, list_off, cells);
  return hipGetLastError();
}

int cell_list_chunks(long box_cells) { return (int)((box_cells + kChunk - 1) / kChunk); }

// mu of a cell from its grid position (as classify_cell computes it)
__device__ __forceinline__ double cell_rcos(int idx, int grid) {
#pragma clang fp contract(off)
  int iy = idx / grid, iz = idx % grid;
  double dg = 2. / grid;
  double y = -1. + iy * dg, z = -1. + iz * dg;
  return sqrt(1. - (y * y + z * z));
}

// ------------------------------------------------------------ shift on a linear grid
struct LinShift {
  bool ident;            // delta == 0: the row itself (SOAP_integration.cu:262-265)
  double opf, fl, c1;    // 1 + fbeta, fbeta lambda_0 / step, 1 - sqrt((1+beta)/(1-beta))
  double rinv;           // 1 / opf (first guess of the gather index only)
};

__device__ __forceinline__ LinShift lin_shift(double delta_kms, double lambda0, double step) {
#pragma clang fp contract(off)
  LinShift s;
  s.ident = delta_kms == 0.0;
  double beta = delta_kms * 1000. / kC;
  double sq = sqrt((1 + beta) / (1 - beta));
  double fbeta = -1 * (1 - sq);
  s.c1 = 1 - sq;
  s.opf = 1 + fbeta;
  s.fl = fbeta * lambda0 / step;
  s.rinv = 1 / s.opf;
  return s;
}

__device__ __forceinline__ LinShift group_shift(const CONSTANT LinGroup &g) {
  LinShift s;
  s.ident = g.ident != 0;
  s.opf = g.opf;
  s.fl = g.fl;
  s.c1 = g.c1;
  s.rinv = g.rinv;
  return s;
}

// a record's shift is none: its fl is 0 (either sign), known on the scalar unit
__device__ __forceinline__ bool no_shift(double fl) { return (__double_as_longlong(fl) << 1) == 0; }

// lambda + Delta_lambda(delta 1000, lambda) (SOAP_integration.cu:240)
__device__ __forceinline__ double lin_lshift(double lam, const LinShift &s) {
#pragma clang fp contract(off)
  return lam + -1 * lam * s.c1;
}

// max{i : ceil(i (1+fbeta) + fbeta lambda_0/step) <= j}: a first guess from the
// reciprocal, then the reference's own expression decides
// (32-bit indices: the launchers refuse grids of 2^31 - 2^12 pixels or more)
__device__ __forceinline__ int lin_gather_index(int j, const LinShift &s) {
#pragma clang fp contract(off)
  int i = (int)floor((j - s.fl) * s.rinv);
  for (int it = 0; it < 8 && (int)ceil(i * s.opf + s.fl) > j; it++) i--;
  for (int it = 0; it < 8 && (int)ceil((i + 1) * s.opf + s.fl) <= j; it++) i++;
  return i;
}

// Staged tile: source indices [base, base + span) of the rows and the wavelengths
// (linear continuation outside the grid, rows 0 there).  The host sizes the window
// from the extreme shifts on the disk with 3-pixel margins on both sides, so every
// i, i + 1 a gather of the tile reads lies inside it; local() clamps all the same,
// so that no index can leave the LDS arrays.
__device__ __forceinline__ int tile_local(int i, int base, int span) {
  int li = i - base;
  return li < 0 ? 0 : (li > span - 2 ? span - 2 : li);
}
constexpr long kLinMaxN = 0x7fffffffL - 4096;

// Window index li and interpolation weight t of pixel j for a shift: i(j) and the
// reference's (lambda_j - ls_i) / (ls_{i+1} - ls_i) of the shifted wavelengths.
// The gathers are bound by vector instructions, so both are formed with few: the index
// is the floor of the inverse map, which the reference's own expression can change only
// where that lies within rounding of a whole number (below 1e-6 at the largest index; the
// exact search runs within 1e-5 of one).  UNI (a grid whose differences are the step to
// 1e-8, as the 0.005 A format is): the reciprocal of ls_{i+1} - ls_i is one Newton step
// from 1 / (step (1 + fbeta)), relative error below 1e-16, in the place of a division.
// Series at the production disk, 100,000 pixels: quiet gather 1304 -> 1079 us, active
// 1315 -> 1004 us.
template <bool UNI>
__device__ __forceinline__ void lin_locate(int j, double lam_j, const LinShift &s, double inv_step, const double *wl,
                                           int base, int span, int &li, double &t) {
  const double est = fma((double)j, s.rinv, -(s.fl * s.rinv)), whole = floor(est), fr = est - whole;
  int i = (int)whole;
  if (!(fr > 1e-5 && fr < 1 - 1e-5)) i = lin_gather_index(j, s);
  li = tile_local(i, base, span);
  const double w0 = wl[li], w1 = wl[li + 1];
  if (UNI) {
    const double ls0 = fma(-w0, s.c1, w0), den = fma(-w1, s.c1, w1) - ls0;
    const double r0 = s.rinv * inv_step, r = fma(r0, fma(-den, r0, 1.0), r0);
    t = (lam_j - ls0) * r;
  } else {
    const double ls0 = lin_lshift(w0, s), ls1 = lin_lshift(w1, s);
    t = (lam_j - ls0) / (ls1 - ls0);
  }
}

__device__ void lin_stage(double *dst, const double *grow, long base, int span, long n) {
  for (int e = threadIdx.x; e < span; e += blockDim.x) {
    long i = base + e;
    dst[e] = (i >= 0 && i < n) ? grow[i] : 0.0;
  }
}

__device__ void lin_stage_wave(double *dst, const double *wave, long base, int span, long n) {
  for (int e = threadIdx.x; e < span; e += blockDim.x) {
    long i = base + e;
    double v;
    if (i < 0)
      v = wave[0] + (double)i * (wave[1] - wave[0]);
    else if (i >= n)
      v = wave[n - 1] + (double)(i - (n - 1)) * (wave[n - 1] - wave[n - 2]);
    else
      v = wave[i];
    dst[e] = v;
  }
}

// ------------------------------------------------------------ shift groups
// Cell c of a segment starts a new group unless the previous cell has the same
// population and a bitwise-equal shift (facula cells in solar mode always start
// one: their intensity depends on the cell's own mu).
__device__ __forceinline__ bool starts_group(const int32_t *cells, long c, const double *delta, int split_fac) {
  int e = cells[c], ep = cells[c - 1];
  int ty = e >> 30;
  if (ty != (ep >> 30) || (split_fac && ty == 1)) return true;
  return delta[e & 0x3fffffff] != delta[ep & 0x3fffffff];
}

// Segment (p, k) = blockIdx.x of a bin-sorted cell list: its runs of equal shift
// become groups with w = sum L and w2 = sum (1 + LB) L over the run, stored from
// the segment's start.  sum_c L_c v(delta) = v(delta) sum_c L_c, so the gathers
// over groups equal the per-cell sums of SOAP_integration.cu:285-307,392-447
// (and itot's, SOAP_initialize.cu:339-395) up to rounding.  The run sums come from
// a segmented scan over each chunk of TPB cells (restarting at run heads, in a fixed
// order: within the waves, then over them) plus the open run carried from the chunk
// before.  25 phases of the production disk: 70 -> 63 us (a scan of ten steps
// through LDS, two barriers each, and the heads' divisions in every wave, before).
template <int TPB>
__global__ __launch_bounds__(TPB) void k_lin_groups(const int32_t *cells, const int64_t *list_off,
                                                    const int32_t *bin_off, int n_mu, const double *delta,
                                                    const double *limb, const double *lbm, double lambda0,
                                                    double step, int split_fac, LinGroup *groups, int32_t *g_n) {
#pragma clang fp contract(off)
  __shared__ int s_wave[TPB / 64];
  __shared__ double s_w[TPB / 64], s_w2[TPB / 64];  // the waves' open runs
  __shared__ int s_f[TPB / 64];                     // a head in the wave
  __shared__ double s_carry[2];
  __shared__ int s_head[TPB];
  const int tid = threadIdx.x;
  int sg = blockIdx.x, p = sg / n_mu, k = sg % n_mu;
  long base = list_off ? list_off[p] : 0;
  const int32_t *bo = bin_off + (long)p * (n_mu + 1);
  long c0 = base + bo[k], c1 = base + bo[k + 1];
  LinGroup *gs = groups + c0;
  int run = 0;                  // groups begun before this chunk
  double cw = 0.0, cw2 = 0.0;   // sums of the run open at the chunk's start
  for (long cb = c0; cb < c1; cb += TPB) {
    long c = cb + tid;
    bool in = c < c1;
    bool head = in && (c == c0 || starts_group(cells, c, delta, split_fac));
    bool last = in && (c + 1 == c1 || starts_group(cells, c + 1, delta, split_fac));
    int e = in ? cells[c] : 0;
    double v = 0.0, v2 = 0.0;
    if (in) {
      int id = e & 0x3fffffff;
      v = limb[id];
      v2 = (1 + lbm[id]) * v;
    }
    int tot;
    int before = block_compact(head, s_wave, &tot);  // heads before this cell in the chunk
    int f = head;
    for (int o = 1; o < 64; o <<= 1) {
      const double u = __shfl_up(v, o, 64), u2 = __shfl_up(v2, o, 64);
      const int uf = __shfl_up(f, o, 64);
      if ((tid & 63) >= o && !f) {
        v = u + v;
        v2 = u2 + v2;
        f = uf;
      }
    }
    if ((tid & 63) == 63) {
      s_w[tid >> 6] = v;
      s_w2[tid >> 6] = v2;
      s_f[tid >> 6] = f;
    }
    __syncthreads();
    if (!f) {  // no head at or before this cell in the wave: the waves before it, back to the carried run
      double b1 = cw, b2 = cw2;
      for (int w = 0; w < tid >> 6; w++) {
        b1 = s_f[w] ? s_w[w] : b1 + s_w[w];
        b2 = s_f[w] ? s_w2[w] : b2 + s_w2[w];
      }
      v = b1 + v;
      v2 = b2 + v2;
    }
    if (head) s_head[before] = e;
    if (last) {  // the run's group: the last head at or before this cell
      LinGroup &g = gs[run + before + (head ? 1 : 0) - 1];
      g.w = v;
      g.w2 = v2;
    }
    long lastc = (cb + TPB < c1 ? cb + TPB : c1) - 1;
    if (c == lastc) {
      s_carry[0] = last ? 0.0 : v;
      s_carry[1] = last ? 0.0 : v2;
    }
    __syncthreads();
    for (int h = tid; h < tot; h += TPB) {  // the heads' shifts, closed up: few waves take the divisions
      LinShift sh = lin_shift(delta[s_head[h] & 0x3fffffff], lambda0, step);
      LinGroup &g = gs[run + h];
      g.opf = sh.opf;
      g.fl = sh.fl;
      g.c1 = sh.c1;
      g.rinv = sh.rinv;
      g.e = s_head[h];
      g.ident = sh.ident ? 1 : 0;
      g.pad[0] = g.pad[1] = 0;
    }
    cw = s_carry[0];
    cw2 = s_carry[1];
    run += tot;
  }
  if (tid == 0) g_n[sg] = run;
}

hipError_t launch_lin_groups(const int32_t *cells, const int64_t *list_off, const int32_t *bin_off, int n_phase,
                             int n_mu, const double *delta, const double *limb, const double *lbm, double lambda0,
                             double step, int split_fac, LinGroup *groups, int32_t *g_n, hipStream_t s) {
  long nseg = (long)n_phase * n_mu;
  if (nseg == 0) return hipSuccess;
  if (nseg > 0x7fffffffL) return hipErrorInvalidValue;
  // 1024-cell chunks: the time goes to the longest segments (the active cells of
  // a phase crowd into the few bins its regions cover)
  k_lin_groups<1024><<<(unsigned)nseg, 1024, 0, s>>>(cells, list_off, bin_off, n_mu, delta, limb, lbm, lambda0, step,
                                                     split_fac, groups, g_n);
  return hipGetLastError();
}

// Quiet star on a linear grid: out[0][j] = sum_cells limb Shift(Sq_k)(j), out[1] for
// the SED cube (itot's cell loop, SOAP_initialize.cu:339-395), per tile of kLTPB
// pixels, bins outer, shift groups of the bin inner.  Block (tile, s) takes bins
// s, s + ns, ... and writes its partial sums to part[s][2][n]; k_quiet_sum adds
// the ns partials in order.
template <bool UNI>
__global__ __launch_bounds__(kLTPB) void k_gather_quiet_linear(LinArgs a, const double *q, const double *qs,
                                                               const LinGroup *groups, const int32_t *bin_off,
                                                               const int32_t *g_n, double *part) {
  extern __shared__ double lds[];  // rows [2][span], wave [span]
  const int ns = gridDim.y, set = blockIdx.y;
  const int j0 = blockIdx.x * kLTPB;
  const int j = j0 + threadIdx.x;
  const int base = j0 + a.off_lo;
  const int span = a.span;
  double *rw = lds, *wl = lds + 2 * span;
  lin_stage_wave(wl, a.wave, base, span, a.n);
  const int lj = j - base;  // inside the window: -off_lo .. kLTPB - 1 - off_lo
  double lam_j = a.wave[j < a.n ? j : a.n - 1];
  double acc_q = 0.0, acc_s = 0.0;
  const CONSTANT LinGroup *gp = gc(groups);
  for (int k = set; k < a.n_mu; k += ns) {
    int c0 = bin_off[k], ng = g_n[k];
    if (ng == 0) continue;  // uniform
    const double *gq = q + (long)k * a.n, *gs = qs + (long)k * a.n;
    __syncthreads();
    lin_stage(rw, gq, base, span, a.n);
    lin_stage(rw + span, gs, base, span, a.n);
    __syncthreads();
    for (int c = c0; c < c0 + ng; c++) {
      const CONSTANT LinGroup &G = gp[c];
      double L = G.w;
      LinShift s = group_shift(G);
      if (s.ident) {
        acc_q += rw[lj] * L;
        acc_s += rw[span + lj] * L;
        continue;
      }
      int li;
      double t;
      lin_locate<UNI>(j, lam_j, s, a.inv_step, wl, base, span, li, t);
      const double a0 = rw[li], a1 = rw[li + 1];
      const double b0 = rw[span + li], b1 = rw[span + li + 1];
      acc_q = fma(fma(a1 - a0, t, a0), L, acc_q);
      acc_s = fma(fma(b1 - b0, t, b0), L, acc_s);
    }
  }
  if (j < a.n) {
    double *o = part + (long)set * 2 * a.n;
    o[j] = acc_q;
    o[a.n + j] = acc_s;
  }
}

__global__ __launch_bounds__(kLTPB) void k_quiet_sum(const double *part, int ns, long n2, double *out) {
  long j = (long)blockIdx.x * kLTPB + threadIdx.x;
  if (j >= n2) return;
  double acc = part[j];
  for (int t = 1; t < ns; t++) acc += part[(long)t * n2 + j];
  out[j] = acc;
}

int quiet_linear_sets(int n_mu) { return n_mu < kQuietSets ? n_mu : kQuietSets; }

hipError_t launch_gather_quiet_linear(const LinArgs &a, const double *q, const double *qs, const LinGroup *groups,
                                      const int32_t *bin_off, const int32_t *g_n, double *part, double *out,
                                      hipStream_t s) {
  size_t lds = (size_t)3 * a.span * sizeof(double);
  if (lds > 65536 || a.span < kLTPB || a.n_mu < 1 || a.n > kLinMaxN) return hipErrorInvalidValue;
  unsigned nb = (unsigned)((a.n + kLTPB - 1) / kLTPB);
  int ns = quiet_linear_sets(a.n_mu);
  if (a.uniform)
    k_gather_quiet_linear<true><<<dim3(nb, ns), kLTPB, lds, s>>>(a, q, qs, groups, bin_off, g_n, part);
  else
    k_gather_quiet_linear<false><<<dim3(nb, ns), kLTPB, lds, s>>>(a, q, qs, groups, bin_off, g_n, part);
  long n2 = 2 * a.n;
  k_quiet_sum<<<(unsigned)((n2 + kLTPB - 1) / kLTPB), kLTPB, 0, s>>>(part, ns, n2, out);
  return hipGetLastError();
}

// ------------------------------------------------------------ quiet star by columns
// Under solid-body rotation delta = y omega sin i is the same along a disk column
// in every mu bin, so the quiet star's shift groups are (bin, column) pairs that
// share their column's index and weight.  k_quiet_columns_maps lays them out as a
// table: per (bin set s, column iy) the weights of the set's kQColBins bins (0
// where the column does not meet the bin), a flag for columns with any weight, and
// the column's shift; k_quiet_columns_pack lists each set's columns with weight, and
// k_gather_quiet_cols computes the index and weight once per (pixel, column) for all
// bins of its set.
constexpr int kQColBins = 4;

// ------------------------------------------------------------ taps on a grid of rounded nodes
// Where the nodes are the grid lambda_0 + i step, rounded (LinArgs::nodes), a shift moves pixel j
// by x(j) = j c1 rinv - fl rinv, and cells share their source pixels: over a tile of 256 pixels,
// all cells of one whole part d and weight w sum to taps at d and d + 1 that are linear in the
// pixel, w (1 - x0 - x' (j - j0)) and w (x0 + x' (j - j0)).  A tile's sum over the cells is then a
// FIR of two coefficients per offset (the value at j0 and the slope) in place of one
// interpolation per pixel and cell: a thousand columns over some forty offsets.  Cells whose
// whole part changes inside the tile (1 % at 10 km/s) are interpolated one by one.  The quiet
// star of the production disk, 100,000 pixels: 1304 us a column at a time -> 75 us; bound by the
// LDS reads of the rows.  Against an 80-bit evaluation its largest error is half of the gather's
// (3.8e-13 and 7.3e-13 at 3001 pixels of 5000 A): that carries the rounding of each shifted
// wavelength.  (Rows of white noise, which lines sampled by this format are not: 0.5-1.2 times
// the gather's at 2 km/s and more, up to 5 times, 6e-11, below 0.2 km/s, where all columns fall
// within a pixel and the rounding of a node is not averaged.)  The active sums keep the gather's weights: they are sums over few cells, compared
// to 1e-12 with the reference's expression and its rounding, 2.6e-12 from these taps.
//  - The nodes' rounding is kept, to first order: a source pixel e from its place enters as the
//    row's value at the place (lin_stage_nodes), a pixel e from its place as its sum's slope
//    times e (node_shift).  What is left is second order, e / step ~ 1e-10 of these terms.
//  - Taps are summed as 64-bit whole numbers at a power of two fitted to the weights (tap_scale:
//    the sum of all |w| below 2^61; slopes, below 1 / 255 of their weight, at 2^8 times that), so
//    that the order of the LDS atomics does not show: 2^-61 of the weights' sum per cell.
//  - A tile with a value that is not finite takes every cell one by one: a tap of 0 must not
//    meet a pixel that no cell reads.
constexpr int kTapPad = 16;  // steps of a FIR turn: taps and rows are padded with zeros

__device__ __forceinline__ double tap_scale(double sum) {  // 0: not finite
  if (!(sum < HUGE_VAL)) return 0.0;
  if (sum == 0.0) return 1.0;
  const int e = 60 - ilogb(sum);
  return ldexp(1.0, e < 1000 ? e : 1000);
}
__device__ __forceinline__ double block_sum(double v, double *s_sum) {  // kLTPB threads, in a fixed order
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = v;
  __syncthreads();
  double all = s_sum[0];
  for (int w = 1; w < kLTPB / 64; w++) all += s_sum[w];
  __syncthreads();
  return all;
}
__device__ __forceinline__ int lin_row_len(int span) { return span + kTapPad; }
__device__ __forceinline__ int lin_tap_len(int span) { return span - kLTPB + kTapPad; }
inline size_t lin_tap_bytes(int rows, int sums, int span) {  // rows and taps, or node_shift's sums
  const size_t fir = (size_t)rows * (span + kTapPad) + 8 * (size_t)(span - kLTPB + kTapPad);
  const size_t shift = (size_t)sums * kLTPB;
  return (fir > shift ? fir : shift) * sizeof(double);
}

// How far node i lies from lambda_0 + i step, in steps.
__device__ __forceinline__ double node_error(const LinArgs &a, long i) {
  return fma(-(double)i, a.step, a.wave[i] - a.lambda0) * a.inv_step;
}

// The rows' values at the grid's places (zeros outside the grid and in the padding); true: one is
// not finite.
template <int R>
__device__ __forceinline__ bool lin_stage_nodes(const LinArgs &a, double *dst, const double *const (&g)[R], long base) {
  const int rl = lin_row_len(a.span);
  bool bad = false;
  for (int e = threadIdx.x; e < rl; e += kLTPB) {
    const long i = base + e;
    const bool in = e < a.span && i >= 0 && i < a.n;
    const long ic = in ? i : 0, up = ic + 1 < a.n ? ic + 1 : ic, dn = ic > 0 ? ic - 1 : ic;
    const double h = -0.5 * node_error(a, ic);
#pragma unroll
    for (int r = 0; r < R; r++) {
      double v = 0.0;
      if (in && g[r]) {
        v = g[r][ic];
        const double x = fma(h, g[r][up] - g[r][dn], v);
        if (isfinite(x)) v = x;
        bad |= !isfinite(v);
      }
      dst[r * rl + e] = v;
    }
  }
  return bad;
}

// sums[r] (pixel j of every thread) moved by the pixel's node error, from the slope of the
// neighbours' sums in the block; buf: R * kLTPB doubles of LDS that nobody reads any more.
template <int R>
__device__ __forceinline__ void node_shift(const LinArgs &a, long j, double (&sums)[R], double *buf) {
  const int t = threadIdx.x;
#pragma unroll
  for (int r = 0; r < R; r++) buf[r * kLTPB + t] = sums[r];
  __syncthreads();
  if (j >= a.n) return;
  const int up = t + 1 < kLTPB && j + 1 < a.n ? t + 1 : t, dn = t > 0 ? t - 1 : t;
  if (up == dn) return;
  const double h = node_error(a, j) / (up - dn);
#pragma unroll
  for (int r = 0; r < R; r++) {
    const double x = fma(h, buf[r * kLTPB + up] - buf[r * kLTPB + dn], sums[r]);
    if (isfinite(x)) sums[r] = x;
  }
}

// The tile's part of one cell: tap index e and the weight's fraction t at j0, slope t1 per pixel;
// false where the whole part changes inside the tile or lies outside the window.
struct LinTap {
  int e;
  double t, t1;
};
__device__ __forceinline__ bool lin_tap(const LinArgs &a, int j0, double fl, double c1, double rinv, LinTap &p) {
  p.t1 = c1 * rinv;
  const double x = fma((double)j0, p.t1, -(fl * rinv)), d = floor(x);
  p.t = x - d;
  p.e = (int)d - a.off_lo;
  return floor(fma((double)(kLTPB - 1), p.t1, x)) == d && p.e >= 0 && p.e < a.span - kLTPB;
}
// One cell at pixel j: window index and fraction (a cell whose taps are not shared).
__device__ __forceinline__ void lin_place(const LinArgs &a, int j, int base, double fl, double c1, double rinv, int &li,
                                          double &t) {
  const double x = fma((double)j, c1 * rinv, -(fl * rinv)), d = floor(x);
  t = x - d;
  li = tile_local(j + (int)d, base, a.span);
}
// w at tap p, scaled: taps[e] (values) and taps[nt + e] (slopes)
__device__ __forceinline__ void tap_add(long long *taps, int nt, const LinTap &p, double w, double scale) {
  const double v = w * scale;
  const long long all = (long long)rint(v), up = (long long)rint(v * p.t), sl = (long long)rint(v * p.t1 * 256.0);
  atomicAdd((unsigned long long *)taps + p.e, (unsigned long long)(all - up));
  atomicAdd((unsigned long long *)taps + p.e + 1, (unsigned long long)up);
  atomicAdd((unsigned long long *)taps + nt + p.e, (unsigned long long)-sl);
  atomicAdd((unsigned long long *)taps + nt + p.e + 1, (unsigned long long)sl);
}

// F += t(lane N of this lane's row of 16) x, one rounding each: the coefficients of 16 steps in
// one register.  Two wait states lie between a vector write of t and its broadcast read.
#define SOAP_BC(F, T, X) "v_fmac_f64_dpp %[" F "], %[" T "], %[" X "] row_newbcast:%[n] row_mask:0xf bank_mask:0xf\n\t"
template <int N>
__device__ __forceinline__ void bc_bins(double &qa, double &qb, double &sa, double &sb, const double (&t)[8],
                                        const double (&x)[8]) {
  asm("s_nop 1\n\t" SOAP_BC("qa", "t0", "x0") SOAP_BC("qb", "t1", "x0") SOAP_BC("sa", "t0", "x1")
          SOAP_BC("sb", "t1", "x1") SOAP_BC("qa", "t2", "x2") SOAP_BC("qb", "t3", "x2") SOAP_BC("sa", "t2", "x3")
              SOAP_BC("sb", "t3", "x3") SOAP_BC("qa", "t4", "x4") SOAP_BC("qb", "t5", "x4") SOAP_BC("sa", "t4", "x5")
                  SOAP_BC("sb", "t5", "x5") SOAP_BC("qa", "t6", "x6") SOAP_BC("qb", "t7", "x6")
                      SOAP_BC("sa", "t6", "x7") SOAP_BC("sb", "t7", "x7")
      : [qa] "+v"(qa), [qb] "+v"(qb), [sa] "+v"(sa), [sb] "+v"(sb)
      : [t0] "v"(t[0]), [t1] "v"(t[1]), [t2] "v"(t[2]), [t3] "v"(t[3]), [t4] "v"(t[4]), [t5] "v"(t[5]), [t6] "v"(t[6]),
        [t7] "v"(t[7]), [x0] "v"(x[0]), [x1] "v"(x[1]), [x2] "v"(x[2]), [x3] "v"(x[3]), [x4] "v"(x[4]), [x5] "v"(x[5]),
        [x6] "v"(x[6]), [x7] "v"(x[7]), [n] "n"(N));
}
#undef SOAP_BC

// step(integral_constant<int, D>) for D = 0 .. 15
template <int D = 0, class F>
__device__ __forceinline__ void steps16(F &&step) {
  if constexpr (D < kTapPad) {
    step(std::integral_constant<int, D>{});
    steps16<D + 1>(step);
  }
}

// The columns of set blockIdx.x with any weight, in order, as records of the shift and the
// weights, with the bins' fixed-point scales (tap_scale).
struct alignas(16) QuietCol {
  double opf, fl, c1, rinv, w[kQColBins];
};
__global__ __launch_bounds__(kLTPB) void k_quiet_columns_pack(int grid, const double *colw, const int32_t *colf,
                                                              const LinGroup *cols, QuietCol *out, double *scale,
                                                              int32_t *count) {
  __shared__ int s_wave[kLTPB / 64];
  __shared__ double s_sum[kLTPB / 64];
  const int set = blockIdx.x;
  double sum[kQColBins] = {};
  QuietCol *o = out + (long)set * grid;
  int n = 0;
  for (int c0 = 0; c0 < grid; c0 += kLTPB) {
    const int iy = c0 + threadIdx.x;
    const bool use = iy < grid && colf[(long)set * grid + iy];
    int tot;
    const int at = n + block_compact(use, s_wave, &tot);
    if (use) {
      const LinGroup &g = cols[iy];
      QuietCol q{g.opf, g.fl, g.c1, g.rinv, {}};
      for (int kk = 0; kk < kQColBins; kk++) {
        q.w[kk] = colw[((long)set * grid + iy) * kQColBins + kk];
        sum[kk] += fabs(q.w[kk]);
      }
      o[at] = q;
    }
    n += tot;
  }
  for (int kk = 0; kk < kQColBins; kk++) {
    const double all = block_sum(sum[kk], s_sum);
    if (threadIdx.x == 0) scale[set * kQColBins + kk] = tap_scale(all);
  }
  if (threadIdx.x == 0) count[set] = n;
}

// The same table straight from the disk maps: block = column iy (one wave), the
// lanes over the column's cells; per bin, each lane sums its cells (z = lane,
// lane + 64, ...) in its own LDS slot, in one pass over the cells, and a fixed butterfly
// adds the 64 partials (one pass per bin before: 68 -> 25 us at 1000 x 1000 cells, 20 bins).  The column's shift
// comes from its first disk cell.
constexpr int kColPass = 32;  // bins whose lane sums are held in LDS together
__global__ __launch_bounds__(64) void k_quiet_columns_maps(const double *limb, const double *delta,
                                                           const int32_t *region, int n_mu, int grid, double lambda0,
                                                           double step, double *colw, int32_t *colf,
                                                           LinGroup *cols) {
#pragma clang fp contract(off)
  __shared__ double s_bin[kColPass][64];
  const int iy = blockIdx.x, lane = threadIdx.x;
  const long row = (long)iy * grid;
  const int ns = (n_mu + kQColBins - 1) / kQColBins;
  int first = -1;
  for (int z0 = 0; z0 < grid && first < 0; z0 += 64) {
    const int iz = z0 + lane;
    const bool disk = iz < grid && !(limb[row + iz] == -999.0 && delta[row + iz] == -999.0);
    const unsigned long long m = __ballot(disk);
    if (m) first = z0 + __ffsll((long long)m) - 1;
  }
  for (int k0 = 0; k0 < ns * kQColBins; k0 += kColPass) {
    for (int kk = 0; kk < kColPass; kk++) s_bin[kk][lane] = 0.0;
    for (int z0 = 0; z0 < grid; z0 += 64) {
      if (z0 + lane >= grid) break;
      const long idx = row + z0 + lane;
      const int kk = region[idx] - k0;
      const double l = limb[idx];
      if (kk >= 0 && kk < kColPass && !(l == -999.0 && delta[idx] == -999.0)) s_bin[kk][lane] += l;
    }
    for (int s = k0 / kQColBins; s < ns && s * kQColBins < k0 + kColPass; s++) {
      int any = 0;
      for (int kk = 0; kk < kQColBins; kk++) {
        const int k = s * kQColBins + kk;
        double w = k < n_mu ? s_bin[k - k0][lane] : 0.0;
        for (int o = 32; o > 0; o >>= 1) w += __shfl_xor(w, o, 64);
        any |= w != 0.0;
        if (lane == 0) colw[((long)s * grid + iy) * kQColBins + kk] = w;
      }
      if (lane == 0) colf[(long)s * grid + iy] = any;
    }
  }
  if (lane == 0) {
    LinGroup g{};
    if (first >= 0) {
      LinShift sh = lin_shift(delta[row + first], lambda0, step);
      g.opf = sh.opf;
      g.fl = sh.fl;
      g.c1 = sh.c1;
      g.rinv = sh.rinv;
      g.e = (int)(row + first);
      g.ident = sh.ident ? 1 : 0;
    } else {  // no disk cell in this column: an identity shift, never used
      g.opf = 1.0;
      g.rinv = 1.0;
      g.ident = 1;
    }
    cols[iy] = g;
  }
}

// Block (tile, s): the rows of bins s * kQColBins .. + kQColBins - 1 staged
// together (rows of bins past n_mu staged as zeros, with weight 0); per column
// with weight, one gather index and weight for all of them.
template <bool UNI>
__global__ __launch_bounds__(kLTPB) void k_gather_quiet_cols(LinArgs a, const double *q, const double *qs,
                                                             const QuietCol *cols, const int32_t *count,
                                                             double *part) {
  extern __shared__ double lds[];  // rows [kQColBins][2][span], wave [span]
  const int set = blockIdx.y;
  const int j0 = blockIdx.x * kLTPB;
  const int j = j0 + threadIdx.x;
  const int base = j0 + a.off_lo;
  const int span = a.span;
  double *rw = lds, *wl = lds + 2 * kQColBins * span;
  lin_stage_wave(wl, a.wave, base, span, a.n);
  for (int kk = 0; kk < kQColBins; kk++) {
    int k = set * kQColBins + kk;
    double *dq = rw + (2 * kk) * span, *ds = dq + span;
    if (k < a.n_mu) {
      lin_stage(dq, q + (long)k * a.n, base, span, a.n);
      lin_stage(ds, qs + (long)k * a.n, base, span, a.n);
    } else {
      for (int e = threadIdx.x; e < 2 * span; e += blockDim.x) dq[e] = 0.0;
    }
  }
  __syncthreads();
  double lam_j = a.wave[j < a.n ? j : a.n - 1];
  double acc_q = 0.0, acc_s = 0.0;
  const QuietCol *cp = cols + (long)set * a.grid;
  // A record of no shift (the column through the rotation axis) has index j and weight exactly 0;
  // still only the row's own pixel is read into it (its neighbour may not be finite).
  const int m = gc(count)[set];
  for (int c = 0; c < m; c++) {
    const CONSTANT double *r = gc((const double *)(cp + c));
    const LinShift s{false, r[0], r[1], r[2], r[3]};
    int li;
    double t;
    lin_locate<UNI>(j, lam_j, s, a.inv_step, wl, base, span, li, t);
    double q0 = 0.0, q1 = 0.0, s0 = 0.0, s1 = 0.0;  // the bins' weighted sums at both ends of the interval
    const bool own = no_shift(s.fl);
#pragma unroll
    for (int kk = 0; kk < kQColBins; kk++) {
      const double *dq = rw + (2 * kk) * span, *ds = dq + span, w = r[4 + kk];
      q0 = fma(dq[li], w, q0);
      q1 = fma(own ? dq[li] : dq[li + 1], w, q1);
      s0 = fma(ds[li], w, s0);
      s1 = fma(own ? ds[li] : ds[li + 1], w, s1);
    }
    acc_q += fma(q1 - q0, t, q0);
    acc_s += fma(s1 - s0, t, s0);
  }
  if (j < a.n) {
    double *o = part + (long)set * 2 * a.n;
    o[j] = acc_q;
    o[a.n + j] = acc_s;
  }
}

// The same sums through taps (above): block (tile, s), the columns over the lanes (neighbouring
// lanes a 64th of the columns apart, so that their atomics seldom meet), then the FIR of the
// bins' rows.
__global__ __launch_bounds__(kLTPB) void k_fir_quiet_cols(LinArgs a, const double *q, const double *qs,
                                                          const QuietCol *cols, const double *scale,
                                                          const int32_t *count, double *part) {
  extern __shared__ double lds[];  // rows [kQColBins][2][rl], taps [kQColBins][2][nt]
  __shared__ unsigned long long s_mask[16];
  __shared__ int s_lo, s_hi;
  const int set = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int j0 = blockIdx.x * kLTPB, j = j0 + tid, base = j0 + a.off_lo;
  const int rl = lin_row_len(a.span), nt = lin_tap_len(a.span);
  double *rw = lds, *taps = lds + 2 * kQColBins * rl;
  long long *ti = (long long *)taps;
  const QuietCol *cp = cols + (long)set * a.grid;
  const int m = count[set];
  double sc[kQColBins];
  const double *g[2 * kQColBins];
  bool bad = false;
  for (int kk = 0; kk < kQColBins; kk++) {
    const int k = set * kQColBins + kk;
    sc[kk] = scale[set * kQColBins + kk];
    bad |= sc[kk] == 0.0;
    g[2 * kk] = k < a.n_mu ? q + (long)k * a.n : nullptr;
    g[2 * kk + 1] = k < a.n_mu ? qs + (long)k * a.n : nullptr;
  }
  for (int i = tid; i < 2 * kQColBins * nt; i += kLTPB) ti[i] = 0;
  if (tid == 0) s_lo = 0x7fffffff, s_hi = -1;
  bad |= lin_stage_nodes<2 * kQColBins>(a, rw, g, base);
  bad = __syncthreads_or(bad);
  double fq[2] = {}, fs[2] = {};
  const int stride = (m + 63) / 64;
  int lo = 0x7fffffff, hi = -1;
  for (int i0 = 0; i0 < stride; i0 += 16) {
    const int i1 = min(i0 + 16, stride);
    for (int it = i0 + wave; it < i1; it += kLTPB / 64) {
      const int c = lane * stride + it;
      bool one = false;
      if (c < m) {
        const QuietCol &r = cp[c];
        LinTap p;
        one = bad || !lin_tap(a, j0, r.fl, r.c1, r.rinv, p);
        if (!one) {
          lo = min(lo, p.e);
          hi = max(hi, p.e + 1);
#pragma unroll
          for (int kk = 0; kk < kQColBins; kk++)
            if (r.w[kk] != 0.0) tap_add(ti + 2 * kk * nt, nt, p, r.w[kk], sc[kk]);
        }
      }
      const unsigned long long ones = __ballot(one);
      if (lane == 0) s_mask[it - i0] = ones;
    }
    __syncthreads();
    for (int it = i0; it < i1; it++) {
      unsigned long long ones = s_mask[it - i0];
      while (ones) {  // the same for the whole block
        const int c = (__ffsll((long long)ones) - 1) * stride + it;
        ones &= ones - 1;
        const QuietCol &r = cp[c];
        int li;
        double t;
        lin_place(a, j, base, r.fl, r.c1, r.rinv, li, t);
        const int up = no_shift(r.fl) ? li : li + 1;
        double q0 = 0.0, q1 = 0.0, s0 = 0.0, s1 = 0.0;
#pragma unroll
        for (int kk = 0; kk < kQColBins; kk++) {
          const double *dq = rw + 2 * kk * rl, *ds = dq + rl, w = r.w[kk];
          q0 = fma(dq[li], w, q0);
          q1 = fma(dq[up], w, q1);
          s0 = fma(ds[li], w, s0);
          s1 = fma(ds[up], w, s1);
        }
        fq[0] += fma(q1 - q0, t, q0);
        fs[0] += fma(s1 - s0, t, s0);
      }
    }
    __syncthreads();
  }
  if (hi >= 0) {
    atomicMin(&s_lo, lo);
    atomicMax(&s_hi, hi);
  }
  for (int kk = 0; kk < kQColBins; kk++) {
    const double inv = 1.0 / (sc[kk] == 0.0 ? 1.0 : sc[kk]);  // a power of two
    for (int i = tid; i < nt; i += kLTPB) {
      const int at = 2 * kk * nt + i;
      taps[at] = (double)ti[at] * inv;
      taps[at + nt] = (double)ti[at + nt] * inv * 0x1p-8;
    }
  }
  __syncthreads();
  lo = s_lo;
  hi = s_hi;
  for (int e0 = lo; e0 <= hi; e0 += kTapPad) {
    double t[2 * kQColBins];
#pragma unroll
    for (int u = 0; u < 2 * kQColBins; u++) t[u] = taps[u * nt + e0 + (lane & 15)];
    const double *r = rw + tid + e0;
    steps16([&](auto D) {
      double x[2 * kQColBins];
#pragma unroll
      for (int u = 0; u < 2 * kQColBins; u++) x[u] = r[u * rl + D()];
      bc_bins<D()>(fq[0], fq[1], fs[0], fs[1], t, x);
    });
  }
  __syncthreads();
  double sums[2] = {fma((double)tid, fq[1], fq[0]), fma((double)tid, fs[1], fs[0])};
  node_shift<2>(a, j, sums, rw);
  if (j < a.n) {
    double *o = part + (long)set * 2 * a.n;
    o[j] = sums[0];
    o[a.n + j] = sums[1];
  }
}

size_t quiet_column_pack_bytes(int n_mu, int grid) {
  return (size_t)quiet_column_sets(n_mu) * (grid * sizeof(QuietCol) + kQColBins * sizeof(double) + sizeof(int32_t));
}

int quiet_column_sets(int n_mu) { return (n_mu + kQColBins - 1) / kQColBins; }

bool quiet_columns_fit(int span) { return (size_t)(2 * kQColBins + 1) * span * sizeof(double) <= 65536; }

hipError_t launch_gather_quiet_cols(const LinArgs &a, const double *q, const double *qs, const int32_t *region,
                                    double *colw, int32_t *colf, LinGroup *cols, void *pack, double *part,
                                    double *out, hipStream_t s) {
  size_t lds = (size_t)(2 * kQColBins + 1) * a.span * sizeof(double);
  if (lds > 65536 || a.span < kLTPB || a.n_mu < 1 || a.n > kLinMaxN || a.grid < 1) return hipErrorInvalidValue;
  k_quiet_columns_maps<<<(unsigned)a.grid, 64, 0, s>>>(a.limb, a.delta, region, a.n_mu, a.grid, a.lambda0, a.step,
                                                       colw, colf, cols);
  unsigned nb = (unsigned)((a.n + kLTPB - 1) / kLTPB);
  int ns = quiet_column_sets(a.n_mu);
  QuietCol *pk = (QuietCol *)pack;
  double *scale = (double *)(pk + (long)ns * a.grid);
  int32_t *count = (int32_t *)(scale + ns * kQColBins);
  k_quiet_columns_pack<<<(unsigned)ns, kLTPB, 0, s>>>(a.grid, colw, colf, cols, pk, scale, count);
  const size_t tap_lds = lin_tap_bytes(2 * kQColBins, 2, a.span);
  if (a.nodes && tap_lds <= 65000)  // 64 KB with the static part: a reach of some 70 pixels either way
    k_fir_quiet_cols<<<dim3(nb, ns), kLTPB, tap_lds, s>>>(a, q, qs, pk, scale, count, part);
  else if (a.uniform)
    k_gather_quiet_cols<true><<<dim3(nb, ns), kLTPB, lds, s>>>(a, q, qs, pk, count, part);
  else
    k_gather_quiet_cols<false><<<dim3(nb, ns), kLTPB, lds, s>>>(a, q, qs, pk, count, part);
  long n2 = 2 * a.n;
  k_quiet_sum<<<(unsigned)((n2 + kLTPB - 1) / kLTPB), kLTPB, 0, s>>>(part, ns, n2, out);
  return hipGetLastError();
}

// Active deltas of phase p on a linear grid (spot_integrate + fast_flux / bconv /
// tot, SOAP_integration.cu:285-307,392-447; solar variant :433 of
// SOAP_integration_solar.cu): per active cell, Q = Shift(Sq_k), QS = Shift(SEDq_k),
// P = Shift(Sspot_k or Sfac_k), all x limb; intensity I = C_spot (spot),
// (1+LB) C_fac or B(T_cell)/B(T_norm) C_fac (facula); flux += QS - I Q,
// bconv += Q - P, tot += QS - I P.  Over a shift group the limb weights sum
// (w = sum L) and the intensity weights too (spot: C_spot w, facula: C_fac
// sum (1+LB) L; solar-mode facula groups are single cells).  Blocks are numbered
// so the phases of a tile run back to back on one XCD.
template <bool UNI>
__global__ __launch_bounds__(kLTPB) void k_gather_active_linear(LinArgs a, FirArgs f, const LinGroup *groups,
                                                                const int64_t *list_off, const int32_t *bin_off,
                                                                const int32_t *g_n, int n_phase, int n_tiles,
                                                                LinSolar sol) {
  extern __shared__ double lds[];  // rows [4][span]: q, qs, spot, facula; wave [span]
  long b = blockIdx.x;
  long slot = b / 8;
  long tile = (slot / n_phase) * 8 + b % 8;
  int p = (int)(slot % n_phase);
  if (tile >= n_tiles) return;  // uniform over the block
  const int j0 = (int)tile * kLTPB;
  const int j = j0 + threadIdx.x;
  const int jc = j < a.n ? j : (int)a.n - 1;
  const int base = j0 + a.off_lo;
  const int span = a.span;
  double *rw = lds, *wl = lds + 4 * span;
  lin_stage_wave(wl, a.wave, base, span, a.n);
  const int lj = j - base;  // inside the window: -off_lo .. kLTPB - 1 - off_lo
  double lam_j = a.wave[jc];
  double cs = f.sps ? f.sps[jc] : 0.0, cf = f.fas ? f.fas[jc] : 0.0;
  double hc = kPlanckH * kC;
  double en = sol.on ? expm1(hc / (lam_j * kBoltzK * (double)sol.t_norm * 1e-10)) : 0.0;
  double flux = 0.0, bconv = 0.0, tot = 0.0;
  const CONSTANT LinGroup *gp = gc(groups + list_off[p]);
  const int32_t *bo = bin_off + (long)p * (a.n_mu + 1);
  const int32_t *gn = g_n + (long)p * a.n_mu;
  for (int k = 0; k < a.n_mu; k++) {
    int c0 = bo[k], ng = gn[k];
    if (ng == 0) continue;  // uniform
    const long ko = (long)k * a.n;
    const double *g[4] = {f.q + ko, f.qs + ko, f.sp ? f.sp + ko : f.q + ko, f.fa ? f.fa + ko : f.q + ko};
    __syncthreads();
    for (int r = 0; r < 4; r++) lin_stage(rw + (long)r * span, g[r], base, span, a.n);
    __syncthreads();
    for (int c = c0; c < c0 + ng; c++) {
      const CONSTANT LinGroup &G = gp[c];
      int e = G.e;
      int idx = e & 0x3fffffff, ty = e >> 30;
      double L = G.w;
      int r_act = ty == 0 ? 2 : 3;
      LinShift s = group_shift(G);
      const double *ra = rw + r_act * span;
      double iq, is, ia;  // shifted rows at pixel j
      if (s.ident) {
        iq = rw[lj];
        is = rw[span + lj];
        ia = ra[lj];
      } else {
        int li;
        double t;
        lin_locate<UNI>(j, lam_j, s, a.inv_step, wl, base, span, li, t);
        double q0 = rw[li], q1 = rw[li + 1];
        double s0 = rw[span + li], s1 = rw[span + li + 1];
        double a0 = ra[li], a1 = ra[li + 1];
        iq = fma(q1 - q0, t, q0);
        is = fma(s1 - s0, t, s0);
        ia = fma(a1 - a0, t, a0);
      }
      // IW = sum over the group of I L
      double IW;
      if (ty == 0) {
        IW = cs * L;  // B(T_spot)/B(int T_spot) = 1
      } else if (sol.on) {
        double T_cell = (double)plage_temp(sol.t_sum, cell_rcos(idx, a.grid));
        IW = en / expm1(hc / (lam_j * kBoltzK * T_cell * 1e-10)) * cf * L;
      } else {
        IW = cf * G.w2;
      }
      flux = fma(-IW, iq, fma(is, L, flux));
      bconv = fma(iq - ia, L, bconv);
      tot = fma(-IW, ia, fma(is, L, tot));
    }
  }
  if (j < a.n) {
    double *o = f.out + (long)p * 3 * a.n;
    o[j] = flux;
    o[a.n + j] = bconv;
    o[2 * a.n + j] = tot;
  }
}

// The same sums where neighbouring groups of a list mostly share their source pixels (solid-body
// rotation: the list is in the order of the columns, some tens of them to a pixel): over a run of
// groups with one whole part of the shift, sum w I(row) = W row_i + T (row_{i+1} - row_i) with
// W = sum w and T = sum w t, so a group costs its own weight t (ten operations, from two
// wavelengths in registers) and the rows are read once per run.  t is lin_locate's, to the bit of
// the shifted wavelengths' rounding that the reference's weights carry.  Every wave finds its
// groups' whole parts with one group per lane; a group whose whole part changes inside the tile,
// comes within 1e-5 of changing, or that has no shift, is interpolated by itself.
// 25 phases of the production disk, 100,000 pixels: 1315 -> 529 us with one set of regions (a
// group at a time, with the reciprocal weights: 1004), 2670-2900 -> 1040-1120 us with bench.py's,
// which hold more groups; two groups' scalar loads at a time, 1 and 4 measured 6 % slower.
__global__ __launch_bounds__(kLTPB) void k_gather_active_runs(LinArgs a, FirArgs f, const LinGroup *groups,
                                                              const int64_t *list_off, const int32_t *bin_off,
                                                              const int32_t *g_n, int n_phase, int n_tiles) {
  extern __shared__ double lds[];  // rows [4][span]: q, qs, spot, facula; wave [span]
  const long b = blockIdx.x, slot = b / 8, tile = (slot / n_phase) * 8 + b % 8;
  const int p = (int)(slot % n_phase);
  if (tile >= n_tiles) return;  // uniform over the block
  const int j0 = (int)tile * kLTPB, tid = threadIdx.x, j = j0 + tid, jc = j < a.n ? j : (int)a.n - 1;
  const int base = j0 + a.off_lo, span = a.span;
  double *rw = lds, *wl = lds + 4 * span;
  lin_stage_wave(wl, a.wave, base, span, a.n);
  const double lam_j = a.wave[jc];
  const double cs = f.sps ? f.sps[jc] : 0.0, cf = f.fas ? f.fas[jc] : 0.0;
  double flux = 0.0, bconv = 0.0, tot = 0.0;
  const int32_t *bo = bin_off + (long)p * (a.n_mu + 1);
  const int32_t *gn = g_n + (long)p * a.n_mu;
  for (int k = 0; k < a.n_mu; k++) {
    const int m = gn[k];
    if (m == 0) continue;  // uniform
    const LinGroup *gv = groups + list_off[p] + bo[k];
    const CONSTANT LinGroup *gp = gc(gv);
    const long ko = (long)k * a.n;
    const double *g[4] = {f.q + ko, f.qs + ko, f.sp ? f.sp + ko : f.q + ko, f.fa ? f.fa + ko : f.q + ko};
    __syncthreads();
    for (int r = 0; r < 4; r++) lin_stage(rw + (long)r * span, g[r], base, span, a.n);
    __syncthreads();
    int run = -1;  // the open run's window index at lane 0 of the block
    double w0 = 0.0, w1 = 0.0;
    double Ws = 0.0, Ts = 0.0, Wf = 0.0, Tf = 0.0, W2 = 0.0, T2 = 0.0;
    auto add = [&](int li, bool own, double Ws, double Ts, double Wf, double Tf, double W2, double T2) {
      const int up = own ? li : li + 1;
      const double q0 = rw[li], dq = rw[up] - q0, s0 = rw[span + li], ds = rw[span + up] - s0;
      const double L = Ws + Wf, T = Ts + Tf;
      const double vs = fma(ds, T, s0 * L);
      flux += vs;
      tot += vs;
      if (Ws != 0.0 || Ts != 0.0) {  // uniform but for the sign of a zero
        const double a0 = rw[2 * span + li], da = rw[2 * span + up] - a0;
        flux = fma(-cs, fma(dq, Ts, q0 * Ws), flux);
        tot = fma(-cs, fma(da, Ts, a0 * Ws), tot);
        bconv += fma(dq - da, Ts, (q0 - a0) * Ws);
      }
      if (Wf != 0.0 || Tf != 0.0 || W2 != 0.0 || T2 != 0.0) {
        const double a0 = rw[3 * span + li], da = rw[3 * span + up] - a0;
        flux = fma(-cf, fma(dq, T2, q0 * W2), flux);
        tot = fma(-cf, fma(da, T2, a0 * W2), tot);
        bconv += fma(dq - da, Tf, (q0 - a0) * Wf);
      }
    };
    auto flush = [&] {
      if (run >= 0) add(tid + run, false, Ws, Ts, Wf, Tf, W2, T2);
      Ws = Ts = Wf = Tf = W2 = T2 = 0.0;
    };
    for (int c0 = 0; c0 < m; c0 += 64) {
      int e = -1;
      if (c0 + (tid & 63) < m) {
        const LinGroup &r = gv[c0 + (tid & 63)];
        const double t1 = r.c1 * r.rinv, x0 = fma((double)j0, t1, -(r.fl * r.rinv));
        const double x1 = fma((double)(kLTPB - 1), t1, x0), d = floor(x0);
        const double f0 = x0 - d, f1 = x1 - d;
        const int at = (int)d - a.off_lo;
        if (f0 > 1e-5 && f0 < 1 - 1e-5 && f1 > 1e-5 && f1 < 1 - 1e-5 && at >= 0 && at <= span - kLTPB - 1) e = at;
      }
      const int n = m - c0 < 64 ? m - c0 : 64;
      // two groups at a time, their scalar loads waited for together
      for (int u0 = 0; u0 < n; u0 += 2) {
        double c1[2], rinv[2], w[2], w2[2];
        int pop[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
          const CONSTANT LinGroup &r = gp[c0 + (u0 + i < n ? u0 + i : u0)];
          c1[i] = r.c1;
          rinv[i] = r.rinv;
          w[i] = r.w;
          w2[i] = r.w2;
          pop[i] = r.e >> 30;
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {  // lanes from n on hold -1; every branch is uniform
          const int at = __builtin_amdgcn_readlane(e, u0 + i);
          if (at < 0) continue;
          if (at != run) {
            flush();
            run = at;
            w0 = wl[tid + run];
            w1 = wl[tid + run + 1];
          }
          const double ls0 = fma(-w0, c1[i], w0), den = fma(-w1, c1[i], w1) - ls0;
          const double r0 = rinv[i] * a.inv_step, t = (lam_j - ls0) * fma(r0, fma(-den, r0, 1.0), r0);
          if (pop[i] == 0) {
            Ws += w[i];
            Ts = fma(w[i], t, Ts);
          } else {
            Wf += w[i];
            Tf = fma(w[i], t, Tf);
            W2 += w2[i];
            T2 = fma(w2[i], t, T2);
          }
        }
      }
      unsigned long long ones = __ballot(e < 0) & (~0ull >> (64 - n));
      while (ones) {
        const CONSTANT LinGroup &r = gp[c0 + __ffsll((long long)ones) - 1];
        ones &= ones - 1;
        const LinShift s = group_shift(r);
        const double w = r.w, w2 = r.w2;
        int li;
        double t;
        lin_locate<true>(j, lam_j, s, a.inv_step, wl, base, span, li, t);
        if (r.e >> 30 == 0)
          add(li, s.ident, w, w * t, 0.0, 0.0, 0.0, 0.0);
        else
          add(li, s.ident, 0.0, 0.0, w, w * t, w2, w2 * t);
      }
    }
    flush();
  }
  if (j < a.n) {
    double *o = f.out + (long)p * 3 * a.n;
    o[j] = flux;
    o[a.n + j] = bconv;
    o[2 * a.n + j] = tot;
  }
}

hipError_t launch_gather_active_linear(const LinArgs &a, const FirArgs &f, const LinGroup *groups,
                                       const int64_t *list_off, const int32_t *bin_off, const int32_t *g_n,
                                       int n_phase, const LinSolar &sol, hipStream_t s) {
  if (n_phase == 0) return hipSuccess;
  size_t lds = (size_t)5 * a.span * sizeof(double);
  if (lds > 65536 || a.span < kLTPB || a.n > kLinMaxN) return hipErrorInvalidValue;
  int n_tiles = (int)((a.n + kLTPB - 1) / kLTPB);
  long tiles8 = ((long)n_tiles + 7) / 8 * 8;
  long blocks = tiles8 * n_phase;
  if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
  if (a.uniform && a.solid && !sol.on)  // solar mode: a facula's intensity depends on its cell
    k_gather_active_runs<<<(unsigned)blocks, kLTPB, lds, s>>>(a, f, groups, list_off, bin_off, g_n, n_phase, n_tiles);
  else if (a.uniform)
    k_gather_active_linear<true><<<(unsigned)blocks, kLTPB, lds, s>>>(a, f, groups, list_off, bin_off, g_n, n_phase,
                                                                      n_tiles, sol);
  else
    k_gather_active_linear<false><<<(unsigned)blocks, kLTPB, lds, s>>>(a, f, groups, list_off, bin_off, g_n, n_phase,
                                                                       n_tiles, sol);
  return hipGetLastError();
}

// ------------------------------------------------------------ resolution
// conv_inst on a linear grid (SOAP_initialize.cu:78-96, SOAP_resolution.cu:76-95):
// o_i = sum_{d=-wid}^{wid-2} w (1 - A_{i+d}) / (sig_i sqrt(2 pi)) exp(-d^2 0.005^2 / (2 sig_i^2)),
// sig_i = Delta_lambda(sigma, lambda_i), for wid < i < n-1-wid (0 elsewhere).
// The Gaussian factors follow g_{d+1} = g_d u_d, u_{d+1} = u_d v from g_0 = 1,
// u_0 = exp(-a), v = exp(-2a), a = 0.005^2 / (2 sig_i^2) (relative error of
// g_d below |d| ulp).  Block = kLTPB pixels of one spectrum; spectrum sp =
// blockIdx.y: A = quiet[sel] - raw (active) or the quiet spectrum itself.
__global__ __launch_bounds__(kLTPB) void k_conv_linear(ConvLinArgs c, const double *quiet, const double *raw,
                                                       double *o_out, double *part) {
  extern __shared__ double xs[];  // 1 - A over [i0 - wid, i0 + kLTPB + wid)
  long sp = blockIdx.y;
  long i0 = (long)blockIdx.x * kLTPB;
  int span = kLTPB + 2 * c.wid;
  const double *Q, *D = nullptr;
  double w;
  if (sp < c.n_active) {
    int t = (int)(sp % 3);
    Q = quiet + (long)(t == 1 ? 0 : 1) * c.n;  // bconv uses the normalised quiet star
    D = raw + sp * c.n;
    w = 0.005;
  } else {
    Q = quiet + (long)c.quiet_sel[sp - c.n_active] * c.n;
    w = c.quiet_weight;
  }
  double amin = HUGE_VAL, omax = -60000.0;
  __shared__ int s_top[kLTPB / 64];
  int top = 0;  // sign-free high word of the window's largest value: its exponent, 2047 if it is not finite
  for (int e = threadIdx.x; e < span; e += blockDim.x) {
    long m = i0 - c.wid + e;
    double v = 1.0;
    if (m >= 0 && m < c.n) {
      double A = D ? Q[m] - D[m] : Q[m];
      v = 1.0 - A;
      if (m >= i0 && m < i0 + kLTPB) amin = A < amin ? A : amin;
    }
    xs[e] = v;
    top = max(top, __double2hiint(v) & 0x7fffffff);
  }
  for (int off = 32; off > 0; off >>= 1) top = max(top, __shfl_xor(top, off));
  if ((threadIdx.x & 63) == 0) s_top[threadIdx.x >> 6] = top;
  __syncthreads();
  for (int k = 0; k < kLTPB / 64; k++) top = max(top, s_top[k]);
  long i = i0 + threadIdx.x;
  double o = 0.0;
  if (i < c.n && i > c.wid && i + c.wid < c.n - 1) {
    double sig = -1 * c.wave[i] * c.c1;  // Delta_lambda(sigma, lambda_i)
    double aa = 0.005 * 0.005 / (2 * sig * sig);
    double v = exp(-2 * aa);
    const double *x = xs + threadIdx.x + c.wid;  // x[d] = 1 - A_{i+d}
    double acc = x[0];
    double g = 1.0, u = exp(-aa);
    // to the offset whose factor times the window's largest value is below 2^-62 of the centre:
    // the window holds 50 widths, most of them below the rounding of the sum (300 -> 134 us).
    // All of it where a value is not finite.
    const int bits = 63 + (top >> 20) - ((__double2hiint(x[0]) >> 20) & 0x7ff);
    const double far = sqrt(0.69314718055994531 * bits / aa);
    const int reach = top < 0x7ff00000 && far < c.wid ? (int)far + 1 : c.wid;
    for (int d = 1; d <= reach; d++) {
      g *= u;
      u *= v;
      double pair = x[-d];
      if (d <= c.wid - 2) pair += x[d];
      acc = fma(g, pair, acc);
    }
    o = w * acc / (sig * sqrt(2. * kPi));
  }
  if (i < c.n) {
    o_out[sp * c.n + i] = o;
    if (o != 0.0 && omax < o) omax = o;
  }
  // block min / max partials
  __shared__ double s_min[kLTPB / 64], s_max[kLTPB / 64];
  for (int off = 32; off > 0; off >>= 1) {
    double x1 = __shfl_xor(amin, off), x2 = __shfl_xor(omax, off);
    amin = x1 < amin ? x1 : amin;
    omax = x2 > omax ? x2 : omax;
  }
  int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0) {
    s_min[wv] = amin;
    s_max[wv] = omax;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double a0 = s_min[0], b0 = s_max[0];
    for (int k = 1; k < kLTPB / 64; k++) {
      a0 = s_min[k] < a0 ? s_min[k] : a0;
      b0 = s_max[k] > b0 ? s_max[k] : b0;
    }
    part[(sp * c.n_tiles + blockIdx.x) * 2] = a0;
    part[(sp * c.n_tiles + blockIdx.x) * 2 + 1] = b0;
  }
}

hipError_t launch_conv_linear(const ConvLinArgs &c, int n_spec, const double *quiet, const double *raw, double *o_out,
                              double *part, hipStream_t s) {
  if (n_spec == 0) return hipSuccess;
  size_t lds = (size_t)(kLTPB + 2 * c.wid) * sizeof(double);
  if (lds > 65536) return hipErrorInvalidValue;
  dim3 grid((unsigned)c.n_tiles, (unsigned)n_spec);
  k_conv_linear<<<grid, kLTPB, lds, s>>>(c, quiet, raw, o_out, part);
  return hipGetLastError();
}

int conv_linear_tile() { return kLTPB; }

// ------------------------------------------------------------ CCF mask
// calc_mask on a linear grid with the reference's literal index arithmetic
// (CCF_func.py:45-91): pixel positions on the extended grid of run_all_SOAP.py:
// 292-295 (no_points = 20000 on each side, step 0.005 in the index formula),
// converted to trimmed-spectrum positions (the slice mask[20000:]); lines with
// aa < 1 or bb + 1 >= n_ext are skipped (len 0).
__device__ __forceinline__ double ext_wave(const double *wt, long n_t, double step, long np, long k) {
  double begin = wt[0] - step * np;
  if (k < np) {
    if (k == np - 1) return wt[0];
    double st = (wt[0] - begin) / (double)(np - 1);
    return (double)k * st + begin;
  }
  if (k < np + n_t) return wt[k - np];
  long kk = k - np - n_t;
  double stop = wt[n_t - 1] + step * np;
  if (kk == np - 1) return stop;
  double st = (stop - wt[n_t - 1]) / (double)(np - 1);
  return (double)kk * st + wt[n_t - 1];
}

__global__ void k_mask_build_linear(const double *line_l, const double *line_w, const int32_t *sorted, int n_lines,
                                    const double *vgrid, int n_v, const double *wave_t, long n_t, double step,
                                    int32_t *m_start, int32_t *m_len, double2 *m_wv) {
  long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long)n_v * n_lines) return;
  int q = (int)(e / n_v), iv = (int)(e % n_v);
  int li = sorted[q];
  const long np = (long)(100.0 / step);
  const long n_ext = n_t + 2 * np;
  double begin_wave = wave_t[0] - step * np;
  double ls = line_l[li] * (1 + vgrid[iv] / kC);
  double beta = 820. / kC;
  double hw = ls * (sqrt((1 + beta) / (1 - beta)) - 1);
  double bgn = ls - hw / 2., end = ls + hw / 2.;
  long aa = (long)ceil((bgn - begin_wave) / 0.005);
  long bb = (long)(ceil((end - begin_wave) / 0.005) - 1);
  double w = line_w[li];
  if (aa < 1 || bb + 1 >= n_ext || bb - aa + 2 > 24 || bb - aa + 2 < 1) {
    m_start[e] = 0;
    m_len[e] = 0;
    m_wv[e] = make_double2(0.0, 0.0);
    return;
  }
  double fb = fabs(ext_wave(wave_t, n_t, step, np, aa) - bgn) /
              (ext_wave(wave_t, n_t, step, np, aa) - ext_wave(wave_t, n_t, step, np, aa - 1));
  double fa = fabs(ext_wave(wave_t, n_t, step, np, bb) - end) /
              (ext_wave(wave_t, n_t, step, np, bb + 1) - ext_wave(wave_t, n_t, step, np, bb));
  m_start[e] = (int32_t)(aa - 1 - 20000);
  m_len[e] = (int32_t)(bb - aa + 2);
  m_wv[e] = make_double2(w * fb, w * fa);
}

hipError_t launch_mask_build_linear(const double *line_l, const double *line_w, const int32_t *sorted, int n_lines,
                                    const double *vgrid, int n_v, const double *wave_t, int64_t n_t, double step,
                                    int32_t *m_start, int32_t *m_len, double2 *m_wv, hipStream_t s) {
  long tot = (long)n_v * n_lines;
  if (tot == 0) return hipSuccess;
  k_mask_build_linear<<<(unsigned)((tot + kLTPB - 1) / kLTPB), kLTPB, 0, s>>>(
      line_l, line_w, sorted, n_lines, vgrid, n_v, wave_t, n_t, step, m_start, m_len, m_wv);
  return hipGetLastError();
}

}  // namespace soap
