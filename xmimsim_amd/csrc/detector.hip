/*
 * detector.hip -- detector response of the simulated spectra on the GPU:
 * the reference's xmi_detector_convolute_all (src/xmi_detector_f.F90:219-580).
 *
 * Per interaction order: window/absorber transmission and crystal absorption
 * per channel (src/xmi_detector_f.F90:404-426), escape peaks from given escape
 * ratios (:582-809), pile-up (:56-217), the Gaussian response with the
 * Si(Li)/SDD low-energy tail (:446-530) and Poisson counting noise (:862-905);
 * the net-line histories get the detector absorption at their line energies
 * (:275-335).
 *
 * Every order of a call goes through the same launches.  k_det_prep, one
 * thread per channel, forms the detection efficiency and the factors of the
 * channel's response that depend on the source energy only; k_det_esc_src
 * and k_det_esc the escape peaks (one workgroup per source, then per
 * target, so that the sums have a fixed order); k_det_cdf and k_det_pileup
 * the pulse trains, each on its own Philox stream; k_det_norm, one workgroup
 * per source channel, the response's normalisation and the source's weight
 * in every order; k_det_conv, one workgroup per target channel, the
 * convolution of every order; k_det_poisson one Poisson variate per channel
 * (inversion for small means, Hormann's PTRS rejection otherwise).
 */
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "../../include/xmimsim_amd.h"
#include "philox.h"
#include "xmi_internal.h"
#include "xrl_model.h"

extern "C" void xmi_set_error(const char *fmt, ...);

#define DET_PHX_SUB 5u /* Philox substream of the detector response */

struct DetResp {
  double zero, gain, a, b, c;
  int nch, type;
};

/* window, absorber or crystal layer of the detector: elements els[first ..
 * first + n) */
struct DetLayer {
  double density, thickness;
  int first, n, crystal, pad;
};
struct DetEl {
  double weight;
  int atom, pad;
};

/* fluorescence line of a crystal element: its energy, the edge of its
 * vacancy's shell, its column in the escape table (line - 1) * ne + element */
struct DetEscLine {
  double energy, edge;
  int col, pad;
};

/* what the escape kernels read: axes of the escape ratios, the lines in
 * the reference's order, and the part of both tables that the sources
 * [i0, i1) of this launch need (rows f0 .. of the fluorescence table; columns
 * c0 .. c0 + nc of the Compton table's rows 0 .. nrow - 1) */
struct DetEsc {
  const double *fe, *ci, *co;
  const DetEscLine *line;
  const double *fluo, *compt;
  double out_diff;
  int nfe, nci, nco, nline, ncol_f; /* ncol_f = 109 * ne */
  int i0, i1, f0, c0, nc;
  int first, last; /* first and last of the launches of a call */
};

/* device buffers of one group of orders: nch entries each (spectra: per
 * order, row k at k * nch) */
struct DetBufs {
  double *A0, *B0, *T, *Q, *alfa;   /* response factors of a source channel */
  double *esum, *eself;             /* escape: summed ratios, self factor of a source */
  int *ep1, *epf;                   /* its positions on the Compton and fluorescence axes, -1 outside */
  double *src, *tmp, *w, *conv;     /* spectra: absorbed (src), after the escape peaks (tmp), weights, result */
  double *cdf;
  unsigned long long *hist;
  int *guide;                       /* [order][DET_GUIDE + 1] */
  struct DetTrains *trains;         /* [order] */
};

/* the pile-up of one order: counts before it, pulses per thread, in all */
struct DetTrains {
  double Nt;
  long each, total;
  unsigned int over, pad;
};

#define DET_GUIDE 1024       /* cells of the pile-up's guide table */
#define DET_PULSE_THREADS 65536
#define DET_NB 4             /* orders of one pass over the pairs */

/* sum over a workgroup of 256, in a fixed order; the result in thread 0 */
__device__ __forceinline__ double det_block_sum(double v, double *red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  const double s = (red[0] + red[1]) + (red[2] + red[3]);
  __syncthreads();
  return s;
}

/* per channel: the detection efficiency (window and absorber transmission
 * times crystal absorption, src/xmi_detector_f.F90:404-426) applied to every
 * order's spectrum, and the response's source factors */
__global__ void __launch_bounds__(64) k_det_prep(DetResp d, DetBufs b, const DetLayer *lay, int n_lay, const DetEl *els,
                                                 const xrl_atom *atoms, int n_ord, int absorb) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= d.nch) return;
  const double E = i * d.gain + d.zero;
  if (absorb) {
    double c = 1.0;
    const xrl_ectx ec = xrl_energy(E);
    for (int l = 0; l < n_lay; l++) {
      double mu = 0.0;
      for (int k = 0; k < lay[l].n; k++) {
        const DetEl e = els[lay[l].first + k];
        mu += xrl_cs_total_c(&atoms[e.atom], &ec) * e.weight;
      }
      const double x = -1.0 * lay[l].density * lay[l].thickness * mu;
      if (lay[l].crystal) c = -1.0 * c * expm1(x);
      else c *= exp(x);
    }
    for (int n = 0; n < n_ord; n++) b.src[(size_t)n * d.nch + i] *= c;
  }
  const double E0 = d.zero + d.gain * i;
  const double B0 = d.c * sqrt(d.a + d.b * E0);
  b.A0[i] = 1.0 / (B0 * 1.7724538509055160273);
  b.B0[i] = B0;
  double T = 0.0, Q = 0.0, alfa = 0.0;
  if (!(E0 > 50.0)) {
    const double tail = d.type == XMI_DETECTOR_CONVOLUTION_PROFILE_SI_SDD ? 0.63 : 2.7;
    T = tail * (2.73E-3 * exp(-0.21 * E0) + 1.E-4);
    Q = 15.0 * (0.000188 * exp(-0.00296 * pow(E0, 0.763)) + 1.355E-5 * exp(0.968 * pow(E0, 0.498)));
    alfa = 1.179 * exp(8.6E-4 * pow(E0, 1.877)) - 7.793 * exp(-3.81 * pow(E0, -0.0716));
  }
  b.T[i] = T;
  b.Q[i] = Q;
  b.alfa[i] = alfa;
}

/* response of channel I to a unit line in channel I0 (before normalisation),
 * from the source factors of I0 */
__device__ __forceinline__ double det_r(const DetResp &d, int I0, int I, double A0, double B0, double T, double Q,
                                        double alfa) {
  const double E0 = d.zero + d.gain * I0, E = d.zero + d.gain * I;
  const double X = (E - E0) / B0;
  return A0 * exp(-X * X) + (T + Q * exp(alfa * (E - E0))) * erfc(X);
}

/* one workgroup per source channel: the sum of its response over the
 * targets, and its weight (content / norm) in every order; the content is
 * the pile-up's histogram where an order has one */
__global__ void __launch_bounds__(256) k_det_norm(DetResp d, DetBufs b, int n_ord, int escape, int pileup) {
  __shared__ double red[4];
  const int I0 = blockIdx.x;
  const double E0 = d.zero + d.gain * I0;
  double s = 0.0;
  if (E0 >= 1.0) {
    const double A0 = b.A0[I0], B0 = b.B0[I0], T = b.T[I0], Q = b.Q[I0], alfa = b.alfa[I0];
    const int last = I0 + 100 < d.nch - 1 ? I0 + 100 : d.nch - 1;
    for (int I = threadIdx.x; I <= last; I += 256) s += det_r(d, I0, I, A0, B0, T, Q, alfa);
  }
  const double norm = det_block_sum(s, red);
  const double *spec = escape ? b.tmp : b.src;
  for (int n = threadIdx.x; n < n_ord; n += 256) {
    const size_t o = (size_t)n * d.nch + I0;
    const double v = pileup && b.trains[n].total > 0 ? (double)b.hist[o] : spec[o];
    b.w[o] = (E0 < 1.0 || v == 0.0) ? 0.0 : v / norm;
  }
}

/* one workgroup per target channel: conv[I] = sum over I0 >= I - 100 of
 * R(I0, I) * w[I0], every order from one evaluation of R (DET_NB at a time).
 * Bound by the exp and erfc of the pairs (about 300 vector instructions a
 * pair); one thread per target, as before, left all but a few CUs idle and
 * formed the source factors' powers again for every pair: 2048 channels of
 * four orders took 4 x 3.4 ms. */
__global__ void __launch_bounds__(256) k_det_conv(DetResp d, DetBufs b, int n_ord) {
  __shared__ double red[4];
  const int I = blockIdx.x, lo = I - 100 > 0 ? I - 100 : 0;
  for (int n0 = 0; n0 < n_ord; n0 += DET_NB) {
    double s[DET_NB];
#pragma unroll
    for (int n = 0; n < DET_NB; n++) s[n] = 0.0;
    for (int I0 = lo + threadIdx.x; I0 < d.nch; I0 += 256) {
      double w[DET_NB];
      int any = 0;
#pragma unroll
      for (int n = 0; n < DET_NB; n++) {
        w[n] = n0 + n < n_ord ? b.w[(size_t)(n0 + n) * d.nch + I0] : 0.0;
        any |= w[n] != 0.0;
      }
      if (!any) continue;
      const double r = det_r(d, I0, I, b.A0[I0], b.B0[I0], b.T[I0], b.Q[I0], b.alfa[I0]);
#pragma unroll
      for (int n = 0; n < DET_NB; n++)
        if (w[n] != 0.0) s[n] += r * w[n];
    }
#pragma unroll
    for (int n = 0; n < DET_NB; n++) {
      const double t = det_block_sum(s[n], red);
      if (threadIdx.x == 0 && n0 + n < n_ord) b.conv[(size_t)(n0 + n) * d.nch + I] = t;
    }
  }
}

/* ---- escape peaks, src/xmi_detector_f.F90:582-809 ------------------------
 * The reference moves, source channel by source channel, a share of its
 * content to lower channels and then scales the source by what stays.  A
 * source's content only changes before its turn through channels above it,
 * which come later, so the result is the content times (1 - sum of shares)
 * plus the shares of the sources above, in any order.  (A line of less than
 * a channel's energy adds to its own source, which the lines after it see:
 * the factors det_esc_self multiplies.) */

__device__ __forceinline__ double det_channel_e(const DetResp &d, int i) { return ((double)i + 0.5) * d.gain + d.zero; }

/* p with a[p] < x <= a[p + 1] (0 when x is within 1e-10 of a[0]) for
 * a[0] <= x < a[n - 1], a increasing */
__device__ __forceinline__ int det_axis_pos(const double *a, int n, double x) {
  if (fabs(x - a[0]) < 1e-10) return 0;
  int lo = 0, hi = n - 1; /* a[lo] < x <= a[hi] */
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (x <= a[mid]) hi = mid;
    else lo = mid;
  }
  return lo;
}

/* share of source i (channel energy e) that escapes with line q, or -1 when
 * the line does not apply; *to = its target channel */
__device__ __forceinline__ double det_esc_line(const DetResp &d, const DetEsc &s, int pf, double e, int q, int *to) {
  const DetEscLine L = s.line[q];
  if (!(e > L.edge) || !((e - L.energy) >= 0.5 * d.gain + d.zero)) return -1.0;
  const double *r = s.fluo + (size_t)(pf - s.f0) * s.ncol_f + L.col;
  const double r0 = r[0], r1 = r[s.ncol_f];
  *to = (int)((e - L.energy - d.zero) / d.gain);
  return r0 + (r1 - r0) * (e - s.fe[pf]) / (s.fe[pf + 1] - s.fe[pf]);
}

/* share of source i that escapes as a Compton photon to channel j */
__device__ __forceinline__ double det_esc_compton(const DetResp &d, const DetEsc &s, int p1, double e, int j) {
  const double diff = e - det_channel_e(d, j);
  if (!(diff >= s.co[0] && diff < s.co[s.nco - 1])) return 0.0;
  const int p2 = det_axis_pos(s.co, s.nco, diff);
  const double x0 = s.ci[p1], x1 = s.ci[p1 + 1], y0 = s.co[p2], y1 = s.co[p2 + 1];
  const double denom = (x1 - x0) * (y1 - y0);
  const double c1 = (x1 - e) * (y1 - diff) / denom, c2 = (e - x0) * (y1 - diff) / denom;
  const double c3 = (x1 - e) * (diff - y0) / denom, c4 = (e - x0) * (diff - y0) / denom;
  const double *g = s.compt + (size_t)p2 * s.nc + (p1 - s.c0);
  return (c1 * g[0] + c2 * g[1] + c3 * g[s.nc] + c4 * g[s.nc + 1]) * d.gain / s.out_diff;
}

/* factor of source i's content that line q sees: the self lines before it
 * (all of them for q = nline) */
__device__ __forceinline__ double det_esc_self(const DetResp &d, const DetEsc &s, int pf, double e, int i, int q) {
  double f = 1.0;
  for (int k = 0; k < q; k++) {
    int to;
    const double r = det_esc_line(d, s, pf, e, k, &to);
    if (r != -1.0 && to == i) f += r * f;
  }
  return f;
}

/* one workgroup per source channel of the launch's range: its positions on
 * the axes and the sum of its shares */
__global__ void __launch_bounds__(256) k_det_esc_src(DetResp d, DetEsc s, DetBufs b) {
  __shared__ double red[4];
  __shared__ int self;
  const int i = s.i0 + blockIdx.x;
  const double e = det_channel_e(d, i);
  const int pf = (e >= s.fe[0] && e < s.fe[s.nfe - 1]) ? det_axis_pos(s.fe, s.nfe, e) : -1;
  const int p1 = (e >= s.ci[0] && e < s.ci[s.nci - 1]) ? det_axis_pos(s.ci, s.nci, e) : -1;
  if (threadIdx.x == 0) self = 0;
  __syncthreads();
  double sum = 0.0;
  if (pf >= 0)
    for (int q = threadIdx.x; q < s.nline; q += 256) {
      int to;
      const double r = det_esc_line(d, s, pf, e, q, &to);
      if (r == -1.0) continue;
      sum += r;
      if (to == i && r != 0.0) self = 1;
    }
  if (p1 >= 0)
    for (int j = threadIdx.x; j < i; j += 256) sum += det_esc_compton(d, s, p1, e, j);
  const double total = det_block_sum(sum, red);
  if (threadIdx.x == 0) {
    b.esum[i] = total;
    b.eself[i] = self ? det_esc_self(d, s, pf, e, i, s.nline) : 1.0;
    b.epf[i] = pf;
    b.ep1[i] = p1;
  }
}

/* one workgroup per target channel j: the shares of the launch's sources
 * above it, for every order (DET_NB per pass), added to b.tmp; the last
 * launch adds what stays of the channel's own content.  A line reaches j
 * from one source channel, at (its energy / gain) channels above: the four
 * channels around it are tested with the reference's expression. */
__global__ void __launch_bounds__(256) k_det_esc(DetResp d, DetEsc s, DetBufs b, int n_ord) {
  __shared__ double red[4];
  const int j = blockIdx.x;
  for (int n0 = 0; n0 < n_ord; n0 += DET_NB) {
    double a[DET_NB];
#pragma unroll
    for (int n = 0; n < DET_NB; n++) a[n] = 0.0;
    auto add = [&](int i, double r) {
#pragma unroll
      for (int n = 0; n < DET_NB; n++)
        if (n0 + n < n_ord) a[n] += r * b.src[(size_t)(n0 + n) * d.nch + i];
    };
    for (int t = threadIdx.x; t < 4 * s.nline; t += 256) {
      const int q = t >> 2;
      const double k = floor(s.line[q].energy / d.gain);
      if (!(k < (double)d.nch)) continue;
      const int i = j + (int)k - 1 + (t & 3);
      if (i <= j || i < s.i0 || i >= s.i1 || b.epf[i] < 0) continue;
      const double e = det_channel_e(d, i);
      int to;
      double r = det_esc_line(d, s, b.epf[i], e, q, &to);
      if (r == -1.0 || to != j) continue;
      if (b.eself[i] != 1.0) r *= det_esc_self(d, s, b.epf[i], e, i, q);
      add(i, r);
    }
    for (int i = (j + 1 > s.i0 ? j + 1 : s.i0) + threadIdx.x; i < s.i1; i += 256) {
      const int p1 = b.ep1[i];
      if (p1 < 0) continue;
      const double r = det_esc_compton(d, s, p1, det_channel_e(d, i), j);
      if (r != 0.0) add(i, r * b.eself[i]);
    }
#pragma unroll
    for (int n = 0; n < DET_NB; n++) {
      const double v = det_block_sum(a[n], red);
      if (threadIdx.x == 0 && n0 + n < n_ord) {
        const size_t o = (size_t)(n0 + n) * d.nch + j;
        double r = s.first ? v : b.tmp[o] + v;
        if (s.last) r += b.src[o] * b.eself[j] * (1.0 - b.esum[j]);
        b.tmp[o] = r;
      }
    }
  }
}

/* Pile-up, src/xmi_detector_f.F90:56-217: trains of pulses whose successive
 * gaps (exponential, mean live_time / N) stay below the pulse width sum into
 * one count.  Trains are independent, so each thread runs its own until it
 * has drawn its share of the pulses (and finishes the train it is in).  As in
 * the reference, a pulse's energy is taken at (channel + 1) * gain + zero and
 * the sum lands in channel (sum - zero) / gain - 1.
 *
 * k_det_cdf, one workgroup per order: the channel contents' cumulative sums
 * normalised to 1, the pulses per thread, the guide table (guide[k]: first
 * channel whose sum exceeds k / DET_GUIDE) and a cleared histogram. */
__global__ void __launch_bounds__(1024) k_det_cdf(int nch, DetBufs b, int escape) {
  __shared__ double wsum[16];
  const int n = blockIdx.x, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const double *t = (escape ? b.tmp : b.src) + (size_t)n * nch;
  double *cdf = b.cdf + (size_t)n * nch;
  const int per = (nch + 1023) / 1024, i0 = threadIdx.x * per, i1 = min(nch, i0 + per);
  double own = 0.0;
  for (int i = i0; i < i1; i++) own += t[i];
  double incl = own;
  for (int off = 1; off < 64; off <<= 1) {
    const double v = __shfl_up(incl, off);
    if (lane >= off) incl += v;
  }
  if (lane == 63) wsum[wv] = incl;
  __syncthreads();
  double base = 0.0, Nt = 0.0;
  for (int k = 0; k < 16; k++) {
    if (k < wv) base += wsum[k];
    Nt += wsum[k];
  }
  const long total = (long)Nt;
  double acc = base + (incl - own);
  for (int i = i0; i < i1; i++) {
    acc += t[i];
    cdf[i] = i == nch - 1 ? 1.0 : acc / Nt;
    b.hist[(size_t)n * nch + i] = 0ull;
  }
  if (threadIdx.x == 0) {
    DetTrains &tr = b.trains[n];
    tr.Nt = Nt;
    tr.total = total > 0 ? total : 0;
    tr.each = total > 0 ? (total + DET_PULSE_THREADS - 1) / DET_PULSE_THREADS : 0;
    tr.over = 0u;
  }
  __syncthreads();
  for (int k = threadIdx.x; k <= DET_GUIDE; k += 1024) {
    const double u = (double)k / DET_GUIDE;
    int lo = 0, hi = nch - 1;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (cdf[mid] > u) hi = mid;
      else lo = mid + 1;
    }
    b.guide[(size_t)n * (DET_GUIDE + 1) + k] = lo;
  }
}

/* DET_PULSE_THREADS threads per order (blockIdx.y).  A pulse's channel is
 * the first whose cumulative sum exceeds the draw, found between the guide
 * table's entries around it; both tables are read from LDS up to
 * DET_PILE_LDS channels.  Bound by the chain of draw, search and logarithm in
 * each thread: all orders in one launch keep four times as many waves in
 * flight as a launch per order, which took 0.64 ms each for 4e6 pulses. */
#define DET_PILE_LDS 4096
__global__ void __launch_bounds__(256) k_det_pileup(int nch, DetBufs b, double live_time, double width, double zero,
                                                    double gain, uint64_t seed, int order0) {
  __shared__ double l_cdf[DET_PILE_LDS];
  __shared__ int guide[DET_GUIDE + 1];
  const int n = blockIdx.y;
  const double *cdf = b.cdf + (size_t)n * nch;
  const DetTrains *tr = &b.trains[n];
  const long n_each = tr->each, n_total = tr->total;
  if (n_total <= 0) return;
  for (int k = threadIdx.x; k <= DET_GUIDE; k += 256) guide[k] = b.guide[(size_t)n * (DET_GUIDE + 1) + k];
  if (nch <= DET_PILE_LDS) {
    for (int k = threadIdx.x; k < nch; k += 256) l_cdf[k] = cdf[k];
    cdf = l_cdf;
  }
  __syncthreads();
  unsigned long long *hist = b.hist + (size_t)n * nch;
  const double mean_gap = live_time / tr->Nt;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long first = t * n_each;
  if (first >= n_total) return;
  const long mine = (first + n_each <= n_total) ? n_each : n_total - first;
  phx_stream s;
  phx_stream_init(&s, seed ^ (0x9E3779B97F4A7C15ull * (uint64_t)(order0 + n + 1)), 0u, 0u, DET_PHX_SUB, (uint64_t)t);
  long done = 0;
  int np = 0, first_ch = 0;
  double esum = 0.0;
  while (done < mine || np > 0) {
    const double u = phx_uniform(&s);
    const int cell = (int)(u * DET_GUIDE);
    int lo = guide[cell], hi = guide[cell + 1];
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (cdf[mid] > u) hi = mid;
      else lo = mid + 1;
    }
    const double gap = -mean_gap * log1p(-phx_uniform(&s));
    np++;
    done++;
    if (np == 1) first_ch = lo;
    esum += (double)(lo + 1) * gain + zero;
    if (np > 100) { /* the reference stops with an error; here the train is dropped and counted */
      atomicAdd(&b.trains[n].over, 1u);
      np = 0;
      esum = 0.0;
      continue;
    }
    if (gap > width) {
      if (np == 1) {
        atomicAdd(&hist[first_ch], 1ull);
      } else {
        const long ps = (long)((esum - zero) / gain);
        if (ps > 0 && ps <= nch) atomicAdd(&hist[ps - 1], 1ull);
      }
      np = 0;
      esum = 0.0;
    }
  }
}

/* Poisson variate of mean lam (lam > 1): inversion below 10, otherwise the
 * transformed rejection with squeeze of W. Hormann, "The transformed
 * rejection method for generating Poisson random variables", Insurance:
 * Mathematics and Economics 12 (1993) 39-45. */
__device__ double det_poisson(double lam, phx_stream *s) {
  if (lam < 10.0) {
    double p = exp(-lam), F = p, u = phx_uniform(s);
    double k = 0.0;
    while (u > F && k < 1000.0) {
      k += 1.0;
      p *= lam / k;
      F += p;
    }
    return k;
  }
  const double slam = sqrt(lam), loglam = log(lam);
  const double b = 0.931 + 2.53 * slam;
  const double a = -0.059 + 0.02483 * b;
  const double inv_alpha = 1.1239 + 1.1328 / (b - 3.4);
  const double vr = 0.9277 - 3.6224 / (b - 2.0);
  for (int it = 0; it < 10000; it++) {
    const double U = phx_uniform(s) - 0.5;
    const double V = phx_uniform(s);
    const double us = 0.5 - fabs(U);
    const double k = floor((2.0 * a / us + b) * U + lam + 0.43);
    if (us >= 0.07 && V <= vr) return k;
    if (k < 0.0 || (us < 0.013 && V > us)) continue;
    if (log(V) + log(inv_alpha) - log(a / (us * us) + b) <= -lam + k * loglam - lgamma(k + 1.0)) return k;
  }
  return floor(lam + 0.5);
}

/* orders order0 + blockIdx.y */
__global__ void k_det_poisson(int nch, double *conv, uint64_t seed, uint32_t order0) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nch) return;
  double *ch = conv + (size_t)blockIdx.y * nch;
  const uint32_t order = order0 + blockIdx.y;
  const double v = ch[i];
  if (v > 4294967295.0 || !(v > 1.0)) return; /* src/xmi_detector_f.F90:891-897 */
  phx_stream s;
  phx_stream_init(&s, seed, 1u, order, DET_PHX_SUB, (uint64_t)i);
  ch[i] = det_poisson(v, &s);
}

/* ------------------------------------------------------------------------ */
/* host */

static double layer_mu(const xmi_layerF *L, double E) {
  double rv = 0.0;
  for (int i = 0; i < L->n_elements; i++) rv += xrl_cs_total(xrl_atom_get(L->Z[i]), E) * L->weight[i];
  return rv;
}

/* detector window/absorber transmission times crystal absorption at E */
static double det_efficiency(const xmi_inputF *in, double E) {
  double c = 1.0;
  for (int l = 0; l < in->n_det_layers; l++)
    c *= exp(-1.0 * in->det_layers[l].density * in->det_layers[l].thickness * layer_mu(&in->det_layers[l], E));
  for (int l = 0; l < in->n_crystal_layers; l++)
    c = -1.0 * c * expm1(-1.0 * in->crystal_layers[l].density * in->crystal_layers[l].thickness *
                         layer_mu(&in->crystal_layers[l], E));
  return c;
}

/* 0-based index p with a[p] < x <= a[p+1] (x == a[0] gives 0), else -1:
 * the findpos of src/xmi_aux_f.F90 used by the escape-peak code */
static int det_findpos(const double *a, int n, double x) {
  if (fabs(x - a[0]) < 1e-10) return 0;
  for (int i = 0; i < n; i++)
    if (x <= a[i]) return i - 1;
  return -1;
}

/* lines of the K, L1, L2 and L3 vacancies that the reference's escape peaks
 * loop over */
static const int esc_shell_first[4] = {1, 32, 60, 86}, esc_shell_last[4] = {29, 58, 85, 109};
static int esc_line_count() {
  int n = 0;
  for (int sh = 0; sh < 4; sh++) n += esc_shell_last[sh] - esc_shell_first[sh] + 1;
  return n;
}

/* escape peaks with given escape ratios, src/xmi_detector_f.F90:582-809, on
 * the host: for axes that are not increasing, a gain that is not positive, a
 * Compton table of over DET_ESC_WORDS / 4 output energies or more lines than
 * DET_ESC_LINES, which the device routine does not take.  fluo_escape_ratios holds the Fortran array (element, line 1..109, input
 * energy) in column-major order; compton_escape_ratios (input, output). */
static void det_escape(std::vector<double> &ch, const xmi_inputF *in, const xmi_escape_ratios *er) {
  const int nch = (int)ch.size();
  const double zero = in->detector.zero, gain = in->detector.gain;
  const double channel_1e = 0.5 * gain + zero;
  const int ne = er->n_elements, nfe = er->n_fluo_input_energies;
  const int nce = er->n_compton_input_energies, nco = er->n_compton_output_energies;
  const double *fe = er->fluo_escape_input_energies;
  const double *ci = er->compton_escape_input_energies, *co = er->compton_escape_output_energies;
  const double compton_out_diff = nco > 1 ? co[1] - co[0] : 1.0;
  const int *shell_first = esc_shell_first, *shell_last = esc_shell_last;
  for (int i = 0; i < nch; i++) {
    const double channel_e = ((double)i + 0.5) * gain + zero;
    double sum_ratio = 0.0;
    for (int j = 0; j < ne; j++) {
      const xrl_atom *a = xrl_atom_get(er->Z[j]);
      for (int sh = 0; sh < 4; sh++) {
        if (!(channel_e > a->edge[sh])) continue;
        for (int line = shell_first[sh]; line <= shell_last[sh]; line++) {
          const double line_e = a->line_energy[line];
          if (!((channel_e - line_e) >= channel_1e && channel_e >= fe[0] && channel_e < fe[nfe - 1])) continue;
          const int pos = det_findpos(fe, nfe, channel_e);
          if (pos < 0) continue;
          const double r0 = er->fluo_escape_ratios[((size_t)pos * 109 + (line - 1)) * ne + j];
          const double r1 = er->fluo_escape_ratios[((size_t)(pos + 1) * 109 + (line - 1)) * ne + j];
          /* interpolate_simple, src/xmi_aux_f.F90:1267-1276 */
          const double ratio = r0 + (r1 - r0) * (channel_e - fe[pos]) / (fe[pos + 1] - fe[pos]);
          sum_ratio += ratio;
          const int escape_i = (int)((channel_e - line_e - zero) / gain);
          if (escape_i >= 0 && escape_i < nch) ch[escape_i] += ratio * ch[i];
        }
      }
    }
    for (int j = 0; j < i; j++) {
      const double channel_c = ((double)j + 0.5) * gain + zero;
      const double compton_diff = channel_e - channel_c;
      if (!(channel_e >= ci[0] && channel_e < ci[nce - 1] && compton_diff >= co[0] && compton_diff < co[nco - 1]))
        continue;
      const int p1 = det_findpos(ci, nce, channel_e), p2 = det_findpos(co, nco, compton_diff);
      if (p1 < 0 || p2 < 0) continue;
      const double denom = (ci[p1 + 1] - ci[p1]) * (co[p2 + 1] - co[p2]);
      const double c1 = (ci[p1 + 1] - channel_e) * (co[p2 + 1] - compton_diff) / denom;
      const double c2 = (channel_e - ci[p1]) * (co[p2 + 1] - compton_diff) / denom;
      const double c3 = (ci[p1 + 1] - channel_e) * (compton_diff - co[p2]) / denom;
      const double c4 = (channel_e - ci[p1]) * (compton_diff - co[p2]) / denom;
      const double *g = er->compton_escape_ratios;
      const double v = c1 * g[(size_t)p2 * nce + p1] + c2 * g[(size_t)p2 * nce + p1 + 1] +
                       c3 * g[(size_t)(p2 + 1) * nce + p1] + c4 * g[(size_t)(p2 + 1) * nce + p1 + 1];
      const double ratio = v * gain / compton_out_diff;
      ch[j] += ratio * ch[i];
      sum_ratio += ratio;
    }
    ch[i] *= (1.0 - sum_ratio);
  }
}

#define DET_TRY(x)                                                          \
  do {                                                                      \
    hipError_t e_ = (x);                                                    \
    if (e_ != hipSuccess) {                                                 \
      xmi_set_error("detector response: %s: %s", #x, hipGetErrorString(e_)); \
      return 0;                                                             \
    }                                                                       \
  } while (0)

extern "C" uint64_t xmi_engine_current_seed(const xmi_main_options *options);

#define DET_ESC_WORDS (1l << 20)  /* doubles of the escape tables of one launch */
#define DET_ESC_AXES (1l << 18)   /* doubles of their axes */
#define DET_LAYER_BYTES (64 << 10) /* detector layers and their elements */
#define DET_ESC_LINES (64 << 10)   /* lines of the escape ratios' elements */

/* what one call uploads once: the detector's layers and elements with their
 * atoms, the escape axes and lines */
struct DetInput {
  std::vector<DetLayer> lay;
  std::vector<DetEl> els;
  std::vector<int> atoms; /* distinct elements */
  std::vector<DetEscLine> lines;
  std::vector<double> axes;
  long nrow = 0;          /* rows of the Compton table that the channels reach */
  int host_front = 0;     /* absorption and escape peaks on the host */
};

static int det_increasing(const double *a, int n) {
  for (int i = 0; i + 1 < n; i++)
    if (!(a[i] < a[i + 1])) return 0;
  return n > 0;
}

static void det_input(const xmi_inputF *in, const xmi_escape_ratios *er, DetInput &q) {
  auto layers = [&](const xmi_layerF *L, int n, int crystal) {
    for (int l = 0; l < n; l++) {
      DetLayer d = {L[l].density, L[l].thickness, (int)q.els.size(), L[l].n_elements, crystal, 0};
      for (int k = 0; k < L[l].n_elements; k++) {
        const auto it = std::find(q.atoms.begin(), q.atoms.end(), L[l].Z[k]);
        q.els.push_back({L[l].weight[k], (int)(it - q.atoms.begin()), 0});
        if (it == q.atoms.end()) q.atoms.push_back(L[l].Z[k]);
      }
      q.lay.push_back(d);
    }
  };
  layers(in->det_layers, in->n_det_layers, 0);
  layers(in->crystal_layers, in->n_crystal_layers, 1);
  if (q.lay.size() * sizeof(DetLayer) + q.els.size() * sizeof(DetEl) > DET_LAYER_BYTES) q.host_front = 1;
  if (!er) return;
  const int nch = in->detector.nchannels;
  const double gain = in->detector.gain, zero = in->detector.zero;
  const int nfe = er->n_fluo_input_energies, nce = er->n_compton_input_energies, nco = er->n_compton_output_energies;
  const double *fe = er->fluo_escape_input_energies, *ci = er->compton_escape_input_energies,
               *co = er->compton_escape_output_energies;
  if (!(gain > 0.0) || !det_increasing(fe, nfe) || !det_increasing(ci, nce) || !det_increasing(co, nco) ||
      (long)nfe + nce + nco > DET_ESC_AXES || er->n_elements > DET_ESC_LINES / esc_line_count()) {
    q.host_front = 1;
    return;
  }
  for (int j = 0; j < er->n_elements; j++) {
    const xrl_atom *a = xrl_atom_get(er->Z[j]);
    for (int sh = 0; sh < 4; sh++)
      for (int line = esc_shell_first[sh]; line <= esc_shell_last[sh]; line++)
        q.lines.push_back({a->line_energy[line], a->edge[sh], (line - 1) * er->n_elements + j, 0});
  }
  q.axes.assign(fe, fe + nfe);
  q.axes.insert(q.axes.end(), ci, ci + nce);
  q.axes.insert(q.axes.end(), co, co + nco);
  /* the largest difference of two channel energies, with a margin for its rounding */
  const double diff = ((double)(nch - 1) * gain) * (1.0 + 1e-9) + 1e-9 * (fabs(zero) + 1.0);
  q.nrow = std::min((long)nco, (long)(std::lower_bound(co, co + nco, diff) - co) + 1);
  if (2 * q.nrow + 2 * 109l * er->n_elements > DET_ESC_WORDS) q.host_front = 1;
}

/* carves the device buffers of n_ord orders out of base; returns their size */
struct DetCarve {
  char *p;
  size_t n;
  template <typename T>
  T *take(size_t count) {
    T *r = (T *)(p + n);
    n += (count * sizeof(T) + 255) & ~(size_t)255;
    return r;
  }
};
struct DetDev {
  DetBufs b;
  DetLayer *lay;
  DetEl *els;
  xrl_atom *atoms;
  DetEscLine *lines;
  double *axes, *tab;
};
static size_t det_carve(void *base, size_t nch, size_t n_ord, const DetInput &q, DetDev *o) {
  DetCarve c = {(char *)base, 0};
  DetBufs &b = o->b;
  for (double **f : {&b.A0, &b.B0, &b.T, &b.Q, &b.alfa, &b.esum, &b.eself}) *f = c.take<double>(nch);
  b.ep1 = c.take<int>(nch);
  b.epf = c.take<int>(nch);
  o->lay = c.take<DetLayer>(q.lay.size());
  o->els = c.take<DetEl>(q.els.size());
  o->atoms = c.take<xrl_atom>(q.atoms.size());
  o->lines = c.take<DetEscLine>(q.lines.size());
  o->axes = c.take<double>(q.axes.size());
  o->tab = c.take<double>(q.axes.empty() ? 0 : DET_ESC_WORDS);
  for (double **f : {&b.src, &b.tmp, &b.w, &b.conv, &b.cdf}) *f = c.take<double>(n_ord * nch);
  b.hist = c.take<unsigned long long>(n_ord * nch);
  b.guide = c.take<int>(n_ord * (DET_GUIDE + 1));
  b.trains = c.take<DetTrains>(n_ord);
  return c.n;
}

/* host memory of the copies: page-locked in a workspace, else the heap's,
 * not cleared (a call writes what it copies; clearing the 8 MB of the escape
 * tables' part took the allocation-free response of 1024 channels from 0.25 to
 * 0.30 ms, its first call from 0.6 to 2.2 ms) */
struct DetStage {
  char *p = nullptr;
  size_t n = 0;
  bool locked = false;
  ~DetStage() { release(); }
  void release() {
    if (p && locked) (void)hipHostFree(p);
    else free(p);
    p = nullptr;
    n = 0;
  }
  hipError_t ensure(size_t bytes) {
    if (bytes <= n) return hipSuccess;
    release();
    hipError_t e = hipSuccess;
    if (locked) e = hipHostMalloc((void **)&p, bytes, hipHostMallocDefault);
    else if (!(p = (char *)malloc(bytes))) e = hipErrorOutOfMemory;
    if (e == hipSuccess) n = bytes;
    else p = nullptr;
    return e;
  }
};

/* the escape peaks of a group of orders: the sources in ranges whose part
 * of the tables fits DET_ESC_WORDS, each uploaded to dv.tab */
static int det_escape_device(const DetResp &d, const DetInput &q, const DetDev &dv, const xmi_escape_ratios *er,
                             int n_ord, double *stage, hipStream_t st) {
  DetEsc s;
  memset(&s, 0, sizeof(s));
  s.nfe = er->n_fluo_input_energies;
  s.nci = er->n_compton_input_energies;
  s.nco = er->n_compton_output_energies;
  s.fe = dv.axes;
  s.ci = s.fe + s.nfe;
  s.co = s.ci + s.nci;
  s.line = dv.lines;
  s.nline = (int)q.lines.size();
  s.ncol_f = 109 * er->n_elements;
  s.out_diff = s.nco > 1 ? q.axes[s.nfe + s.nci + 1] - q.axes[s.nfe + s.nci] : 1.0;
  /* position of source i on an axis, -1 outside (det_axis_pos on the host) */
  auto pos = [&](const double *a, int n, int i) -> int {
    const double e = ((double)i + 0.5) * d.gain + d.zero;
    if (!(e >= a[0] && e < a[n - 1])) return -1;
    if (fabs(e - a[0]) < 1e-10) return 0;
    return (int)(std::lower_bound(a, a + n, e) - a) - 1;
  };
  const double *fe = q.axes.data(), *ci = fe + s.nfe;
  int i0 = 0;
  while (i0 < d.nch) {
    int f0 = -1, f1 = -1, c0 = -1, c1 = -1, i1 = i0;
    for (; i1 < d.nch; i1++) {
      const int f = pos(fe, s.nfe, i1), c = pos(ci, s.nci, i1);
      const int nf0 = f0 < 0 ? f : f0, nf1 = f >= 0 ? f : f1, nc0 = c0 < 0 ? c : c0, nc1 = c >= 0 ? c : c1;
      const long words = (nf0 >= 0 ? (long)(nf1 - nf0 + 2) * s.ncol_f : 0) +
                         (nc0 >= 0 ? (long)(nc1 - nc0 + 2) * q.nrow : 0);
      if (words > DET_ESC_WORDS) break;
      f0 = nf0;
      f1 = nf1;
      c0 = nc0;
      c1 = nc1;
    }
    const size_t wf = f0 >= 0 ? (size_t)(f1 - f0 + 2) * s.ncol_f : 0;
    s.i0 = i0;
    s.i1 = i1;
    s.f0 = f0 >= 0 ? f0 : 0;
    s.c0 = c0 >= 0 ? c0 : 0;
    s.nc = c0 >= 0 ? c1 - c0 + 2 : 0;
    s.first = i0 == 0;
    s.last = i1 == d.nch;
    if (!s.first) DET_TRY(hipStreamSynchronize(st)); /* the staging memory is still being copied */
    if (wf) memcpy(stage, er->fluo_escape_ratios + (size_t)f0 * s.ncol_f, wf * sizeof(double));
    for (long r = 0; s.nc && r < q.nrow; r++)
      memcpy(stage + wf + (size_t)r * s.nc, er->compton_escape_ratios + (size_t)r * s.nci + c0, s.nc * sizeof(double));
    const size_t words = wf + (size_t)s.nc * q.nrow;
    if (words) DET_TRY(hipMemcpyAsync(dv.tab, stage, words * sizeof(double), hipMemcpyHostToDevice, st));
    s.fluo = dv.tab;
    s.compt = dv.tab + wf;
    hipLaunchKernelGGL(k_det_esc_src, dim3(i1 - i0), dim3(256), 0, st, d, s, dv.b);
    hipLaunchKernelGGL(k_det_esc, dim3(d.nch), dim3(256), 0, st, d, s, dv.b, n_ord);
    DET_TRY(hipGetLastError());
    i0 = i1;
  }
  return 1;
}

/* the response of every order into channels_conv[n] (nch doubles each,
 * owned by the caller), src/xmi_detector_f.F90:219-580; 1 on success.  block:
 * device memory for the buffers of `group` orders (det_carve) */
static int det_convolute(const xmi_inputF *in, double **channels_noconv, double **channels_conv,
                         double *brute_history, double *var_red_history, const xmi_main_options *options,
                         const xmi_escape_ratios *er, int n_interactions_all, int zero_interaction, const DetInput &q,
                         void *block, int group, DetStage &stage, hipStream_t st) {
  const int nch = in->detector.nchannels;
  const int n_int = in->general.n_interactions_trajectory;
  DetResp d;
  d.zero = in->detector.zero;
  d.gain = in->detector.gain;
  d.a = in->detector.noise * in->detector.noise;
  /* the reference writes (2.3548)**2 * 3.85 with default-real literals */
  d.b = (double)((2.3548f * 2.3548f) * 3.85f) * in->detector.fano / 1000.0;
  d.c = sqrt(2.0) / (2.0 * sqrt(2.0 * log(2.0)));
  d.nch = nch;
  d.type = (int)in->detector.detector_type;
  const uint64_t seed = xmi_engine_current_seed(options);
  const int escape = er && !q.host_front;
  /* without an order the device has nothing to do, and no copy may be under
   * way when the staging memory goes back to its owner */
  const int first = zero_interaction ? 0 : 1, any_order = first <= n_interactions_all;
  std::vector<double> eff;
  if (q.host_front && any_order) {
    eff.resize(nch);
    for (int i = 0; i < nch; i++) eff[i] = det_efficiency(in, i * d.gain + d.zero);
  }
  /* staging: inputs that every group shares, the group's spectra, the escape
   * tables, the results */
  auto up = [](size_t bytes) { return (bytes + 255) & ~(size_t)255; };
  DetDev dv;
  (void)det_carve(block, nch, group, q, &dv);
  const size_t n_const = (size_t)((char *)dv.tab - (char *)dv.lay), n_spec = up((size_t)group * nch * sizeof(double));
  const size_t n_tab = escape ? DET_ESC_WORDS * sizeof(double) : 0;
  if (any_order) DET_TRY(stage.ensure(n_const + n_spec + n_tab + n_spec + up(group * sizeof(DetTrains))));
  char *s_spec = stage.p + n_const, *s_tab = s_spec + n_spec, *s_out = s_tab + n_tab, *s_tr = s_out + n_spec;
  if (any_order) {
    auto put = [&](const void *dst, const void *src, size_t bytes) {
      if (bytes) memcpy(stage.p + ((const char *)dst - (const char *)dv.lay), src, bytes);
    };
    put(dv.lay, q.lay.data(), q.lay.size() * sizeof(DetLayer));
    put(dv.els, q.els.data(), q.els.size() * sizeof(DetEl));
    for (size_t k = 0; k < q.atoms.size(); k++) put(dv.atoms + k, xrl_atom_get(q.atoms[k]), sizeof(xrl_atom));
    put(dv.lines, q.lines.data(), q.lines.size() * sizeof(DetEscLine));
    put(dv.axes, q.axes.data(), q.axes.size() * sizeof(double));
    if (n_const) DET_TRY(hipMemcpyAsync(dv.lay, stage.p, n_const, hipMemcpyHostToDevice, st));
  }
  /* net-line histories: rows with counts and the detector absorption at
   * their line energies, formed while the device works */
  std::vector<std::pair<double *, double>> rows;
  bool rows_done = false;
  auto absorb_rows = [&]() {
    for (double *hist : {var_red_history, brute_history}) {
      if (!hist) continue;
      for (int Z = 1; Z <= 100 && Z <= XMI_MAXZ; Z++) {
        const xrl_atom *a = xrl_atom_get(Z);
        if (!a) continue;
        for (int line = 1; line <= 383; line++) {
          double *c = hist + ((size_t)(Z - 1) * 385 + (line - 1)) * n_int;
          bool any = false;
          for (int i = 0; i < n_int; i++) any |= c[i] > 0.0;
          if (any && a->line_energy[line] > 0.0) rows.push_back({c, det_efficiency(in, a->line_energy[line])});
        }
      }
    }
    rows_done = true;
  };
  const int nb = (nch + 255) / 256;
  for (int n0 = first; n0 <= n_interactions_all; n0 += group) {
    const int n_ord = std::min(group, n_interactions_all - n0 + 1);
    for (int n = 0; n < n_ord; n++) {
      double *t = (double *)s_spec + (size_t)n * nch;
      memcpy(t, channels_noconv[n0 + n], nch * sizeof(double));
      if (q.host_front) {
        std::vector<double> temp(t, t + nch);
        for (int i = 0; i < nch; i++) temp[i] *= eff[i];
        if (er) det_escape(temp, in, er);
        memcpy(t, temp.data(), nch * sizeof(double));
      }
    }
    DET_TRY(hipMemcpyAsync(dv.b.src, s_spec, (size_t)n_ord * nch * sizeof(double), hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_det_prep, dim3((nch + 63) / 64), dim3(64), 0, st, d, dv.b, dv.lay, (int)q.lay.size(), dv.els,
                       dv.atoms, n_ord, q.host_front ? 0 : 1);
    DET_TRY(hipGetLastError());
    if (escape && !det_escape_device(d, q, dv, er, n_ord, (double *)s_tab, st)) return 0;
    if (options->use_sum_peaks) {
      hipLaunchKernelGGL(k_det_cdf, dim3(n_ord), dim3(1024), 0, st, nch, dv.b, escape);
      hipLaunchKernelGGL(k_det_pileup, dim3(DET_PULSE_THREADS / 256, n_ord), dim3(256), 0, st, nch, dv.b,
                         in->detector.live_time, in->detector.pulse_width, d.zero, d.gain, seed, n0);
      DET_TRY(hipGetLastError());
      DET_TRY(hipMemcpyAsync(s_tr, dv.b.trains, n_ord * sizeof(DetTrains), hipMemcpyDeviceToHost, st));
    }
    hipLaunchKernelGGL(k_det_norm, dim3(nch), dim3(256), 0, st, d, dv.b, n_ord, escape, options->use_sum_peaks ? 1 : 0);
    hipLaunchKernelGGL(k_det_conv, dim3(nch), dim3(256), 0, st, d, dv.b, n_ord);
    if (options->use_poisson)
      hipLaunchKernelGGL(k_det_poisson, dim3(nb, n_ord), dim3(256), 0, st, nch, dv.b.conv, seed, (uint32_t)n0);
    DET_TRY(hipGetLastError());
    DET_TRY(hipMemcpyAsync(s_out, dv.b.conv, (size_t)n_ord * nch * sizeof(double), hipMemcpyDeviceToHost, st));
    if (!rows_done) absorb_rows();
    DET_TRY(hipStreamSynchronize(st));
    if (options->use_sum_peaks)
      for (int n = 0; n < n_ord; n++)
        if (((const DetTrains *)s_tr)[n].over) { /* src/xmi_detector_f.F90:152-156 stops the program here */
          xmi_set_error("detector response: pulse train maximum (100 pulses) reached %u times; adjust the pulse "
                        "width or disable the pile-up generation", ((const DetTrains *)s_tr)[n].over);
          return 0;
        }
    for (int n = 0; n < n_ord; n++)
      memcpy(channels_conv[n0 + n], (double *)s_out + (size_t)n * nch, nch * sizeof(double));
  }
  if (!zero_interaction) memset(channels_conv[0], 0, nch * sizeof(double));
  if (!rows_done) absorb_rows();
  for (const auto &r : rows)
    for (int i = 0; i < n_int; i++)
      if (r.first[i] > 0.0) r.first[i] *= r.second;
  return 1;
}

/* workspaces of xmi_detector_convolute_all: a stream, device memory and
 * page-locked staging, each taken by one call at a time.  At most
 * DET_POOL wait for the next call, with at most DET_KEEP bytes each; the
 * others are released when their call ends, the waiting ones by
 * xmi_detector_release_workspaces.  A workspace's memory is used on its own
 * stream only, which therefore need not be ordered with the null stream: it
 * is created non-blocking, so that a waiting workspace does not take part in
 * other work's synchronisations. */
#define DET_POOL 4
#define DET_KEEP ((size_t)64 << 20)
struct DetWork {
  int dev = -1;
  hipStream_t st = nullptr;
  void *block = nullptr;
  size_t n = 0;
  DetStage stage;
  ~DetWork() {
    if (block) (void)hipFree(block);
    stage.release();
    if (st) (void)hipStreamDestroy(st);
  }
};
static std::mutex g_pool_mutex;
static std::vector<DetWork *> *g_det_pool = new std::vector<DetWork *>(); /* not destroyed: the runtime may end first */

static DetWork *det_take_work(size_t bytes, hipError_t *e) {
  int dev = 0;
  if ((*e = hipGetDevice(&dev)) != hipSuccess) return nullptr;
  DetWork *w = nullptr;
  {
    std::lock_guard<std::mutex> g(g_pool_mutex);
    for (size_t k = 0; k < g_det_pool->size(); k++)
      if ((*g_det_pool)[k]->dev == dev) {
        w = (*g_det_pool)[k];
        g_det_pool->erase(g_det_pool->begin() + k);
        break;
      }
  }
  if (!w) {
    w = new DetWork();
    w->dev = dev;
    w->stage.locked = true;
    *e = hipStreamCreateWithFlags(&w->st, hipStreamNonBlocking);
  }
  if (*e == hipSuccess && w->n < bytes) {
    if (w->block) (void)hipFree(w->block);
    w->block = nullptr;
    w->n = 0;
    if ((*e = hipMalloc(&w->block, bytes)) == hipSuccess) w->n = bytes;
  }
  if (*e != hipSuccess) {
    delete w;
    return nullptr;
  }
  return w;
}

static void det_give_work(DetWork *w, bool ok) {
  if (ok && w->n <= DET_KEEP && w->stage.n <= DET_KEEP) {
    std::lock_guard<std::mutex> g(g_pool_mutex);
    if (g_det_pool->size() < DET_POOL) {
      g_det_pool->push_back(w);
      return;
    }
  }
  (void)hipStreamSynchronize(w->st);
  delete w;
}

extern "C" int64_t xmi_detector_release_workspaces(void) {
  std::vector<DetWork *> idle;
  int64_t bytes = 0;
  {
    std::lock_guard<std::mutex> g(g_pool_mutex);
    idle.swap(*g_det_pool);
  }
  for (DetWork *w : idle) {
    bytes += (int64_t)(w->n + w->stage.n);
    delete w; /* their calls have synchronised */
  }
  return bytes;
}

/* orders of one group: as many as `bytes` of device memory hold, at least one */
static int det_group(size_t nch, int n_ord, const DetInput &q, size_t bytes) {
  DetDev dv;
  int g = n_ord < 1 ? 1 : n_ord;
  while (g > 1 && det_carve(nullptr, nch, g, q, &dv) > bytes) g--;
  return g;
}

extern "C" void xmi_detector_convolute_all(xmi_inputFPtr inputFPtr, double **channels_noconv, double **channels_conv,
                                           double *brute_history, double *var_red_history, xmi_main_options *options,
                                           xmi_escape_ratios *escape_ratios, int n_interactions_all,
                                           int zero_interaction) {
  const xmi_inputF *in = (const xmi_inputF *)inputFPtr;
  const size_t nch = (size_t)in->detector.nchannels;
  for (int n = 0; n <= n_interactions_all; n++) channels_conv[n] = nullptr;
  const xmi_escape_ratios *er = options->use_escape_peaks ? escape_ratios : nullptr;
  DetInput q;
  det_input(in, er, q);
  const int group = det_group(nch, n_interactions_all + 1 - (zero_interaction ? 0 : 1), q, DET_KEEP);
  DetDev dv;
  hipError_t e = hipSuccess;
  int ok = 0;
  DetWork *w = det_take_work(det_carve(nullptr, nch, group, q, &dv), &e);
  if (!w) {
    xmi_set_error("detector response: device allocation: %s", hipGetErrorString(e));
  } else {
    for (int n = 0; n <= n_interactions_all; n++) channels_conv[n] = (double *)malloc(nch * sizeof(double));
    ok = det_convolute(in, channels_noconv, channels_conv, brute_history, var_red_history, options, er,
                       n_interactions_all, zero_interaction, q, w->block, group, w->stage, w->st);
    det_give_work(w, ok);
  }
  if (!ok) /* no partial result: every order's pointer is NULL after a failure */
    for (int n = 0; n <= n_interactions_all; n++) {
      free(channels_conv[n]);
      channels_conv[n] = nullptr;
    }
}

/* ---- the allocation-free variant ------------------------------------------
 * The buffers live in this file-scope array; each device holds its own copy,
 * found once per device through hipGetSymbolAddress.  Calls that overlap on
 * one device share the array and race.  It holds one order of
 * DET_NOALLOC_MAX_CHANNELS channels with every element's atom and the escape
 * tables of one launch (22 MB); orders beyond what fits go in groups. */
#define DET_NOALLOC_MAX_CHANNELS 65536
#define DET_SCRATCH_BYTES ((size_t)32 << 20)
static __device__ __align__(256) unsigned char scratch[DET_SCRATCH_BYTES];
/* one order of the largest spectrum with the largest tables fits (det_carve:
 * 24 arrays, each rounded up to 256 bytes; its bounds are det_input's) */
static_assert((size_t)DET_NOALLOC_MAX_CHANNELS * (13 * sizeof(double) + 2 * sizeof(int)) + DET_LAYER_BYTES +
                      94 * sizeof(xrl_atom) + DET_ESC_LINES * sizeof(DetEscLine) +
                      (DET_ESC_AXES + DET_ESC_WORDS) * sizeof(double) + (DET_GUIDE + 1) * sizeof(int) +
                      sizeof(DetTrains) + 24 * 256 <=
                  DET_SCRATCH_BYTES,
              "the allocation-free response's buffers fit its array");

#define DET_MAX_DEVICES 64
static void *g_scratch_ptr[DET_MAX_DEVICES];
static std::mutex g_scratch_mutex;

extern "C" int xmi_detector_convolute_all_noalloc(xmi_inputFPtr inputFPtr, double **channels_noconv,
                                                  double **channels_conv, double *brute_history,
                                                  double *var_red_history, xmi_main_options *options,
                                                  xmi_escape_ratios *escape_ratios, int n_interactions_all,
                                                  int zero_interaction) {
  const xmi_inputF *in = (const xmi_inputF *)inputFPtr;
  if (!in || !channels_noconv || !channels_conv || !options) {
    xmi_set_error("xmi_detector_convolute_all_noalloc: NULL argument");
    return 0;
  }
  const int nch = in->detector.nchannels;
  if (nch < 1 || nch > DET_NOALLOC_MAX_CHANNELS) {
    xmi_set_error("xmi_detector_convolute_all_noalloc: %d channels; the allocation-free response holds at most %d",
                  nch, DET_NOALLOC_MAX_CHANNELS);
    return 0;
  }
  for (int n = 0; n <= n_interactions_all; n++)
    if (!channels_conv[n]) {
      xmi_set_error("xmi_detector_convolute_all_noalloc: channels_conv[%d] is NULL (the caller owns the outputs)", n);
      return 0;
    }
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= DET_MAX_DEVICES) {
    xmi_set_error("xmi_detector_convolute_all_noalloc: no usable device (%s)", hipGetErrorString(e));
    return 0;
  }
  void *base = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
      void *p = nullptr;
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess || !p) {
        xmi_set_error("xmi_detector_convolute_all_noalloc: scratch address: %s", hipGetErrorString(e));
        return 0;
      }
      g_scratch_ptr[dev] = p;
    }
    base = g_scratch_ptr[dev];
  }
  const xmi_escape_ratios *er = options->use_escape_peaks ? escape_ratios : nullptr;
  DetInput q;
  det_input(in, er, q);
  const int group = det_group((size_t)nch, n_interactions_all + 1 - (zero_interaction ? 0 : 1), q, DET_SCRATCH_BYTES);
  DetStage stage;
  const int ok = det_convolute(in, channels_noconv, channels_conv, brute_history, var_red_history, options, er,
                               n_interactions_all, zero_interaction, q, base, group, stage, (hipStream_t)0);
  if (!ok) (void)hipStreamSynchronize((hipStream_t)0); /* copies out of the staging memory may be under way */
  return ok;
}

/* the name under which the reference loads a custom detector response
 * (bin/xmimsim.c:516) */
extern "C" void xmi_detector_convolute_all_custom(xmi_inputFPtr inputFPtr, double **channels_noconv,
                                                  double **channels_conv, double *brute_history,
                                                  double *var_red_history, xmi_main_options *options,
                                                  xmi_escape_ratios *escape_ratios, int n_interactions_all,
                                                  int zero_interaction) {
  xmi_detector_convolute_all(inputFPtr, channels_noconv, channels_conv, brute_history, var_red_history, options,
                             escape_ratios, n_interactions_all, zero_interaction);
}
