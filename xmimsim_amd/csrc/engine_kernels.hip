/*
 * engine_kernels.hip -- gfx950 kernels of the photon-history engine.
 *
 * Event-based transport of one batch of histories (reference loop
 * src/xmi_main.F90:1223-1681, variance-reduction branch):
 *
 *   k_source        primary energy, direction, polarisation, entry point
 *                   (src/xmi_main.F90:319-716, 957-1186)
 *   per interaction order n = 1..n_int:
 *     k_step        forced interaction (src/xmi_main.F90:1414-1518), atom and
 *                   interaction-type selection (:1558-1652); appends the
 *                   photon to one of three queues (Rayleigh, Compton, photo),
 *                   counts each wave's events per layer, and computes the
 *                   estimator's geometry of the new point (d_vr_geom)
 *     k_layer_scan, k_layer_base   offsets of the per-layer event lists
 *     k_vr_list, k_vr_cone, k_vr_scatter, k_vr_lines
 *                   detection-weight estimator of every photon at order n
 *                   (src/xmi_variance_reduction.F90:29-726, 949-1101)
 *     k_interact    one launch over the three interaction queues:
 *                   Rayleigh src/xmi_main.F90:1986-2101, Compton :2103-2229
 *                   and 4985-5069, photo-absorption :2231-2411, 5184-5437
 *
 * Random numbers: Philox streams per history (philox.h); the transport stream
 * of order n is consumed as: step, atom, type, then the interaction kernel
 * continues at draw 3.  The estimator has its own stream per order.
 *
 * Regrouping by interaction type keeps every wavefront of the interaction
 * kernels on one code path.  All kernels are FP64 VALU work; nothing here is
 * a dense contraction, so no MFMA is used.
 */
#include <stdlib.h>

#include "engine_kernels.h"


/* read-only tables through the constant address space: wave-uniform reads
 * become scalar loads (the tables are not written while a kernel runs) */
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(4))) T *d_const(const T *p) {
  return (const __attribute__((address_space(4))) T *)p;
}

/* ------------------------------------------------------------------------ */
/* elementary functions on the ranges the kernels use */

/* square root of x > 0 (no scaling: x far from the ends of the range): the
 * hardware's reciprocal root, one coupled Newton step and a residual
 * correction; NaN at 0 */
__device__ __forceinline__ double d_sqrt_pos(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = fma(-h, g, 0.5);
  g = fma(g, r, g);
  h = fma(h, r, h);
  return fma(fma(-g, g, x), h, g);
}

/* sin(pi w) for |w| <= 1/2: w times the polynomial in w^2 that interpolates
 * sin(pi w) / w at the Chebyshev nodes of the interval (relative error below
 * 4e-19 before rounding) */
__device__ __forceinline__ double d_sinpi_core(double w) {
  const double z = w * w;
  double p = fma(z, 0x1.9d462020fcc78p-21, -0x1.6f7acdb8f6580p-16);
  p = fma(z, p, 0x1.e8f3675ee37ddp-12);
  p = fma(z, p, -0x1.e3074dfaf87afp-8);
  p = fma(z, p, 0x1.5078348551854p-4);
  p = fma(z, p, -0x1.32d2cce627c86p-1);
  p = fma(z, p, 0x1.466bc6775aa7dp+1);
  p = fma(z, p, -0x1.4abbce625be52p+2);
  p = fma(z, p, 0x1.921fb54442d18p+1);
  return w * p;
}

/* sin(pi t) and cos(pi t) for |t| <= 1: the sine folded to [0, 1/2], the
 * cosine as the sine of 1/2 - |t| (both differences exact) */
__device__ __forceinline__ double d_sinpi1(double t) {
  const double w = fabs(t);
  return copysign(d_sinpi_core(fmin(w, 1.0 - w)), t);
}
__device__ __forceinline__ double d_cospi1(double t) { return d_sinpi_core(0.5 - fabs(t)); }

/* reciprocal square root of x > 0 far from the ends of the range: the
 * hardware's estimate (2^-24 or better) and one third-order step */
__device__ __forceinline__ double d_rsqrt_pos(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}

/* 1 / x for normal x away from the range's ends: the instruction's seed and
 * one cubic step, a third of an IEEE division's issue */
__device__ __forceinline__ double d_rcp(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, y, 1.0);
  return fma(y, fma(e, e, e), y);
}

/* E^-p of the photo-ionisation cross sections (p = 11/4) for an energy in the
 * provider's range: E^(-1/2) cubed twice times E^(1/4), from two reciprocal
 * square roots; 0 for E <= 0, as xrl_energy */
static_assert(XRL_PHOTO_EXPONENT == 2.75, "d_photo_pe forms E^-11/4");
__device__ __forceinline__ double d_photo_pe(double E) {
  const double a = d_rsqrt_pos(E), a2 = a * a;
  return E > 0.0 ? a2 * a2 * (a2 * d_rsqrt_pos(a)) : 0.0;
}

/* the provider's energy context (xrl_energy) with E^-p as d_photo_pe */
__device__ __forceinline__ xrl_ectx d_energy(double E) {
  xrl_ectx c;
  c.E = E;
  c.pe = c.cf = 0.0;
  c.ci = 0;
  if (!(E > 0.0)) return c;
  const double inv_h = (double)(XRL_NCS - 1) / (XRL_CS_LNE1 - XRL_CS_LNE0);
  const double x = (log(E) - XRL_CS_LNE0) * inv_h;
  int i = (int)floor(x);
  i = i < 0 ? 0 : (i > XRL_NCS - 2 ? XRL_NCS - 2 : i);
  c.ci = i;
  c.cf = x - (double)i;
  c.pe = d_photo_pe(E);
  return c;
}

/* ---- directions ----------------------------------------------------------
 * A photon's frame is e_theta = (ct cp, ct sp, -st), e_phi = (-sp, cp, 0) and
 * its direction d = (st cp, st sp, ct).  The reference keeps the angles and
 * takes their sines and cosines back; here they are read off d itself: ct =
 * dz, st = sqrt(1 - dz^2) (what sin(acos(dz)) gives: beside the axis it
 * carries dz's rounding, as the reference's does), cp and sp from (dx, dy)
 * (cp = 1, sp = 0 on the axis, as atan2(0, 0) = 0).  A turn takes two square
 * roots where it took six sines and cosines, an acos and an atan2, and two
 * words of photon state less: k_interact 193 -> 135 us for 2^21 slots. */
struct DFrame {
  double et[3], ep0, ep1;
  double d[3];
};

/* sqrt(1 - c^2), 0 where rounding has taken |c| to 1 or beyond */
__device__ __forceinline__ double d_sin_of(double c) {
  const double x = (1.0 - c) * (1.0 + c);
  return x > 0.0 ? d_sqrt_pos(x) : 0.0;
}

__device__ __forceinline__ DFrame d_frame(const double *d) {
  const double s2 = fma(d[0], d[0], d[1] * d[1]);
  const double is = d_rsqrt_pos(s2), st = d_sin_of(d[2]);
  const int axis = !(s2 > 0.0);
  const double cp = axis ? 1.0 : d[0] * is, sp = axis ? 0.0 : d[1] * is;
  DFrame f;
  f.et[0] = d[2] * cp;
  f.et[1] = d[2] * sp;
  f.et[2] = -st;
  f.ep0 = -sp;
  f.ep1 = cp;
  f.d[0] = st * cp;
  f.d[1] = st * sp;
  f.d[2] = d[2];
  return f;
}

/* the direction of a frame turned by the polar angle (cosine c, sine s) with
 * the azimuth (cosine ca, sine sa), of unit length again: the length is 1 up
 * to rounding, so one linear step restores it */
__device__ __forceinline__ void d_turn(double *d, const DFrame &f, double c, double s, double ca, double sa) {
  const double v0 = s * ca, v1 = s * sa;
  const double n0 = fma(v0, f.et[0], fma(v1, f.ep0, c * f.d[0]));
  const double n1 = fma(v0, f.et[1], fma(v1, f.ep1, c * f.d[1]));
  const double n2 = fma(v0, f.et[2], c * f.d[2]);
  const double k = fma(-0.5, fma(n0, n0, fma(n1, n1, n2 * n2)), 1.5);
  d[0] = n0 * k;
  d[1] = n1 * k;
  d[2] = n2 * k;
}

/* the polarisation after a turn: its part normal to the new direction */
__device__ __forceinline__ void d_update_elecv(const double *d, double *e) {
  const double c = d_dot(d, e);
  for (int i = 0; i < 3; i++) e[i] = fma(-c, d[i], e[i]);
  const double k = d_rsqrt_pos(d_dot(e, e));
  for (int i = 0; i < 3; i++) e[i] *= k;
}

/* azimuth (cosine, sine) of phi, measured from the polarisation e, in the
 * frame of the direction (src/xmi_main.F90:2034-2060: phi0 + phi, phi0 the
 * arc cosine of e . e_theta with the sign of e . e_phi) */
__device__ __forceinline__ void d_from_polarisation(const DFrame &f, const double *e, double *ca, double *sa) {
  double c0 = e[0] * f.et[0] + e[1] * f.et[1] + e[2] * f.et[2];
  c0 = fmin(fmax(c0, -1.0), 1.0);
  const double s0 = e[0] * f.ep0 + e[1] * f.ep1 < 0.0 ? -d_sin_of(c0) : d_sin_of(c0);
  const double c = *ca, s = *sa;
  *ca = c * c0 - s * s0;
  *sa = s * c0 + c * s0;
}

/* cosine and sine of an azimuth table's angle in [0, 2 pi] */
__device__ __forceinline__ void d_azimuth(double phi, double *c, double *s) {
  const double t = fma(phi, 1.0 / ENG_PI, -1.0);
  *c = -d_cospi1(t);
  *s = -d_sinpi1(t);
}

/* cosine and sine of 2 pi u, u in [0, 1) (2 u - 1 is exact) */
__device__ __forceinline__ void d_turns(double u, double *c, double *s) {
  const double t = fma(2.0, u, -1.0);
  *c = -d_cospi1(t);
  *s = -d_sinpi1(t);
}

/* ------------------------------------------------------------------------ */
/* physics helpers on the device */

/* mass attenuation of a layer, sum_i w_i CS_Total(Z_i, E) (src/xmi_aux_f.F90:1109-1141),
 * from the per-layer tables: equal to the element sum up to rounding, since
 * the layer sums are formed once on the host */
__device__ __forceinline__ double d_cell_mu(const EngineParams &P, int layer0, const LayCell &r, const xrl_ectx &c) {
  double pb = r.pb;
  if (!r.edge_free) {
    /* an edge inside the cell: count the edges above E */
    const int eo = P.lay_eoff[layer0], ne = P.lay_eoff[layer0 + 1] - eo;
    int K = r.K;
    while (K < ne && P.lay_edge[eo + K] > c.E) K++;
    pb = P.lay_pb[eo + layer0 + K];
  }
  return fma(c.pe, pb, fma(c.cf, r.dT, r.T0));
}

__device__ __forceinline__ double d_layer_mu_tab(const EngineParams &P, int layer0, const xrl_ectx *c) {
  if (!(c->E > 0.0)) return 0.0;
  return d_cell_mu(P, layer0, P.lay_cell[(size_t)c->ci * P.n_layers + layer0], *c);
}

__device__ __forceinline__ void d_mu_all(const EngineParams &P, double E, double *mus, size_t stride, size_t idx) {
  xrl_ectx c = d_energy(E);
  for (int l = 0; l < P.n_layers; l++) mus[(size_t)l * stride + idx] = d_layer_mu_tab(P, l, &c);
}

/* this wavefront's sub-counter of a counter slot (1-D launches) */
__device__ __forceinline__ unsigned long long *d_ctr(const EngineParams &P, int slot) {
  const unsigned int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  return &P.counters[(size_t)slot * ENG_SPREAD + (wave & (ENG_SPREAD - 1))];
}

/* wavefront-aggregated counter: call from converged code only */
__device__ __forceinline__ void d_wave_count(unsigned long long *ctr, int pred) {
  unsigned long long m = __ballot(pred);
  if (m != 0ull && __lane_id() == 0) atomicAdd(ctr, (unsigned long long)__popcll(m));
}

/* table value at (x1, x2), rows along x1: on the uniform grids of the
 * generator the cell and the fraction come from the coordinate itself (its
 * rounding, 2e-13 of a cell, is far below the table's), without reading the
 * grids; other grids (a table file may hold any) take d_bilinear */
__device__ __forceinline__ double d_table(int uniform, const double *arr, const double *a1, int n1, double a10,
                                          double a1inv, const double *a2, int n2, double a20, double a2inv, double x1,
                                          double x2) {
  if (!uniform) return d_bilinear(arr, a1, n1, a10, a1inv, a2, n2, a20, a2inv, x1, x2);
  const double t1 = (x1 - a10) * a1inv, t2 = (x2 - a20) * a2inv;
  int p1 = (int)floor(t1), p2 = (int)floor(t2);
  p1 = p1 < 0 ? 0 : (p1 > n1 - 2 ? n1 - 2 : p1);
  p2 = p2 < 0 ? 0 : (p2 > n2 - 2 ? n2 - 2 : p2);
  const double f1 = t1 - (double)p1, f2 = t2 - (double)p2;
  const double *r0 = arr + (size_t)p1 * n2 + p2, *r1 = r0 + n2;
  const double v0 = fma(f2, r0[1] - r0[0], r0[0]), v1 = fma(f2, r1[1] - r1[0], r1[0]);
  return fma(f1, v1 - v0, v0);
}

/* cone-sampling estimate of the detector solid angle seen from (r1, theta1),
 * src/xmi_solid_angle_f.F90:432-710 (same estimator as src/xmi_kernels.cl:219-452).
 * Split in a set-up and a per-trial test: trial i consumes exactly the words
 * 2i and 2i+1 of the stream, so a wavefront can run the trials of one
 * estimate on all its lanes and count exactly the hits of the sequential loop.
 *
 * A trial's direction (c0, c1, x) in the cone's frame, with x = cos theta,
 * c0 = sin theta cos phi and c1 = sin theta sin phi, turns to (c0, v1, v2)
 * with v1 = -st c1 - ct x and v2 = ct c1 - st x, and the ray from (0, l1, l2)
 * meets the plane h below it at (-h c0, l1 v2 - h v1) / v2.  The distance
 * test against a radius is multiplied through by v2^2 (v2 < 0 is tested
 * first) and c0 enters squared only, c0^2 = sin^2 theta - c1^2: one square
 * root and one sine per trial, no division.  q = l1 v2 - h v1 is linear in c1
 * and x; its two factors are formed once per cone.  Bound by vector issue,
 * about 40 % of it the Philox multiplies: 1024 x 1024 cells of 5000 trials
 * take 14.0 ms (25.7 ms with the general sine and cosine, two divisions and
 * two square roots per trial), the off-grid points of a batch 31 us (54). */
struct SaCone {
  double cone_sa;
  double k, k2;             /* (1 - cos apex) per word unit, and half of it */
  double st, ct;
  double qa, qb, l2, R2;    /* window: q = qa c1 + qb x, l2 = h^2, R^2 */
  double oa, ob, oh2, Rc2;  /* collimator top, when the point is outside */
  int outside;
};

/* detector window radius and collimator (radius, height, present) */
struct SaGeom {
  double R, Rc, H;
  int coll;
};

__device__ __forceinline__ SaGeom d_sa_geom(const EngineParams &P) {
  SaGeom g;
  g.R = P.det_radius;
  g.Rc = P.coll_radius;
  g.H = P.coll_height;
  g.coll = P.coll_present;
  return g;
}

/* returns 0 when the collimator hides the detector (estimate 0, no draws) */
__device__ __forceinline__ int d_sa_setup(const SaGeom g, double r1, double theta1, SaCone *c) {
  double r, fcbr, st, ct, s1, c1;
  const double R = g.R, Rc = g.Rc, H = g.H;
  sincos(theta1, &s1, &c1);
  const double l1 = r1 * c1, l2 = r1 * s1;
  int top = 0, outside = 0; /* top: the cone is seen from the collimator's top */
  if (g.coll) {
    if (fabs(Rc - R) < 0.000001) {
      top = !(l1 <= R);
    } else if (!(l1 <= R && l2 <= H * (l1 - R) / (Rc - R))) {
      if (l2 <= H) return 0;
      top = 1;
    }
    outside = l2 > H;
  }
  if (top) {
    r = sqrt(r1 * r1 - 2.0 * l2 * H + H * H);
    ct = l1 / r;
    st = fabs(l2 - H) / r;
    fcbr = Rc;
  } else {
    r = r1;
    ct = c1;
    st = s1;
    fcbr = R;
  }
  /* the larger of the cone's two half angles, as the reference takes it: the
   * cone's size is one minus the rounded cosine, an ulp of which is 1e-14 of
   * the size in cells far from the window.  (A quotient for the cosine would save
   * 1 % of the grid's time; its roundings fall to the other side in 40 % of
   * those cells.) */
  const double beta = atan(fcbr / r);
  double alpha = atan(fcbr * st / (r - fcbr * ct));
  if (alpha <= 0.0) alpha += ENG_PI;
  const double om = 1.0 - cos(beta > alpha ? beta : alpha);
  c->cone_sa = 2.0 * ENG_PI * om;
  c->k = om * (1.0 / 4294967296.0);
  c->k2 = 0.5 * c->k;
  c->st = st;
  c->ct = ct;
  c->qa = l1 * ct + l2 * st;
  c->qb = l2 * ct - l1 * st;
  c->l2 = l2 * l2;
  c->R2 = R * R;
  const double h = l2 - H;
  c->oa = l1 * ct + h * st;
  c->ob = h * ct - l1 * st;
  c->oh2 = h * h;
  c->Rc2 = Rc * Rc;
  c->outside = outside;
  return 1;
}

/* one cone direction from two words at their midpoints, u1 = 1 - cos theta
 * over 1 - cos apex and u2 = phi over 2 pi; 1 if it reaches the window */
__device__ __forceinline__ int d_sa_trial(const SaCone &c, uint32_t w1, uint32_t w2) {
  const double y = fma((double)w1, c.k, c.k2), x = 1.0 - y; /* y = 1 - cos theta */
  const double s2 = y * (2.0 - y);
  /* sin(2 pi u2) = -sin(pi (2 u2 - 1)), 2 u2 - 1 exact */
  const double c1 = -d_sqrt_pos(s2) * d_sinpi1(fma((double)w2, 0x1.0p-31, 0x1.0p-32 - 1.0));
  const double v2 = fma(c.ct, c1, -c.st * x);
  if (!(v2 < 0.0)) return 0;
  const double c0s = fma(-c1, c1, s2), v2s = v2 * v2;
  if (c.outside) {
    const double q = fma(c.oa, c1, c.ob * x);
    if (fma(c.oh2, c0s, q * q) > c.Rc2 * v2s) return 0;
  }
  const double q = fma(c.qa, c1, c.qb * x);
  return fma(c.l2, c0s, q * q) <= c.R2 * v2s;
}

/* cone trials 2 b and 2 b + 1 from block b of a stream (its counter
 * word 0 advanced by b): words 0, 1 and 2, 3, one uniform each */
__device__ __forceinline__ int d_sa_trial_pair(const SaCone &c, const uint32_t *ctr, const uint32_t *key, uint32_t b,
                                               int both) {
  uint32_t o[4];
  const uint32_t cc[4] = {ctr[0] + b, ctr[1], ctr[2], ctr[3]};
  phx_4x32_10(cc, key, o);
  int n = d_sa_trial(c, o[0], o[1]);
  if (both) n += d_sa_trial(c, o[2], o[3]);
  return n;
}

/* sequential estimate (one thread per grid cell): hits trials from blocks
 * 0 .. ceil(hits / 2) - 1 of the cell's stream */
__device__ __forceinline__ double d_single_solid_angle_impl(const SaGeom g, double r1, double theta1, long hits,
                                                           phx_stream *rng) {
  SaCone c;
  if (!d_sa_setup(g, r1, theta1, &c)) return 0.0;
  long nhit = 0;
  for (long i = 0; i < hits; i += 2) nhit += d_sa_trial_pair(c, rng->ctr, rng->key, (uint32_t)(i >> 1), i + 1 < hits);
  return c.cone_sa * (double)nhit / (double)hits;
}


/* ------------------------------------------------------------------------ */
/* solid-angle grid: one thread per (r, theta) cell, Philox stream per cell */

__global__ void __launch_bounds__(ENG_BLOCK) k_solid_angle_grid(EngineParams P, double *grid, const double *rv,
                                                                 const double *tv, int n_r, int n_t, long hits,
                                                                 uint64_t seed) {
  long total = (long)n_r * n_t;
  for (long cell = blockIdx.x * (long)blockDim.x + threadIdx.x; cell < total; cell += (long)gridDim.x * blockDim.x) {
    int jt = (int)(cell / n_r), ir = (int)(cell % n_r);
    phx_stream s = {};
    phx_stream_init(&s, seed, 0u, 0u, PHX_SUB_GRID, (uint64_t)cell);
    grid[cell] = d_single_solid_angle_impl(d_sa_geom(P), rv[ir], tv[jt], hits, &s);
  }
}

/* ------------------------------------------------------------------------ */
/* source */

__device__ double d_gauss(phx_stream *s, double sigma) {
  double u1 = phx_uniform(s), u2 = phx_uniform(s);
  return sigma * sqrt(-2.0 * log(1.0 - u1)) * -d_cospi1(fma(2.0, u2, -1.0));
}

__device__ double d_exc_corr(const SourceTable &S, double E) {
  double corr = 1.0;
  const double *p = S.exc_layers;
  for (int k = 0; k < S.n_exc; k++) {
    double dens = p[0], thick = p[1];
    int nel = (int)p[2];
    double mu = 0.0;
    for (int i = 0; i < nel; i++) mu += xrl_cs_total(&S.exc_atoms[(int)p[3 + i]], E) * p[3 + nel + i];
    corr *= exp(-1.0 * dens * thick * mu);
    p += 3 + 2 * nel;
  }
  return corr;
}

/* trapezoid sampler, src/xmi_aux_f.F90:1836-1941; returns 0 on failure */
__device__ int d_ran_trap(double x1, double x2, double y1, double y2, double u, double *out) {
  double m = (y2 - y1) / (x2 - x1);
  double denom = (x2 - x1) * (y1 - x1 * m) + m * (x2 * x2 - x1 * x1) / 2.0;
  double a = m / 2.0, b = y1 - x1 * m, c = -x1 * y1 + m * x1 * x1 / 2.0 - denom * u;
  double r1 = 0.0, r2 = 0.0;
  int nr;
  if (a == 0.0) {
    if (b == 0.0) return 0;
    r1 = -1.0 * c / b;
    nr = 1;
  } else {
    double delta = b * b - 4.0 * a * c;
    if (delta < 0.0) return 0;
    if (delta == 0.0) {
      r1 = r2 = -b / 2.0 / a;
    } else {
      double sd = sqrt(delta);
      double t1 = (-b + sd) / 2.0 / a, t2 = (-b - sd) / 2.0 / a;
      r1 = t1 < t2 ? t1 : t2;
      r2 = t1 < t2 ? t2 : t1;
    }
    nr = 2;
  }
  if (x1 <= r1 && r1 <= x2) {
    *out = r1;
    return 1;
  }
  if (nr == 2 && x1 <= r2 && r2 <= x2) {
    *out = r2;
    return 1;
  }
  return 0;
}

/* one primary photon; returns 1 when it enters the sample */
__device__ int d_source_one(const EngineParams &P, const PhotonSoA &S, const SourceTable &T, uint64_t batch_start,
                            int i) {
  const uint64_t run = batch_start + (uint64_t)i;
  /* last source with run0 <= run (empty sources share their successor's run0
   * and are skipped): a wave's photons are neighbours in the run order, so the
   * search for its first photon is scalar and the others walk on from there */
  const auto *run0 = d_const(T.run0);
  const uint64_t run_w = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)run) |
                         ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(run >> 32)) << 32);
  int lo = 0, hi = T.n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (run0[mid] <= run_w) lo = mid;
    else hi = mid - 1;
  }
  while (lo + 1 < T.n && T.run0[lo + 1] <= run) lo++;
  const SourceDesc &d = T.d[lo];
  const uint64_t hid = d.hid0 + (run - d.run0);
  const size_t cap = (size_t)P.cap;
  S.layer[i] = 0;
  S.hid[i] = hid; /* the last interaction's line and element are written by the interactions */
  if (P.brute) {
    S.cflags[i] = P.casc;
    if (P.off_half) S.layer[i + P.off_half] = 0; /* no offspring yet */
  }
  if (!d.valid) return 0;
  const long j = (long)(hid - d.hid0);
  phx_stream s;
  phx_stream_init(&s, P.seed, P.sample, 0u, PHX_SUB_SOURCE, hid);

  double E, w, hor = 0.0;
  if (d.kind == 0) {
    if (!d_ran_trap(d.x1, d.x2, d.y1, d.y2, phx_uniform(&s), &E)) {
      atomicAdd(d_ctr(P, ENG_CNT_ERRORS), 1ull);
      atomicAdd(d_ctr(P, ENG_CNT_ERR_SOURCE), 1ull);
      return 0;
    }
    hor = d_interp(d.x1, d.h1, d.x2, d.h2, E) / d_interp(d.x1, d.y1, d.x2, d.y2, E);
    w = d.weight * d_exc_corr(T, E);
    d_mu_all(P, E, S.mus, cap, i);
  } else {
    if (d.dist == 1) {
      E = d_gauss(&s, d.scale) + d.energy;
      if (E <= 1.0 || E > 200.0) return 0;
      d_mu_all(P, E, S.mus, cap, i);
    } else if (d.dist == 2) {
      E = d.scale * tan(ENG_PI * (phx_uniform(&s) - 0.5)) + d.energy;
      if (E <= 1.0 || E > 200.0) return 0;
      d_mu_all(P, E, S.mus, cap, i);
    } else {
      E = d.energy;
      for (int l = 0; l < P.n_layers; l++) S.mus[(size_t)l * cap + i] = T.line_mus[(size_t)lo * P.n_layers + l];
    }
    w = d.weight;
  }

  /* xmi_coords_dir, src/xmi_main.F90:957-1136 */
  double dirv[3], coords[3], x1, y1;
  if (fabs(d.sx * d.sy) < 1.0e-20) {
    x1 = P.slit_ax * (-1.0 + 2.0 * phx_uniform(&s));
    y1 = P.slit_ay * (-1.0 + 2.0 * phx_uniform(&s));
    coords[0] = coords[1] = coords[2] = 0.0;
  } else {
    x1 = d_gauss(&s, d.sxp);
    y1 = d_gauss(&s, d.syp);
    coords[0] = d_gauss(&s, d.sx) - P.d_source_slit * sin(x1);
    coords[1] = d_gauss(&s, d.sy) - P.d_source_slit * sin(y1);
    coords[2] = 0.0;
  }
  if (fabs(x1) < 0.5 * ENG_PI && fabs(y1) < 0.5 * ENG_PI) {
    const double tx = x1 * (1.0 / ENG_PI), ty = y1 * (1.0 / ENG_PI);
    dirv[0] = d_sinpi_core(tx) / d_cospi1(tx);
    dirv[1] = d_sinpi_core(ty) / d_cospi1(ty);
  } else {
    dirv[0] = tan(x1);
    dirv[1] = tan(y1);
  }
  dirv[2] = 1.0;
  d_normalize(dirv); /* rounded as the reference's: the frame of a beam along z hangs on the last bit of dz */

  double ev[3];
  if (d.pol == 1) {
    /* escape-ratio runs: a random polarisation azimuth in the x-y plane */
    d_turns(phx_uniform(&s), &ev[0], &ev[1]);
    ev[2] = 0.0;
  } else {
    int horizontal;
    if (d.kind == 0) horizontal = phx_uniform(&s) <= hor;
    else horizontal = (double)(j + 1) <= d.hor_ver_ratio;
    ev[0] = horizontal ? 0.0 : 1.0;
    ev[1] = horizontal ? 1.0 : 0.0;
    ev[2] = 0.0;
  }
  double cosalfa = d_dot(ev, dirv);
  if (fabs(cosalfa) > 1.0) {
    atomicAdd(d_ctr(P, ENG_CNT_ERRORS), 1ull);
      atomicAdd(d_ctr(P, ENG_CNT_ERR_SOURCE), 1ull);
    return 0;
  }
  const double c_ae = d_rsqrt_pos((1.0 - cosalfa) * (1.0 + cosalfa));
  for (int k = 0; k < 3; k++) ev[k] = c_ae * fma(-cosalfa, dirv[k], ev[k]);

  /* xmi_photon_shift_first_layer */
  int layer = 0;
  if (coords[2] >= P.layer_zb[0]) {
    for (int l = 0; l < P.n_layers; l++)
      if (coords[2] < P.layer_ze[l]) {
        layer = l + 1;
        break;
      }
    if (layer == 0) {
      atomicAdd(d_ctr(P, ENG_CNT_ERRORS), 1ull);
      atomicAdd(d_ctr(P, ENG_CNT_ERR_SOURCE), 1ull);
      return 0;
    }
  } else {
    double pp[3] = {0.0, 0.0, P.layer_zb[0]}, ip[3];
    if (!d_intersect(pp, P.n_sample, coords, dirv, ip)) {
      atomicAdd(d_ctr(P, ENG_CNT_ERRORS), 1ull);
      atomicAdd(d_ctr(P, ENG_CNT_ERR_SOURCE), 1ull);
      return 0;
    }
    coords[0] = ip[0];
    coords[1] = ip[1];
    coords[2] = ip[2];
    layer = 1;
  }
  S.x[i] = coords[0];
  S.y[i] = coords[1];
  S.z[i] = coords[2];
  S.dx[i] = dirv[0];
  S.dy[i] = dirv[1];
  S.dz[i] = dirv[2];
  S.ex[i] = ev[0];
  S.ey[i] = ev[1];
  S.ez[i] = ev[2];
  S.energy[i] = E;
  S.weight[i] = w;
  S.layer[i] = layer;
  return 1;
}

/* the batch's primaries: positions batch_start .. batch_start + count - 1
 * of the run order, or, with a batch queue Q, those of the batch that
 * k_batch_next popped; then slots count .. limit - 1 (limit: the launch's
 * count argument) are marked empty */
__global__ void __launch_bounds__(ENG_BLOCK) k_source(EngineParams P, PhotonSoA S, SourceTable T,
                                                       uint64_t batch_start, int count, const BatchQueue *Q) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, limit = count;
  if (Q) {
    batch_start = Q->start;
    count = Q->count;
  }
  int alive = 0;
  if (i < count) {
    alive = d_source_one(P, S, T, batch_start, i);
  } else if (i < limit) {
    S.layer[i] = 0;
    if (P.off_half) S.layer[i + P.off_half] = 0;
  }
  d_wave_count(d_ctr(P, ENG_CNT_HISTORIES), alive);
}

/* the device batch queue: k_batch_init before a run's first replay, then
 * k_batch_next, the first node of every replay, pops the next batch of at
 * most cap positions (one thread each) */
__global__ void k_batch_init(BatchQueue *Q, unsigned long long total) {
  Q->next = 0ull;
  Q->total = total;
  Q->start = 0ull;
  Q->count = 0;
}

__global__ void k_batch_next(BatchQueue *Q, int cap) {
  const unsigned long long s = Q->next, left = Q->total > s ? Q->total - s : 0ull;
  const int c = left < (unsigned long long)cap ? (int)left : cap;
  Q->start = s;
  Q->count = c;
  Q->next = s + (unsigned long long)c;
}

/* ------------------------------------------------------------------------ */
/* queues */

__global__ void k_reset_queues(EngineParams P) {
  if (threadIdx.x < ENG_NQUEUES * ENG_SPREAD) P.qcount[threadIdx.x] = 0ull;
  if (threadIdx.x == 0 && P.ocount_out) *P.ocount_out = 0u;
}

/* wavefront-aggregated append of the lanes with pred to queue t, in this
 * wave's sub-queue: one atomic per wave, spread over ENG_SPREAD counters.  A
 * sub-queue receives the photons of every ENG_SPREAD-th wave of a launch with
 * one thread per photon slot, so qreg = ceil(waves / ENG_SPREAD) * 64 entries
 * cannot overflow.  Call from converged code. */
__device__ __forceinline__ void d_append(const EngineParams &P, int t, int pred, int idx) {
  const unsigned int j = ((blockIdx.x * blockDim.x + threadIdx.x) >> 6) & (ENG_SPREAD - 1);
  unsigned long long mask = __ballot(pred);
  if (mask == 0ull) return;
  int lane = __lane_id();
  int leader = __ffsll((long long)mask) - 1;
  unsigned int base = 0;
  if (lane == leader)
    base = (unsigned int)atomicAdd(&P.qcount[(size_t)t * ENG_SPREAD + j], (unsigned long long)__popcll(mask));
  base = __shfl(base, leader);
  if (pred) {
    unsigned long long below = mask & ((1ull << lane) - 1ull);
    P.queue[((size_t)t * ENG_SPREAD + j) * P.qreg + base + __popcll(below)] = idx;
  }
}

/* the interaction-type queues (Rayleigh, Compton, photo) */
__device__ __forceinline__ void d_enqueue(const EngineParams &P, int type, int idx) {
  for (int t = 0; t < 3; t++) d_append(P, t, type == t, idx);
}

/* layer lists: k_step stores each wave's number of events per layer (0 = no
 * event), k_layer_scan turns them into offsets, k_vr_list writes the slots.
 * Both launches run one thread per slot with the same workgroups, so a slot
 * has the same wave and lane in both.  Call from converged code. */
__device__ __forceinline__ void d_layer_count(const EngineParams &P, int layer) {
  const unsigned int w = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  for (int L = 1; L <= P.n_layers; L++) {
    const unsigned long long m = __ballot(layer == L);
    if (__lane_id() == 0) P.lay_woff[(size_t)(L - 1) * P.n_waves + w] = __popcll(m);
  }
}

__device__ __forceinline__ void d_layer_list(const EngineParams &P, int layer, int idx) {
  const unsigned int w = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const unsigned long long below = (1ull << __lane_id()) - 1ull;
  for (int L = 1; L <= P.n_layers; L++) {
    const unsigned long long m = __ballot(layer == L);
    if (layer == L) {
      const int pos = P.lay_woff[(size_t)(L - 1) * P.n_waves + w] +
                      P.lay_segbase[(L - 1) * ENG_SCAN_NSEG + (int)(w / ENG_SCAN_SEG)] + __popcll(m & below);
      if ((unsigned int)pos < (unsigned int)P.cap) P.lay_list[(size_t)(L - 1) * P.cap + pos] = idx;
      else atomicAdd(d_ctr(P, ENG_CNT_ERRORS), 1ull); /* counts of k_step and k_vr_list disagree */
    }
  }
}

/* ------------------------------------------------------------------------ */
/* forced interaction + atom and interaction-type selection */

/* CS_Total_Kissel of element slot j of the layers (xrl_cs_total_c, the same
 * operations on the same values), from its cell record r: the photo sum of the
 * cell's edge count where no edge of the element lies in the cell, else
 * counted from the atom's edges */
__device__ __forceinline__ double d_elem_cs_total(const EngineParams &P, int j, const LayCell &r,
                                                 const xrl_ectx *c) {
  if (!(c->E > 0.0)) return 0.0;
  double pb = r.pb;
  if (!r.edge_free) {
    const xrl_atom *a = &P.atoms[P.el_u[j]];
    pb = a->photo_Bsum[xrl_edges_above(a, c->E)];
  }
  return c->pe * pb + (r.T0 + c->cf * r.dT);
}

/* atom selection and interaction type of the photon in slot i (energy E, now
 * in layer my, whose mass attenuation is mu_cur), from its transport stream
 * after the step's number: S.elem set, the type returned (0 Rayleigh, 1
 * Compton, 2 photo-absorption).  Both choices compare products instead of
 * quotients: one division in all */
__device__ __forceinline__ int d_select(const EngineParams &P, const PhotonSoA &S, int i, double E, int my,
                                        double mu_cur, phx_stream *sp) {
  phx_stream &s = *sp;
  /* atom selection, src/xmi_main.F90:1558-1572 */
  const double target = phx_uniform(&s) * mu_cur;
  int off = P.layer_off[my - 1], nel = P.layer_nel[my - 1];
  double thr = 0.0;
  int sel = nel - 1;
  xrl_ectx ec = d_energy(E);
  {
    /* the next element's record is loaded before this one's test */
    const LayCell *cell = P.el_cell + (size_t)ec.ci * P.n_lay_el + off;
    LayCell rn = cell[0];
    double wn = P.el_w[off];
    for (int k = 0; k < nel; k++) {
      const LayCell r = rn;
      const double w = wn;
      if (k + 1 < nel) {
        rn = cell[k + 1];
        wn = P.el_w[off + k + 1];
      }
      thr = fma(w, d_elem_cs_total(P, off + k, r, &ec), thr);
      if (target < thr) {
        sel = k;
        break;
      }
    }
  }
  S.elem[i] = sel;
  /* interaction type, src/xmi_main.F90:1591-1652 */
  double R3 = phx_uniform(&s);
  int u = P.el_u[off + sel];
  const double *ie = P.ip_E + P.ip_off[u];
  int len = P.ip_off[u + 1] - P.ip_off[u];
  int pos;
  if (fabs(E - ie[0]) < 1e-10) pos = 0;
  else {
    int cell = (int)floor((E - P.ip_acc_E0) * P.ip_acc_inv);
    if (cell < 0) cell = 0;
    if (cell > ENG_IP_ACC - 1) cell = ENG_IP_ACC - 1;
    pos = P.ip_acc[(size_t)u * ENG_IP_ACC + cell];
    while (pos + 2 < len && ie[pos + 1] < E) pos++;
  }
  const double *ir = P.ip_r + P.ip_off[u], *irc = P.ip_rc + P.ip_off[u];
  const double f = (E - ie[pos]) / (ie[pos + 1] - ie[pos]);
  const double pr = fma(ir[pos + 1] - ir[pos], f, ir[pos]);
  const double pc = fma(irc[pos + 1] - irc[pos], f, irc[pos]);
  return (R3 < pr) ? 0 : ((R3 < pc) ? 1 : 2);
}

#define VR_ACTIVE 1
#define VR_UP 2

/* path lengths through the layers from a point of layer cur along the unit
 * direction d, itn = d . n_sample, in travel order: entry k is layer k upwards
 * and layer NL - 1 - k downwards (planes and predicate are then selects of
 * wave-uniform values), 0 where not crossed.  From plane to plane through the
 * rounded points, with the reference's divisions: with z about 100 cm the
 * points carry 1e-14 cm, and a photon that leaves a dense layer from 1e-7 cm
 * below its surface shows another rounding of them at 1e-7 */
template <int NL>
__device__ __forceinline__ void d_layer_walk(const EngineParams &P, const double *from, const double *d, double itn,
                                             int up, int cur, double *dist) {
  double lp[3] = {from[0], from[1], from[2]};
#pragma unroll
  for (int k = 0; k < NL; k++) {
    const double z = up ? P.layer_ze[k] : P.layer_zb[NL - 1 - k];
    const int crossed = up ? k >= cur - 1 && k < P.n_layers : NL - 1 - k <= cur - 1;
    const double diff[3] = {0.0 - lp[0], 0.0 - lp[1], z - lp[2]};
    const double t = d_dot(diff, P.n_sample) / itn;
    const double p[3] = {t * d[0] + lp[0], t * d[1] + lp[1], t * d[2] + lp[2]};
    dist[k] = crossed ? d_distance(lp, p) : 0.0;
#pragma unroll
    for (int j = 0; j < 3; j++) lp[j] = crossed ? p[j] : lp[j];
  }
}

/* the geometry of the detection-weight estimator for the photon of slot i,
 * at its interaction point coords (lab frame) with direction dirv_l in layer
 * cur (src/xmi_variance_reduction.F90:29-330): a point of the detector
 * window, the scattering angle and polarisation azimuth towards it, the path
 * through the layers and its escape probability, the solid angle from the
 * grid (or the slot queued for a cone estimate: *need_sa).  mus: the layers'
 * mass attenuation at the photon's energy.  Writes the photon's estimator
 * record; returns 1 when there is an event (*info set), 0 for a point behind
 * the window plane.
 *
 * The scattering angle enters the cross sections through its cosine c (the
 * half angle's sine is sqrt((1 - c) / 2)) and the azimuth through sin^2 theta
 * cos^2 phi: those two are stored and no angle is formed.  The detector frame
 * is orthonormal, so c and the distance to the window's centre are taken in
 * the lab frame. */
template <int NL>
__device__ __forceinline__ int d_vr_geom(const EngineParams &P, const PhotonSoA &S, const VrSoA &V, int n, int i,
                                         const double *coords, const double *dirv_l, int cur, const double *mus,
                                         int *need_sa, int *info) {
  const size_t cap = (size_t)P.cap;
  phx_stream s;
  phx_stream_init(&s, P.seed, P.sample, (uint32_t)n, PHX_SUB_VARRED, S.hid[i]);
  const double radius = sqrt(phx_uniform(&s)) * P.det_radius;
  double ca, sa;
  d_turns(phx_uniform(&s), &ca, &sa);
  const double rel[3] = {coords[0] - P.p_det[0], coords[1] - P.p_det[1], coords[2] - P.p_det[2]};
  double lpnt[3];
  d_matvec(P.det_inv, rel, lpnt);
  double ld[3] = {-lpnt[0], ca * radius - lpnt[1], sa * radius - lpnt[2]};
  if (ld[0] >= 0.0) return 0;
  const double d2 = d_dot(ld, ld), id = d_rsqrt_pos(d2);
  for (int k = 0; k < 3; k++) ld[k] *= id;
  double nd[3];
  d_matvec(P.det_new, ld, nd);
  const double c0 = d_dot(dirv_l, nd);
  const double c = c0 > 1.0 ? 1.0 : (c0 < -1.0 ? -1.0 : c0);
  /* cosine of the angle between the polarisation and the part of nd normal
   * to the direction, times sin theta, squared */
  double q;
  {
    double proj[3];
    for (int k = 0; k < 3; k++) proj[k] = fma(-c0, dirv_l[k], nd[k]);
    const double ev[3] = {S.ex[i], S.ey[i], S.ez[i]};
    const double pe = d_dot(proj, ev), pp = d_dot(proj, proj) * d_dot(ev, ev);
    double cf = pp > 0.0 ? pe * d_rsqrt_pos(pp) : 0.0;
    cf = cf > 1.0 ? 1.0 : (cf < -1.0 ? -1.0 : cf);
    q = (1.0 - c) * (1.0 + c) * cf * cf;
  }
  const double itn = d_dot(nd, P.n_sample);
  const int up = itn > 0.0;
  /* path to the detector through the layers (0 where not crossed); the layer
   * holding the detector point ends the walk */
  double murhod = 0.0;
  {
    double dd[NL], rest = d2 * id;
    d_layer_walk<NL>(P, coords, nd, itn, up, cur, dd);
#pragma unroll
    for (int k = 0; k < NL; k++) {
      dd[k] = dd[k] <= rest ? dd[k] : rest;
      rest -= dd[k];
      murhod = fma(up ? mus[k] * P.layer_density[k] : mus[NL - 1 - k] * P.layer_density[NL - 1 - k], dd[k], murhod);
    }
#pragma unroll
    for (int l = 0; l < NL; l++)
      if (l < P.n_layers) V.dist[(size_t)l * cap + i] = up ? dd[l] : dd[NL - 1 - l];
  }
  /* solid angle, src/xmi_solid_angle_f.F90:712-801 */
  double omega = 0.0;
  const double r = sqrt(d_dot(rel, rel));
  double tt = acos(fmin(fmax(d_dot(rel, P.n_det) / r, -1.0), 1.0));
  if (tt > ENG_PI / 2.0) tt = ENG_PI - tt;
  const double sth = ENG_PI / 2.0 - tt;
  if (sth >= P.sa_t[0]) {
    if (r > P.sa_r[P.sa_nr - 1] || sth > P.sa_t[P.sa_nt - 1]) {
      *need_sa = 1;
      V.sar[i] = r;
      V.sat[i] = sth;
    } else {
      omega = d_table(P.sa_uniform, P.sa_grid, P.sa_t, P.sa_nt, P.sa_t0, P.sa_tinv, P.sa_r, P.sa_nr, P.sa_r0, P.sa_rinv,
                      sth, r);
    }
  }
  V.ct[i] = c;
  V.q[i] = q;
  V.omega[i] = omega;
  V.pesc[i] = exp(-murhod);
  V.blk[i] = s.ctr[0]; /* two uniforms drawn: block 1, nothing buffered */
  *info = VR_ACTIVE | (up ? VR_UP : 0);
  return 1;
}

/* the layer lists of an order's estimator events: one thread per slot, as
 * the step kernel, whose per-wave counts k_layer_scan has turned into
 * offsets (a photon of layer l with energy above the threshold is listed,
 * with or without an event) */
__global__ void __launch_bounds__(ENG_BLOCK) k_vr_list(EngineParams P, PhotonSoA S, int count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int ev_layer = (i < count && S.layer[i] > 0 && S.energy[i] > 1.0) ? S.layer[i] : 0;
  d_layer_list(P, ev_layer, i);
}

/* NL bounds the layer count; the layers' attenuation is kept by layer and the
 * path lengths in travel order (d_layer_walk), so that register arrays have
 * compile-time indices and the layers' constants are wave-uniform; layers
 * the path does not cross add nothing.
 * EST: the estimator's geometry of the new interaction point follows in the
 * same thread (d_vr_geom), while the photon's record is in registers.
 * Occupancy: as many waves as the registers allow without spills (80 VGPRs up
 * to three layers, 96 for four, 115 for five, 161 for eight).
 * Bound by double-precision issue: 1768 vector instructions at three layers
 * (2487 with angles, a division per layer and choice): 40.9 -> 31.7 ms of the
 * 1e8-history tube run on three layers */
template <int NL, bool EST>
__global__ void __launch_bounds__(ENG_BLOCK) __attribute__((amdgpu_waves_per_eu(NL <= 3 ? 6 : NL <= 4 ? 5 : NL <= 5 ? 4 : 1)))
k_step(EngineParams P, PhotonSoA S, VrSoA V, int n, int count) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  int type = -1, ev_layer = 0, need_sa = 0, info = 0, vr_active = 0;
  const size_t cap = (size_t)P.cap;
  const int cur = i < count ? S.layer[i] : 0;
  if (cur > 0) {
    const double E = S.energy[i];
    if (E < 1.0) {
      S.layer[i] = 0;
    } else {
      phx_stream s;
      phx_stream_init(&s, P.seed, P.sample, (uint32_t)n, PHX_SUB_TRANSPORT, S.hid[i]);
      const double R = phx_uniform(&s);
      const double dirv[3] = {S.dx[i], S.dy[i], S.dz[i]};
      const double coords[3] = {S.x[i], S.y[i], S.z[i]};
      const double itn = d_dot(dirv, P.n_sample);
      const int up = itn > 0.0;
      double mus[NL], md[NL], dist[NL]; /* md: by travel order, as dist */
#pragma unroll
      for (int l = 0; l < NL; l++) mus[l] = l < P.n_layers ? S.mus[(size_t)l * cap + i] : 0.0;
      d_layer_walk<NL>(P, coords, dirv, itn, up, cur, dist);
      double Pabs = 0.0;
#pragma unroll
      for (int k = 0; k < NL; k++) {
        md[k] = up ? mus[k] * P.layer_density[k] : mus[NL - 1 - k] * P.layer_density[NL - 1 - k];
        Pabs = fma(md[k], dist[k], Pabs);
      }
      const double Pabs2 = -expm1(-Pabs);
      const double negln = -log1p(-1.0 * R * Pabs2);
      /* layer of the interaction: first where the optical depth exceeds negln
       * (rounding may leave none: then the own layer) */
      int km = up ? cur - 1 : NL - cur, found = 0;
      double sum = 0.0;
#pragma unroll
      for (int k = 0; k < NL; k++) {
        sum = fma(md[k], dist[k], sum);
        if (!found && sum > negln) {
          km = k;
          found = 1;
        }
      }
      const int my = up ? km + 1 : NL - km;
      double mu_my = mus[0], mrm = md[0];
#pragma unroll
      for (int l = 1; l < NL; l++) {
        if (l == my - 1) mu_my = mus[l];
        if (l == km) mrm = md[l];
      }
      double tsum = 0.0;
#pragma unroll
      for (int k = 0; k < NL; k++)
        if (k < km) tsum += (1.0 - (md[k] / mrm)) * dist[k];
      tsum = tsum + negln / mrm;
      const double pt[3] = {coords[0] + tsum * dirv[0], coords[1] + tsum * dirv[1], coords[2] + tsum * dirv[2]};
      S.x[i] = pt[0];
      S.y[i] = pt[1];
      S.z[i] = pt[2];
      S.weight[i] *= Pabs2;
      S.layer[i] = my;
      /* an estimator event of this order */
      ev_layer = E > 1.0 ? my : 0;

      /* atom and type serve the interaction, which the last order of the
       * estimator path does not launch */
      if (!EST || n < P.n_int) type = d_select(P, S, i, E, my, mu_my, &s);
      if (EST && ev_layer) vr_active = d_vr_geom<NL>(P, S, V, n, i, pt, dirv, my, mus, &need_sa, &info);
    }
  }
  d_enqueue(P, type, i);
  d_layer_count(P, ev_layer);
  if (EST) {
    if (i < count) V.info[i] = info;
    d_append(P, ENG_CNT_Q_SA, need_sa, i);
    d_wave_count(d_ctr(P, ENG_CNT_FALLBACKS), need_sa);
    d_wave_count(d_ctr(P, ENG_CNT_VR), vr_active);
    for (int L = 1; L <= P.n_layers; L++) d_wave_count(d_ctr(P, ENG_CNT_LAYER0 + L - 1), vr_active && ev_layer == L);
  }
}

/* exclusive scan of the per-wave counts in segments of ENG_SCAN_SEG waves:
 * workgroup (segment, layer) scans its segment in place (coalesced, one
 * count per thread) and stores the segment's total; k_layer_base then turns
 * the totals into segment offsets and each layer's total.  nw = waves of the
 * k_step launch, at most ENG_SCAN_SEG * ENG_SCAN_NSEG. */
__global__ void __launch_bounds__(ENG_SCAN_SEG) k_layer_scan(EngineParams P, int nw) {
  __shared__ int wsum[ENG_SCAN_SEG / 64];
  const int seg = blockIdx.x, L0 = blockIdx.y;
  int *row = P.lay_woff + (size_t)L0 * P.n_waves;
  const int k = seg * ENG_SCAN_SEG + threadIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int v = k < nw ? row[k] : 0;
  int incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int t = __shfl_up(incl, off);
    if (lane >= off) incl += t;
  }
  if (lane == 63) wsum[w] = incl;
  __syncthreads();
  int base = 0;
  for (int j = 0; j < w; j++) base += wsum[j];
  if (k < nw) row[k] = base + incl - v;
  if (threadIdx.x == ENG_SCAN_SEG - 1) P.lay_segbase[L0 * ENG_SCAN_NSEG + seg] = base + incl;
}

/* segment totals -> segment offsets, and each layer's total: one workgroup
 * of ENG_SCAN_NSEG threads per layer */
__global__ void __launch_bounds__(ENG_SCAN_NSEG) k_layer_base(EngineParams P, int nseg) {
  __shared__ int first;
  const int L0 = blockIdx.x, s = threadIdx.x, lane = s & 63;
  int *seg = P.lay_segbase + L0 * ENG_SCAN_NSEG;
  const int v = s < nseg ? seg[s] : 0;
  int incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int t = __shfl_up(incl, off);
    if (lane >= off) incl += t;
  }
  if (s == 63) first = incl;
  __syncthreads();
  if (s >= 64) incl += first;
  if (s < nseg) seg[s] = incl - v;
  if (s == ENG_SCAN_NSEG - 1) P.lay_total[L0] = incl;
}

/* ------------------------------------------------------------------------ */
/* detection-weight estimator of every photon at order n
 * (src/xmi_variance_reduction.F90:29-726, xmi_compton_varred2 :949-1101),
 * after its geometry in the step kernel (d_vr_geom: detector point, angles,
 * path through the layers to the detector, escape probability, solid angle
 * from the grid; off-grid points go to a queue), as kernels with their own
 * register and LDS budgets:
 *
 *   k_vr_list     one lane per slot: the per-layer event lists
 *   k_vr_cone     one wavefront per queued photon: the cone estimate of
 *                 src/xmi_solid_angle_f.F90:432-710 with the trials split over
 *                 the lanes (same draws, same hit count as the serial loop)
 *   k_vr_scatter  one lane per photon: Rayleigh and Compton terms of every
 *                 element of the photon's layer; the Compton Doppler draws
 *                 continue the photon's estimator stream in element order
 *   k_vr_lines    a few photons per lane; the wavefront walks the layer's
 *                 (element, fluorescence line) entries with the line data in
 *                 scalar registers and sums each line's terms over its photons
 *
 * Path lengths are kept by layer, 0 where the path does not cross it, so that
 * register arrays have compile-time indices only (NL bounds the layer count).  Tallies are 128-bit fixed point, privatised in LDS when they fit;
 * integer adds commute, so totals do not depend on the order of the adds. */

__device__ __forceinline__ double d_readlane(double v, int lane) {
  long long b = __double_as_longlong(v);
  unsigned int lo = (unsigned int)__builtin_amdgcn_readlane((int)(b & 0xffffffffll), lane);
  unsigned int hi = (unsigned int)__builtin_amdgcn_readlane((int)(b >> 32), lane);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

/* one DPP lane move of a double (two 32-bit moves); lanes the row mask
 * leaves out, or whose source lane lies outside the row, read 0 */
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double d_dpp0(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), CTRL, ROW_MASK, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROW_MASK, 0xf, true);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned int)hi << 32) | (unsigned int)lo));
}

/* the wavefront's sums of a and of b, in a fixed order (row prefix sums, then
 * the row totals), returned wave-uniform: the halves exchanged first (a's sums
 * then live in lanes 0 to 31, b's in 32 to 63), so that one row reduction
 * serves both.  DPP moves keep it in the VALU, without the LDS round trips of a
 * shuffle butterfly */
__device__ __forceinline__ void d_wave_total2(double a, double b, double *ta, double *tb) {
  const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  double v = __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])) +
             __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
  v += d_dpp0<0x111, 0xf>(v); /* row_shr:1 */
  v += d_dpp0<0x112, 0xf>(v); /* row_shr:2 */
  v += d_dpp0<0x114, 0xf>(v); /* row_shr:4 */
  v += d_dpp0<0x118, 0xf>(v); /* row_shr:8: lane 15 of a row holds its sum */
  v += d_dpp0<0x142, 0xa>(v); /* row_bcast:15 into rows 1 and 3 */
  *ta = d_readlane(v, 31);
  *tb = d_readlane(v, 63);
}

/* The scattering kernel's tables in LDS: 2^(j/64) for the exponential and,
 * for a mantissa m in [1 + j/128, 1 + (j+1)/128), the rounded reciprocal of
 * the interval's middle with its logarithm in cells of the ln E grid (from
 * the grid's first node) and its power 11/4. */
#define ENG_LOG_LOG2 7
#define ENG_LOG_N (1 << ENG_LOG_LOG2)
struct ScatterTab {
  double exp2t[64];
  double inv[ENG_LOG_N], cell[ENG_LOG_N], pw[ENG_LOG_N];
};

__device__ __forceinline__ void d_scatter_tab(ScatterTab *t) {
  const int j = threadIdx.x;
  if (j < 64) t->exp2t[j] = exp2((double)j / 64.0);
  if (j < ENG_LOG_N) {
    const double inv = 1.0 / (1.0 + ((double)j + 0.5) / ENG_LOG_N);
    t->inv[j] = inv;
    t->cell[j] = (-log(inv) - XRL_CS_LNE0) * ((double)(XRL_NCS - 1) / (XRL_CS_LNE1 - XRL_CS_LNE0));
    t->pw[j] = pow(inv, XRL_PHOTO_EXPONENT);
  }
}

/* the provider's energy context (xrl_energy) by table: E = 2^k m, r = m inv_j
 * - 1 with |r| <= 1/256, so that ln E = k ln 2 - ln inv_j + ln(1 + r) and E^-p =
 * 2^(-11 k / 4) inv_j^p (1 + r)^-p; both series to r^7 (1e-20 and 1e-18).
 * Table-driven as P. T. P. Tang, "Table-driven implementation of the
 * logarithm function in IEEE floating-point arithmetic", ACM TOMS 16(4),
 * 1990.  The logarithm carries 2e-16 absolute, as a correctly rounded one
 * does in these cells' units. */
__device__ __forceinline__ xrl_ectx d_energy_tab(double E, const ScatterTab &t) {
  xrl_ectx c;
  c.E = E;
  c.pe = c.cf = 0.0;
  c.ci = 0;
  if (!(E > 0.0)) return c;
  constexpr double inv_h = (double)(XRL_NCS - 1) / (XRL_CS_LNE1 - XRL_CS_LNE0);
  const long long b = __double_as_longlong(E);
  const int hi = (int)(b >> 32), k = (hi >> 20) - 1023, j = (hi >> (20 - ENG_LOG_LOG2)) & (ENG_LOG_N - 1);
  const double m = __longlong_as_double((b & 0x000fffffffffffffll) | 0x3ff0000000000000ll);
  const double r = fma(m, t.inv[j], -1.0);
  double q = fma(r, inv_h / 7.0, -inv_h / 6.0);
  q = fma(r, q, inv_h / 5.0);
  q = fma(r, q, -inv_h / 4.0);
  q = fma(r, q, inv_h / 3.0);
  q = fma(r, q, -inv_h / 2.0);
  q = fma(r, q, inv_h);
  const double x = fma(r, q, fma((double)k, 0.6931471805599453 * inv_h, t.cell[j]));
  int i = (int)x;
  i = i < 0 ? 0 : (i > XRL_NCS - 2 ? XRL_NCS - 2 : i);
  c.ci = i;
  c.cf = x - (double)i;
  /* binomial series of exponent -11/4 */
  constexpr double p = XRL_PHOTO_EXPONENT, b1 = -p, b2 = b1 * (-p - 1.0) / 2.0, b3 = b2 * (-p - 2.0) / 3.0,
                   b4 = b3 * (-p - 3.0) / 4.0, b5 = b4 * (-p - 4.0) / 5.0, b6 = b5 * (-p - 5.0) / 6.0,
                   b7 = b6 * (-p - 6.0) / 7.0;
  double w = fma(r, b7, b6);
  w = fma(r, w, b5);
  w = fma(r, w, b4);
  w = fma(r, w, b3);
  w = fma(r, w, b2);
  w = fma(r, w, b1);
  const double s = t.pw[j] * t.exp2t[(k & 3) * 16];
  c.pe = ldexp(fma(s, w * r, s), (k >> 2) - 3 * k); /* -11 k / 4 = -3 k + k / 4 */
  return c;
}

/* e^-m from t = -m ENG_EXP64 (m >= 0), table-driven (P. T. P. Tang, "Table-
 * driven implementation of the exponential function in IEEE floating-point
 * arithmetic", ACM TOMS 15(2), 1989): t = 64 k + j + f with |f| <= 1/2, the
 * value 2^k 2^(j/64) 2^(f/64), the last factor its Taylor polynomial of
 * degree 5 (4e-17); ldexp underflows to 0 by itself */
#define ENG_EXP64 92.33248261689366 /* 64 / ln 2 */
__device__ __forceinline__ double d_exp64(double t, const ScatterTab &tab) {
  constexpr double h = 0.6931471805599453 / 64.0;
  const double n = rint(t), f = t - n;
  const int ni = (int)n;
  double q = fma(f, h * h * h * h * h / 120.0, h * h * h * h / 24.0);
  q = fma(f, q, h * h * h / 6.0);
  q = fma(f, q, h * h / 2.0);
  q = fma(f, q, h);
  const double T = tab.exp2t[ni & 63];
  return ldexp(fma(T, q * f, T), ni >> 6);
}

/* e^-m from t = -m ENG_EXP_UNIT, for a factor that tables and coefficients
 * hold in these units: t = 512 k + j + f with |f| <= 1/2, so the value is
 * 2^k * tab[j] * 2^(f/512), tab[j] = 2^(j/512) in LDS (4 KB) and the last
 * factor minus 1 its Taylor polynomial of degree 4 (1.2e-18); two
 * instructions fewer than the 64-entry table's reduction and degree 5, and
 * the unit saves the scaling and the clamp: ldexp underflows to 0 by itself */
__device__ __forceinline__ double d_exp_unit_poly(double f) {
  constexpr double h = 0.6931471805599453 / ENG_EXP_N;
  double p = fma(f, h * h * h * h / 24.0, h * h * h / 6.0);
  p = fma(f, p, h * h / 2.0);
  p = fma(f, p, h);
  return f * p;
}

/* persistent: the off-grid queue's photons (entries flattened over the
 * ENG_SPREAD sub-queues) times ENG_CONE_SEGS(hits) segments of
 * ENG_CONE_SEG trials are the work items; a wavefront takes items w, w + W,
 * ...  Trials 2 b and 2 b + 1 of a photon use block ctr0 + b of its
 * estimator stream (one 32-bit word per uniform), as the serial loop does,
 * and each segment adds its integer hit count and one
 * completion to the photon's packed accumulator (completions in bits 40 and
 * up); the wavefront that completes the photon writes its estimate and clears
 * the accumulator for the next launch.  Integer sums: the estimate equals the
 * serial one whatever the order of the segments. */
#define ENG_CONE_SEG 1024
#define ENG_CONE_DONE_SHIFT 40
__global__ void __launch_bounds__(ENG_BLOCK) k_vr_cone(EngineParams P, PhotonSoA S, VrSoA V, int n) {
  const int lane = __lane_id();
  const unsigned int wave = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  const unsigned int waves = (gridDim.x * blockDim.x) >> 6;
  /* sub-queue sizes, one per lane, and their inclusive prefix sums */
  const unsigned long long sz = P.qcount[(size_t)ENG_CNT_Q_SA * ENG_SPREAD + lane];
  unsigned long long incl = sz;
  for (int off = 1; off < 64; off <<= 1) {
    const unsigned long long v = __shfl_up(incl, off);
    if (lane >= off) incl += v;
  }
  const unsigned long long total = __shfl(incl, 63);
  const long hits = P.hits_per_single;
  const unsigned long long nseg = hits > 0 ? (unsigned long long)((hits + ENG_CONE_SEG - 1) / ENG_CONE_SEG) : 1ull;
  const SaGeom g = d_sa_geom(P);
  for (unsigned long long item = wave; item < total * nseg; item += waves) {
    const unsigned long long e = item / nseg, sg = item - e * nseg;
    /* sub-queue holding entry e: first lane whose inclusive prefix exceeds e */
    const int j = __ffsll((long long)__ballot(incl > e)) - 1;
    const unsigned long long before = __shfl(incl - sz, j);
    const int i = P.queue[((size_t)ENG_CNT_Q_SA * ENG_SPREAD + j) * P.qreg + (e - before)];
    phx_stream s;
    phx_stream_init(&s, P.seed, P.sample, (uint32_t)n, PHX_SUB_VARRED, S.hid[i]);
    const uint32_t ctr0 = V.blk[i];
    SaCone cone;
    const int open = d_sa_setup(g, V.sar[i], V.sat[i], &cone);
    unsigned long long nhit = 0;
    if (open) {
      /* trial pairs (2 b, 2 b + 1) from block ctr0 + b; segments start at
       * even trials (ENG_CONE_SEG is even) */
      const long t1 = min((long)((sg + 1) * ENG_CONE_SEG), hits);
      const uint32_t cs[4] = {ctr0, s.ctr[1], s.ctr[2], s.ctr[3]};
      for (long t = (long)(sg * ENG_CONE_SEG) + 2 * lane; t < t1; t += 128)
        nhit += d_sa_trial_pair(cone, cs, s.key, (uint32_t)(t >> 1), t + 1 < t1);
    }
    for (int off = 32; off > 0; off >>= 1) nhit += __shfl_xor(nhit, off);
    if (lane == 0) {
      unsigned long long *acc = P.cone_acc + e;
      const unsigned long long old = atomicAdd(acc, (1ull << ENG_CONE_DONE_SHIFT) + nhit);
      if ((old >> ENG_CONE_DONE_SHIFT) + 1ull == nseg) {
        const unsigned long long all = (old & ((1ull << ENG_CONE_DONE_SHIFT) - 1ull)) + nhit;
        V.omega[i] = open ? cone.cone_sa * (double)all / (double)hits : 0.0;
        if (open) V.blk[i] = ctr0 + (uint32_t)((hits + 1) / 2);
        *acc = 0ull;
      }
    }
  }
}

/* walk over the layer lists in chunks of 64 entries: chunk c of the
 * concatenation of every layer's chunks (layer 1 first); a wavefront takes
 * chunks in increasing order, so the layer only moves forward (wave-uniform) */
struct LayerChunks {
  int L, tot;
  long long c_begin, c_end;
};

__device__ __forceinline__ bool d_chunk_next(const EngineParams &P, LayerChunks &w, long long c, int csz = 64) {
  while (c >= w.c_end && w.L < P.n_layers) {
    w.L++;
    w.tot = P.lay_total[w.L - 1];
    w.c_begin = w.c_end;
    w.c_end += (w.tot + csz - 1) / csz;
  }
  return c < w.c_end;
}

/* row[] at x >= 0 of a grid whose cells start near x * inv: on the uniform
 * grids of the generator cell and fraction come from x itself (d_table) */
__device__ __forceinline__ double d_grid_lookup(int uniform, const double *grid, const double *row, int len, double inv,
                                               double x) {
  const double t = x * inv;
  int pos = (int)t;
  if (pos > len - 2) pos = len - 2;
  const double f = uniform ? t - (double)pos : (x - grid[pos]) * d_rcp(grid[pos + 1] - grid[pos]);
  return fma(row[pos + 1] - row[pos], f, row[pos]);
}

/* the Compton profile's CDF at momentum pz from its grid (the
 * xmi_profile_cdf_grid table of the element; gs grid points per unit
 * momentum), clamped to the grid's last point, 0 for pz <= 0; in two parts,
 * so that the grid values of one element can be loaded while the previous
 * element is scored: the two grid values and the fraction of the lookup, then
 * the interpolation */
struct CdfPair {
  double v0, v1, f;
};

__device__ __forceinline__ void d_profile_cdf_load(const double *g, double gs, double pz, CdfPair *p) {
  p->v0 = p->v1 = p->f = 0.0;
  if (!(pz > 0.0)) return;
  const double x = fmin(pz * gs, (double)(XMI_CP_GRID - 1));
  int j = (int)x;
  j = j > XMI_CP_GRID - 2 ? XMI_CP_GRID - 2 : j;
  p->v0 = g[j];
  p->v1 = g[j + 1];
  p->f = x - (double)j;
}

__device__ __forceinline__ double d_profile_cdf_eval(const CdfPair &p) { return fma(p.v1 - p.v0, p.f, p.v0); }

/* ---- the advanced Compton model (use_advanced_compton) ------------------
 * src/xmi_main.F90:4785-4983 (transport) and src/xmi_variance_reduction.F90:
 * 752-947 (estimator) with src/xmi_aux_f.F90:1951-2057 (kinematics) */

/* the largest projected momentum an electron of binding energy Ii can carry
 * for scattering by the angle of cosine ct (xmi_get_qimax) */
__device__ __forceinline__ double d_qimax(double energy, double Ii, double ct) {
  if (Ii != 0.0 && energy < Ii) return 0.0;
  const double EminIi = energy - Ii;
  const double Q = 137.0 * (EminIi * energy * (1.0 - ct) * (1.0 / ENG_MEC2) - Ii);
  return Q * d_rsqrt_pos(EminIi * EminIi + energy * energy - 2.0 * EminIi * energy * ct);
}

/* the projected momentum of an energy E1, without its positive denominator
 * (xmi_get_q_from_energy's sign) */
__device__ __forceinline__ double d_q_from_energy(double E0, double E1, double ct) {
  return 137.0 * (E1 - E0 + (1.0 - ct) * E0 * E1 * (1.0 / ENG_MEC2));
}

__device__ __forceinline__ double d_q_denom(double E0, double E1, double ct) {
  return sqrt(E1 * E1 + E0 * E0 - 2.0 * E0 * E1 * ct);
}

/* xmi_get_energy_from_q: the root of the quadratic whose momentum has Q's
 * sign; 0 in the reference's exceptions, -1 when no root has it (the
 * reference stops there) */
__device__ double d_energy_from_q(double E0, double Q, double c) {
  if (fabs(c - 1.0) < 1e-8) return 0.0;
  if (fabs(Q) < 1e-4) return E0 * d_rcp(1.0 + E0 * (1.0 - c) * (1.0 / ENG_MEC2));
  const double d = 1.0 + E0 * (1.0 / ENG_MEC2) - E0 * c * (1.0 / ENG_MEC2);
  const double aq = 137.0 * 137.0 * d * d - Q * Q;
  const double bq = -2.0 * 137.0 * 137.0 * E0 * d + 2.0 * E0 * c * Q * Q;
  const double cq = 137.0 * 137.0 * E0 * E0 - E0 * E0 * Q * Q;
  double E1, E2;
  if (aq == 0.0) {
    if (bq == 0.0) return 0.0;
    E1 = E2 = -1.0 * cq / bq;
  } else {
    const double delta = bq * bq - 4.0 * aq * cq;
    if (delta < 0.0) return 0.0;
    const double ia = 0.5 * d_rcp(aq);
    if (delta == 0.0) {
      E1 = E2 = -bq * ia;
    } else {
      const double sd = d_sqrt_pos(delta);
      const double t1 = (-bq + sd) * ia, t2 = (-bq - sd) * ia;
      E1 = t1 < t2 ? t1 : t2;
      E2 = t1 < t2 ? t2 : t1;
    }
  }
  const double N1 = d_q_from_energy(E0, E1, c), N2 = d_q_from_energy(E0, E2, c);
  if (Q * N1 > 0.0) return E1;
  if (Q * N2 > 0.0) return E2;
  if (fabs(E1 - E2) < 1e-10 || fabs(N1 / d_q_denom(E0, E1, c) - N2 / d_q_denom(E0, E2, c)) < 1e-10) return E1;
  return -1.0;
}

/* subshell g's two-sided partial-profile CDF at its Qimax (binding energy Ii) */
__device__ __forceinline__ double d_adv_cdf(const EngineParams &P, double Ii, int g, double energy, double ct) {
  const double q = d_qimax(energy, Ii, ct);
  if (q < -100.0) return 0.0;
  if (q > 100.0) return 1.0;
  const double v = d_grid_lookup(P.cp_adv_uniform, P.cp_Qs, P.cp_pcdf + (size_t)g * P.cp_len, P.cp_len, P.cp_Qs_rcp, fabs(q));
  return q < 0.0 ? 1.0 - (0.5 + v) : 0.5 + v;
}

/* the projected momentum at a value cdf of subshell g's two-sided profile */
__device__ __forceinline__ double d_adv_q(const EngineParams &P, int g, double cdf) {
  const double cp = cdf < 0.5 ? 0.5 - cdf : cdf - 0.5;
  const double Q = d_grid_lookup(P.cp_adv_uniform, P.cp_inv, P.cp_qinv + (size_t)g * P.cp_len, P.cp_len, P.cp_inv_rcp, cp);
  return cdf < 0.5 ? -Q : Q;
}

/* - ENG_EXP64 times the mass path of a photon of the given energy to the
 * detector from layer L, the records of several crossed layers loaded before
 * the first is used.  Up to five layers rd holds the layers' factors; beyond
 * (register budget) the wave's layers lo .. hi are walked four at a time, a
 * lane taking those on its side of L (up or down) from slot i's record. */
template <int NL>
__device__ __forceinline__ double d_mass_path(const EngineParams &P, const VrSoA &V, double energy, int L, int up, int lo,
                                              int hi, int i, const double *rd, const ScatterTab &tab) {
  const xrl_ectx ce = d_energy_tab(energy, tab);
  if (!(energy > 0.0)) return 0.0;
  const LayCell *cell = P.lay_cell + (size_t)ce.ci * P.n_layers;
  double t = 0.0;
  if constexpr (NL <= 5) {
    LayCell r[NL];
#pragma unroll
    for (int l = 0; l < NL; l++)
      if (rd[l] < 0.0) r[l] = cell[l];
#pragma unroll
    for (int l = 0; l < NL; l++)
      if (rd[l] < 0.0) t = fma(d_cell_mu(P, l, r[l], ce), rd[l], t);
  } else {
    for (int l0 = lo; l0 <= hi; l0 += 4) {
      LayCell r[4];
      double d[4];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int l = l0 + k;
        if (l <= hi && (up ? l >= L - 1 : l <= L - 1)) {
          r[k] = cell[l];
          d[k] = V.dist[(size_t)l * P.cap + i];
        }
      }
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int l = l0 + k;
        if (l <= hi && (up ? l >= L - 1 : l <= L - 1)) t = fma(d_cell_mu(P, l, r[k], ce) * P.layer_density[l], d[k], t);
      }
    }
    t *= -ENG_EXP64;
  }
  return t;
}

/* Bound by vector issue (50 % of the cycles) and the address unit's work on
 * per-lane table reads (66 %): per photon and element one profile CDF, one
 * inverse CDF and one record per crossed layer.  Hence uniform grids are not
 * read, an energy's layer records lie side by side and are loaded together,
 * and logarithm, power, exponential and quotients are the short forms above.
 * 1e8 histories of the three-layer tube run: 43.6 -> 33.0 ms; the advanced
 * model on 3e5 photons in seven layers 559 -> 449 us an order (38 % issue;
 * bound by the last round of its 4700 chunks on 3072 resident waves).
 * Occupancy: four waves per SIMD (128 VGPRs) measured 2 % faster than three
 * up to three layers, where few registers spill; three elsewhere. */
template <int NL, bool use_lds, bool ADV>
__global__ void __launch_bounds__(ENG_BLOCK) __attribute__((amdgpu_waves_per_eu(!ADV && NL <= 3 ? 4 : 3)))
k_vr_scatter(EngineParams P, PhotonSoA S, VrSoA V, int n) {
  /* LDS tallies (when they fit): channels [nch][2], Rayleigh/Compton rows
   * [nZ][2][2]; flushed once per workgroup */
  extern __shared__ unsigned long long lds[];
  __shared__ ScatterTab tab;
  const size_t n_ch2 = (size_t)P.nch * 2, n_rc2 = (size_t)P.nZ * 4;
  const size_t cap = (size_t)P.cap;
  unsigned long long *gch = P.t_ch + (size_t)(n - 1) * n_ch2;
  unsigned long long *grc = P.t_rc + (size_t)(n - 1) * n_rc2;
  unsigned long long *tch = gch, *trc = grc;
  d_scatter_tab(&tab);
  if (use_lds) {
    tch = lds;
    trc = lds + n_ch2;
    for (size_t k = threadIdx.x; k < n_ch2 + n_rc2; k += blockDim.x) lds[k] = 0ull;
  }
  __syncthreads();
  const int shift = P.tally_shift;
  const int lane = __lane_id();
  const double inv_gain = 1.0 / P.gain;
  const double r_end = d_const(P.cp_rn)[P.cp_len - 2];
  /* single-precision literals of src/xmi_variance_reduction.F90:949-1008 */
  const double cc = (double)1.2399e-6f, c0 = (double)4.85e-12f, c1 = (double)1.456e-2f;
  /* wave index through readfirstlane: wave-uniform for the compiler too,
   * so that the chunk walk and the layer's data stay in scalar registers */
  const long long wave = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6),
                  waves = (gridDim.x * blockDim.x) >> 6;
  LayerChunks lc = {0, 0, 0, 0};
  for (long long c = wave; d_chunk_next(P, lc, c); c += waves) {
    const int L = lc.L;
    const int e = (int)((c - lc.c_begin) * 64) + lane;
    const int i = e < lc.tot ? P.lay_list[(size_t)(L - 1) * cap + e] : 0;
    const int info = e < lc.tot ? V.info[i] : 0;
    const int mine = info & VR_ACTIVE;
    /* per-photon factors, shared by every element of the layer */
    double E = 0.0, wo = 0.0, pesc = 0.0, inv_mu = 0.0, c_lamb0 = 1.0, A0 = 0.0, A1 = 0.0, ct_e = 0.0;
    phx_stream sd; /* advanced model: uniforms from the same stream position */
    /* - rho * path * ENG_EXP64 by layer (0 where not crossed): in registers for
     * up to five layers, read from the records beyond (register budget) */
    constexpr int NR = NL <= 5 ? NL : 1;
    double rd[NR];
    xrl_dcsp_ctx dc = {0.0, 0.0, 0.0};
    int ch_r = -1;
    uint32_t ww[4] = {0u, 0u, 0u, 0u}; /* the current block's words */
    uint32_t ctr0 = 0u, hid_lo = 0u, hid_hi = 0u;
#pragma unroll
    for (int k = 0; k < NR; k++) rd[k] = 0.0;
    if (mine) {
      E = S.energy[i];
      const double ct = V.ct[i], q = V.q[i], mct = 1.0 - ct;
      wo = V.omega[i] * S.weight[i];
      pesc = V.pesc[i];
      inv_mu = d_rcp(S.mus[(size_t)(L - 1) * cap + i]);
      if (NL <= 5) {
#pragma unroll
        for (int l = 0; l < NR; l++)
          if (l < P.n_layers) rd[l] = (-ENG_EXP64 * P.layer_density[l]) * V.dist[(size_t)l * cap + i];
      }
      /* the estimator stream from the block after the geometry and cone
       * draws, as words: element k takes word k */
      ctr0 = V.blk[i];
      {
        const unsigned long long hid = S.hid[i];
        hid_lo = (uint32_t)hid;
        hid_hi = (uint32_t)(hid >> 32);
      }
      if (ADV) {
        phx_stream_init(&sd, P.seed, P.sample, (uint32_t)n, PHX_SUB_VARRED, S.hid[i]);
        sd.ctr[0] = ctr0;
      }
      ct_e = ct;
      /* xrl_dcsp_setup from cos theta and sin^2 theta cos^2 phi */
      const double sth2 = mct > 0.0 ? d_sqrt_pos(0.5 * mct) : 0.0, k1 = 1.0 + E * (1.0 / XRL_MEC2) * mct, kk = d_rcp(k1);
      dc.x = E * (1.0 / XRL_KEV_ANGSTROM) * sth2;
      dc.thomson = XRL_RE2 * (1.0 - q);
      dc.kn = XRL_RE2 * 0.5 * kk * kk * (kk + k1 - 2.0 * q);
      c_lamb0 = cc * d_rcp(E * 1000.0);
      A0 = c0 * sth2 * sth2;
      A1 = c1 * c_lamb0 * sth2;
      ch_r = E >= 1.0 ? (int)((E - P.zero) * inv_gain) : -1;
    }
    const int lo = __ballot(mine && !(info & VR_UP)) ? 0 : L - 1, hi = __ballot(mine && (info & VR_UP)) ? P.n_layers - 1 : L - 1;
    const int off = __builtin_amdgcn_readfirstlane(P.layer_off[L - 1]);
    const int nel = __builtin_amdgcn_readfirstlane(P.layer_nel[L - 1]);
    double twr_sum = 0.0; /* Rayleigh keeps the energy: one channel per photon */
    double rsum = 0.0;    /* lane 2j + kind: row total of element k0 + j of this group */
    /* the accepted momenta's bounds of the Doppler draw (per photon), and
     * the profile-CDF values at them of the next element, loaded one
     * element ahead */
    const double iA1 = A1 > 0.0 ? d_rcp(A1) : 0.0, pz_max = A0 * iA1, pz_neg = (c_lamb0 + A0) * iA1;
    CdfPair cdf_max = {0.0, 0.0, 0.0}, cdf_neg = {0.0, 0.0, 0.0};
    if (!ADV && mine && A1 > 0.0 && nel > 0) {
      const int u0 = d_const(P.el_u)[off];
      const double *gr = P.cp_cdfg + (size_t)u0 * XMI_CP_GRID;
      const double gs = d_const(P.cp_gscale)[u0];
      d_profile_cdf_load(gr, gs, pz_max, &cdf_max);
      d_profile_cdf_load(gr, gs, pz_neg, &cdf_neg);
    }
    for (int k = 0; k < nel; k++) {
      const int u = d_const(P.el_u)[off + k];
      const auto *a = d_const(P.atoms) + u;
      const double Pconv = d_const(P.el_w)[off + k] * inv_mu;
      double f_max = 0.0, f_neg = 0.0;
      if (!ADV && mine && A1 > 0.0) {
        f_max = d_profile_cdf_eval(cdf_max);
        f_neg = d_profile_cdf_eval(cdf_neg);
        if (k + 1 < nel) {
          const int u1 = d_const(P.el_u)[off + k + 1];
          const double *gr = P.cp_cdfg + (size_t)u1 * XMI_CP_GRID;
          const double gs = d_const(P.cp_gscale)[u1];
          d_profile_cdf_load(gr, gs, pz_max, &cdf_max);
          d_profile_cdf_load(gr, gs, pz_neg, &cdf_neg);
        }
      }
      /* Rayleigh, and the element's factor of its Compton terms
       * (xrl_dcsp_rayl_c and xrl_dcsp_compt_c: 1 / d1^4 and 1 - 1 / d2^2 =
       * v (2 + v) / d2^2 from one reciprocal) */
      double twr = 0.0, dcw = 0.0;
      if (mine) {
        const double u1 = dc.x * a->inv_ff_x0, u2 = dc.x * a->inv_sf_x0, v = u2 * u2;
        const double d1 = fma(3.0 * u1, u1, 1.0), d2 = 1.0 + v, d12 = d1 * d1, d14 = d12 * d12, d22 = d2 * d2;
        const double t = d_rcp(d14 * d22), Z = (double)a->Z, pw = Pconv * wo * a->barn_per_A;
        twr = (pw * dc.thomson) * (Z * Z) * (t * d22) * pesc;
        dcw = (pw * dc.kn) * Z * (v * (2.0 + v)) * (t * d14);
        twr_sum += twr;
      }
      /* Compton, xmi_compton_varred2: Doppler-broadened energy from the
       * element's Compton profile, continuing the photon's estimator stream */
      double twc = 0.0;
      if (ADV && mine) {
        /* every occupied subshell with weight count * CDF(Qimax) / sum, one
         * uniform each (xmi_compton_varred) */
        const int g0 = d_const(P.cp_sh_off)[u], g1 = d_const(P.cp_sh_off)[u + 1];
        double csum = 0.0;
        for (int g = g0; g < g1; g++) {
          const int sh = d_const(P.cp_sh_idx)[g];
          csum += a->occupancy[sh] * d_adv_cdf(P, a->edge[sh], g, E, ct_e);
        }
        const double icsum = csum != 0.0 ? d_rcp(csum) : 0.0;
        for (int g = g0; csum != 0.0 && g < g1; g++) {
          const int sh = d_const(P.cp_sh_idx)[g];
          const double cdf = d_adv_cdf(P, a->edge[sh], g, E, ct_e);
          const double sw = a->occupancy[sh] * cdf * icsum;
          if (sw == 0.0) continue;
          const double energy = d_energy_from_q(E, d_adv_q(P, g, phx_uniform(&sd) * cdf), ct_e);
          if (!(energy > 0.0)) continue;
          const double tw = dcw * d_exp64(d_mass_path<NL>(P, V, energy, L, info & VR_UP, lo, hi, i, rd, tab), tab) * sw;
          twc += tw;
          const int ch = energy >= 1.0 ? (int)((energy - P.zero) * inv_gain) : -1;
          if (ch >= 0 && ch <= P.nch - 1 && tw > 0.0) fx_add_global(&tch[2 * ch], tw, shift);
        }
      }
      if (!ADV && mine) {
        /* xmi_compton_varred2 (src/xmi_variance_reduction.F90:949-1008)
         * redraws the momentum until E' <= E; the accepted momenta are pz <=
         * A0/A1 and, where E' turns negative, pz > (c_lamb0 + A0)/A1.  They
         * are drawn here directly from that part of the profile, one word
         * each (the same distribution, and no wavefront waits on its lanes'
         * longest rejection run); r ranges over [0, r_end), the inverse
         * table without its last interval */
        const double *icdf = P.cp_icdf + (size_t)u * P.cp_len;
        if (!(A1 > 0.0)) f_max = f_neg = r_end; /* the profile CDFs at A0 / A1 were loaded ahead */
        const double m_pos = f_max + (r_end - f_neg);
        if ((k & 3) == 0) {
          uint32_t c4[4] = {ctr0 + (uint32_t)(k >> 2), (P.sample << 12) | (((uint32_t)n & 0xFFu) << 4) | PHX_SUB_VARRED, hid_lo,
                            hid_hi};
          const uint32_t key[2] = {(uint32_t)P.seed, (uint32_t)(P.seed >> 32)};
          phx_4x32_10(c4, key, ww);
        }
        const uint32_t wd = ww[0];
        ww[0] = ww[1];
        ww[1] = ww[2];
        ww[2] = ww[3];
        const double uu = (double)wd * 0x1.0p-32 * (r_end + m_pos);
        double r, sgn;
        if (uu < r_end) {
          r = uu;
          sgn = -1.0;
        } else {
          const double v = uu - r_end;
          r = v < f_max ? v : v - f_max + f_neg;
          sgn = 1.0;
        }
        const double pz = sgn * d_grid_lookup(P.cp_rn_uniform, P.cp_rn, icdf, P.cp_len - 1, P.cp_rn_inv, r);
        const double energy = (cc / 1000.0) * d_rcp(c_lamb0 + (A0 - A1 * pz));
        twc = dcw * d_exp64(d_mass_path<NL>(P, V, energy, L, info & VR_UP, lo, hi, i, rd, tab), tab);
        const int ch = energy >= 1.0 ? (int)((energy - P.zero) * inv_gain) : -1;
        if (ch >= 0 && ch <= P.nch - 1 && twc > 0.0) fx_add_global(&tch[2 * ch], twc, shift);
      }
      /* history rows: wave totals collected in lanes, 32 elements a group */
      double tr, tc;
      d_wave_total2(twr, twc, &tr, &tc);
      const int j = k & 31;
      if (lane == 2 * j) rsum = tr;
      if (lane == 2 * j + 1) rsum = tc;
      if (j == 31 || k == nel - 1) {
        const int kl = k - j + (lane >> 1);
        if (kl <= k && rsum > 0.0) {
          const int ul = d_const(P.el_u)[off + kl];
          fx_add_global(&trc[((size_t)ul * 2 + (lane & 1)) * 2], rsum, shift);
        }
        rsum = 0.0;
      }
    }
    if (ch_r >= 0 && ch_r <= P.nch - 1 && twr_sum > 0.0) fx_add_global(&tch[2 * ch_r], twr_sum, shift);
  }
  if (use_lds) {
    __syncthreads();
    for (size_t k = threadIdx.x; k < n_ch2 / 2; k += blockDim.x)
      if (tch[2 * k] | tch[2 * k + 1]) fx_merge_global(&gch[2 * k], tch[2 * k], tch[2 * k + 1]);
    for (size_t k = threadIdx.x; k < n_rc2 / 2; k += blockDim.x)
      if (trc[2 * k] | trc[2 * k + 1]) fx_merge_global(&grc[2 * k], trc[2 * k], trc[2 * k + 1]);
  }
}

/* Bound by vector issue of the pairs (line, photon): 15 instructions each
 * with three layers (three for the attenuation, rint, difference, conversion,
 * two for the table's index, four for the polynomial, one each for the table,
 * the exponent and the sum).  2^21 histories of the three-layer tube run took
 * 250 us with the 64-entry table, four-layer rows and one entry loaded ahead
 * of its use; in batches of 2^23 they take 180.
 *
 * lines phase: KP photons per lane, a chunk of 64 KP photons (all in layer
 * L); the wavefront walks the layer's (element, line) entries.  Per (line t,
 * photon) term
 *   wf_t * P_shell(t, photon) * g * exp(-sum_l mu_rho(t, l) * d_l)
 * with g = Omega / 4 pi * weight / mu(E) and d_l the photon's path in layer l
 * on its way to the detector.  The line's data are wave-uniform (scalar
 * loads); P_shell is formed once per (element, shell) of the walk: a first
 * interaction (or a photon not coming from fluorescence) uses
 * E^-p * shell_C[cascade][edges above E][shell], a fluorescence photon the
 * precalculated cascade table (src/xmi_variance_reduction.F90:540-580).  The
 * terms of a line are summed over each lane's photons, then over the lanes in
 * a fixed order (deterministic), and added once to the line's fixed-point
 * bin: one wavefront sum per line and 64 KP photons.  The lane sums go
 * through LDS eight lines at a time: the lanes store their terms of eight
 * lines, then eight lanes per line add its 64 terms (eight each, then three
 * DPP steps), instead of a six-step DPP reduction per line. */
#define ENG_LRED_STRIDE 72 /* doubles per line row of the staging: 8 mod 32, conflict-free reads */
template <int NL, int KP, bool use_lds>
__global__ void __launch_bounds__(ENG_BLOCK) k_vr_lines(EngineParams P, PhotonSoA S, VrSoA V, int n) {
  /* LDS tallies (when they fit): compact line bins [n_lbins][2] */
  extern __shared__ unsigned long long lds[];
  __shared__ double exp_tab[ENG_EXP_N];
  /* per wavefront: the lanes' terms of 8 lines, row j = line j of the group */
  __shared__ double lred[ENG_BLOCK / 64][8 * ENG_LRED_STRIDE];
  const size_t n_line2 = (size_t)P.n_lbins * 2;
  const size_t cap = (size_t)P.cap;
  unsigned long long *gline = P.t_line + (size_t)(n - 1) * P.nZ * ENG_MAX_ACT * 2;
  unsigned long long *tline = gline;
  for (int k = threadIdx.x; k < ENG_EXP_N; k += ENG_BLOCK) exp_tab[k] = exp2((double)k / ENG_EXP_N);
  if (use_lds) {
    tline = lds;
    for (size_t k = threadIdx.x; k < n_line2; k += blockDim.x) lds[k] = 0ull;
  }
  __syncthreads();
  const int shift = P.tally_shift;
  const int smax = P.use_M_lines ? 8 : 3;
  /* wave index through readfirstlane: wave-uniform for the compiler too,
   * so that the chunk walk and the layer's data stay in scalar registers */
  const long long wave = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6),
                  waves = (gridDim.x * blockDim.x) >> 6;
  LayerChunks lc = {0, 0, 0, 0};
  for (long long c = wave; d_chunk_next(P, lc, c, 64 * KP); c += waves) {
    const int L = lc.L;
    /* the lane's KP photons: list entries e0, e0 + 64, ... of layer L */
    const int e0 = (int)((c - lc.c_begin) * (64 * KP)) + __lane_id();
    double E[KP], g[KP], x[KP];
    /* path length per layer, by layer index (0 where not crossed) */
    double dl[KP][NL];
    int fo[KP], px[KP], kE[KP];
    int any_act = 0;
#pragma unroll
    for (int k = 0; k < KP; k++) {
      const int e = e0 + 64 * k;
      const int i = e < lc.tot ? P.lay_list[(size_t)(L - 1) * cap + e] : 0;
      const int info = e < lc.tot ? V.info[i] : 0;
      const int act = info & VR_ACTIVE;
      any_act |= act;
      E[k] = 2.0;
      g[k] = x[k] = 0.0;
      fo[k] = 1;
      px[k] = kE[k] = 0;
#pragma unroll
      for (int l = 0; l < NL; l++) dl[k][l] = 0.0;
      if (act) {
        E[k] = S.energy[i];
        g[k] = V.omega[i] / 4.0 / ENG_PI * S.weight[i] / S.mus[(size_t)(L - 1) * cap + i];
        const int pl = S.prev_line[i];
        fo[k] = !(n > 1 && pl > 0);
        /* E^-p goes with the weight factor; a fluorescence photon has its
         * place in the rows of the cascade table instead */
        if (fo[k]) g[k] *= d_photo_pe(E[k]);
        else px[k] = S.prev_u[i] * XMI_NLINES_VR_DEV + (pl - 1);
#pragma unroll
        for (int l = 0; l < NL; l++)
          if (l < P.n_layers) dl[k][l] = V.dist[(size_t)l * cap + i];
      }
    }
    if (__ballot(any_act) == 0ull) continue;
    const int t0 = __builtin_amdgcn_readfirstlane(P.fl_off[L - 1]), t1 = __builtin_amdgcn_readfirstlane(P.fl_off[L]);
    int u_cur = -1, z_cur = -1, any = 0;
    double *wred = lred[threadIdx.x >> 6];
    const int lane = __lane_id();
    /* the entries' scalars come two ahead, in two buffers by the entry's
     * parity (the tables end with two zero entries; one rotated buffer would
     * copy, and so wait for, what was just asked for).  Scalar and LDS loads
     * complete out of order with each other, so a wait for an LDS value waits
     * for every scalar load under way: they are issued behind an entry's LDS
     * reads, where the next wait is a whole entry's arithmetic away.  Two
     * buffers of more than four layers would not fit the scalar registers:
     * there the next entry's are issued first */
    constexpr int AH = NL <= 4 ? 2 : 1;
    const auto *ent = d_const(P.fl_ent) + (size_t)t0 * (NL + 1);
    double nx[AH][NL + 1]; /* {element, shell} packed, attenuation by layer */
    auto fetch = [&](double *to, int t) {
#pragma unroll
      for (int l = 0; l <= NL; l++) to[l] = ent[(t - t0) * (NL + 1) + l];
    };
#pragma unroll
    for (int a = 0; a < AH; a++) fetch(nx[a], t0 + a);
    auto entry = [&](double *buf, int t) {
      const long long uz = __double_as_longlong(buf[0]);
      const int2 it = make_int2((int)uz, (int)(uz >> 32));
      double mr[NL];
#pragma unroll
      for (int l = 0; l < NL; l++) mr[l] = buf[l + 1];
      if (AH == 1) fetch(buf, t + 1);
      if (it.x != u_cur) {
        /* edges of the element above each photon's energy */
        const auto *a = d_const(&P.atoms[it.x]);
#pragma unroll
        for (int k = 0; k < KP; k++) {
          kE[k] = 0;
#pragma unroll
          for (int q = 0; q < 9; q++) kE[k] += a->edge[q] > E[k] ? 1 : 0;
        }
        u_cur = it.x;
        z_cur = -1;
      }
      if (it.y != z_cur) {
        z_cur = it.y;
        int nz = 0;
        const double *sc = &P.atoms[u_cur].shell_C[P.cascade - 1][0][z_cur];
        const double *pc = P.precalc_xrf + ((size_t)u_cur * 9 + z_cur) * P.nZ * XMI_NLINES_VR_DEV;
#pragma unroll
        for (int k = 0; k < KP; k++) {
          double v;
          if (fo[k]) v = (!P.use_M_lines && z_cur >= 4) ? 0.0 : sc[9 * kE[k]];
          else v = z_cur <= smax ? pc[px[k]] : 0.0;
          /* shell factor times the photon's weight factor; 0 for lanes
           * without a photon, so that their terms vanish */
          x[k] = v * g[k];
          nz |= x[k] != 0.0;
        }
        any = __ballot(nz) != 0ull;
      }
      const int j = (t - t0) & 7;
      double acc = 0.0;
      if (any) {
        /* attenuation rows are padded to NL entries (zeros past the stack),
         * in units of the table exponential; the lane's photons are summed
         * before the wavefront sum */
        double T[KP], p[KP];
        int ni[KP];
#pragma unroll
        for (int k = 0; k < KP; k++) {
          double m = mr[0] * dl[k][0];
#pragma unroll
          for (int l = 1; l < NL; l++) m = fma(mr[l], dl[k][l], m);
          const double r = rint(m);
          ni[k] = (int)r;
          T[k] = exp_tab[ni[k] & (ENG_EXP_N - 1)];
          p[k] = d_exp_unit_poly(m - r);
        }
#pragma unroll
        for (int k = 0; k < KP; k++) acc = fma(x[k], ldexp(fma(T[k], p[k], T[k]), ni[k] >> 9), acc);
      }
      wred[j * ENG_LRED_STRIDE + lane] = acc;
      if (AH == 2) {
        __builtin_amdgcn_sched_barrier(0);
        fetch(buf, t + 2);
      }
      if (j == 7 || t == t1 - 1) {
        /* line m of the group (m <= j): lane 8m + q adds the terms of lanes
         * 8r + q (r = 0..7), then the eight lanes of m are summed (xor 1,
         * xor 2 in quads, then the half-row mirror joins the two quads); the
         * staging of the next group is written after these reads (one
         * wavefront's LDS accesses complete in order) */
        __builtin_amdgcn_wave_barrier();
        const int m = lane >> 3, q = lane & 7;
        double sum = 0.0;
#pragma unroll
        for (int r = 0; r < 8; r++) sum += wred[m * ENG_LRED_STRIDE + 8 * r + q];
        sum += d_dpp0<0xB1, 0xf>(sum);  /* quad_perm [1, 0, 3, 2] */
        sum += d_dpp0<0x4E, 0xf>(sum);  /* quad_perm [2, 3, 0, 1] */
        sum += d_dpp0<0x141, 0xf>(sum); /* row_half_mirror */
        __builtin_amdgcn_wave_barrier();
        const int tl = t - j + m;
        if (q == 0 && tl <= t && sum > 0.0) {
          const int4 il = P.fl_info[tl];
          unsigned long long *bin =
              use_lds ? &tline[(size_t)il.w * 2] : &tline[((size_t)il.x * ENG_MAX_ACT + il.y) * 2];
          fx_add_global(bin, sum * P.fl_wf[tl], shift);
        }
      }
    };
    for (int t = t0; t < t1; t += 2) {
      entry(nx[0], t);
      if (t + 1 < t1) entry(nx[AH - 1], t + 1);
    }
  }
  if (use_lds) {
    __syncthreads();
    for (size_t k = threadIdx.x; k < n_line2 / 2; k += blockDim.x)
      if (tline[2 * k] | tline[2 * k + 1])
        fx_merge_global(&gline[(size_t)P.lbin_g[k] * 2], tline[2 * k], tline[2 * k + 1]);
  }
}

/* ------------------------------------------------------------------------ */
/* interactions */

/* transport substream of slot i: a cascade's offspring photon has its own */
__device__ __forceinline__ uint32_t d_tr_sub(const EngineParams &P, int i) {
  return (P.off_half && i >= P.off_half) ? PHX_SUB_OFFSPRING : PHX_SUB_TRANSPORT;
}

/* the interaction routines are compiled twice: BRUTE (brute-force runs)
 * adds the history rows of Rayleigh and Compton, the analogue yield and the
 * cascades, which the variance-reduction path does without */

template <bool BRUTE>
__device__ __forceinline__ void d_rayleigh_one(const EngineParams &P, const PhotonSoA &S, int n, int i) {
  const size_t cap = (size_t)P.cap;
  int L = S.layer[i];
  int u = P.el_u[P.layer_off[L - 1] + S.elem[i]];
  phx_stream s;
  phx_stream_init(&s, P.seed, P.sample, (uint32_t)n, BRUTE ? d_tr_sub(P, i) : PHX_SUB_TRANSPORT, S.hid[i]);
  d_stream_seek(&s, 3u);
  double E = S.energy[i];
  double r = phx_uniform(&s);
  const double h = d_table(P.tab_uniform, P.ray_icdf + (size_t)u * P.n_e * P.n_r, P.tab_E, P.n_e, P.tab_E0, P.tab_Einv,
                           P.tab_R, P.n_r, P.tab_R0, P.tab_Rinv, E, r) * (0.5 / ENG_PI);
  /* half the scattering angle, over pi */
  const double sh = d_sinpi_core(h), ct = fma(-2.0 * sh, sh, 1.0), st = 2.0 * sh * d_cospi1(h);
  const double s2 = st * st, tt = s2 / (4.0 - 2.0 * s2);
  const double phi_i = d_table(P.tab_uniform, P.phi_icdf, P.phi_T, P.phi_nt, P.phi_T0, P.phi_Tinv, P.phi_R, P.phi_nr,
                               P.phi_R0, P.phi_Rinv, tt, phx_uniform(&s));
  double ev[3] = {S.ex[i], S.ey[i], S.ez[i]}, dirv[3] = {S.dx[i], S.dy[i], S.dz[i]}, ca, sa;
  const DFrame f = d_frame(dirv);
  d_azimuth(phi_i, &ca, &sa);
  d_from_polarisation(f, ev, &ca, &sa);
  d_turn(dirv, f, ct, st, ca, sa);
  d_update_elecv(dirv, ev);
  S.dx[i] = dirv[0];
  S.dy[i] = dirv[1];
  S.dz[i] = dirv[2];
  S.ex[i] = ev[0];
  S.ey[i] = ev[1];
  S.ez[i] = ev[2];
  /* brute force: the history row of the last interaction, and its element */
  S.prev_line[i] = BRUTE ? 384 : 0;
  if (BRUTE) S.prev_u[i] = u;
  (void)cap;
}

template <bool BRUTE, bool ADV>
__device__ __forceinline__ void d_compton_one(const EngineParams &P, const PhotonSoA &S, int n, int i) {
  const size_t cap = (size_t)P.cap;
  int L = S.layer[i];
  int u = P.el_u[P.layer_off[L - 1] + S.elem[i]];
  phx_stream s;
  phx_stream_init(&s, P.seed, P.sample, (uint32_t)n, BRUTE ? d_tr_sub(P, i) : PHX_SUB_TRANSPORT, S.hid[i]);
  d_stream_seek(&s, 3u);
  double E = S.energy[i];
  const double theta_i = d_table(P.tab_uniform, P.comp_icdf + (size_t)u * P.n_e * P.n_r, P.tab_E, P.n_e, P.tab_E0,
                                 P.tab_Einv, P.tab_R, P.n_r, P.tab_R0, P.tab_Rinv, E, phx_uniform(&s));
  /* half the scattering angle, over pi */
  const double h = theta_i * (0.5 / ENG_PI), sth2 = d_sinpi_core(h), mct = 2.0 * sth2 * sth2; /* 1 - cos theta */
  const double ct = 1.0 - mct, st = 2.0 * sth2 * d_cospi1(h);
  const double K0K = 1.0 + E * mct / ENG_MEC2, st2 = st * st;
  const double tt = st2 / (K0K + (1.0 / K0K) - st2) / 2.0;
  const double phi_i = d_table(P.tab_uniform, P.phi_icdf, P.phi_T, P.phi_nt, P.phi_T0, P.phi_Tinv, P.phi_R, P.phi_nr,
                               P.phi_R0, P.phi_Rinv, tt, phx_uniform(&s));
  if (ADV) {
    /* xmi_update_photon_energy_compton: the subshell by count * CDF(Qimax),
     * Q from its profile below Qimax, the energy from Q; 0 ends the photon */
    const xrl_atom *a = &P.atoms[u];
    const int g0 = P.cp_sh_off[u], g1 = P.cp_sh_off[u + 1];
    double csum = 0.0;
    for (int g = g0; g < g1; g++)
      csum += a->occupancy[P.cp_sh_idx[g]] * d_adv_cdf(P, a->edge[P.cp_sh_idx[g]], g, E, ct);
    if (csum == 0.0) {
      S.energy[i] = 0.0;
      return;
    }
    const double r = phx_uniform(&s);
    double ts = 0.0, cdf_sel = 0.0;
    int sel = -1, last = g0;
    for (int g = g0; g < g1; g++) {
      const double w = a->occupancy[P.cp_sh_idx[g]] * d_adv_cdf(P, a->edge[P.cp_sh_idx[g]], g, E, ct);
      if (w > 0.0) last = g;
      ts += w / csum;
      if (r <= ts) {
        sel = g;
        break;
      }
    }
    if (sel < 0) sel = last; /* rounding left the running sum just below r */
    cdf_sel = d_adv_cdf(P, a->edge[P.cp_sh_idx[sel]], sel, E, ct);
    const double e = d_energy_from_q(E, d_adv_q(P, sel, phx_uniform(&s) * cdf_sel), ct);
    if (!(e > 0.0)) {
      S.energy[i] = 0.0;
      return;
    }
    E = e;
    S.energy[i] = E;
    d_mu_all(P, E, S.mus, cap, i);
  } else {
  /* xmi_update_photon_energy_compton2 */
  const double cc = (double)1.2399e-6f, c0 = (double)4.85e-12f, c1 = (double)1.456e-2f;
  double energy = E * 1000.0;
  double c_lamb0 = cc / energy;
  const double *icdf = P.cp_icdf + (size_t)u * P.cp_len;
  /* the reference loops until acceptance; every draw with pz <= 0 is accepted,
   * so the bound below is never reached by valid data and only turns a
   * corrupted table into a counted error instead of a hung wave */
  int accepted = 0;
  for (int it = 0; it < 4096; it++) {
    double r = phx_uniform(&s);
    double pz = d_grid_lookup(P.cp_rn_uniform, P.cp_rn, icdf, P.cp_len, P.cp_rn_inv, r);
    if (phx_uniform(&s) < 0.5) pz = -pz;
    double dlamb = c0 * sth2 * sth2 - c1 * c_lamb0 * sth2 * pz;
    energy = cc / (c_lamb0 + dlamb) / 1000.0;
    if (energy <= E) {
      accepted = 1;
      break;
    }
  }
  if (!accepted) {
    atomicAdd(d_ctr(P, ENG_CNT_ERRORS), 1ull);
    atomicAdd(d_ctr(P, ENG_CNT_ERR_DOPPLER), 1ull);
    S.energy[i] = 0.0;
    return;
  }
  E = energy;
  S.energy[i] = E;
  d_mu_all(P, E, S.mus, cap, i);
  if (E == 0.0) return;
  }
  double ev[3] = {S.ex[i], S.ey[i], S.ez[i]}, dirv[3] = {S.dx[i], S.dy[i], S.dz[i]};
  double cph, sph;
  d_azimuth(phi_i, &cph, &sph);
  {
    const DFrame f = d_frame(dirv);
    double ca = cph, sa = sph;
    d_from_polarisation(f, ev, &ca, &sa);
    d_turn(dirv, f, ct, st, ca, sa);
  }
  d_update_elecv(dirv, ev);
  double pp = 2.0 * ((ct * cph) * (ct * cph) + sph * sph);
  double rat = 1.0 / (1.0 + mct * E / (double)510.998910f);
  double rk = rat - 2.0 + 1.0 / rat;
  pp = pp / (rk + pp);
  double r = phx_uniform(&s);
  double w_h = (1.0 + pp) / 2.0;
  if (r > w_h) {
    double c0x = dirv[1] * ev[2] - dirv[2] * ev[1];
    double c1x = dirv[2] * ev[0] - dirv[0] * ev[2];
    double c2x = dirv[0] * ev[1] - dirv[1] * ev[0];
    ev[0] = c0x;
    ev[1] = c1x;
    ev[2] = c2x;
  }
  S.dx[i] = dirv[0];
  S.dy[i] = dirv[1];
  S.dz[i] = dirv[2];
  S.ex[i] = ev[0];
  S.ey[i] = ev[1];
  S.ez[i] = ev[2];
  S.prev_line[i] = BRUTE ? 385 : 0;
  if (BRUTE) S.prev_u[i] = u;
}

/* Coster-Kronig vacancy shift, src/xmi_main.F90:5184-5323 */
__device__ int d_coster_kronig(const xrl_atom *a, phx_stream *s, int shell) {
  const double *f = a->ck;
  if (shell == 1 || shell == 2) {
    for (;;) {
      double r = phx_uniform(s);
      if (shell == 2) {
        if (r < f[XRL_FL23]) shell = 3;
        return shell;
      }
      if (r < f[XRL_FL12]) {
        shell = 2;
        continue;
      }
      if (r < f[XRL_FL12] + f[XRL_FL13]) shell = 3;
      return shell;
    }
  } else if (shell >= 4 && shell <= 7) {
    for (;;) {
      double r = phx_uniform(s);
      if (shell == 7) {
        if (r < f[XRL_FM45]) shell = 8;
        return shell;
      } else if (shell == 6) {
        if (r < f[XRL_FM34]) {
          shell = 7;
          continue;
        }
        if (r < f[XRL_FM34] + f[XRL_FM35]) shell = 8;
        return shell;
      } else if (shell == 5) {
        double sum = f[XRL_FM23];
        if (r < sum) {
          shell = 6;
          continue;
        }
        sum += f[XRL_FM24];
        if (r < sum) {
          shell = 7;
          continue;
        }
        sum += f[XRL_FM25];
        if (r < sum) shell = 8;
        return shell;
      } else {
        double sum = f[XRL_FM12];
        if (r < sum) {
          shell = 5;
          continue;
        }
        sum += f[XRL_FM13];
        if (r < sum) {
          shell = 6;
          continue;
        }
        sum += f[XRL_FM14];
        if (r < sum) {
          shell = 7;
          continue;
        }
        sum += f[XRL_FM15];
        if (r < sum) shell = 8;
        return shell;
      }
    }
  }
  return shell;
}

/* first and last line of a vacancy's shell 0 (K) .. 8 (M5), one byte each
 * (xrl_shell_lines: a shell's last line precedes the next one's first) */
__device__ __forceinline__ int d_shell_first(int shell) {
  constexpr unsigned long long f = (unsigned long long)XRL_KL1 | (unsigned long long)XRL_L1_FIRST << 8 |
                                   (unsigned long long)XRL_L2_FIRST << 16 | (unsigned long long)XRL_L3_FIRST << 24 |
                                   (unsigned long long)XRL_M1_FIRST << 32 | (unsigned long long)XRL_M2_FIRST << 40 |
                                   (unsigned long long)XRL_M3_FIRST << 48 | (unsigned long long)XRL_M4_FIRST << 56;
  return shell < 8 ? (int)((f >> (8 * shell)) & 0xffull) : (shell == 8 ? XRL_M5_FIRST : XRL_M5_LAST + 1);
}
static_assert(XRL_KP5 + 1 == XRL_L1_FIRST && XRL_L1_LAST + 1 == XRL_L2_FIRST && XRL_L2_LAST + 1 == XRL_L3_FIRST &&
              XRL_L3_LAST + 1 == XRL_M1_FIRST && XRL_M1_LAST + 1 == XRL_M2_FIRST && XRL_M2_LAST + 1 == XRL_M3_FIRST &&
              XRL_M3_LAST + 1 == XRL_M4_FIRST && XRL_M4_LAST + 1 == XRL_M5_FIRST && XRL_M5_LAST < 255,
              "the shells' lines are consecutive");

/* the line that the number r selects among a shell's by the radiative rates
 * (first whose cumulative rate exceeds r), 0 for none; rate_cum holds each
 * shell's running sums, so five probes replace up to 29 dependent ones */
__device__ __forceinline__ int d_pick_line(const EngineParams &P, int u, int shell, double r) {
  if (shell < 0 || shell > 8) return 0;
  int lo = d_shell_first(shell), hi = d_shell_first(shell + 1);
  const double *cum = P.rate_cum + (size_t)u * (XMI_NLINES_VR_DEV + 1);
  const int end = hi;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (r < cum[mid]) hi = mid;
    else lo = mid + 1;
  }
  return lo < end ? lo : 0;
}

/* ------------------------------------------------------------------------ */
/* cascades of brute-force runs, src/xmi_main.F90:2413-4783 */

/* xmi_fluorescence_yield_check (src/xmi_main.F90:5325-5350): 1 when the
 * vacancy fluoresces.  Shells beyond M5 never do (the reference reads past
 * the end of its nine corrected yields there); the number is drawn all the
 * same. */
__device__ __forceinline__ int d_yield_check(const EngineParams &P, int u, int shell, phx_stream *s) {
  const double r = phx_uniform(s);
  const double y = (shell >= 0 && shell <= 8) ? P.fycorr[(size_t)u * 9 + shell] : 0.0;
  return !(r > y);
}

/* xmi_fluorescence_line_check (src/xmi_main.F90:5352-5437): the line of a
 * vacancy by the radiative rates, its energy, or 0 and line 0 */
__device__ double d_line_check(const EngineParams &P, int u, int shell, phx_stream *s, int *line) {
  *line = d_pick_line(P, u, shell, phx_uniform(s));
  return *line ? P.line_E[(size_t)u * XMI_NLINES_VR_DEV + (*line - 1)] : 0.0;
}

/* a cascade's photon in slot j: energy and attenuation, isotropic direction,
 * random polarisation made orthogonal to it, history row of its line, no
 * cascades left (src/xmi_main.F90:4330-4370,4720-4765) */
__device__ void d_cascade_emit(const EngineParams &P, const PhotonSoA &S, int j, double E, int line, int u,
                               phx_stream *s) {
  S.energy[j] = E;
  d_mu_all(P, E, S.mus, (size_t)P.cap, j);
  S.cflags[j] = 0;
  const double ct = 2.0 * phx_uniform(s) - 1.0, st = sqrt((1.0 - ct) * (1.0 + ct));
  double cp, sp, ev[3] = {0.0, 0.0, 0.0};
  d_turns(phx_uniform(s), &cp, &sp);
  const double dirv[3] = {st * cp, st * sp, ct};
  d_turns(phx_uniform(s), &ev[0], &ev[1]);
  d_update_elecv(dirv, ev);
  S.dx[j] = dirv[0];
  S.dy[j] = dirv[1];
  S.dz[j] = dirv[2];
  S.ex[j] = ev[0];
  S.ey[j] = ev[1];
  S.ez[j] = ev[2];
  S.prev_line[j] = line;
  S.prev_u[j] = u;
}

/* the offspring of slot i starts at the parent's interaction point, in its
 * layer, with its weight and history id */
__device__ __forceinline__ int d_offspring(const EngineParams &P, const PhotonSoA &S, int i) {
  const int j = i + P.off_half;
  S.x[j] = S.x[i];
  S.y[j] = S.y[i];
  S.z[j] = S.z[i];
  S.layer[j] = S.layer[i];
  S.elem[j] = S.elem[i];
  S.weight[j] = S.weight[i];
  S.hid[j] = S.hid[i];
  return j;
}

/* xmi_simulate_photon_cascade_auger (src/xmi_main.F90:2413-4594): the
 * vacancy's Auger transition (the provider's rates) leaves two vacancies;
 * the first may fluoresce as the parent photon, the second as the
 * offspring.  M vacancies count with use_M_lines only. */
__device__ int d_cascade_auger(const EngineParams &P, const PhotonSoA &S, int i, int u, const xrl_atom *a,
                               int shell, phx_stream *s) {
  int first, last, spawned = 0;
  if (!xrl_auger_range(shell, &first, &last)) return 0;
  const double r = phx_uniform(s);
  /* the first transition whose running sum exceeds r; five or six probes of
   * the table replace up to 64 rates of several divisions each, formed by the
   * few lanes of a wave whose vacancies decay so: the brute-force interactions
   * of 8e6 photons 578 -> 249 us a launch */
  const double *cum = P.auger_cum + (size_t)u * XRL_AUGER_N;
  int t = first, hi = last + 1;
  while (t < hi) {
    const int mid = (t + hi) >> 1;
    if (r < cum[mid]) hi = mid;
    else t = mid + 1;
  }
  if (t > last) return 0;
  int sh[2];
  xrl_auger_shells(t, &sh[0], &sh[1]);
  for (int k = 0; k < 2; k++) {
    const int m_shell = sh[k] >= XRL_M1_SHELL && sh[k] <= XRL_M5_SHELL;
    if ((m_shell && !P.use_M_lines) || !d_yield_check(P, u, sh[k], s)) continue;
    const int v = d_coster_kronig(a, s, sh[k]);
    int line;
    const double e = d_line_check(P, u, v, s, &line);
    if (e <= 1.0) continue;
    d_cascade_emit(P, S, k == 0 ? i : d_offspring(P, S, i), e, line, u, s);
    spawned = k == 1;
  }
  return spawned;
}

/* xmi_simulate_photon_cascade_radiative (src/xmi_main.F90:4596-4783): the
 * line the parent emitted leaves a vacancy in its other shell (K -> L or M;
 * L -> M with use_M_lines), which may fluoresce as the offspring; then the
 * parent has no cascades left either */
__device__ int d_cascade_radiative(const EngineParams &P, const PhotonSoA &S, int i, int u, const xrl_atom *a,
                                   int shell, int line, phx_stream *s) {
  int sn = -1;
  if (shell == XRL_K_SHELL) {
    if (line >= xrl_line_KL(0) && line <= xrl_line_KM(4)) sn = line; /* KL1..KL3, KM1..KM5 -> L1..M5 */
  } else if (shell >= XRL_L1_SHELL && shell <= XRL_L3_SHELL && P.use_M_lines) {
    const int base = xrl_line_LM(shell - 1, 0);
    if (line >= base && line <= base + 4) sn = XRL_M1_SHELL + (line - base);
  } else {
    return 0;
  }
  if (sn < 0) return 0;
  if (sn >= XRL_M1_SHELL && sn <= XRL_M5_SHELL && !P.use_M_lines) return 0;
  if (!d_yield_check(P, u, sn, s)) return 0;
  sn = d_coster_kronig(a, s, sn);
  int ln;
  const double e = d_line_check(P, u, sn, s, &ln);
  if (e <= 1.0) return 0;
  S.cflags[i] = 0;
  d_cascade_emit(P, S, d_offspring(P, S, i), e, ln, u, s);
  return 1;
}

/* returns 1 when a cascade started an offspring photon (brute force) */
template <bool BRUTE>
__device__ __forceinline__ int d_photo_one(const EngineParams &P, const PhotonSoA &S, int n, int i) {
  const size_t cap = (size_t)P.cap;
  int L = S.layer[i];
  int u = P.el_u[P.layer_off[L - 1] + S.elem[i]];
  const xrl_atom *a = &P.atoms[u];
  phx_stream s;
  phx_stream_init(&s, P.seed, P.sample, (uint32_t)n, BRUTE ? d_tr_sub(P, i) : PHX_SUB_TRANSPORT, S.hid[i]);
  d_stream_seek(&s, 3u);
  double E = S.energy[i];
  /* the shell by its share of the photo-ionisation: the cross sections are
   * E^-p times the shells' constants, so E^-p cancels */
  const double r_sh = phx_uniform(&s);
  const int max_shell = P.use_M_lines ? 8 : 3;
  int shell = -1;
  {
    int k = 0;
#pragma unroll
    for (int sh = 0; sh < 9; sh++) k += a->edge[sh] > E ? 1 : 0;
    const double target = r_sh * a->photo_Bsum[k];
    double sum = 0.0;
#pragma unroll
    for (int sh = 0; sh < 9; sh++) {
      const double e = a->edge[sh];
      if (sh <= max_shell && e > 0.0 && E >= e) sum += a->photo_B[sh];
      if (shell < 0 && target < sum) shell = sh;
    }
  }
  S.prev_line[i] = 0;
  if (shell < 0) {
    S.energy[i] = 0.0;
    return 0;
  }
  const double ry = phx_uniform(&s); /* unused by the reference's yield weighting */
  if (BRUTE) {
    /* the analogue yield, perhaps an Auger cascade (src/xmi_main.F90:2298-2315) */
    if (ry > P.fycorr[(size_t)u * 9 + shell]) {
      S.energy[i] = 0.0;
      return (S.cflags[i] & 1) ? d_cascade_auger(P, S, i, u, a, shell, &s) : 0;
    }
  } else {
    S.weight[i] *= P.fycorr[(size_t)u * 9 + shell];
  }
  shell = d_coster_kronig(a, &s, shell);
  const int line = d_pick_line(P, u, shell, phx_uniform(&s));
  if (line == 0) {
    S.energy[i] = 0.0;
    return 0;
  }
  E = P.line_E[(size_t)u * XMI_NLINES_VR_DEV + (line - 1)];
  S.energy[i] = E;
  for (int l = 0; l < P.n_layers; l++)
    S.mus[(size_t)l * cap + i] = P.precalc_mu[((size_t)l * P.nZ + u) * XMI_NLINES_VR_DEV + (line - 1)];
  /* isotropic: cos theta = 1 - 2 u */
  const double ui = phx_uniform(&s), ct = fma(-2.0, ui, 1.0), st = 2.0 * sqrt(ui * (1.0 - ui));
  double ca, sa;
  d_turns(phx_uniform(&s), &ca, &sa);
  double ev[3] = {S.ex[i], S.ey[i], S.ez[i]}, dirv[3] = {S.dx[i], S.dy[i], S.dz[i]};
  d_turn(dirv, d_frame(dirv), ct, st, ca, sa);
  d_update_elecv(dirv, ev);
  S.dx[i] = dirv[0];
  S.dy[i] = dirv[1];
  S.dz[i] = dirv[2];
  S.ex[i] = ev[0];
  S.ey[i] = ev[1];
  S.ez[i] = ev[2];
  S.prev_line[i] = line;
  S.prev_u[i] = u;
  if (BRUTE && (S.cflags[i] & 2)) return d_cascade_radiative(P, S, i, u, a, shell, line, &s);
  return 0;
}

/* exclusive prefix sums of the 3 x ENG_SPREAD sub-queue lengths of the
 * interaction queues into off[0..3 ENG_SPREAD], off[3 ENG_SPREAD] = total
 * (first wave of the workgroup; the caller synchronises) */
__device__ __forceinline__ void d_queue_offsets(const unsigned long long *qc, unsigned int *off) {
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    unsigned int base = 0;
    for (int t = 0; t < 3; t++) {
      const unsigned int c = (unsigned int)qc[(size_t)t * ENG_SPREAD + lane];
      unsigned int x = c;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const unsigned int y = __shfl_up(x, d);
        if (lane >= d) x += y;
      }
      off[t * ENG_SPREAD + lane] = base + x - c;
      base += __shfl(x, 63);
    }
    if (lane == 0) off[3 * ENG_SPREAD] = base;
  }
}

/* wavefront-aggregated append of the lanes with pred to a list (one atomic
 * per wave; for rare entries such as a cascade's offspring) */
__device__ __forceinline__ void d_list_append(int *list, unsigned int *cnt, int pred, int idx) {
  const unsigned long long m = __ballot(pred);
  if (!m) return;
  const int lane = __lane_id(), leader = __ffsll((long long)m) - 1;
  unsigned int base = 0;
  if (lane == leader) base = atomicAdd(cnt, (unsigned int)__popcll(m));
  base = __shfl(base, leader);
  if (pred) list[base + __popcll(m & ((1ull << lane) - 1ull))] = idx;
}

/* entry q of the concatenated interaction queues (Rayleigh, Compton, photo;
 * each queue's ENG_SPREAD sub-queues in order; off: their prefix sums): the
 * photon's slot, and the queue in *type */
__device__ __forceinline__ int d_queue_entry(const EngineParams &P, const unsigned int *off, unsigned int q, int *type) {
  int lo = 0, hi = 3 * ENG_SPREAD;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= q) lo = mid;
    else hi = mid;
  }
  *type = lo / ENG_SPREAD;
  return P.queue[(size_t)lo * P.qreg + (q - off[lo])];
}

/* the interaction of the photon in slot i from queue `type`; returns 1 when a
 * cascade started an offspring */
template <bool BRUTE, bool ADV>
__device__ __forceinline__ int d_interact_one(const EngineParams &P, const PhotonSoA &S, int n, int type, int i) {
  if (type == 0) d_rayleigh_one<BRUTE>(P, S, n, i);
  else if (type == 1) d_compton_one<BRUTE, ADV>(P, S, n, i);
  else return d_photo_one<BRUTE>(P, S, n, i);
  return 0;
}

/* one launch serves the three interaction queues: thread q takes entry q of
 * their concatenation, so the grid's empty waves are only those beyond the
 * photons that interact at this order, and a wavefront straddles two queues
 * at two places at most.  Each photon is one thread's, with its own random
 * stream, so results do not depend on the assignment. */
/* bound by the latency of its gathers (78 % of the wave cycles wait, 31 % of
 * the vector issue): eight waves per SIMD, 63 VGPRs without spills, measured
 * 2 % faster than seven.  ADV: the advanced Compton model, compiled apart */
template <bool ADV>
__global__ void __launch_bounds__(ENG_BLOCK) __attribute__((amdgpu_waves_per_eu(8)))
k_interact(EngineParams P, PhotonSoA S, int n) {
  __shared__ unsigned int off[3 * ENG_SPREAD + 1];
  d_queue_offsets(P.qcount, off);
  __syncthreads();
  const unsigned int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= off[3 * ENG_SPREAD]) return;
  int type;
  const int i = d_queue_entry(P, off, q, &type);
  (void)d_interact_one<false, ADV>(P, S, n, type, i);
}

/* the brute-force interactions (analogue yields, cascades), one thread per
 * queue entry as in k_interact; the offspring that cascades start join the
 * offspring list.  (A fixed grid striding over the entries would keep the
 * kernel's many table pointers live across the loop: at five waves per SIMD
 * that spills 200 VGPRs instead of about 50.)  Four waves per SIMD run 3 %
 * faster than five here. */
template <bool ADV>
__global__ void __launch_bounds__(ENG_BLOCK) __attribute__((amdgpu_waves_per_eu(4)))
k_interact_brute(EngineParams P, PhotonSoA S, int n) {
  __shared__ unsigned int off[3 * ENG_SPREAD + 1];
  d_queue_offsets(P.qcount, off);
  __syncthreads();
  const unsigned int total = off[3 * ENG_SPREAD], q = blockIdx.x * blockDim.x + threadIdx.x;
  if (blockIdx.x * blockDim.x >= total) return;
  int i = -1, spawned = 0;
  if (q < total) {
    int type;
    i = d_queue_entry(P, off, q, &type);
    spawned = d_interact_one<true, ADV>(P, S, n, type, i);
  }
  d_list_append(P.olist_out, P.ocount_out, spawned, i + P.off_half);
}

/* ------------------------------------------------------------------------ */
/* escape-ratio runs (src/xmi_main.F90:5473-5801 with the analogue step of
 * :1274-1407): after its forced first interaction a photon leaves the crystal
 * when the analogue step's random number (the first draw of the next order's
 * transport stream) exceeds the probability of interacting on the way out;
 * escaped Compton photons are tallied by energy, fluorescence photons by
 * element and line (weight times fluorescence yield), and the weight after
 * the forced step of every interacted photon normalises its input energy.
 * One thread per queue entry of the three interaction queues. */

/* integer sum of v over the wavefront, wave-uniform (the row steps of
 * d_wave_total2, then row_bcast:31 into rows 2 and 3: lane 63 holds it) */
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ unsigned long long d_dpp0_u64(unsigned long long v) {
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)v, CTRL, ROW_MASK, 0xf, true);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(v >> 32), CTRL, ROW_MASK, 0xf, true);
  return ((unsigned long long)hi << 32) | lo;
}
__device__ __forceinline__ unsigned long long d_wave_total_u64(unsigned long long v) {
  v += d_dpp0_u64<0x111, 0xf>(v);
  v += d_dpp0_u64<0x112, 0xf>(v);
  v += d_dpp0_u64<0x114, 0xf>(v);
  v += d_dpp0_u64<0x118, 0xf>(v);
  v += d_dpp0_u64<0x142, 0xa>(v);
  v += d_dpp0_u64<0x143, 0xc>(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)v, 63);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(v >> 32), 63);
  return ((unsigned long long)hi << 32) | lo;
}

/* exact wave-aggregated fixed-point add: every lane with key >= 0 adds
 * value to bin key of tally; the lanes of one key are summed as integers
 * (three 42-bit limbs, which 64 lanes cannot overflow) and added once, so
 * that thousands of photons of one bin do not serialise on its address and
 * the sum does not depend on which photons share a wavefront.  From the first
 * key with fewer than FEW lanes on, the remaining lanes add for themselves
 * (Compton energies: nearly every lane its own bin).  Call from converged
 * code. */
template <int FEW>
__device__ __forceinline__ void d_fx_add_keyed(unsigned long long *tally, long key, double value, int shift) {
  unsigned long long pending = __ballot(key >= 0);
  if (!pending) return;
  unsigned long long lo = 0ull, hi = 0ull;
  if (key >= 0) fx_split(value, shift, &lo, &hi);
  const unsigned long long M42 = (1ull << 42) - 1ull;
  const unsigned long long l0 = lo & M42, l1 = (lo >> 42) | ((hi & ((1ull << 20) - 1ull)) << 22), l2 = hi >> 20;
  while (pending) {
    const int leader = __ffsll((long long)pending) - 1;
    const long k = (long)(((unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(key >> 32), leader) << 32) |
                          (unsigned)__builtin_amdgcn_readlane((int)key, leader));
    const int mine = key == k;
    const unsigned long long group = __ballot(mine);
    if (FEW > 1 && __popcll(group) < FEW) {
      if ((pending >> __lane_id()) & 1ull) fx_merge_global(&tally[(size_t)key * 2], lo, hi);
      return;
    }
    const unsigned long long a0 = d_wave_total_u64(mine ? l0 : 0ull), a1 = d_wave_total_u64(mine ? l1 : 0ull),
                             a2 = d_wave_total_u64(mine ? l2 : 0ull);
    if (__lane_id() == leader) {
      const unsigned __int128 t = (unsigned __int128)a0 + ((unsigned __int128)a1 << 42) + ((unsigned __int128)a2 << 84);
      fx_merge_global(&tally[(size_t)k * 2], (unsigned long long)t, (unsigned long long)(t >> 64));
    }
    pending &= ~group;
  }
}

/* interaction and way out in one thread, so that the photon's record stays in
 * the caches between them: a launch of its own over the record of 8e6 photons
 * took 555 us after the interactions' 520 and a copy of the weights; together
 * 831 (four waves per SIMD; six spill and take 879) */
__global__ void __launch_bounds__(ENG_BLOCK) __attribute__((amdgpu_waves_per_eu(4)))
k_interact_escape(EngineParams P, PhotonSoA S, EscParams Q) {
  __shared__ unsigned int off[3 * ENG_SPREAD + 1];
  d_queue_offsets(P.qcount, off);
  __syncthreads();
  const unsigned int total = off[3 * ENG_SPREAD], q = blockIdx.x * blockDim.x + threadIdx.x;
  if (blockIdx.x * blockDim.x >= total) return;
  const int shift = P.tally_shift;
  long key_n = -1, key_c = -1, key_f = -1;
  double w_n = 0.0, w = 0.0;
  if (q < total) {
    int type;
    const int i = d_queue_entry(P, off, q, &type);
    w_n = S.weight[i];
    (void)d_interact_one<false, false>(P, S, 1, type, i);
    const int iE = (int)(S.hid[i] / (uint64_t)Q.n_photons);
    if (iE >= 0 && iE < Q.nE) {
      /* the photon's weight after the forced step (w_n) normalises; the
       * photo-absorption step has multiplied S.weight by the fluorescence
       * yield, which an escape-ratio run applies to the escape tally only
       * (src/xmi_variance_reduction.F90:742-746) */
      key_n = iE;
      w = S.weight[i];
      const double E = S.energy[i];
      const int cur = S.layer[i];
      int escaped = E >= 1.0 && cur >= 1; /* below the energy threshold: stays inside */
      if (escaped) {
        phx_stream s;
        phx_stream_init(&s, P.seed, P.sample, 2u, PHX_SUB_TRANSPORT, S.hid[i]);
        const double R = phx_uniform(&s);
        const double dirv[3] = {S.dx[i], S.dy[i], S.dz[i]};
        const int up = d_dot(dirv, P.n_sample) > 0.0;
        double lp[3] = {S.x[i], S.y[i], S.z[i]};
        double max_r = 0.0, blbs = 1.0;
        const size_t cap = (size_t)P.cap;
        for (int l = cur - 1; up ? l < P.n_layers : l >= 0; l += up ? 1 : -1) {
          double pp[3] = {0.0, 0.0, up ? P.layer_ze[l] : P.layer_zb[l]}, ip[3];
          d_intersect(pp, P.n_sample, lp, dirv, ip);
          const double dist = d_distance(lp, ip);
          const double temp_prod = -1.0 * dist * P.layer_density[l] * S.mus[(size_t)l * cap + i];
          const double tempexp = exp(temp_prod);
          max_r = max_r - blbs * expm1(temp_prod);
          if (R <= max_r) { /* interacts on the way out: inside */
            escaped = 0;
            break;
          }
          lp[0] = ip[0];
          lp[1] = ip[1];
          lp[2] = ip[2];
          blbs = blbs * tempexp;
        }
      }
      if (escaped && type == 1) {
        const int idx = (int)((E - Q.out0) / Q.dOut) + 1;
        if (idx >= 1 && idx <= Q.nOut) key_c = (long)(idx - 1) * Q.nE + iE;
      } else if (escaped && type == 2) {
        const int line = S.prev_line[i], u = S.prev_u[i];
        if (line >= 1 && line <= ENG_ESC_LINES && u >= 0) key_f = ((long)iE * ENG_ESC_LINES + (line - 1)) * P.nZ + u;
      }
    }
  }
  d_fx_add_keyed<1>(Q.interacted, key_n, w_n, shift);
  d_fx_add_keyed<4>(Q.compton, key_c, w, shift);
  d_fx_add_keyed<1>(Q.fluo, key_f, w, shift);
}

/* ------------------------------------------------------------------------ */
/* host-side launch wrappers */

static size_t lds_if_fits(size_t words) {
  size_t b = words * sizeof(unsigned long long);
  return b <= ENG_LDS_BYTES ? b : 0;
}
static size_t scatter_lds_bytes(const EngineParams *P) { return lds_if_fits((size_t)P->nch * 2 + (size_t)P->nZ * 4); }
static size_t lines_lds_bytes(const EngineParams *P) { return lds_if_fits((size_t)P->n_lbins * 2); }

/* Workgroups of a grid-stride kernel: as many as can be resident at once,
 * since every workgroup ends with one flush of its LDS tallies to global
 * memory.  per_cu > 0 (the run's launch configuration) overrides the
 * resident count per CU. */
static int resident_blocks(const void *kernel, size_t lds, int n_cu, int blocks, int per_cu = 0) {
  if (per_cu <= 0 &&
      (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, ENG_BLOCK, lds) != hipSuccess || per_cu < 1))
    per_cu = 1;
  int vb = n_cu * per_cu;
  if (vb > blocks) vb = blocks;
  return vb < 1 ? 1 : vb;
}

/* ------------------------------------------------------------------------ */
/* brute-force runs (use_variance_reduction = 0): the analogue step of
 * src/xmi_main.F90:1274-1407 with the detector tests of every path segment,
 * one thread per photon slot; a photon that reaches the detector is tallied
 * by its energy and its last interaction (src/xmi_main.F90:445-535) and its
 * history ends, as it does when it leaves the sample elsewhere or hits the
 * collimator */

/* lab -> detector frame: x along the detector axis towards the sample, the
 * window at x = 0 */
__device__ __forceinline__ void d_det_frame(const EngineParams &P, const double *x, double *o) {
  const double d[3] = {x[0] - P.p_det[0], x[1] - P.p_det[1], x[2] - P.p_det[2]};
  d_matvec(P.det_inv, d, o);
}

/* xmi_check_detector_intersection (src/xmi_aux_f.F90:1622-1833) of the path
 * segment b -> e: 0 none, 1 collimator, 2 window, 3 window from behind.
 * Without a collimator the reference's line direction is norm(e - b), a
 * scalar assigned to all three components (src/xmi_aux_f.F90:1668): the line
 * (L, L, L) crosses x = 0 at (0, e_y - e_x, e_z - e_x), always as a crossing
 * from behind.  Kept as computed there.  A line parallel to the window,
 * where the reference stops the program, counts as no crossing. */
template <bool COLL>
__device__ __forceinline__ int d_detector_segment(const EngineParams &P, const double *b, const double *e) {
  double bd[3], ed[3], ip[3];
  d_det_frame(P, b, bd);
  d_det_frame(P, e, ed);
  const double o[3] = {0.0, 0.0, 0.0}, nx[3] = {1.0, 0.0, 0.0};
  if (!COLL) {
    if (bd[0] * ed[0] > 0.0) return 0;
    const double L = d_distance(ed, bd);
    const double ld[3] = {L, L, L};
    if (!d_intersect(o, nx, ed, ld, ip)) return 0;
    ip[0] = 0.0;
    if (d_norm(ip) <= P.det_radius) return ld[0] >= 0.0 ? 3 : 2;
    return 0;
  }
  const double ld[3] = {ed[0] - bd[0], ed[1] - bd[1], ed[2] - bd[2]};
  const double t_begin = (bd[0] - ed[0]) / ld[0], t_end = (ed[0] - ed[0]) / ld[0];
  const double t_hi = t_begin > t_end ? t_begin : t_end, t_lo = t_begin < t_end ? t_begin : t_end;
  const double c2t = P.det_cos2;
  const double m[3] = {1.0 - c2t, -c2t, -c2t};
  const double delta[3] = {ed[0] - P.det_vertex[0], ed[1] - P.det_vertex[1], ed[2] - P.det_vertex[2]};
  const double dM[3] = {ld[0] * m[0], ld[1] * m[1], ld[2] * m[2]};
  const double deltaM[3] = {delta[0] * m[0], delta[1] * m[1], delta[2] * m[2]};
  const double c2 = d_dot(dM, ld), c1 = d_dot(dM, delta), c0 = d_dot(deltaM, delta);
  const double disc = c1 * c1 - c0 * c2;
  if (disc < 0.0) return 0;
  const double t1 = (-c1 + sqrt(disc)) / c2, t2 = (-c1 - sqrt(disc)) / c2;
  const double x1 = ed[0] + t1 * ld[0], x2 = ed[0] + t2 * ld[0];
  const int v1 = -(x1 - P.det_vertex[0]) >= 0.0, v2 = -(x2 - P.det_vertex[0]) >= 0.0;
  const double h = P.coll_height;
  if (!v1 && !v2) return 0;
  if (v1 && v2) {
    if (t1 <= t_hi && t1 >= t_lo && x1 <= h) return 1;
    if (t2 <= t_hi && t2 >= t_lo && x2 <= h) return 1;
    return 0;
  }
  const double t = v1 ? t1 : t2, xx = v1 ? x1 : x2;
  if (t <= t_hi && t >= t_lo && xx <= h) return 1;
  if (!d_intersect(o, nx, ed, ld, ip)) return 0;
  ip[0] = 0.0;
  if (d_norm(ip) <= P.det_radius && d_distance(bd, ip) <= d_distance(bd, ed)) return ld[0] >= 0.0 ? 3 : 2;
  return 0;
}

/* xmi_check_photon_detector_hit (src/xmi_main.F90:1920-1984): a photon that
 * left the sample reaches the detector when it moves against the detector
 * normal and crosses the window (and the collimator's top) within their
 * radii */
template <bool COLL>
__device__ __forceinline__ int d_escape_hits_detector(const EngineParams &P, const double *coords, const double *dirv) {
  if (d_dot(dirv, P.n_det) >= 0.0) return 0;
  double dd[3], cd[3], ip[3];
  d_matvec(P.det_inv, dirv, dd);
  d_det_frame(P, coords, cd);
  const double o[3] = {0.0, 0.0, 0.0}, nx[3] = {1.0, 0.0, 0.0};
  if (!d_intersect(o, nx, cd, dd, ip)) return 0;
  if (d_norm(ip) > P.det_radius) return 0;
  if (!COLL) return 1;
  const double pc[3] = {P.coll_height, 0.0, 0.0};
  if (!d_intersect(pc, nx, cd, dd, ip)) return 0;
  ip[0] = 0.0;
  return d_norm(ip) <= P.coll_radius;
}

/* the analogue step of photon i at order n: a photon alive after n - 1
 * interactions takes its step; one that stays in the sample with fewer than
 * n_int interactions gets its atom and interaction type (*type), the others
 * end, those that reach the detector tallied (*key_ch, *key_h, *w_hit) */
template <bool COLL>
__device__ __forceinline__ void d_brute_step(const EngineParams &P, const PhotonSoA &S, int n, int i, int *type,
                                             int *stepped, int *reached, long *key_ch, long *key_h, double *w_hit) {
  const size_t cap = (size_t)P.cap;
  const double E = S.energy[i];
  if (E < 1.0) {
    S.layer[i] = 0;
    return;
  }
  *stepped = 1;
  phx_stream s;
  phx_stream_init(&s, P.seed, P.sample, (uint32_t)n, d_tr_sub(P, i), S.hid[i]);
  const double R = phx_uniform(&s);
  const double dirv[3] = {S.dx[i], S.dy[i], S.dz[i]};
  double c[3] = {S.x[i], S.y[i], S.z[i]};
  const int cur = S.layer[i];
  const int up = d_dot(dirv, P.n_sample) > 0.0;
  const int last = up ? P.n_layers : 1, dir = up ? 1 : -1;
  double max_r = 0.0, min_r = 0.0, blbs = 1.0;
  int inside = 0, hit = 0, ended = 0;
  for (int l = cur; up ? l <= last : l >= last; l += dir) {
    const int l0 = l - 1;
    const double pp[3] = {0.0, 0.0, up ? P.layer_ze[l0] : P.layer_zb[l0]};
    double ip[3];
    d_intersect(pp, P.n_sample, c, dirv, ip);
    const double mu = S.mus[(size_t)l0 * cap + i];
    double dist = d_distance(c, ip);
    const double temp_prod = -1.0 * dist * P.layer_density[l0] * mu;
    const double em = expm1(temp_prod); /* e^t = 1 + em to the rounding that max_r carries */
    min_r = max_r;
    max_r = max_r - blbs * em;
    if (R <= max_r) {
      dist = -1.0 * log1p(-1.0 * (R - min_r) / blbs) / mu / P.layer_density[l0];
      const double to[3] = {c[0] + dist * dirv[0], c[1] + dist * dirv[1], c[2] + dist * dirv[2]};
      const int rc = d_detector_segment<COLL>(P, c, to);
      c[0] = to[0];
      c[1] = to[1];
      c[2] = to[2];
      if (rc) {
        ended = 1;
        hit = rc == 2;
      } else {
        inside = l;
      }
      break;
    }
    const int rc = d_detector_segment<COLL>(P, c, ip);
    if (rc) {
      ended = 1;
      hit = rc == 2;
      break;
    }
    c[0] = ip[0];
    c[1] = ip[1];
    c[2] = ip[2];
    blbs = fma(blbs, em, blbs);
  }
  if (!inside && !ended) hit = d_escape_hits_detector<COLL>(P, c, dirv);
  if (hit) {
    /* channels(n_interactions:, channel) and the history row of the last
     * interaction; the host sums the orders into the cumulative rows */
    *reached = 1;
    *w_hit = S.weight[i];
    const int ch = (int)((E - P.zero) / P.gain);
    if (ch >= 0 && ch < P.nch) *key_ch = (long)(n - 1) * P.nch + ch;
    if (n >= 2 && S.prev_line[i] > 0 && S.prev_u[i] >= 0)
      *key_h = ((long)(n - 2) * P.nZ + S.prev_u[i]) * 385 + (S.prev_line[i] - 1);
  }
  if (!inside || n > P.n_int) {
    S.layer[i] = 0;
  } else {
    S.x[i] = c[0];
    S.y[i] = c[1];
    S.z[i] = c[2];
    S.layer[i] = inside;
    *type = d_select(P, S, i, E, inside, S.mus[(size_t)(inside - 1) * cap + i], &s);
  }
}

/* order n of a brute-force run.  The photons alive at its start are the
 * batch's primaries at n = 1; afterwards the entries of order n - 1's
 * interaction queues (those that interacted) followed by the offspring that
 * its cascades started.  A fixed grid strides over them, every lane of a
 * wave taking the same trips, so that the queue appends, counters and
 * tallies see converged waves.  COLL: with a detector collimator, whose cone
 * test takes the registers (163 VGPRs, three waves per SIMD); without one four
 * waves (128 VGPRs) run 7 % faster than three and 10 % than five, whose spills
 * cost more: 371 us a launch over the orders of 8e6 photons, 414 with the cone
 * test compiled in and two exponentials a layer. */
template <bool COLL>
__global__ void __launch_bounds__(ENG_BLOCK) __attribute__((amdgpu_waves_per_eu(COLL ? 3 : 4)))
k_step_brute(EngineParams P, PhotonSoA S, int n, int count) {
  constexpr int NS = 3 * ENG_SPREAD;
  __shared__ unsigned int off[NS + 1];
  unsigned int nq = 0, total = (unsigned int)count;
  if (n >= 2) {
    d_queue_offsets(P.pqcount, off);
    __syncthreads();
    nq = off[NS];
    total = nq + (P.off_half ? *P.ocount_in : 0u);
  }
  const unsigned int stride = gridDim.x * blockDim.x;
  for (unsigned int base = blockIdx.x * blockDim.x; base < total; base += stride) {
    const unsigned int q = base + threadIdx.x;
    int type = -1, stepped = 0, reached = 0, i = -1;
    long key_ch = -1, key_h = -1;
    double w_hit = 0.0;
    if (q < total) {
      if (n == 1) {
        i = (int)q;
      } else if (q < nq) {
        int lo = 0, hi = NS;
        while (hi - lo > 1) {
          const int mid = (lo + hi) >> 1;
          if (off[mid] <= q) lo = mid;
          else hi = mid;
        }
        i = P.pqueue[(size_t)lo * P.qreg + (q - off[lo])];
      } else {
        i = P.olist_in[q - nq];
      }
      if (S.layer[i] > 0) d_brute_step<COLL>(P, S, n, i, &type, &stepped, &reached, &key_ch, &key_h, &w_hit);
    }
    d_enqueue(P, type, i);
    d_wave_count(d_ctr(P, ENG_CNT_STEPS), stepped);
    d_wave_count(d_ctr(P, ENG_CNT_HITS), reached);
    d_fx_add_keyed<4>(P.t_bch, key_ch, w_hit, P.tally_shift);
    d_fx_add_keyed<4>(P.t_bhist, key_h, w_hit, P.tally_shift);
  }
}

static void launch_interact(const EngineParams *P, const PhotonSoA *S, int n, int blocks, hipStream_t st) {
  if (P->adv_compton) hipLaunchKernelGGL(k_interact<true>, dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, n);
  else hipLaunchKernelGGL(k_interact<false>, dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, n);
}

static void launch_interact_brute(const EngineParams *P, const PhotonSoA *S, int n, int blocks, hipStream_t st) {
  if (P->adv_compton) hipLaunchKernelGGL(k_interact_brute<true>, dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, n);
  else hipLaunchKernelGGL(k_interact_brute<false>, dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, n);
}

template <int NL, int KP>
static void launch_lines_kp(const EngineParams *P, const PhotonSoA *S, const VrSoA *V, int n, int n_cu, int blocks,
                            hipStream_t st) {
  const size_t ll = lines_lds_bytes(P);
  if (ll) {
    int vb = resident_blocks((const void *)k_vr_lines<NL, KP, true>, ll, n_cu, blocks, P->wg_per_cu);
    hipLaunchKernelGGL((k_vr_lines<NL, KP, true>), dim3(vb), dim3(ENG_BLOCK), ll, st, *P, *S, *V, n);
  } else {
    int vb = resident_blocks((const void *)k_vr_lines<NL, KP, false>, 0, n_cu, blocks, P->wg_per_cu);
    hipLaunchKernelGGL((k_vr_lines<NL, KP, false>), dim3(vb), dim3(ENG_BLOCK), 0, st, *P, *S, *V, n);
  }
}

/* photons per lane of k_vr_lines (P->lines_kp, 0: the default): an entry's
 * loads, staging and reduction then serve 64 KP photons; fewer where the
 * per-photon path lengths take more registers.  Four up to three layers
 * (107 VGPRs, four waves per SIMD; three photons run 3 % slower on the
 * three-layer tube run, 10 % on one layer), three up to five (three against
 * four on four layers: 2 % faster), two up to eight */
template <int NL>
static void launch_lines(const EngineParams *P, const PhotonSoA *S, const VrSoA *V, int n, int n_cu, int blocks,
                         hipStream_t st) {
  const int kp = P->lines_kp;
  if constexpr (NL <= 4) {
    if (kp == 2) launch_lines_kp<NL, 2>(P, S, V, n, n_cu, blocks, st);
    else if (kp == 3 || (kp != 4 && NL == 4)) launch_lines_kp<NL, 3>(P, S, V, n, n_cu, blocks, st);
    else launch_lines_kp<NL, 4>(P, S, V, n, n_cu, blocks, st);
  } else if constexpr (NL <= 5) {
    if (kp == 1) launch_lines_kp<NL, 1>(P, S, V, n, n_cu, blocks, st);
    else if (kp == 2) launch_lines_kp<NL, 2>(P, S, V, n, n_cu, blocks, st);
    else launch_lines_kp<NL, 3>(P, S, V, n, n_cu, blocks, st);
  } else if constexpr (NL <= 8) {
    if (kp == 1) launch_lines_kp<NL, 1>(P, S, V, n, n_cu, blocks, st);
    else launch_lines_kp<NL, 2>(P, S, V, n, n_cu, blocks, st);
  } else {
    launch_lines_kp<NL, 1>(P, S, V, n, n_cu, blocks, st);
  }
}

template <int NL, bool ADV>
static void launch_scatter(const EngineParams *P, const PhotonSoA *S, const VrSoA *V, int n, int n_cu, int blocks,
                           size_t ls, hipStream_t st) {
  if (ls) {
    int vb = resident_blocks((const void *)k_vr_scatter<NL, true, ADV>, ls, n_cu, blocks, P->wg_per_cu);
    hipLaunchKernelGGL((k_vr_scatter<NL, true, ADV>), dim3(vb), dim3(ENG_BLOCK), ls, st, *P, *S, *V, n);
  } else {
    int vb = resident_blocks((const void *)k_vr_scatter<NL, false, ADV>, 0, n_cu, blocks, P->wg_per_cu);
    hipLaunchKernelGGL((k_vr_scatter<NL, false, ADV>), dim3(vb), dim3(ENG_BLOCK), 0, st, *P, *S, *V, n);
  }
}

static void launch_cone(const EngineParams *P, const PhotonSoA *S, const VrSoA *V, int n, int n_cu, hipStream_t st) {
  /* one resident round: the trial segments are of equal size, so a second,
   * partial round of workgroups would only add a tail */
  const int cb = resident_blocks((const void *)k_vr_cone, 0, n_cu, n_cu * 4);
  hipLaunchKernelGGL(k_vr_cone, dim3(cb), dim3(ENG_BLOCK), 0, st, *P, *S, *V, n);
}

/* the estimator of order n after the step and the layer scan, each kernel
 * timed with ev.  (The line kernel on a second stream beside the scatter
 * kernel, and the off-grid solid angles beside the layer lists, measured no
 * faster: 9.50 and 9.21 s per step against 9.20 on one stream.) */
template <int NL>
static void launch_estimator_nl(const EngineParams *P, const PhotonSoA *S, const VrSoA *V, int n, int count,
                                int n_cu, int blocks, hipStream_t st, hipEvent_t *ev) {
  const size_t ls = scatter_lds_bytes(P);
  hipLaunchKernelGGL(k_vr_list, dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, count);
  if (ev) (void)hipEventRecord(ev[0], st);
  launch_cone(P, S, V, n, n_cu, st);
  if (ev) (void)hipEventRecord(ev[1], st);
  if (P->adv_compton)
    launch_scatter<NL, true>(P, S, V, n, n_cu, blocks, ls, st);
  else
    launch_scatter<NL, false>(P, S, V, n, n_cu, blocks, ls, st);
  if (ev) (void)hipEventRecord(ev[2], st);
  launch_lines<NL>(P, S, V, n, n_cu, blocks, st);
  if (ev) (void)hipEventRecord(ev[3], st);
}

/* NL, the layer-count bound of the estimator and the step: the smallest of
 * 1 to 5, 8, 16 that holds n_layers */
static void launch_estimator(const EngineParams *P, const PhotonSoA *S, const VrSoA *V, int n, int count, int n_cu,
                             int blocks, hipStream_t st, hipEvent_t *ev) {
  const int nl = P->n_layers;
  if (nl <= 1) launch_estimator_nl<1>(P, S, V, n, count, n_cu, blocks, st, ev);
  else if (nl <= 2) launch_estimator_nl<2>(P, S, V, n, count, n_cu, blocks, st, ev);
  else if (nl <= 3) launch_estimator_nl<3>(P, S, V, n, count, n_cu, blocks, st, ev);
  else if (nl <= 4) launch_estimator_nl<4>(P, S, V, n, count, n_cu, blocks, st, ev);
  else if (nl <= 5) launch_estimator_nl<5>(P, S, V, n, count, n_cu, blocks, st, ev);
  else if (nl <= 8) launch_estimator_nl<8>(P, S, V, n, count, n_cu, blocks, st, ev);
  else launch_estimator_nl<16>(P, S, V, n, count, n_cu, blocks, st, ev);
}

extern "C" {

hipError_t eng_launch_grid(const EngineParams *P, double *grid, const double *rv, const double *tv, int n_r, int n_t,
                           long hits, uint64_t seed, hipStream_t st) {
  long total = (long)n_r * n_t;
  int blocks = (int)((total + ENG_BLOCK - 1) / ENG_BLOCK);
  hipLaunchKernelGGL(k_solid_angle_grid, dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, grid, rv, tv, n_r, n_t, hits, seed);
  return hipGetLastError();
}

hipError_t eng_launch_source(const EngineParams *P, const PhotonSoA *S, const SourceTable *T, uint64_t start,
                             int count, hipStream_t st) {
  int blocks = (count + ENG_BLOCK - 1) / ENG_BLOCK;
  hipLaunchKernelGGL(k_source, dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *T, start, count,
                     (const BatchQueue *)nullptr);
  return hipGetLastError();
}

hipError_t eng_launch_batch_init(BatchQueue *Q, unsigned long long total, hipStream_t st) {
  hipLaunchKernelGGL(k_batch_init, dim3(1), dim3(1), 0, st, Q, total);
  return hipGetLastError();
}

hipError_t eng_launch_source_queued(const EngineParams *P, const PhotonSoA *S, const SourceTable *T, BatchQueue *Q,
                                    int cap, hipStream_t st) {
  hipLaunchKernelGGL(k_batch_next, dim3(1), dim3(1), 0, st, Q, cap);
  const int blocks = (cap + ENG_BLOCK - 1) / ENG_BLOCK;
  hipLaunchKernelGGL(k_source, dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *T, (uint64_t)0, cap,
                     (const BatchQueue *)Q);
  return hipGetLastError();
}

/* one escape-ratio batch: the forced step, then the interaction with the
 * escape test and its tallies */
hipError_t eng_launch_escape(const EngineParams *P, const PhotonSoA *S, const VrSoA *V, const EscParams *Q,
                             int count, hipStream_t st) {
  int blocks = (count + ENG_BLOCK - 1) / ENG_BLOCK;
  hipLaunchKernelGGL(k_reset_queues, dim3(1), dim3(ENG_NQUEUES * ENG_SPREAD), 0, st, *P);
  {
    const int nl = P->n_layers;
    if (nl <= 1) hipLaunchKernelGGL((k_step<1, false>), dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *V, 1, count);
    else if (nl <= 2) hipLaunchKernelGGL((k_step<2, false>), dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *V, 1, count);
    else if (nl <= 4) hipLaunchKernelGGL((k_step<4, false>), dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *V, 1, count);
    else if (nl <= 8) hipLaunchKernelGGL((k_step<8, false>), dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *V, 1, count);
    else hipLaunchKernelGGL((k_step<16, false>), dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *V, 1, count);
  }
  hipLaunchKernelGGL(k_interact_escape, dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *Q);
  return hipGetLastError();
}

hipError_t eng_launch_order_brute(const EngineParams *P, const PhotonSoA *S, int n, int count, int blocks,
                                  hipStream_t st, hipEvent_t *ev) {
  hipLaunchKernelGGL(k_reset_queues, dim3(1), dim3(ENG_NQUEUES * ENG_SPREAD), 0, st, *P);
  if (ev) (void)hipEventRecord(ev[0], st);
  if (P->coll_present) hipLaunchKernelGGL(k_step_brute<true>, dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, n, count);
  else hipLaunchKernelGGL(k_step_brute<false>, dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, n, count);
  if (ev) (void)hipEventRecord(ev[1], st);
  /* the interactions: one thread per photon that may be alive */
  const int alive = (n == 1 || !P->off_half) ? count : 2 * count;
  if (n <= P->n_int) launch_interact_brute(P, S, n, (alive + ENG_BLOCK - 1) / ENG_BLOCK, st);
  if (ev) (void)hipEventRecord(ev[2], st);
  return hipGetLastError();
}

int eng_brute_blocks(int n_cu, int coll) {
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, coll ? (const void *)k_step_brute<true> : (const void *)k_step_brute<false>,
                                                   ENG_BLOCK, 0) != hipSuccess ||
      per_cu < 1)
    per_cu = 1;
  return n_cu * per_cu;
}

hipError_t eng_launch_order(const EngineParams *P, const PhotonSoA *S, const VrSoA *V, int n, int count, int n_cu,
                            hipStream_t st, hipEvent_t *ev /* ENG_ORDER_EVENTS events or NULL */) {
  int blocks = (count + ENG_BLOCK - 1) / ENG_BLOCK;
  if (ev) (void)hipEventRecord(ev[0], st);
  hipLaunchKernelGGL(k_reset_queues, dim3(1), dim3(ENG_NQUEUES * ENG_SPREAD), 0, st, *P);
  {
    const int nl = P->n_layers;
    if (nl <= 1) hipLaunchKernelGGL((k_step<1, true>), dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *V, n, count);
    else if (nl <= 2) hipLaunchKernelGGL((k_step<2, true>), dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *V, n, count);
    else if (nl <= 3) hipLaunchKernelGGL((k_step<3, true>), dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *V, n, count);
    else if (nl <= 4) hipLaunchKernelGGL((k_step<4, true>), dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *V, n, count);
    else if (nl <= 5) hipLaunchKernelGGL((k_step<5, true>), dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *V, n, count);
    else if (nl <= 8) hipLaunchKernelGGL((k_step<8, true>), dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *V, n, count);
    else hipLaunchKernelGGL((k_step<16, true>), dim3(blocks), dim3(ENG_BLOCK), 0, st, *P, *S, *V, n, count);
  }
  {
    const int nw = blocks * (ENG_BLOCK / 64), nseg = (nw + ENG_SCAN_SEG - 1) / ENG_SCAN_SEG;
    hipLaunchKernelGGL(k_layer_scan, dim3(nseg, P->n_layers), dim3(ENG_SCAN_SEG), 0, st, *P, nw);
    hipLaunchKernelGGL(k_layer_base, dim3(P->n_layers), dim3(ENG_SCAN_NSEG), 0, st, *P, nseg);
  }
  if (ev) (void)hipEventRecord(ev[1], st);
  launch_estimator(P, S, V, n, count, n_cu, blocks, st, ev ? ev + 2 : nullptr);
  /* the interactions of the last order change only photon states that no
   * later step reads (the estimator has scored this order): not launched */
  if (n < P->n_int) launch_interact(P, S, n, (count + ENG_BLOCK - 1) / ENG_BLOCK, st);
  if (ev) (void)hipEventRecord(ev[6], st);
  return hipGetLastError();
}

} /* extern "C" */
