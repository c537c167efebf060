// eif_suspensions.hip -- ellipses coupled to the fluid on gfx950:
// Eulerian IBM weights, inertia integrals, momentum exchange and its
// box-local deposit, soft-sphere collisions, Crank-Nicolson increments.
//
// Per-element arithmetic follows NaokiHori/EllipsesInFlows:
//   ellipse geometry      src/ellipse.c:7-65
//   IBM weights / boxes   src/suspensions/auxiliary.c:11-75
//   inertia               src/suspensions/inertia.c:9-70
//   momentum exchange     src/suspensions/exchange.c:13-88
//   field update          src/suspensions/update.c:36-59
//   collisions            src/suspensions/collision.c:75-367
//   increments / update   src/suspensions/increment.c:10-72, update.c:8-34
//
// Work decomposition (gfx950):
//   * one wave per slice of 64 to 256 cells of a particle's boxes for the IBM
//     integrals (its three periodic images' boxes flattened), the slices' sums
//     added per particle in a fixed tree;
//   * the signed distance of every box cell is cached per particle with the
//     position it belongs to; the reference evaluates it three times at
//     identical positions in every RK stage (inertia(0), exchange and the
//     first inertia(1), src/main.c:21-38), the cache serves the repeats with
//     the same bits;
//   * the exchange writes each box cell's forcing to box-local scratch and
//     registers the box with the 64x4 tiles it touches; a gather over the
//     tiles then adds the contributions cell by cell in the reference's
//     particle/image order and applies them to ux/uy (no atomics, no
//     full-field pass);
//   * collisions: one wave per particle finds the partners whose bounding
//     circles reach it (all others, or the neighbours of a cell list), solves
//     the contacts with two lanes each and adds their forces in the
//     reference's pair order.
#include "eif_ellipse.hpp"
#include "eif_internal.hpp"
#include <hip/hip_ext.h>
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <type_traits>

namespace eif {

#define TRY_S(x)          \
  do {                    \
    const int _r = (x);   \
    if (_r) return _r;    \
  } while (0)

#define NEXTRA 3
#define BETA 2.

// src/suspensions/auxiliary.c:11-17
// ih = 1/h, used when h is a power of two (pow2): then x * ih == x / h
__device__ inline void loop_size(int lb, int ub, double h, double ih, bool pow2, double r,
                                 double c, int &mn, int &mx) {
  mn = (int)(floor(pow2 ? (c - r) * ih : (c - r) / h) - NEXTRA);
  mx = (int)(ceil(pow2 ? (c + r) * ih : (c + r) / h) + NEXTRA);
  mn = mn < lb ? lb : mn;
  mx = mx > ub ? ub : mx;
}

// src/ellipse.c:30-65
__device__ double find_normal_t(const EllipseShape &e, double x_, double y_, int &iters) {
  const double px = fabs(x_), py = fabs(y_);
  double t = 0.25 * EIF_PI;
  int n;
  for (n = 0;; n++) {
    double s, c;
    sincos(t, &s, &c);
    const double x = e.a * c, y = e.b * s;
    const double ex = e.kex * cube(c), ey = e.key * cube(s);
    const double rx = x - ex, ry = y - ey;
    const double qx = px - ex, qy = py - ey;
    const double r = sqrt(ry * ry + rx * rx);
    const double q = sqrt(qy * qy + qx * qx);
    const double dc = r * asin((rx * qy - ry * qx) / (r * q));
    const double dt = dc / sqrt(e.a2b2 - x * x - y * y);
    t += dt;
    t = fmin(0.5 * EIF_PI, t);
    t = fmax(0., t);
    if (fabs(dt) < 1.e-8) break;
    if (n > 100) break;
  }
  iters += n + 1;
  if (x_ < 0.) t = EIF_PI - t;
  if (y_ < 0.) t = -t;
  return t;
}

// compute_signed_dist, src/suspensions/auxiliary.c:19-47; (cr, sr) are
// cos(-paz), sin(-paz)
__device__ inline double signed_dist(const EllipseShape &e, double grid_size,
                                     double px, double py, double cr, double sr,
                                     double x, double y, int &iters) {
  const double ddx = x - px, ddy = y - py;
  const double x_ = cr * ddx - sr * ddy;
  const double y_ = sr * ddx + cr * ddy;
  const double xa = x_ / e.a, yb = y_ / e.b;
  const double f0 = 1. - xa * xa - yb * yb;
  const double sign = f0 > 0. ? +1. : -1.;
  const double t = find_normal_t(e, x_, y_, iters);
  double st, ct;
  sincos(t, &st, &ct);
  const double ex = e.a * ct - x_, ey = e.b * st - y_;
  const double dist = sign * sqrt(+ex * ex + ey * ey);
  return dist / grid_size;
}

// ---------------------------------------------------------------------
// Foot of the normal for the IBM weights.
//
// src/ellipse.c:30-65 iterates t <- clamp(t + dt) from t = pi/4 until
// |dt| < 1e-8, every iteration in FP64 with sin, cos, asin and three
// square roots.  The iteration converges quadratically to the unique foot
// on the first-quadrant arc, so here it starts in FP32 (foot_fp32: hardware
// sin/cos, stopped at |dt| < 1e-3, where the FP32 rounding noise takes over)
// and finishes with the reference's FP64 iteration and stopping rule
// (foot_fp64), which then needs one or two iterations instead of about four
// (1.51 per evaluated cell at 2048x4096, 1024 ellipses).  After the first
// FP64 step every update of t is below 2^-10, so cos and sin of the new t
// follow from the old ones by the addition theorem with the Taylor series
// of cos(delta) and sin(delta) (truncation below 1e-21), and only one FP64
// sincos is evaluated per cell.  The converged (cos t, sin t) agree with
// the reference's to a few units in the last place.
//
// The weights use only the distance, which is stationary in t for a cell
// centre off the boundary, but the stopping rule cannot be loosened for that:
// on the boundary an error of t enters linearly, with a factor that grows as
// b / a falls.  Ended at |dt| < 2^-17 with the length factors and the
// starting cos t, sin t in FP32, 60 steps took 119.5 ms instead of 126.6
// (2048x4096, 1024 ellipses) and 6 steps 12.8 instead of 13.8 (1024x2048,
// 4096 ellipses), but distances were off by 1e-11 (b/a = 1) to 3e-10 cells
// (b/a = 0.1) at 20 cells, against 5e-15 here.
// ---------------------------------------------------------------------

// compute_signed_dist (src/suspensions/auxiliary.c:19-47) with the foot
// from foot_fp32 / foot_fp64; the unfolding of ellipse.c:62-63 maps
// (cos t, sin t) of the folded foot to (-cos t, sin t) for x_ < 0 and
// (cos t, -sin t) for y_ < 0.  t: the foot's parameter on return; where the
// search starts if warm, the parameter this cell's foot had at the particle's
// previous evaluation in the same RK stage, which the particle has barely
// moved from (else from the FP32 estimate).  The root on the first-quadrant
// arc is unique, so the start changes only the number of iterations.
__device__ inline double signed_dist_from(const EllipseShape &e, const EllipseShape32 &f,
                                          double inv_grid, double px, double py, double cr,
                                          double sr, double x, double y, bool warm, double &t,
                                          int &it32, int &it64) {
  const double ddx = x - px, ddy = y - py;
  const double x_ = cr * ddx - sr * ddy;
  const double y_ = sr * ddx + cr * ddy;
  const double xa = x_ * e.ia, yb = y_ * e.ib;
  const double f0 = 1. - xa * xa - yb * yb;
  const double sign = f0 > 0. ? +1. : -1.;
  const double ax = fabs(x_), ay = fabs(y_);
  if (!warm) t = (double)foot_fp32(f, ax, ay, it32);
  double ct, st;
  foot_fp64(e, ax, ay, t, ct, st, it64);
  const double fx = x_ < 0. ? -(e.a * ct) : e.a * ct;
  const double fy = y_ < 0. ? -(e.b * st) : e.b * st;
  const double ex = fx - x_, ey = fy - y_;
  const double dist = sign * sqrt(+ex * ex + ey * ey);
  return dist * inv_grid;
}

// src/suspensions/auxiliary.c:49-59.  tanh(x) as 1 - 2 / (exp(2|x|) + 1)
// with the sign of x: like the libm routine it rounds to exactly +-1 once
// 2 / (exp(2|x|) + 1) drops below half an ulp of 1, so the weights are
// exactly 0 or 1 on the same cells.
__device__ inline double tanh_w(double x) {
  const double th = 1. - 2. / (exp(2. * fabs(x)) + 1.);
  return copysign(th, x);
}
// Both weights are functions of th = tanh(BETA d); the per-cell cache keeps
// th, so a cached cell needs no exp.
__device__ inline double weight_th(double d) { return tanh_w(BETA * d); }
__device__ inline double v_weight_th(double th) { return 0.5 * (1. + th); }
__device__ inline double s_weight_th(double th) { return 0.5 * BETA * (1. - th * th); }

// mass and moment of inertia, src/suspensions/auxiliary.c:63-75
__device__ inline double p_mass(const double *q) {
  const double vol = EIF_PI * q[R_A] * q[R_B];
  return q[R_DEN] * vol;
}
__device__ inline double p_moi(const double *q) {
  const double m = p_mass(q);
  return 0.25 * m * (q[R_A] * q[R_A] + q[R_B] * q[R_B]);
}

// ---------------------------------------------------------------------
// IBM integrals
// ---------------------------------------------------------------------
constexpr int IBM_THREADS = 256;
// Box cells per wave of the inertia / exchange kernels (a.slice): 256, or 128
// or 64 where longer slices leave fewer than IBM_WAVES waves.  A wave takes
// its cells four, two or one a lane in turn, so a launch too small to fill
// the GPU is as long as that turn: with 64 cells k_inertia_collide took 10.0
// -> 7.0 us and k_ibm_dist 10.2 -> 6.1 at 64 ellipses on 512x1024 (2600
// waves), 8.5 -> 5.1 and 10.7 -> 5.2 at one on 128x128 (with a shorter foot
// search than now, when the launches take 7.4, 6.1, 5.0 and 5.2); at 11600 waves
// (1024 ellipses on 2048x4096) shorter slices only repeat the waves' prologue.
constexpr int IBM_SLICE = 256;
constexpr int IBM_WAVES = 2048;
constexpr int SLICE_VALS = 5;   // per-slice partials: 3 sums, FP64 and FP32 iterations

// Sub-iteration `sub` of a stage's speculatively queued Crank-Nicolson
// loop (src/main.c:37-50) runs unless the previous one converged (residual
// below 1e-8) or the stage has already run 101 of them.  res[s] is the
// residual of sub-iteration s, cleared at the stage start, so a sub-iteration
// that did not run leaves 0 and closes every later one.  res == nullptr:
// not gated.
__device__ inline bool sub_open(const double *res, int sub) {
  return !res || sub == 0 || (!(res[sub - 1] < 1.e-8) && sub <= 101);
}

// The IBM, deposit and collision kernels give each wave its own slice, tile or
// particle, one wave a workgroup: four made the collision launch 28 -> 41 us
// and left the others as they were (2048x4096, 1024 ellipses; the dispatch of
// 11600 one-wave workgroups takes 3.6 us).
constexpr int WAVE = 64;
__device__ inline int wave_lane() { return threadIdx.x & 63; }
// the wave's place in the launch, known uniform
__device__ inline int wave_index(const VB &vb) { return __builtin_amdgcn_readfirstlane(vb.bx); }
// LDS written by the wave's lanes is visible to its other lanes
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

struct SliceHead;

struct IbmArgs {
  Layout L;
  int nx, ny;
  double ly, dx, dy, grid_size;
  double idx, idy;  // 1/dx, 1/dy
  int pow2;         // dx, dy powers of two: divisions by them are products with idx, idy
  const double *xc, *yc;
  const double *ux, *uy;
  double *prt;
  const double *dscal;
  Box *boxes;
  const long *box_off;
  double *sc_fx, *sc_fy;
  double *sc_dist;  // per box cell: tanh(BETA d) of the signed distance d
  double *sc_pos;
  double *sc_t;   // per box cell: foot parameter of the last evaluation
  int *sc_key;    // per particle: boxes of that evaluation (8 ints)
  int *tile_cnt, *tile_list;
  int ntx, nty;
  int *flags;
  unsigned long long *stats;  // per particle: cells, cells evaluated, FP64 and FP32 iterations
  double *cpos;               // np x 4: the broad phase's packed positions and radii
  int np;
  int slice;               // box cells of each slice
  const int *slice_first;  // np+1: first slice of each particle
  const int4 *slice_rec;   // of each slice: its particle, the particle's first slice and slices
  long *slice_info;        // np x 2: box cells, cells evaluated (this call)
  const double *res;       // sub-iteration residuals (null: not gated)
  int sub;                 // sub-iteration index
  // k_exchange only: with us_x, also inertia(0) of the stage-start
  // velocity (us_x, us_y), its slice sums into slice_part0
  const double *us_x, *us_y;
  double *slice_part0;
  double *slice_part;
  const int *halt;   // graph-step stop flag
  SliceHead *heads;  // per particle: the pass's position, shape, boxes, cache state
};

// x of lane i + n of the same row of 16 lanes (DPP row_shl:n, CTRL = 0x100 + n);
// lanes whose source leaves the row get 0
template <int CTRL>
__device__ inline double row_shl_f64(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// fixed-order tree over the 64 lanes of a wave (lane 0 receives the sum):
// v[i] += v[i + off] for off = 32, 16, 8, 4, 2, 1; the last four levels stay
// inside lanes 0-15 and move through DPP instead of LDS permutes
__device__ inline double wave_sum(double v) {
  v += __shfl_down(v, 32, 64);
  v += __shfl_down(v, 16, 64);
  v += row_shl_f64<0x108>(v);
  v += row_shl_f64<0x104>(v);
  v += row_shl_f64<0x102>(v);
  v += row_shl_f64<0x101>(v);
  return v;
}

// the same tree over integers
__device__ inline int wave_sum(int v) {
  v += __shfl_down(v, 32, 64);
  v += __shfl_down(v, 16, 64);
  v += __builtin_amdgcn_update_dpp(0, v, 0x108, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x104, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x102, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x101, 0xf, 0xf, false);
  return v;
}

// the lanes' FP64 and FP32 iteration counts added as one integer: a slice's
// 256 cells take at most 102 and 8 each, sums below 2^16
__device__ inline void sum_counts(int it64, int it32, double &c64, double &c32) {
  const int c = wave_sum(it64 + (it32 << 16));
  c64 = (double)(c & 0xffff);
  c32 = (double)(c >> 16);
}

// lane l's x, l the same on every lane of the wave
__device__ inline double lane_value(double x, int l) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_readlane((int)b, l);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// A slice's partial sums (lane 0); slice_sums adds them per particle after
// the kernel has finished, so no fence or atomic is needed.
__device__ inline void slice_store(const IbmArgs &a, int slice, const double v[SLICE_VALS]) {
  if (wave_lane() == 0)
    for (int k = 0; k < SLICE_VALS; k++) a.slice_part[SLICE_VALS * (long)slice + k] = v[k];
}

// box of one periodic image (auxiliary.c:11-17); three separate members
// rather than an array, so that selecting an image stays in registers
struct Img {
  int imin, imax, jmin, jmax;
  int cnt;
  float inv_w;  // 1 / box width, for the quotient in cell_of
};
struct BoxSet {
  Img b0, b1, b2;
  int total;
};

__device__ inline Img make_img(const IbmArgs &a, double px, double py_, double r) {
  Img m;
  loop_size(1, a.nx, a.dx, a.idx, a.pow2, r, px, m.imin, m.imax);
  loop_size(1, a.ny, a.dy, a.idy, a.pow2, r, py_ - 0., m.jmin, m.jmax);
  const int w = m.imax - m.imin + 1, h = m.jmax - m.jmin + 1;
  m.cnt = (w > 0 && h > 0) ? w * h : 0;
  m.inv_w = w > 0 ? 1.f / (float)w : 0.f;
  return m;
}

__device__ inline void make_boxes(const IbmArgs &a, double px, double py,
                                  double r, BoxSet &bs) {
  bs.b0 = make_img(a, px, py + a.ly * (0 - 1), r);
  bs.b1 = make_img(a, px, py + a.ly * (1 - 1), r);
  bs.b2 = make_img(a, px, py + a.ly * (2 - 1), r);
  bs.total = bs.b0.cnt + bs.b1.cnt + bs.b2.cnt;
}

__device__ inline Img pick(const BoxSet &bs, int k) {
  Img m = bs.b0;
  if (k == 1) m = bs.b1;
  if (k == 2) m = bs.b2;
  return m;
}

// image k and cell (i, j) of flattened box cell t.  single: the particle has
// cells in the middle image only, which is the same for the whole wave;
// otherwise the image's fields are blended arithmetically (a select between
// struct members can be turned into a load from a stack copy).  The quotient
// by the box width comes from a float reciprocal, corrected once (exact for
// t < 2^24).
__device__ inline bool single_image(const BoxSet &bs) { return bs.b1.cnt == bs.total; }
__device__ inline void cell_of(const BoxSet &bs, int t, int &k, int &i, int &j,
                               bool single = false) {
  int tk = t, imin = bs.b1.imin, imax = bs.b1.imax, jmin = bs.b1.jmin;
  k = 1;
  if (!single) {
    const int c0 = bs.b0.cnt, c01 = c0 + bs.b1.cnt;
    const int g1 = t >= c0, g2 = t >= c01;
    k = g1 + g2;
    tk = t - g1 * c0 - g2 * bs.b1.cnt;
    imin = bs.b0.imin + g1 * (bs.b1.imin - bs.b0.imin) + g2 * (bs.b2.imin - bs.b1.imin);
    imax = bs.b0.imax + g1 * (bs.b1.imax - bs.b0.imax) + g2 * (bs.b2.imax - bs.b1.imax);
    jmin = bs.b0.jmin + g1 * (bs.b1.jmin - bs.b0.jmin) + g2 * (bs.b2.jmin - bs.b1.jmin);
  }
  const int w = imax - imin + 1;
  int q = (int)((float)tk * __builtin_amdgcn_rcpf((float)w));
  int r = tk - q * w;
  if (r < 0) {
    q--;
    r += w;
  } else if (r >= w) {
    q++;
    r -= w;
  }
  j = jmin + q;
  i = imin + r;
}
// the U cells of a lane of a slice, t0 + lane + 64 u (the last cell, t1 - 1,
// in the place of those past it)
template <int U>
__device__ inline void lane_cells(const BoxSet &bs, int t0, int t1, int lane, int (&k)[U],
                                  int (&i)[U], int (&j)[U]) {
  if (single_image(bs)) {
#pragma unroll
    for (int u = 0; u < U; u++)
      cell_of(bs, min(t0 + lane + 64 * u, t1 - 1), k[u], i[u], j[u], true);
  } else {
#pragma unroll
    for (int u = 0; u < U; u++)
      cell_of(bs, min(t0 + lane + 64 * u, t1 - 1), k[u], i[u], j[u]);
  }
}

// the x and y faces west of and south of cell (i, j) in the velocity arrays
// (fewer than 2^31 values: the context bounds the grid)
__device__ inline unsigned face_x(const Layout &L, int i, int j) {
  return (unsigned)j * (unsigned)(L.nx + 1) + (unsigned)(i - 1);
}
__device__ inline unsigned face_y(const Layout &L, int i, int j) {
  return (unsigned)j * (unsigned)(L.nx + 2) + (unsigned)i;
}

// What every slice wave of one IBM pass needs of its particle: computed
// once per particle and pass, by the kernel that last moved the particle
// or updated its cache (k_reset, the finalise passes, k_increment, or
// k_heads), instead of by each of the particle's waves.  The arithmetic is
// that the waves would do themselves.
struct SliceHead {
  EllipseShape e;
  double px, py, paz;  // position of the pass
  double cr, sr;       // cos, sin of -paz
  double inv_pm, inv_pim;
  long off, cap;       // the particle's per-cell scratch range
  BoxSet bs;
  EllipseShape32 f;
  int cached;          // the distance cache holds this position
  int warm;            // the foot parameters hold these boxes
};

// lane l's integer, l the same on every lane of the wave
__device__ inline int lane_int(int x, int l) { return __builtin_amdgcn_readlane(x, l); }

// The pass whose distances and foot parameters a particle's cache holds, as
// the lanes of its wave see it: the position on every lane, the box corner
// of image min(lane, 2)
struct CachedPass {
  double px, py, paz;
  int imin, jmin, total;
  bool pos, boxes;  // recorded
};
// ... from the records (sc_pos, sc_key)
__device__ inline CachedPass cached_records(const IbmArgs &a, int n, int lane) {
  const double *cp = a.sc_pos + 4 * (long)n;
  const int *key = a.sc_key + 8 * (long)n;
  const int k = min(lane, 2);
  return {cp[0], cp[1], cp[2], key[2 * k], key[2 * k + 1], key[6], cp[3] != 0., key[7] != 0};
}

// The position-dependent parts of a particle's header, by the lanes of one
// wave: lanes 0, 1, 2 make the boxes of the three images.  rad: the
// particle's larger semi-axis
__device__ inline void write_head(const IbmArgs &a, SliceHead *h, int lane, double px, double py,
                                  double paz, double rad, const CachedPass &prev) {
  const Img m = make_img(a, px, py + a.ly * (min(lane, 2) - 1), rad);
  const int total = lane_int(m.cnt, 0) + lane_int(m.cnt, 1) + lane_int(m.cnt, 2);
  const bool same = __ballot(m.imin != prev.imin || m.jmin != prev.jmin) == 0ull &&
                    total == prev.total;
  double sr, cr;
  sincos(-paz, &sr, &cr);
  if (lane < 3) (&h->bs.b0)[lane] = m;
  if (lane == 0) {
    h->px = px;
    h->py = py;
    h->paz = paz;
    h->cr = cr;
    h->sr = sr;
    h->bs.total = total;
    h->cached = prev.pos && prev.px == px && prev.py == py && prev.paz == paz;
    h->warm = prev.boxes && same;
  }
}

// the parts that depend only on the particle's shape and mass (written at
// every stage start, so records changed between calls are picked up)
__device__ inline void write_head_shape(const IbmArgs &a, SliceHead *h, int n, int lane,
                                        const double *q) {
  if (lane != 0) return;
  const EllipseShape e = make_shape(q[R_A], q[R_B]);
  h->e = e;
  h->f = shape32(e);
  h->inv_pm = 1. / p_mass(q);
  h->inv_pim = 1. / p_moi(q);
  h->off = a.box_off[n];
  h->cap = a.box_off[n + 1] - h->off;
}

// heads at the particles' positions, with the increments when with_dx; one
// wave per particle, four per workgroup
struct HeadsB {
  static constexpr int T = 256, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, IbmArgs a, int with_dx) {
    if (halted(a.halt)) return;
    const int n = vb.bx * 4 + (int)(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (n >= a.np) return;
    const double *q = a.prt + (long)n * R_N;
    const double w = with_dx ? 1. : 0.;  // x + 0 is x
    SliceHead *h = a.heads + n;
    const CachedPass prev = cached_records(a, n, lane);
    write_head_shape(a, h, n, lane, q);
    write_head(a, h, lane, q[R_X] + w * q[R_DX], q[R_Y] + w * q[R_DY], q[R_AZ] + w * q[R_DAZ],
               fmax(q[R_A], q[R_B]), prev);
  }
};
__global__ __launch_bounds__(256) void k_heads(IbmArgs a, int with_dx) {
  HeadsB::run(VB::here(), a, with_dx);
}

// src/suspensions/inertia.c:9-70.  One wave per slice of 64 U box cells of
// one particle (its three images' boxes flattened); the increment adds the
// slices' sums.
// open: the sub-iteration gate, evaluated by the caller; tested after this
// slice's own loads are issued, so the gate's load is not waited for alone
template <int U>
__device__ __forceinline__ void inertia_slice(const IbmArgs &a, int cnstep, int slice,
                                              bool open = true) {
  const int lane = wave_lane();
  const int4 rec = a.slice_rec[slice];
  const int n = rec.x, s0 = rec.y, nsl = rec.z;
  const SliceHead &hd = a.heads[n];
  const BoxSet bs = hd.bs;
  const int total = bs.total;
  if (!open) return;
  if (total > hd.cap || total > nsl * (64 * U)) {
    if (lane == 0) atomicOr(&a.flags[0], 1);
    return;
  }
  const EllipseShape e = hd.e;
  const EllipseShape32 f = hd.f;
  const double px = hd.px, py = hd.py;
  const double inv_pm = hd.inv_pm, inv_pim = hd.inv_pim;
  const bool cached = hd.cached, warm = hd.warm;
  double *dist = a.sc_dist + hd.off;
  double *tcell = a.sc_t + hd.off;
  const double cr = hd.cr, sr = hd.sr;
  const double dxdy = a.dx * a.dy;
  double acc[3] = {0., 0., 0.};  // iux, iuy, ivz
  int it64 = 0, it32 = 0;
  const int t0 = (slice - s0) * (64 * U);
  const int t1 = t0 + 64 * U < total ? t0 + 64 * U : total;
  auto add = [&](int k, double x, double y, double th, double vx0, double vx1, double vy0,
                 double vy1) {
    const double py_ = py + a.ly * (k - 1);
    const double w = v_weight_th(th);
    const double valx = w * 0.5 * (vx0 + vx1) * dxdy;
    const double valy = w * 0.5 * (vy0 + vy1) * dxdy;
    acc[0] += valx * inv_pm;
    acc[2] += -(y - py_) * valx * inv_pim;
    acc[1] += valy * inv_pm;
    acc[2] += +(x - px) * valy * inv_pim;
  };
  if (cached) {
    // all loads of the lane's cells first (a cell past t1 loads the last cell
    // instead and is not added), then the sums in cell order
    if (t0 < t1) {
      double th_[U], x_[U], y_[U], vx0[U], vx1[U], vy0[U], vy1[U];
      int k_[U], i_[U], j_[U];
      lane_cells<U>(bs, t0, t1, lane, k_, i_, j_);
#pragma unroll
      for (int u = 0; u < U; u++) {
        const unsigned fx = face_x(a.L, i_[u], j_[u]), fy = face_y(a.L, i_[u], j_[u]);
        x_[u] = a.xc[i_[u]];
        y_[u] = a.yc[j_[u] - 1];
        th_[u] = dist[min(t0 + lane + 64 * u, t1 - 1)];
        vx0[u] = a.ux[fx];
        vx1[u] = a.ux[fx + 1];
        vy0[u] = a.uy[fy];
        vy1[u] = a.uy[fy + (unsigned)(a.nx + 2)];
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (t0 + lane + 64 * u < t1)
          add(k_[u], x_[u], y_[u], th_[u], vx0[u], vx1[u], vy0[u], vy1[u]);
    }
  } else {
    // G cells at a time, their loads first (they do not depend on the
    // distance).  Of U = 4 one: four cells' loads held through four searches
    // take more than the 128 VGPRs there are, and 60 steps at 2048x4096 with
    // 1024 ellipses 127.4 ms instead of 124.3.  Of U = 2 both: eight cases
    // advanced together take 34.3 ms, 35.0 one at a time
    constexpr int G = U > 2 ? 1 : U;
#pragma nounroll
    for (int c0 = 0; c0 < U; c0 += G) {
      const int b0 = t0 + 64 * c0;
      if (b0 >= t1) break;
      double tf[G] = {}, x_[G], y_[G], vx0[G], vx1[G], vy0[G], vy1[G];
      int k_[G], i_[G], j_[G];
      lane_cells<G>(bs, b0, t1, lane, k_, i_, j_);
#pragma unroll
      for (int u = 0; u < G; u++) {
        const unsigned fx = face_x(a.L, i_[u], j_[u]), fy = face_y(a.L, i_[u], j_[u]);
        x_[u] = a.xc[i_[u]];
        y_[u] = a.yc[j_[u] - 1];
        vx0[u] = a.ux[fx];
        vx1[u] = a.ux[fx + 1];
        vy0[u] = a.uy[fy];
        vy1[u] = a.uy[fy + (unsigned)(a.nx + 2)];
      }
      if (warm) {
#pragma unroll
        for (int u = 0; u < G; u++) tf[u] = tcell[min(b0 + lane + 64 * u, t1 - 1)];
      }
#pragma unroll
      for (int u = 0; u < G; u++) {
        const int t = b0 + lane + 64 * u;
        if (t >= t1) continue;
        const double th = weight_th(signed_dist_from(e, f, 1. / a.grid_size, px,
                                                     py + a.ly * (k_[u] - 1), cr, sr, x_[u], y_[u],
                                                     warm, tf[u], it32, it64));
        tcell[t] = tf[u];
        dist[t] = th;
        add(k_[u], x_[u], y_[u], th, vx0[u], vx1[u], vy0[u], vy1[u]);
      }
    }
  }
  double part[SLICE_VALS] = {wave_sum(acc[0]), wave_sum(acc[1]), wave_sum(acc[2])};
  sum_counts(it64, it32, part[3], part[4]);
  slice_store(a, slice, part);
  if (slice == s0 && lane == 0) {
    a.slice_info[2 * (long)n] = total;
    a.slice_info[2 * (long)n + 1] = cached ? 0 : total;
  }
}

// U: cells a lane, slices of 64 U
template <int U>
struct InertiaB {
  static constexpr int T = WAVE, M = 4;
  static __device__ __forceinline__ void run(const VB &vb, IbmArgs a, int cnstep) {
  if (halted(a.halt)) return;
  inertia_slice<U>(a, cnstep, wave_index(vb), sub_open(a.res, a.sub));
}
};
template <int U>
__global__ __launch_bounds__(WAVE, 4) void k_inertia(IbmArgs a, int cnstep) {
  InertiaB<U>::run(VB::here(), a, cnstep);
}

// Per-particle totals of the sliced inertia / exchange kernels, by the 64
// lanes of one wave: lane l adds slices l, l + 64, ... and the lanes' sums are
// added in a fixed tree (every lane gets them).  In slice order through
// readlane, three instructions a slice and value one behind the other, 41
// slices took 3.5 us of the increment.
__device__ inline void slice_sums(const IbmArgs &a, int s0, int s1, double tot[SLICE_VALS]) {
  double v[SLICE_VALS] = {0., 0., 0., 0., 0.};
  for (int s = s0 + wave_lane(); s < s1; s += 64)
    for (int k = 0; k < SLICE_VALS; k++) v[k] += a.slice_part[SLICE_VALS * (long)s + k];
  for (int k = 0; k < SLICE_VALS; k++) tot[k] = lane_value(wave_sum(v[k]), 0);
}

// The cache records of the pass with header h and the work counters, by the
// lanes of one wave: their old values and the pass's boxes are loaded by
// load(), early, and stored by store()
struct PassRecord {
  double px, py, paz;
  Img img;  // of image min(lane, 2)
  int total;
  unsigned long long stat, info;  // lanes 0..3
  __device__ void load(const IbmArgs &a, int n, int lane) {
    const SliceHead *h = a.heads + n;
    px = h->px;
    py = h->py;
    paz = h->paz;
    img = (&h->bs.b0)[min(lane, 2)];
    total = h->bs.total;
    stat = a.stats[4 * (long)n + min(lane, 3)];
    info = (unsigned long long)a.slice_info[2 * (long)n + min(lane, 1)];
  }
  __device__ void store(const IbmArgs &a, int n, int lane, const double tot[SLICE_VALS]) const {
    if (lane < 4) {
      a.sc_pos[4 * (long)n + lane] = lane == 0 ? px : lane == 1 ? py : lane == 2 ? paz : 1.;
      a.stats[4 * (long)n + lane] =
          stat + (lane < 2 ? info : (unsigned long long)(lane == 2 ? tot[3] : tot[4]));
      int *key = a.sc_key + 8 * (long)n + 2 * lane;
      key[0] = lane < 3 ? img.imin : total;
      key[1] = lane < 3 ? img.jmin : 1;
      if (n == 0 && lane == 0) a.stats[4 * (long)a.np] += 1ull;  // IBM calls
    }
  }
  __device__ CachedPass pass() const { return {px, py, paz, img.imin, img.jmin, total, true, true}; }
};

__device__ void finalize_particle(const IbmArgs &a, int n, int which) {
  const int lane = threadIdx.x & 63;
  PassRecord pr;
  pr.load(a, n, lane);
  double tot[SLICE_VALS];
  slice_sums(a, a.slice_first[n], a.slice_first[n + 1], tot);
  pr.store(a, n, lane, tot);
  if (lane != 0) return;
  double *q = a.prt + (long)n * R_N;
  if (which < 2) {
    q[R_IUX + which] = tot[0];
    q[R_IUY + which] = tot[1];
    q[R_IVZ + which] = tot[2];
  } else {
    q[R_FUX] = tot[0];
    q[R_FUY] = tot[1];
    q[R_TVZ] = tot[2];
  }
}

// The exchange's sums of particle n and those of the inertia(0) computed
// beside it, by one wave; the exchange's call records the distance cache
// and the counters.  The first sub-iteration's pass is at the same
// positions (the increments are zero), whose distances are now cached.
__device__ inline void finalize_x0_particle(const IbmArgs &a, int n) {
  const int lane = threadIdx.x & 63;
  finalize_particle(a, n, 2);
  IbmArgs a0 = a;
  a0.slice_part = a.slice_part0;
  double tot[SLICE_VALS];
  slice_sums(a0, a.slice_first[n], a.slice_first[n + 1], tot);
  if (lane != 0) return;
  double *q = a.prt + (long)n * R_N;
  q[R_IUX] = tot[0];
  q[R_IUY] = tot[1];
  q[R_IVZ] = tot[2];
  SliceHead *h = a.heads + n;
  h->cached = 1;
  h->warm = 1;
}

// one wave per particle, four per workgroup
struct IbmFinalizeB {
  static constexpr int T = 256, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, IbmArgs a, int which) {
  if (halted(a.halt)) return;
  if (!sub_open(a.res, a.sub)) return;
  const int n = vb.bx * 4 + (int)(threadIdx.x >> 6);
  if (n < a.np) finalize_particle(a, n, which);
}
};
__global__ __launch_bounds__(256) void k_ibm_finalize(IbmArgs a, int which) {
  IbmFinalizeB::run(VB::here(), a, which);
}

// Measurement only: the reference's FP64 iteration (find_normal_t,
// src/ellipse.c:30-65) at every cell of the particles' current inertia
// boxes, counting cells and iterations into out[0], out[1].
__global__ __launch_bounds__(IBM_THREADS) void k_ref_iterations(IbmArgs a,
                                                                unsigned long long *out) {
  __shared__ BoxSet bs;
  __shared__ unsigned long long sum;
  const int n = blockIdx.x;
  const double *q = a.prt + (long)n * R_N;
  const double pa = q[R_A], pb = q[R_B];
  const double px = q[R_X] + q[R_DX];
  const double py = q[R_Y] + q[R_DY];
  const double paz = q[R_AZ] + q[R_DAZ];
  const EllipseShape e = make_shape(pa, pb);
  if (threadIdx.x == 0) {
    make_boxes(a, px, py, fmax(pa, pb), bs);
    sum = 0;
  }
  __syncthreads();
  double cr, sr;
  sincos(-paz, &sr, &cr);
  int iters = 0;
  for (long t = threadIdx.x; t < bs.total; t += IBM_THREADS) {
    int k, i, j;
    cell_of(bs, t, k, i, j);
    const double py_ = py + a.ly * (k - 1);
    (void)signed_dist(e, a.grid_size, px, py_, cr, sr, a.xc[i], a.yc[j - 1], iters);
  }
  if (iters) atomicAdd(&sum, (unsigned long long)iters);
  __syncthreads();
  if (threadIdx.x == 0) {
    atomicAdd(&out[0], (unsigned long long)bs.total);
    atomicAdd(&out[1], sum);
  }
}

// Tiles reached by a box's forcing in the field update (update.c:42-57:
// UX(i) reads DUX(i-1), UY(j) reads DUY(j-1), and DUY(i,0) is the periodic
// copy of DUY(i,jtot)).  Up to two rectangles of tiles per box.
struct TileRange {
  int tx0, tx1, ty0, ty1;
  __device__ int count() const { return tx1 < tx0 || ty1 < ty0 ? 0 : (tx1 - tx0 + 1) * (ty1 - ty0 + 1); }
};

__device__ inline void box_tile_ranges(const IbmArgs &a, int imin, int imax, int jmin,
                                       int jmax, TileRange &r0, TileRange &r1) {
  const int i_hi = imax + 1 > a.nx ? a.nx : imax + 1;
  const int j_hi = jmax + 1 > a.ny ? a.ny : jmax + 1;
  r0 = {(imin - 1) / TILE_X, (i_hi - 1) / TILE_X, (jmin - 1) / TILE_Y, (j_hi - 1) / TILE_Y};
  if (jmax == a.ny && jmin > 1)
    r1 = {(imin - 1) / TILE_X, (imax - 1) / TILE_X, 0, 0};
  else
    r1 = {0, -1, 0, -1};
}

__device__ inline void register_tile(const IbmArgs &a, int tile, int box_id) {
  const int slot = atomicAdd(&a.tile_cnt[tile], 1);
  if (slot < TILE_CAP)
    a.tile_list[(long)tile * TILE_CAP + slot] = box_id;
  else
    atomicOr(&a.flags[0], 2);
}

// Signed distances of the box cells at the particles' positions (with the
// increments dx, dy, daz when with_dx) where the per-particle cache does not
// already hold them; sliced like k_inertia.  Used before k_exchange when
// the cache may be stale.
struct IbmDistB {
  static constexpr int T = WAVE, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, IbmArgs a) {
  if (halted(a.halt)) return;
  if (!sub_open(a.res, a.sub)) return;
  const int slice = wave_index(vb), lane = wave_lane();
  const int4 rec = a.slice_rec[slice];
  const int n = rec.x, s0 = rec.y, nsl = rec.z;
  const SliceHead &hd = a.heads[n];
  const BoxSet bs = hd.bs;
  const int total = bs.total;
  if (total > hd.cap || total > nsl * a.slice) {
    if (lane == 0) atomicOr(&a.flags[0], 1);
    return;
  }
  const bool cached = hd.cached;
  const double px = hd.px, py = hd.py;
  int it64 = 0, it32 = 0;
  if (!cached) {
    const EllipseShape e = hd.e;
    const EllipseShape32 f = hd.f;
    const bool warm = hd.warm, single = single_image(bs);
    double *dist = a.sc_dist + hd.off;
    double *tcell = a.sc_t + hd.off;
    const double cr = hd.cr, sr = hd.sr;
    const int t0 = (slice - s0) * a.slice;
    const int t1 = t0 + a.slice < total ? t0 + a.slice : total;
    for (int t = t0 + lane; t < t1; t += 64) {
      int k, i, j;
      cell_of(bs, t, k, i, j, single);
      const double py_ = py + a.ly * (k - 1);
      double tp = warm ? tcell[t] : 0.;
      dist[t] = weight_th(signed_dist_from(e, f, 1. / a.grid_size, px, py_, cr, sr, a.xc[i],
                                           a.yc[j - 1], warm, tp, it32, it64));
      tcell[t] = tp;
    }
  }
  double c64, c32;
  sum_counts(it64, it32, c64, c32);
  if (lane == 0) {
    a.slice_part[SLICE_VALS * (long)slice + 3] = c64;
    a.slice_part[SLICE_VALS * (long)slice + 4] = c32;
    if (slice == s0) a.slice_info[2 * (long)n + 1] = cached ? 0 : total;
  }
}
};
__global__ __launch_bounds__(WAVE) void k_ibm_dist(IbmArgs a) {
  IbmDistB::run(VB::here(), a);
}

// src/suspensions/exchange.c:13-88, sliced like k_inertia, on distances
// already in the per-particle cache (the position is the one of the
// preceding inertia(0) or k_ibm_dist).  The first slice of a particle also
// publishes its boxes and registers them with the tiles they reach.
// own_counts: no k_ibm_dist ran before, so this kernel reports no
// distance work.
// The heads hold the particles' positions without increments.
template <int U>
struct ExchangeB {
  static constexpr int T = WAVE, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, IbmArgs a, int own_counts) {
  if (halted(a.halt)) return;
  const int slice = wave_index(vb), lane = wave_lane();
  const int4 rec = a.slice_rec[slice];
  const int n = rec.x, s0 = rec.y, nsl = rec.z;
  const double *q = a.prt + (long)n * R_N;
  const SliceHead &hd = a.heads[n];
  const double dt = a.dscal[S_DT];
  const double inv_dt = 1. / dt;
  const double inv_pm = hd.inv_pm, inv_pim = hd.inv_pim;
  const double px = hd.px, py = hd.py;
  const double pux = q[R_UX], puy = q[R_UY], pvz = q[R_VZ];
  const BoxSet bs = hd.bs;
  const int total = bs.total;
  if (total > hd.cap || total > nsl * (64 * U)) {
    if (lane == 0) atomicOr(&a.flags[0], 1);
    return;
  }
  if (slice == s0) {
    if (lane == 0) {
      long off = hd.off;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const Img m = pick(bs, k);
        Box b;
        b.imin = m.imin;
        b.imax = m.imax;
        b.jmin = m.jmin;
        b.jmax = m.jmax;
        b.off = off;
        a.boxes[(long)n * 3 + k] = b;
        off += m.cnt;
      }
    }
    // register the boxes with their tiles, one tile per lane: the first
    // tile of each of the six ranges is claimed by atomics issued together,
    // then the list entries stored (the registrations of one range do not
    // wait for those of the range before); a range of more than 64 tiles
    // registers the rest one by one
    int tile_[6], slot_[6];
#pragma unroll
    for (int r = 0; r < 6; r++) {
      tile_[r] = -1;
      const Img m = pick(bs, r / 2);
      if (m.cnt <= 0) continue;
      TileRange tr[2];
      box_tile_ranges(a, m.imin, m.imax, m.jmin, m.jmax, tr[0], tr[1]);
      const TileRange &rg = tr[r & 1];
      const int cnt = rg.count();
      const int w = rg.tx1 - rg.tx0 + 1;
      if (lane < cnt) tile_[r] = (rg.ty0 + lane / w) * a.ntx + rg.tx0 + lane % w;
      for (int e_ = lane + 64; e_ < cnt; e_ += 64)
        register_tile(a, (rg.ty0 + e_ / w) * a.ntx + rg.tx0 + e_ % w, n * 3 + r / 2);
    }
#pragma unroll
    for (int r = 0; r < 6; r++) slot_[r] = tile_[r] >= 0 ? atomicAdd(&a.tile_cnt[tile_[r]], 1) : -1;
#pragma unroll
    for (int r = 0; r < 6; r++) {
      if (tile_[r] < 0) continue;
      if (slot_[r] < TILE_CAP)
        a.tile_list[(long)tile_[r] * TILE_CAP + slot_[r]] = n * 3 + r / 2;
      else
        atomicOr(&a.flags[0], 2);
    }
  }
  const double *dist = a.sc_dist + hd.off;
  double *fxo = a.sc_fx + hd.off;
  double *fyo = a.sc_fy + hd.off;
  const double dx = a.dx, dy = a.dy;
  const double dxdy = a.dx * a.dy;
  double acc[3] = {0., 0., 0.};  // fux, fuy, tvz
  double ai[3] = {0., 0., 0.};   // inertia(0): iux, iuy, ivz
  const int t0 = (slice - s0) * (64 * U);
  const int t1 = t0 + 64 * U < total ? t0 + 64 * U : total;
  // all loads of the lane's cells first (a cell past t1 loads the last cell
  // instead and is skipped), then the forcing and the sums in cell order
  if (t0 < t1) {
    double th_[U], x_[U], y_[U], fx0[U], fx1[U], fy0[U], fy1[U], sx0[U], sx1[U], sy0[U],
        sy1[U];
    int k_[U], i_[U], j_[U];
    lane_cells<U>(bs, t0, t1, lane, k_, i_, j_);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const unsigned fx = face_x(a.L, i_[u], j_[u]), fy = face_y(a.L, i_[u], j_[u]);
      x_[u] = a.xc[i_[u]];
      y_[u] = a.yc[j_[u] - 1];
      th_[u] = dist[min(t0 + lane + 64 * u, t1 - 1)];
      fx0[u] = a.ux[fx];
      fx1[u] = a.ux[fx + 1];
      fy0[u] = a.uy[fy];
      fy1[u] = a.uy[fy + (unsigned)(a.nx + 2)];
      if (a.us_x) {
        sx0[u] = a.us_x[fx];
        sx1[u] = a.us_x[fx + 1];
        sy0[u] = a.us_y[fy];
        sy1[u] = a.us_y[fy + (unsigned)(a.nx + 2)];
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int t = t0 + lane + 64 * u;
      if (t >= t1) continue;
      const double py_ = py + a.ly * (k_[u] - 1);
      const double x = x_[u], y = y_[u];
      const double th = th_[u];
      if (a.us_x) {  // inertia(0), src/suspensions/inertia.c:55-60, at dx = 0
        const double wv = v_weight_th(th);
        const double valx = wv * 0.5 * (sx0[u] + sx1[u]) * dxdy;
        const double valy = wv * 0.5 * (sy0[u] + sy1[u]) * dxdy;
        ai[0] += valx * inv_pm;
        ai[2] += -(y - py_) * valx * inv_pim;
        ai[1] += valy * inv_pm;
        ai[2] += +(x - px) * valy * inv_pim;
      }
      const double w = s_weight_th(th);
      const double ux_p = pux - pvz * (y - py_);
      const double uy_p = puy + pvz * (x - px);
      const double ux_f = 0.5 * (fx0[u] + fx1[u]);
      const double uy_f = 0.5 * (fy0[u] + fy1[u]);
      const double fx = w * (ux_p - ux_f) * inv_dt;
      const double fy = w * (uy_p - uy_f) * inv_dt;
      fxo[t] = fx * dt;
      fyo[t] = fy * dt;
      acc[0] -= +(fx * dx * dy) * inv_pm;
      acc[2] -= -(y - py_) * (fx * dx * dy) * inv_pim;
      acc[1] -= +(fy * dx * dy) * inv_pm;
      acc[2] -= +(x - px) * (fy * dx * dy) * inv_pim;
    }
  }
  const double s0v = wave_sum(acc[0]), s1v = wave_sum(acc[1]), s2v = wave_sum(acc[2]);
  if (a.us_x) {
    const double i0 = wave_sum(ai[0]), i1 = wave_sum(ai[1]), i2 = wave_sum(ai[2]);
    if (lane == 0) {
      double *pp = a.slice_part0 + SLICE_VALS * (long)slice;
      pp[0] = i0;
      pp[1] = i1;
      pp[2] = i2;
      pp[3] = 0.;
      pp[4] = 0.;
    }
  }
  if (lane == 0) {
    double *pp = a.slice_part + SLICE_VALS * (long)slice;
    pp[0] = s0v;
    pp[1] = s1v;
    pp[2] = s2v;
    if (own_counts) {
      pp[3] = 0.;
      pp[4] = 0.;
    }
    if (slice == s0) {
      a.slice_info[2 * (long)n] = total;
      if (own_counts) a.slice_info[2 * (long)n + 1] = 0;
    }
  }
}
};
template <int U>
__global__ __launch_bounds__(WAVE) void k_exchange(IbmArgs a, int own_counts) {
  ExchangeB<U>::run(VB::here(), a, own_counts);
}

// ---------------------------------------------------------------------
// deposit + apply over active tiles (update.c:36-59)
// ---------------------------------------------------------------------
struct TileArgs {
  Layout L;
  int nx, ny, ntx;
  const Box *boxes;
  const double *sc_fx, *sc_fy;
  const int *tile_cnt, *tile_list;
  double *ux, *uy;
  double *dux, *duy;  // materialisation target (or null)
  int apply;
  const int *halt;
};

__device__ inline double box_value(const Box &b, const double *sc, int i, int j) {
  if (i < b.imin || i > b.imax || j < b.jmin || j > b.jmax) return 0.;
  const long w = b.imax - b.imin + 1;
  return sc[b.off + (long)(j - b.jmin) * w + (i - b.imin)];
}

// One 64-lane wave per active tile (lane = tile column, all TILE_Y rows),
// so that many tiles are in flight per CU.  The tile's box registrations
// (in registration order) are ranked in parallel into the reference's order
// (particle index, then image; a box registered twice counts once), the
// boxes are staged in LDS, and every cell sums its boxes' values in that
// order.
static_assert(TILE_X == 64, "one lane per tile column");
static_assert(TILE_CAP <= 64, "one lane per registration");

__device__ __forceinline__ void tile_body(const TileArgs &a, int tile) {
  __shared__ int raw[TILE_CAP];
  __shared__ bool rep[TILE_CAP];
  __shared__ Box sbox[TILE_CAP];
  // tiles in grid order, so neighbouring workgroups touch neighbouring
  // memory; tiles no box reaches return at once
  const int cnt = min(a.tile_cnt[tile], TILE_CAP);
  if (cnt == 0) return;
  const int lane = wave_lane();
  const Layout L = a.L;
  const int tx = tile % a.ntx, ty = tile / a.ntx;
  const int i0 = tx * TILE_X + 1, j0 = ty * TILE_Y + 1;
  if (lane < cnt) raw[lane] = a.tile_list[(long)tile * TILE_CAP + lane];
  wave_sync();
  int v = 0;
  bool dup = false;
  if (lane < cnt) {
    v = raw[lane];
    for (int s = 0; s < lane; s++) dup |= raw[s] == v;
    rep[lane] = dup;
  }
  wave_sync();
  if (lane < cnt && !dup) {
    int pos = 0;
    for (int s = 0; s < cnt; s++) pos += raw[s] < v && !rep[s];
    sbox[pos] = a.boxes[v];
  }
  wave_sync();
  const int nl = __popcll(__ballot(lane < cnt && !dup));  // every box once
  // column i0-1+lane of DUX and column i0+lane of DUY on rows j0-1 .. j0+3
  // (DUY's row j0-1 = 0 is row jtot), then column i0+lane of the tile.
  // Boxes outermost: the 13 loads of one box are in flight together, and
  // every cell still adds its boxes in list order.
  const int i = i0 + lane;
  double dxw[TILE_Y], dxc[TILE_Y], dy[TILE_Y + 1];
  int jy[TILE_Y + 1];
#pragma unroll
  for (int r = 0; r < TILE_Y; r++) dxw[r] = dxc[r] = 0.;
#pragma unroll
  for (int r = 0; r <= TILE_Y; r++) {
    dy[r] = 0.;
    jy[r] = j0 - 1 + r == 0 ? a.ny : j0 - 1 + r;
  }
  const bool iw = i - 1 >= 1 && i - 1 <= a.nx, ic = i <= a.nx;
  for (int s = 0; s < nl; s++) {
    const Box b = sbox[s];
    double tw[TILE_Y], tc[TILE_Y], ty_[TILE_Y + 1];
#pragma unroll
    for (int r = 0; r < TILE_Y; r++) {
      const bool rin = j0 + r <= a.ny;
      tw[r] = rin && iw ? box_value(b, a.sc_fx, i - 1, j0 + r) : 0.;
      tc[r] = rin && ic ? box_value(b, a.sc_fx, i, j0 + r) : 0.;
    }
#pragma unroll
    for (int r = 0; r <= TILE_Y; r++)
      ty_[r] = ic && jy[r] <= a.ny ? box_value(b, a.sc_fy, i, jy[r]) : 0.;
#pragma unroll
    for (int r = 0; r < TILE_Y; r++) {
      dxw[r] += tw[r];
      dxc[r] += tc[r];
    }
#pragma unroll
    for (int r = 0; r <= TILE_Y; r++) dy[r] += ty_[r];
  }
  if (i > a.nx) return;
#pragma unroll
  for (int r = 0; r < TILE_Y; r++) {
    const int j = j0 + r;
    if (j > a.ny) break;
    const double dux_w = dxw[r], dux_c = dxc[r], duy_s = dy[r], duy_c = dy[r + 1];
    if (a.apply) {
      // cells no box reaches get an increment of exactly zero: adding it
      // changes no value (a -0.0 could become +0.0), so they are skipped
      if (i >= 2 && (dux_w != 0. || dux_c != 0.)) {
        const long k = L.ux(i, j);
        const double u = a.ux[k] + 0.5 * (dux_w + dux_c);
        a.ux[k] = u;
        if (j == a.ny) a.ux[L.ux(i, 0)] = u;
        if (j == 1) a.ux[L.ux(i, a.ny + 1)] = u;
      }
      if (duy_s != 0. || duy_c != 0.) {
        const long k = L.p(i, j);
        const double u = a.uy[k] + 0.5 * (duy_s + duy_c);
        a.uy[k] = u;
        if (j == a.ny) a.uy[L.p(i, 0)] = u;
        if (j == 1) a.uy[L.p(i, a.ny + 1)] = u;
      }
    } else {
      a.dux[L.p(i, j)] = dux_c;
      a.duy[L.p(i, j)] = duy_c;
    }
  }
}

struct TilesB {
  static constexpr int T = WAVE, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, TileArgs a) {
  if (halted(a.halt)) return;
  tile_body(a, wave_index(vb));
}
};
__global__ __launch_bounds__(WAVE) void k_tiles(TileArgs a) {
  TilesB::run(VB::here(), a);
}

// The stage start's deposit with the exchange's per-particle sums (and
// inertia(0)'s) in the same launch: the first np workgroups finalise one
// particle each, the rest are the tiles.  Neither reads what the other
// writes.
struct TilesX0B {
  static constexpr int T = WAVE, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, TileArgs t, IbmArgs a) {
  if (halted(a.halt)) return;
  const int k = wave_index(vb);
  if (k < a.np)
    finalize_x0_particle(a, k);
  else
    tile_body(t, k - a.np);
}
};
__global__ __launch_bounds__(WAVE) void k_tiles_x0(TileArgs t, IbmArgs a) {
  TilesX0B::run(VB::here(), t, a);
}

// ---------------------------------------------------------------------
// collisions, src/suspensions/collision.c:75-367
// ---------------------------------------------------------------------
struct EllD {
  double a, b, x, y, angle;
};

// compute_evolute (collision.c:75-109) with the foot from foot_fp64,
// started at tw, the folded parameter of the previous fit in the same
// fixed-point iteration (or the FP32 estimate when tw < 0); the root on
// the first-quadrant arc is unique, so the start only changes the number
// of iterations.  (cm, sm) = cos/sin(-angle), (cp, sp) = cos/sin(+angle).
// (ct, st): cosine and sine of the foot's parameter (ellipse.c:62-63).
__device__ void evolute_fit_fast(const EllD &e, const EllipseShape &s,
                                 const EllipseShape32 &f, double cm, double sm, double cp,
                                 double sp, double x, double y, double &ex, double &ey,
                                 double &ct, double &st, double &tw) {
  double x_, y_;
  {
    const double x__ = x - e.x, y__ = y - e.y;
    x_ = cm * x__ - sm * y__;
    y_ = sm * x__ + cm * y__;
  }
  const double px = fabs(x_), py = fabs(y_);
  int it32 = 0, it64 = 0;
  if (tw < 0.) tw = (double)foot_fp32(f, px, py, it32);
  double c, sn;
  foot_fp64(s, px, py, tw, c, sn, it64);
  ct = x_ < 0. ? -c : c;
  st = y_ < 0. ? -sn : sn;
  x_ = s.kex * cube(ct);
  y_ = s.key * cube(st);
  ex = cp * x_ - sp * y_;
  ey = sp * x_ + cp * y_;
  ex = ex + e.x;
  ey = ey + e.y;
}

// what compute_evolute returns besides the centre: the radius of curvature
// at the foot and the foot itself, which only the last fit of the
// fixed-point iteration has to give
__device__ inline void evolute_radius(const EllD &e, double cp, double sp, double ct, double st,
                                      double &ix, double &iy, double &r) {
  // compute_curvature, ellipse.c:15-25
  const double ct2 = ct * ct, st2 = st * st;
  const double a2 = e.a * e.a, b2 = e.b * e.b;
  const double num = e.a * e.b * (ct2 + st2);
  const double den = +a2 * st2 + b2 * ct2;
  r = 1. / fmax(num / (den * sqrt(den)), DBL_EPSILON);
  const double x_ = e.a * ct, y_ = e.b * st;
  ix = cp * x_ - sp * y_;
  iy = sp * x_ + cp * y_;
}

struct CollArgs {
  const double *res;  // sub-iteration residuals (null: not gated)
  int sub;            // sub-iteration index
  int np;
  double lx, ly;
  double *prt;
  int cnstep;
  int *rows;       // np x CONTACT_CAP: colliding partners of each particle, ascending
  int *row_cnt;    // np
  int *wall_hit;   // np x 2
  int *flags;
  const int *halt;
  // the cell list (use_cells): partners are sought in a particle's cell and
  // its eight neighbours (periodic in y) instead of among all particles
  int use_cells;
  int ncx, ncy;
  double hx, hy;
  int *cl_start, *cl_items, *cl_cell, *cl_slot;
  double *cpos;  // np x 4: x + dx, y + dy, max(a, b) (written by k_reset, k_increment, k_coll_pack)
};

__device__ inline double harmonic(double v0, double v1) {
  const double r = 0.5 * (1. / v0 + 1. / v1);
  return 1. / r;
}

__device__ inline double min_image_offset(double p0y, double p1y, double ly) {
  double yoffset = 0., minval = DBL_MAX;
  for (int periodic = -1; periodic <= 1; periodic++) {
    const double val = fabs((p1y + ly * periodic) - p0y);
    if (val < minval) {
      minval = val;
      yoffset = ly * periodic;
    }
  }
  return yoffset;
}

// a particle's bounding circle, from the packed cpos (the same values as the
// records give)
struct Circle {
  double x, y, r;
};
__device__ inline Circle circle_of(const CollArgs &a, int n) {
  const double *p = a.cpos + 4 * (long)n;
  return {p[0], p[1], p[2]};
}

// The early exit of collision.c:156-189 for the pair n0 < n1: the bounding
// circles (radius max(a, b)) of the minimum image overlap
__device__ inline bool pair_candidate(const Circle &p0, const Circle &p1, double ly) {
  const double y1 = p1.y + min_image_offset(p0.y, p1.y, ly);
  const double dx = p1.x - p0.x, dy = y1 - p0.y, r = p0.r + p1.r;
  // far apart by the squares, with a margin far above their rounding: the
  // exact test would say so too (and NaN goes on to it)
  if (dx * dx + dy * dy > r * r * (1. + 1e-12)) return false;
  const double norm = fmax(hypot(dx, dy), DBL_EPSILON);
  return !(r - norm < 0.);
}

// the packed positions and radii of the broad phase, from the records
struct CollPackB {
  static constexpr int T = 256, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, CollArgs a) {
    if (halted(a.halt)) return;
    if (!sub_open(a.res, a.sub)) return;
    const int n = vb.bx * blockDim.x + threadIdx.x;
    if (n >= a.np) return;
    const double *q = a.prt + (long)n * R_N;
    double *o = a.cpos + 4 * (long)n;
    o[0] = q[R_X] + q[R_DX];
    o[1] = q[R_Y] + q[R_DY];
    o[2] = fmax(q[R_A], q[R_B]);
    o[3] = 0.;
  }
};
__global__ __launch_bounds__(256) void k_coll_pack(CollArgs a) {
  CollPackB::run(VB::here(), a);
}

// One contact of collision.c:156-304, by the two lanes l and l^1.
// A pair n0 < n1 (wall < 0): the lane of side 0 fits ellipse n0 and the
// lane of side 1 ellipse n1, each towards the other's current equivalent-
// circle centre, exchanged every iteration (the reference evaluates both
// fits from the previous centres too).  A wall (wall = 0: x = 0, 1: x = lx)
// of particle n0: both lanes fit n0 towards its mirror image.  Returns
// whether the circles overlap, with the contributions to n0 in v[0..2] and,
// for a pair, to n1 in v[3..5]; both lanes return the same values.
__device__ bool contact_force(const CollArgs &a, int n0, int n1, int wall, int side,
                              double v[6]) {
  const double wallx = wall == 0 ? 0. : a.lx;
  const double *p0 = a.prt + (long)n0 * R_N;
  const double *p1 = wall < 0 ? a.prt + (long)n1 * R_N : p0;
  const double *pm = side && wall < 0 ? p1 : p0;
  double yoffset = 0.;
  if (wall < 0) {
    yoffset = min_image_offset(p0[R_Y] + p0[R_DY], p1[R_Y] + p1[R_DY], a.ly);
  } else {  // wall early exit, collision.c:259-266
    const double x = p0[R_X] + p0[R_DX];
    const double r = fmax(p0[R_A], p0[R_B]);
    const double norm = fabs(wallx - x);
    if (r - norm < 0.) return false;
  }
  const double ym = pm[R_Y] + pm[R_DY];
  const EllD e = {pm[R_A], pm[R_B], pm[R_X] + pm[R_DX],
                  side && wall < 0 ? ym + yoffset : ym, pm[R_AZ]};
  // find_equivalent_circles, collision.c:111-135 (guarded iteration count)
  const EllipseShape sh = make_shape(e.a, e.b);
  const EllipseShape32 f = shape32(sh);
  double cp, sp;
  sincos(e.angle, &sp, &cp);
  const double cm = cp, sm = -sp;
  double tw = -1.;
  double cx = e.x, cy = e.y, ct = 0., st = 0.;
  for (int it = 0;; it++) {
    const double ox = __shfl_xor(cx, 1), oy = __shfl_xor(cy, 1);
    const double tx = wall < 0 ? ox : 2. * wallx - cx, ty = wall < 0 ? oy : cy;
    double nx, ny;
    evolute_fit_fast(e, sh, f, cm, sm, cp, sp, tx, ty, nx, ny, ct, st, tw);
    const double dx = nx - cx, dy = ny - cy;
    cx += dx;
    cy += dy;
    const double dm = fmax(fabs(dx), fabs(dy));
    const double dmo = __shfl_xor(dm, 1);
    const double dmax = wall >= 0 ? dm : side ? fmax(dmo, dm) : fmax(dm, dmo);
    if (dmax < 1.e-8) break;
    if (it >= EQC_ITER_CAP) {
      if (side == 0) atomicOr(&a.flags[0], 8);
      break;
    }
  }
  double ix, iy, cr;
  evolute_radius(e, cp, sp, ct, st, ix, iy, cr);
  const double ocx = __shfl_xor(cx, 1), ocy = __shfl_xor(cy, 1), ocr = __shfl_xor(cr, 1);
  const double oix = __shfl_xor(ix, 1), oiy = __shfl_xor(iy, 1);
  if (wall >= 0) {  // collision.c:268-304
    const double m = p_mass(p0), im = p_moi(p0);
    double nxv = wallx - cx;
    const double norm = fabs(nxv);
    nxv /= norm;
    const double overlap = cr - norm;
    if (!(overlap > 0.)) return false;
    double k;
    {
      const double mass = m;
      const double r = sqrt(p0[R_A] * p0[R_B]);
      const double reft = pow(r, 1.5);
      k = mass * (EIF_PI * EIF_PI) / (reft * reft);
    }
    const double cfx = k * overlap * nxv;
    const double cfy = 0.;
    v[0] = 1. / m * (-cfx);
    v[1] = 1. / m * (-cfy);
    v[2] = 1. / im * (ix * (-cfy) - iy * (-cfx));
    return true;
  }
  const double c0x = side ? ocx : cx, c0y = side ? ocy : cy, c0r = side ? ocr : cr;
  const double c1x = side ? cx : ocx, c1y = side ? cy : ocy, c1r = side ? cr : ocr;
  const double ix0 = side ? oix : ix, iy0 = side ? oiy : iy;
  const double ix1 = side ? ix : oix, iy1 = side ? iy : oiy;
  double nxv = c1x - c0x, nyv = c1y - c0y;
  const double norm = fmax(hypot(nxv, nyv), DBL_EPSILON);
  nxv /= norm;
  nyv /= norm;
  const double overlap = c0r + c1r - norm;
  if (!(overlap > 0.)) return false;
  const double m0 = p_mass(p0), m1 = p_mass(p1);
  const double i0 = p_moi(p0), i1 = p_moi(p1);
  double k;
  {
    const double mass = harmonic(m0, m1);
    const double r0 = sqrt(p0[R_A] * p0[R_B]);
    const double r1 = sqrt(p1[R_A] * p1[R_B]);
    const double reft = pow(harmonic(r0, r1), 1.5);
    k = mass * (EIF_PI * EIF_PI) / (reft * reft);
  }
  const double cfx = k * overlap * nxv;
  const double cfy = k * overlap * nyv;
  v[0] = 1. / m0 * (-cfx);
  v[1] = 1. / m0 * (-cfy);
  v[2] = 1. / i0 * (ix0 * (-cfy) - iy0 * (-cfx));
  v[3] = 1. / m1 * (+cfx);
  v[4] = 1. / m1 * (+cfy);
  v[5] = 1. / i1 * (ix1 * (+cfy) - iy1 * (+cfx));
  return true;
}

// The collision force of particle n (collision.c:306-367), by one wave:
// the lanes test all partners, then fit the candidate pairs and the two
// walls in parallel, two lanes per contact (each pair is fitted by both of
// its particles' waves, with the same operands), and the contributions are
// added in the order of the reference's loops: partners in ascending
// index, then wall x = 0, then wall x = lx.
//
// The launch is as long as one wave's chain of dependent loads and FP64
// operations, so loads are taken together (four partners a lane; the nine
// cells as three runs), the wave goes before others on its SIMD, and what
// only the last fit or an overlap needs is left to the end: k_inertia_collide
// 38.2 -> 35.3 us at 4096 ellipses on 1024x2048, 33.0 -> 31.6 at 1024 on
// 2048x4096 (with a shorter foot search than now: 43 and 46 us).
constexpr int COLL_CAND_CAP = 256;  // candidate partners per particle

// the lanes' partners that hit, appended to s_cand
__device__ inline void add_candidates(int lane, int m, bool hit, int *s_cand, int &cnt) {
  const unsigned long long b = __ballot(hit);
  if (hit) {
    const int pos = cnt + __popcll(b & ((1ull << lane) - 1ull));
    if (pos < COLL_CAND_CAP) s_cand[pos] = m;
  }
  cnt += __popcll(b);
}

// whether particle n (circle me) and m may touch
__device__ inline bool candidate(const CollArgs &a, int n, const Circle &me, int m,
                                 const Circle &q) {
  return m != n && pair_candidate(n < m ? me : q, n < m ? q : me, a.ly);
}

__device__ void collide_particle(const CollArgs &a, int n) {
  __shared__ int s_cand[COLL_CAND_CAP];
  __shared__ int s_sorted[COLL_CAND_CAP];
  // a long chain of dependent operations beside waves of short ones
  __builtin_amdgcn_s_setprio(3);
  const int lane = wave_lane();
  int cnt = 0;
  const int *cand = s_cand;
  const Circle me = circle_of(a, n);
  if (a.use_cells) {
    // the cell and its neighbours (ncy >= 3: the three rows are distinct);
    // two particles within reach are in the same or adjacent cells.  A row's
    // neighbouring cells are one run of the items; the three runs are taken
    // as one list, a partner a lane.
    const int c0 = a.cl_cell[n], cx0 = c0 % a.ncx, cy0 = c0 / a.ncx;
    const int xa = max(cx0 - 1, 0), xb = min(cx0 + 1, a.ncx - 1);
    int r0[3], r1[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const int row = (cy0 + d - 1 + a.ncy) % a.ncy * a.ncx;
      r0[d] = a.cl_start[row + xa];
      r1[d] = a.cl_start[row + xb + 1];
    }
    const int e0 = r1[0] - r0[0], e1 = e0 + r1[1] - r0[1], e2 = e1 + r1[2] - r0[2];
    for (int base = 0; base < e2; base += 64) {
      const int t = base + lane;
      const int k = t < e0 ? r0[0] + t : t < e1 ? r0[1] + (t - e0) : r0[2] + (t - e1);
      const int m = t < e2 ? a.cl_items[k] : n;
      add_candidates(lane, m, candidate(a, n, me, m, circle_of(a, m)), s_cand, cnt);
    }
    if (cnt > COLL_CAND_CAP) {
      if (lane == 0) atomicOr(&a.flags[0], 4);
      cnt = COLL_CAND_CAP;
    }
    wave_sync();
    // ascending partner order, as the scan over all particles finds them:
    // each candidate's rank is the number of smaller ones (all distinct)
    for (int k = lane; k < cnt; k += 64) {
      const int v = s_cand[k];
      int r = 0;
      for (int j = 0; j < cnt; j++) r += s_cand[j] < v;
      s_sorted[r] = v;
    }
    cand = s_sorted;
  } else {
    // four partners a lane in flight
    for (int base = 0; base < a.np; base += 256) {
      Circle q[4];
#pragma unroll
      for (int u = 0; u < 4; u++) q[u] = circle_of(a, min(base + 64 * u + lane, a.np - 1));
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int m = base + 64 * u + lane;
        add_candidates(lane, m, m < a.np && candidate(a, n, me, m, q[u]), s_cand, cnt);
      }
    }
    if (cnt > COLL_CAND_CAP) {
      if (lane == 0) atomicOr(&a.flags[0], 4);
      cnt = COLL_CAND_CAP;
    }
  }
  wave_sync();
  double fx = 0., fy = 0., tz = 0.;
  int ncont = 0;
  int *row = a.rows + (long)n * CONTACT_CAP;
  const int njobs = cnt + 2;  // the candidates, then the two walls
  for (int r = 0; r < njobs; r += 32) {
    const int k = r + (lane >> 1), side = lane & 1;
    int m = -1;
    bool hit = false;
    double w0 = 0., w1 = 0., w2 = 0.;
    if (k < njobs) {
      const int wall = k < cnt ? -1 : k - cnt;
      if (wall < 0) m = cand[k];
      double v[6] = {0., 0., 0., 0., 0., 0.};
      hit = contact_force(a, wall < 0 ? min(n, m) : n, wall < 0 ? max(n, m) : n, wall, side, v);
      const bool first = wall >= 0 || n < m;  // n's own contributions
      w0 = first ? v[0] : v[3];
      w1 = first ? v[1] : v[4];
      w2 = first ? v[2] : v[5];
      if (wall >= 0 && side == 0) a.wall_hit[2 * (long)n + wall] = hit ? 1 : 0;
    }
    unsigned long long hb = __ballot(hit && side == 0);
    while (hb) {
      const int l = __ffsll((long long)hb) - 1;
      hb &= hb - 1ull;
      const double u0 = lane_value(w0, l), u1 = lane_value(w1, l), u2 = lane_value(w2, l);
      const int mm = __builtin_amdgcn_readlane(m, l);
      if (mm >= 0) {  // a partner
        if (ncont >= CONTACT_CAP) {
          if (lane == 0) atomicOr(&a.flags[0], 16);
          continue;
        }
        if (lane == 0) row[ncont] = mm;
        ncont++;
      }
      fx += u0;
      fy += u1;
      tz += u2;
    }
  }
  if (lane == 0) {
    a.row_cnt[n] = ncont;
    double *q = a.prt + (long)n * R_N;
    q[R_CFX + a.cnstep] = fx;
    q[R_CFY + a.cnstep] = fy;
    q[R_CTZ + a.cnstep] = tz;
  }
}

// one wave per particle
struct CollideB {
  static constexpr int T = WAVE, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, CollArgs a) {
  if (halted(a.halt)) return;
  if (!sub_open(a.res, a.sub)) return;
  collide_particle(a, wave_index(vb));
}
};
__global__ __launch_bounds__(WAVE) void k_collide(CollArgs a) {
  CollideB::run(VB::here(), a);
}

// The cell list of the collision broad phase at the particles' current
// positions (x + dx, y + dy, from cpos).  The order within a cell follows
// atomics; the broad phase sorts each particle's candidates.  Up to
// CELL_BUILD_MAX particles one workgroup builds it in one launch, gated like
// the collisions it serves (CellBuildB: 14.4 -> 8.0 us at 4096 in a step; 7.5
// against the three launches' 15.2 at 8192).  Above, by three launches:
//  - count: each particle's cell, and its place in the cell from a device
//    atomic on the cell's count;
//  - scan: one workgroup turns the counts into offsets and clears them, so
//    that every build starts from zero counts;
//  - place: each particle's index stored at its cell's offset plus its place.
// Count and place are gated like the collisions they serve; the scan only
// by the sub-iteration (not by the halt flag, which another stream may
// raise between the launches), so it runs whenever the count ran.

// the cell of a particle at (x, y): reciprocals may move a cell boundary by
// rounding, which the 1e-6 margin of the cell size covers
__device__ inline int cell_of(const CollArgs &a, double x, double y) {
  const double yw = y - floor(y * (1. / a.ly)) * a.ly;  // into [0, ly), for the cell only
  const int cx = min(max((int)floor(x * (1. / a.hx)), 0), a.ncx - 1);
  const int cy = min(max((int)floor(yw * (1. / a.hy)), 0), a.ncy - 1);
  return cy * a.ncx + cx;
}

// sums of up to 16 waves at part[0] and their scan at part[32]
constexpr int CELL_SCAN = 64;

// cnt (nc counts in LDS) turned into exclusive offsets by the workgroup's
// threads, part their partial sums; returns the total.  Each thread sums a
// contiguous run; the runs' sums are scanned within each wave by lane
// shuffles, the waves' totals by the first wave.
__device__ inline int cell_offsets(int *cnt, int *part, int nc) {
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int per = (nc + blockDim.x - 1) / blockDim.x;
  const int k0 = min(t * per, nc), k1 = min(k0 + per, nc);
  int sum = 0;
  for (int k = k0; k < k1; k++) sum += cnt[k];
  int inc = sum;  // inclusive scan of the wave's run sums
  for (int d = 1; d < 64; d <<= 1) {
    const int v = __shfl_up(inc, d, 64);
    if (lane >= d) inc += v;
  }
  if (lane == 63) part[w] = inc;
  __syncthreads();
  if (w == 0) {
    const int nw = blockDim.x >> 6;
    int tot = lane < nw ? part[lane] : 0;
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(tot, d, 64);
      if (lane >= d) tot += v;
    }
    if (lane < nw) part[32 + lane] = tot;  // inclusive totals of waves
  }
  __syncthreads();
  int run = (w > 0 ? part[32 + w - 1] : 0) + inc - sum;  // exclusive offset of this run
  for (int k = k0; k < k1; k++) {
    const int v = cnt[k];
    cnt[k] = run;
    run += v;
  }
  __syncthreads();
  return part[32 + (blockDim.x >> 6) - 1];
}

// The whole list in one launch, by one workgroup with the counts in LDS.
struct CellBuildB {
  static constexpr int T = 1024, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, CollArgs a) {
    if (halted(a.halt)) return;
    if (!sub_open(a.res, a.sub)) return;
    extern __shared__ int cl_lds[];
    const int nc = a.ncx * a.ncy, t = threadIdx.x;
    int *cnt = cl_lds, *part = cl_lds + nc;
    int cell[CELL_BUILD_MAX / T], slot[CELL_BUILD_MAX / T];
#pragma unroll
    for (int u = 0; u < CELL_BUILD_MAX / T; u++) {
      const double *p = a.cpos + 4 * (long)min(t + u * T, a.np - 1);
      cell[u] = cell_of(a, p[0], p[1]);
    }
    for (int k = t; k < nc; k += T) cnt[k] = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < CELL_BUILD_MAX / T; u++) {
      const int n = t + u * T;
      if (n >= a.np) continue;
      a.cl_cell[n] = cell[u];
      slot[u] = atomicAdd(&cnt[cell[u]], 1);
    }
    __syncthreads();
    const int total = cell_offsets(cnt, part, nc);
    for (int k = t; k < nc; k += T) a.cl_start[k] = cnt[k];
    if (t == 0) a.cl_start[nc] = total;
#pragma unroll
    for (int u = 0; u < CELL_BUILD_MAX / T; u++) {
      const int n = t + u * T;
      if (n < a.np) a.cl_items[cnt[cell[u]] + slot[u]] = n;
    }
  }
};
__global__ __launch_bounds__(1024) void k_cell_build(CollArgs a) {
  CellBuildB::run(VB::here(), a);
}

struct CellCountB {
  static constexpr int T = 256, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, CollArgs a, int *counts) {
    if (halted(a.halt)) return;
    if (!sub_open(a.res, a.sub)) return;
    const int n = vb.bx * blockDim.x + threadIdx.x;
    if (n >= a.np) return;
    const double *q = a.prt + (long)n * R_N;
    const int c = cell_of(a, q[R_X] + q[R_DX], q[R_Y] + q[R_DY]);
    a.cl_cell[n] = c;
    a.cl_slot[n] = atomicAdd(&counts[c], 1);
  }
};
__global__ __launch_bounds__(256) void k_cell_count(CollArgs a, int *counts) {
  CellCountB::run(VB::here(), a, counts);
}

struct CellScanB {
  static constexpr int T = 1024, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, CollArgs a, int *counts) {
    if (!sub_open(a.res, a.sub)) return;
    extern __shared__ int cl_lds[];
    const int nc = a.ncx * a.ncy;
    int *cnt = cl_lds;          // nc counts
    int *part = cl_lds + nc;    // CELL_SCAN sums of the waves
    for (int k = threadIdx.x; k < nc; k += blockDim.x) {
      cnt[k] = counts[k];
      counts[k] = 0;
    }
    __syncthreads();
    const int total = cell_offsets(cnt, part, nc);
    for (int k = threadIdx.x; k < nc; k += blockDim.x) a.cl_start[k] = cnt[k];
    if (threadIdx.x == 0) a.cl_start[nc] = total;
  }
};
__global__ __launch_bounds__(1024) void k_cell_scan(CollArgs a, int *counts) {
  CellScanB::run(VB::here(), a, counts);
}

struct CellPlaceB {
  static constexpr int T = 256, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, CollArgs a) {
    if (halted(a.halt)) return;
    if (!sub_open(a.res, a.sub)) return;
    const int n = vb.bx * blockDim.x + threadIdx.x;
    if (n >= a.np) return;
    a.cl_items[a.cl_start[a.cl_cell[n]] + a.cl_slot[n]] = n;
  }
};
__global__ __launch_bounds__(256) void k_cell_place(CollArgs a) {
  CellPlaceB::run(VB::here(), a);
}

// One launch for a sub-iteration's inertia(1) and collision(1), which read
// the same positions and write disjoint particle members: the first np
// waves are the collisions (long, started first), the rest the IBM
// slices.  Bounded to 4 waves per SIMD (128 VGPRs): the collision path
// alone needs more and spills a little, which costs less than the
// occupancy its registers would take from the slices.
template <int U>
struct InertiaCollideB {
  static constexpr int T = WAVE, M = 4;
  static __device__ __forceinline__ void run(const VB &vb, IbmArgs a, CollArgs ca, int cnstep) {
  if (halted(a.halt)) return;
  const bool open = sub_open(a.res, a.sub);
  const int k = wave_index(vb);
  if (k < ca.np) {
    if (open) collide_particle(ca, k);
  } else {
    inertia_slice<U>(a, cnstep, k - ca.np, open);
  }
}
};
template <int U>
__global__ __launch_bounds__(WAVE, 4) void k_inertia_collide(IbmArgs a, CollArgs ca,
                                                                      int cnstep) {
  InertiaCollideB<U>::run(VB::here(), a, ca, cnstep);
}

struct ZeroIntB {
  static constexpr int T = 1024, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, int *p, int n) {
  const int t = vb.bx * blockDim.x + threadIdx.x;
  if (t < n) p[t] = 0;
}
};
__global__ void k_zero_int(int *p, int n) {
  ZeroIntB::run(VB::here(), p, n);
}


// ---------------------------------------------------------------------
// particle increments / update / reset
// ---------------------------------------------------------------------
__device__ inline void atomic_max_nonneg(double *addr, double v) {
  atomicMax(reinterpret_cast<unsigned long long *>(addr),
            (unsigned long long)__double_as_longlong(v));
}

struct ZeroResidualB {
  static constexpr int T = 1024, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, double *dscal) { dscal[S_RESIDUAL] = 0.; }
};
__global__ void k_zero_residual(double *dscal) {
  ZeroResidualB::run(VB::here(), dscal);
}

// src/suspensions/increment.c:10-64
// fin: also finalises the preceding inertia(1) call (its slice sums and
// cache records) for this particle first, saving a launch per sub-iteration.
//
// One wave per particle, four per workgroup, sixteen from INC_WIDE particles
// on: every workgroup ends with an atomic maximum on one address, and 1024
// of those take 8 us (4096 particles 15.4 -> 9.3 us by the wide workgroups;
// 1024 particles 8.7 -> 9.9, 64 particles 5.2 -> 8.6, where the sixteen waves
// share a CU's issue).  The launch is as long as one wave's chain of loads and dependent operations, so the wave issues every
// load before it tests the gate, holds the record one member a lane (read
// back by readlane), and spreads what is independent over lanes: the three
// images' boxes, the cache records and the counters.  With its
// predecessor's chain on lane 0 (and the header copied through scratch) it
// took 9.7 us at 1024 particles, 7.2 at 64, 16.7 at 4096.
constexpr int INC_WIDE = 2048;
struct IncrementB {
  static constexpr int T = 1024, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, double *prt, int np, const double *dscal,
                                                   double ga, double Fr, double *res_out,
                                                   IbmArgs ia, int fin) {
  __shared__ double red[16];
  const int waves = blockDim.x >> 6;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n = vb.bx * waves + w, nc = min(n, np - 1);
  double *p = prt + (long)nc * R_N;
  const int stop = ia.halt ? *ia.halt : 0;
  const double res_prev = ia.res && ia.sub > 0 ? ia.res[ia.sub - 1] : 1.;
  const double dt = dscal[S_DT];
  const double rec = p[min(lane, R_N - 1)];
  int s0 = 0, s1 = 0;
  PassRecord pr;
  CachedPass prev;
  if (fin) {
    s0 = ia.slice_first[nc];
    s1 = ia.slice_first[nc + 1];
    pr.load(ia, nc, lane);
  } else {
    prev = cached_records(ia, nc, lane);
  }
  // all threads of the workgroup see the same gate
  if (stop || (ia.res && ia.sub > 0 && (res_prev < 1.e-8 || ia.sub > 101))) return;
  auto member = [&](int m) { return lane_value(rec, m); };
  double res = 0.;
  if (n < np) {
    double iux1, iuy1, ivz1;
    if (fin) {  // inertia(1) of this sub-iteration: its sums and cache records
      double tot[SLICE_VALS];
      slice_sums(ia, s0, s1, tot);
      iux1 = tot[0];
      iuy1 = tot[1];
      ivz1 = tot[2];
      pr.store(ia, n, lane, tot);
      prev = pr.pass();
    } else {
      iux1 = member(R_IUX + 1);
      iuy1 = member(R_IUY + 1);
      ivz1 = member(R_IVZ + 1);
    }
    const double cfx0 = member(R_CFX), cfy0 = member(R_CFY), ctz0 = member(R_CTZ);
    // sub-iteration 0: collision(1) at the stage-start positions
    const bool first = ia.res && ia.sub == 0;
    const double cfx1 = first ? cfx0 : member(R_CFX + 1);
    const double cfy1 = first ? cfy0 : member(R_CFY + 1);
    const double ctz1 = first ? ctz0 : member(R_CTZ + 1);
    const double den = member(R_DEN);
    const double dux = +0.5 * ga * dt * (cfx0 + cfx1) + dt * member(R_FUX) + (iux1 - member(R_IUX))
                       + 1.0 * ga * dt * (1. - den) / (Fr * Fr);
    const double duy = +0.5 * ga * dt * (cfy0 + cfy1) + dt * member(R_FUY) + (iuy1 - member(R_IUY));
    const double dvz = +0.5 * ga * dt * (ctz0 + ctz1) + dt * member(R_TVZ) + (ivz1 - member(R_IVZ));
    res = fmax(res, fabs(dux - member(R_DUX)));
    res = fmax(res, fabs(duy - member(R_DUY)));
    res = fmax(res, fabs(dvz - member(R_DVZ)));
    const double ux0 = member(R_UX), uy0 = member(R_UY), vz0 = member(R_VZ);
    const double ux1 = ux0 + dux, uy1 = uy0 + duy, vz1 = vz0 + dvz;
    const double dxn = 0.5 * ga * dt * (ux0 + ux1);
    const double dyn = 0.5 * ga * dt * (uy0 + uy1);
    const double dazn = 0.5 * ga * dt * (vz0 + vz1);
    const double x = member(R_X) + dxn, y = member(R_Y) + dyn, az = member(R_AZ) + dazn;
    const double rad = fmax(member(R_A), member(R_B));
    if (lane == 0) {
      if (fin) {
        p[R_IUX + 1] = iux1;
        p[R_IUY + 1] = iuy1;
        p[R_IVZ + 1] = ivz1;
      }
      if (first) {
        p[R_CFX + 1] = cfx1;
        p[R_CFY + 1] = cfy1;
        p[R_CTZ + 1] = ctz1;
      }
      p[R_DUX] = dux;
      p[R_DUY] = duy;
      p[R_DVZ] = dvz;
      p[R_DX] = dxn;
      p[R_DY] = dyn;
      p[R_DAZ] = dazn;
      // the broad phase's packed position for the next sub-iteration's collisions
      double *cp = ia.cpos + 4 * (long)n;
      cp[0] = x;
      cp[1] = y;
      cp[2] = rad;
    }
    // the next sub-iteration's inertia pass
    write_head(ia, ia.heads + n, lane, x, y, az, rad, prev);
  }
  if (lane == 0) red[w] = res;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < waves; k++) res = fmax(res, red[k]);
    atomic_max_nonneg(res_out, res);
  }
}
};
__global__ __launch_bounds__(1024) void k_increment(double *prt, int np, const double *dscal,
                                                   double ga, double Fr, double *res_out,
                                                   IbmArgs ia, int fin) {
  IncrementB::run(VB::here(), prt, np, dscal, ga, Fr, res_out, ia, fin);
}

// src/suspensions/update.c:8-34
struct UpdateParticlesB {
  static constexpr int T = 1024, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, double *prt, int np, double ly, const int *halt) {
  if (halted(halt)) return;
  const int n = vb.bx * blockDim.x + threadIdx.x;
  if (n >= np) return;
  double *p = prt + (long)n * R_N;
  p[R_UX] += p[R_DUX];
  p[R_UY] += p[R_DUY];
  p[R_VZ] += p[R_DVZ];
  p[R_X] += p[R_DX];
  p[R_Y] += p[R_DY];
  p[R_AZ] += p[R_DAZ];
  if (p[R_Y] < 0.) p[R_Y] += ly;
  if (p[R_Y] > ly) p[R_Y] -= ly;
  if (p[R_AZ] < 0.) p[R_AZ] += 2. * EIF_PI;
  if (p[R_AZ] > 2. * EIF_PI) p[R_AZ] -= 2. * EIF_PI;
}
};
__global__ void k_update_particles(double *prt, int np, double ly, const int *halt) {
  UpdateParticlesB::run(VB::here(), prt, np, ly, halt);
}

// src/suspensions/reset.c:7-18, by one wave per particle, four per workgroup
// update: the previous stage's particle update (UpdateParticlesB's
// operations) first, in the same launch
// res (RES_SLOTS sub-iteration residuals) and tile_cnt (ntiles): cleared
// when given, for the stage's sub-iterations and the next exchange's tile
// registrations
// Also the heads of the stage-start pass (positions without increments).
struct ResetB {
  static constexpr int T = 256, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, IbmArgs a, double *res, int *tile_cnt,
                                             int ntiles, int update) {
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int n = vb.bx * 4 + w, nc = max(min(n, a.np - 1), 0);
    const int stop = a.halt ? *a.halt : 0;
    double rec = 0.;
    CachedPass prev{};
    double *p = a.prt + (long)nc * R_N;
    if (a.np > 0) {
      rec = p[min(lane, R_N - 1)];
      prev = cached_records(a, nc, lane);
    }
    if (stop) return;
    const int t = vb.bx * blockDim.x + threadIdx.x;
    if (res && t < RES_SLOTS) res[t] = 0.;
    if (tile_cnt)
      for (int k = t; k < ntiles; k += vb.gx * blockDim.x) tile_cnt[k] = 0;
    if (n >= a.np) return;
    auto member = [&](int m) { return lane_value(rec, m); };
    double x = member(R_X), y = member(R_Y), az = member(R_AZ);
    if (update) {
      x += member(R_DX);
      y += member(R_DY);
      az += member(R_DAZ);
      if (y < 0.) y += a.ly;
      if (y > a.ly) y -= a.ly;
      if (az < 0.) az += 2. * EIF_PI;
      if (az > 2. * EIF_PI) az -= 2. * EIF_PI;
    }
    SliceHead *h = a.heads + n;
    const double pa = member(R_A), pb = member(R_B);
    if (lane == 0) {
      if (update) {
        p[R_UX] = member(R_UX) + member(R_DUX);
        p[R_UY] = member(R_UY) + member(R_DUY);
        p[R_VZ] = member(R_VZ) + member(R_DVZ);
        p[R_X] = x;
        p[R_Y] = y;
        p[R_AZ] = az;
      }
      p[R_DUX] = 0.;
      p[R_DUY] = 0.;
      p[R_DVZ] = 0.;
      p[R_DX] = 0.;
      p[R_DY] = 0.;
      p[R_DAZ] = 0.;
      // foot-point warm starts reach back no further than the stage start, so
      // that a run restarted from a save repeats the same operations
      a.sc_key[8 * (long)n + 7] = 0;
      // the broad phase's packed position
      double *cp = a.cpos + 4 * (long)n;
      cp[0] = x;
      cp[1] = y;
      cp[2] = fmax(pa, pb);
    }
    prev.boxes = false;
    double q[3] = {member(R_DEN), pa, pb};  // the members that the shape needs
    write_head_shape(a, h, n, lane, q);
    write_head(a, h, lane, x, y, az, fmax(pa, pb), prev);
  }
};
__global__ __launch_bounds__(256) void k_reset(IbmArgs a, double *res, int *tile_cnt, int ntiles,
                                               int update) {
  ResetB::run(VB::here(), a, res, tile_cnt, ntiles, update);
}

// ---------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------
static IbmArgs ibm_args(Ctx *c) {
  IbmArgs a;
  a.L = c->L;
  a.nx = c->nx;
  a.ny = c->ny;
  a.ly = c->ly;
  a.dx = c->dx;
  a.dy = c->dy;
  a.grid_size = fmin(c->dx, c->dy);
  a.idx = 1. / c->dx;
  a.idy = 1. / c->dy;
  a.pow2 = c->pow2_grid ? 1 : 0;
  a.xc = c->xc;
  a.yc = c->yc;
  a.ux = c->ux;
  a.uy = c->uy;
  a.prt = c->prt;
  a.dscal = c->dscal;
  a.boxes = c->boxes;
  a.box_off = c->box_off;
  a.sc_fx = c->sc_fx;
  a.sc_fy = c->sc_fy;
  a.sc_dist = c->sc_dist;
  a.sc_pos = c->sc_pos;
  a.sc_t = c->sc_t;
  a.sc_key = c->sc_key;
  a.tile_cnt = c->tile_cnt;
  a.tile_list = c->tile_list;
  a.ntx = c->ntx;
  a.nty = c->nty;
  a.flags = c->flags;
  a.stats = c->ibm_pp;
  a.cpos = c->cpos;
  a.np = c->np;
  a.slice = c->slice_len;
  a.slice_first = c->slice_first;
  a.slice_rec = c->slice_rec;
  a.slice_info = c->slice_info;
  a.res = nullptr;
  a.sub = 0;
  a.us_x = a.us_y = nullptr;
  a.slice_part0 = c->slice_part0;
  a.slice_part = c->slice_part;
  a.heads = static_cast<SliceHead *>(c->heads);
  a.halt = c->halt;
  return a;
}

// f(cells a lane) for the context's slices
template <class F>
static void by_slice(const Ctx *c, F f) {
  switch (c->slice_len) {
    case 64: f(std::integral_constant<int, 1>{}); break;
    case 128: f(std::integral_constant<int, 2>{}); break;
    default: f(std::integral_constant<int, IBM_SLICE / 64>{}); break;
  }
}
static void go_inertia(Ctx *c, const IbmArgs &a, int cnstep, hipStream_t st) {
  by_slice(c, [&](auto u) {
    constexpr int U = decltype(u)::value;
    go<InertiaB<U>>(k_inertia<U>, dim3(c->nslices), dim3(WAVE), 0, st, a, cnstep);
  });
}
static void go_exchange(Ctx *c, const IbmArgs &a, int own_counts) {
  by_slice(c, [&](auto u) {
    constexpr int U = decltype(u)::value;
    go<ExchangeB<U>>(k_exchange<U>, dim3(c->nslices), dim3(WAVE), 0, c->stream, a,
                     own_counts);
  });
}

int launch_ref_iterations(Ctx *c, unsigned long long *dout) {
  if (c->np == 0) return EIF_OK;
  IbmArgs a = ibm_args(c);
  hipLaunchKernelGGL(k_ref_iterations, dim3(c->np), dim3(IBM_THREADS), 0, c->stream, a, dout);
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

int susp_init(Ctx *c) {
  // per-particle scratch capacity: three images of a box no wider than
  // floor(2r/h)+10 cells in each direction
  std::vector<double> rec((size_t)c->np * R_N);
  EIF_HIP(hipMemcpy(rec.data(), c->prt, rec.size() * sizeof(double), hipMemcpyDeviceToHost));
  std::vector<long> off(c->np + 1, 0);
  // slices of slice_len cells per particle: the boxes of at most two images
  // meet the domain when ly > 2r + 8 dy, and two clipped images together
  // are at most two rows taller than one box; otherwise allow three images
  std::vector<int> first(c->np + 1, 0);
  std::vector<long> box(c->np, 0);
  long all = 0;
  for (int n = 0; n < c->np; n++) {
    const double r = fmax(rec[(size_t)n * R_N + R_A], rec[(size_t)n * R_N + R_B]);
    const long cx = (long)(2. * r / c->dx) + 10, cy = (long)(2. * r / c->dy) + 10;
    const long wx = cx < c->nx ? cx : c->nx, wy = cy < c->ny ? cy : c->ny;
    off[n + 1] = off[n] + 3 * wx * wy;
    box[n] = c->ly > 2. * r + 16. * c->dy ? wx * (wy + 4) : 3 * wx * wy;
    all += box[n];
  }
  c->slice_len = IBM_SLICE;
  while (c->slice_len > 64 && all / c->slice_len < IBM_WAVES) c->slice_len /= 2;
  // room for whole slices of IBM_SLICE whatever the length: bodies that grow
  // by an upload of their records fit or do not at the same sizes
  for (int n = 0; n < c->np; n++)
    first[n + 1] = first[n] + (int)((box[n] + IBM_SLICE - 1) / IBM_SLICE) * (IBM_SLICE / c->slice_len);
  c->scratch_cells = off[c->np];
  c->nslices = first[c->np];
  TRY_S(coll_cells_setup(c, rec.data()));
  EIF_HIP(hipMalloc(&c->slice_first, (c->np + 1) * sizeof(int)));
  EIF_HIP(hipMemcpy(c->slice_first, first.data(), (c->np + 1) * sizeof(int), hipMemcpyHostToDevice));
  {
    std::vector<int4> rec(c->nslices > 0 ? c->nslices : 1, int4{0, 0, 0, 0});
    for (int n = 0; n < c->np; n++)
      for (int sl = first[n]; sl < first[n + 1]; sl++)
        rec[sl] = int4{n, first[n], first[n + 1] - first[n], 0};
    EIF_HIP(hipMalloc(&c->slice_rec, rec.size() * sizeof(int4)));
    EIF_HIP(hipMemcpy(c->slice_rec, rec.data(), rec.size() * sizeof(int4), hipMemcpyHostToDevice));
  }
  EIF_HIP(hipMalloc(&c->slice_info, 2 * (size_t)(c->np > 0 ? c->np : 1) * sizeof(long)));
  EIF_HIP(hipMemset(c->slice_info, 0, 2 * (size_t)(c->np > 0 ? c->np : 1) * sizeof(long)));
  EIF_HIP(hipMalloc(&c->slice_part, SLICE_VALS * (size_t)(c->nslices > 0 ? c->nslices : 1) * sizeof(double)));
  EIF_HIP(hipMalloc(&c->slice_part0, SLICE_VALS * (size_t)(c->nslices > 0 ? c->nslices : 1) * sizeof(double)));
  EIF_HIP(hipMalloc(&c->heads, sizeof(SliceHead) * (size_t)(c->np > 0 ? c->np : 1)));
  EIF_HIP(hipMalloc(&c->ibm_pp, (4 * (size_t)c->np + 1) * sizeof(unsigned long long)));
  EIF_HIP(hipMemset(c->ibm_pp, 0, (4 * (size_t)c->np + 1) * sizeof(unsigned long long)));
  EIF_HIP(hipMalloc(&c->box_off, (c->np + 1) * sizeof(long)));
  EIF_HIP(hipMemcpy(c->box_off, off.data(), (c->np + 1) * sizeof(long), hipMemcpyHostToDevice));
  const size_t sc = (size_t)(c->scratch_cells > 0 ? c->scratch_cells : 1) * sizeof(double);
  EIF_HIP(hipMalloc(&c->sc_fx, sc));
  EIF_HIP(hipMalloc(&c->sc_fy, sc));
  EIF_HIP(hipMalloc(&c->sc_dist, sc));
  EIF_HIP(hipMalloc(&c->sc_t, sc));
  EIF_HIP(hipMalloc(&c->sc_key, 8 * (size_t)(c->np > 0 ? c->np : 1) * sizeof(int)));
  EIF_HIP(hipMemset(c->sc_key, 0, 8 * (size_t)(c->np > 0 ? c->np : 1) * sizeof(int)));
  EIF_HIP(hipMalloc(&c->sc_pos, 4 * (size_t)(c->np > 0 ? c->np : 1) * sizeof(double)));
  EIF_HIP(hipMemset(c->sc_pos, 0, 4 * (size_t)(c->np > 0 ? c->np : 1) * sizeof(double)));
  EIF_HIP(hipMalloc(&c->boxes, 3 * (size_t)(c->np > 0 ? c->np : 1) * sizeof(Box)));
  EIF_HIP(hipMemset(c->boxes, 0, 3 * (size_t)(c->np > 0 ? c->np : 1) * sizeof(Box)));
  c->ntx = (c->nx + TILE_X - 1) / TILE_X;
  c->nty = (c->ny + TILE_Y - 1) / TILE_Y;
  const size_t ntiles = (size_t)c->ntx * c->nty;
  EIF_HIP(hipMalloc(&c->tile_cnt, ntiles * sizeof(int)));
  EIF_HIP(hipMemset(c->tile_cnt, 0, ntiles * sizeof(int)));
  EIF_HIP(hipMalloc(&c->tile_list, ntiles * TILE_CAP * sizeof(int)));
  // collisions
  {
    const size_t npp = (size_t)(c->np > 0 ? c->np : 1);
    EIF_HIP(hipMalloc(&c->rows, npp * CONTACT_CAP * sizeof(int)));
    EIF_HIP(hipMalloc(&c->cpos, 4 * npp * sizeof(double)));
    EIF_HIP(hipMemset(c->cpos, 0, 4 * npp * sizeof(double)));
    EIF_HIP(hipMalloc(&c->row_cnt, npp * sizeof(int)));
    EIF_HIP(hipMemset(c->row_cnt, 0, npp * sizeof(int)));
  }
  EIF_HIP(hipMalloc(&c->wall_hit, 2 * (size_t)(c->np > 0 ? c->np : 1) * sizeof(int)));
  EIF_HIP(hipMemset(c->wall_hit, 0, 2 * (size_t)(c->np > 0 ? c->np : 1) * sizeof(int)));
  return EIF_OK;
}

int launch_reset(Ctx *c, hipStream_t st, bool clear_tiles, bool update) {
  if (!st) st = c->stream;
  // also clears the sub-iteration residuals, so it runs without particles too
  const int ntiles = c->np > 0 && clear_tiles ? c->ntx * c->nty : 0;
  const int grid = std::max({(c->np + 3) / 4, (ntiles + 1023) / 1024, 1});
  go<ResetB>(k_reset, dim3(grid), dim3(256), 0, st, ibm_args(c),
                     c->res_slots, ntiles > 0 ? c->tile_cnt : nullptr, ntiles, update ? 1 : 0);
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

int launch_inertia(Ctx *c, int cnstep, hipStream_t st, bool defer_finalize) {
  if (c->np == 0) return EIF_OK;
  if (!st) st = c->stream;
  ProfScope ps(c, "ibm_inertia", st);
  IbmArgs a = ibm_args(c);
  go<HeadsB>(k_heads, dim3((c->np + 3) / 4), dim3(256), 0, st, a, 1);
  go_inertia(c, a, cnstep, st);
  if (!defer_finalize)
    go<IbmFinalizeB>(k_ibm_finalize, dim3((c->np + 3) / 4), dim3(256), 0, st, a, cnstep);
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

int launch_exchange(Ctx *c, bool cached_known, bool tiles_clear, bool defer_finalize) {
  if (c->np == 0) return EIF_OK;
  ProfScope ps(c, "ibm_exchange");
  const size_t ntiles = (size_t)c->ntx * c->nty;
  if (!tiles_clear) {  // clear the previous call's tile registrations
    go<ZeroIntB>(k_zero_int, dim3((unsigned)((ntiles + 255) / 256)), dim3(256), 0,
                       c->stream, c->tile_cnt, (int)ntiles);
  }
  IbmArgs a = ibm_args(c);
  go<HeadsB>(k_heads, dim3((c->np + 3) / 4), dim3(256), 0, c->stream, a, 0);
  if (!cached_known)
    go<IbmDistB>(k_ibm_dist, dim3(c->nslices), dim3(WAVE), 0, c->stream, a);
  go_exchange(c, a, cached_known ? 1 : 0);
  EIF_HIP(hipGetLastError());
  if (!defer_finalize) return launch_exchange_finalize(c, c->stream);
  return EIF_OK;
}

// Signed distances (as tanh(BETA d)) of the box cells at the particles'
// positions without increments, into the per-cell cache
int launch_ibm_dist(Ctx *c, hipStream_t st) {
  if (c->np == 0) return EIF_OK;
  go<IbmDistB>(k_ibm_dist, dim3(c->nslices), dim3(WAVE), 0, st ? st : c->stream,
                     ibm_args(c));
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

// The exchange at the stage start (distances cached by launch_ibm_dist, tile
// registrations cleared by the reset) with inertia(0) of the stage-start
// velocity (us_x, us_y) in the same pass over the cells; the sums are added
// by the deposit launch (launch_update_momentum_x0)
int launch_exchange_inertia0(Ctx *c, const double *us_x, const double *us_y) {
  if (c->np == 0) return EIF_OK;
  ProfScope ps(c, "ibm_exchange");
  IbmArgs a = ibm_args(c);
  a.us_x = us_x;
  a.us_y = us_y;
  go_exchange(c, a, 0);
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

// the exchange's per-particle sums; nothing on the fluid side
// reads them, so this may run on another stream after the exchange
int launch_exchange_finalize(Ctx *c, hipStream_t st) {
  if (c->np == 0) return EIF_OK;
  go<IbmFinalizeB>(k_ibm_finalize, dim3((c->np + 3) / 4), dim3(256), 0, st, ibm_args(c), 2);
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

static TileArgs tile_args(Ctx *c, int apply) {
  TileArgs t;
  t.L = c->L;
  t.nx = c->nx;
  t.ny = c->ny;
  t.ntx = c->ntx;
  t.boxes = c->boxes;
  t.sc_fx = c->sc_fx;
  t.sc_fy = c->sc_fy;
  t.tile_cnt = c->tile_cnt;
  t.tile_list = c->tile_list;
  t.ux = c->ux;
  t.uy = c->uy;
  t.dux = c->dux;
  t.duy = c->duy;
  t.apply = apply;
  t.halt = c->halt;
  return t;
}

static long tile_count(const Ctx *c) { return (long)c->ntx * c->nty; }

int launch_update_momentum(Ctx *c) {
  if (c->np == 0) return EIF_OK;
  ProfScope ps(c, "ibm_apply");
  TileArgs t = tile_args(c, 1);
  go<TilesB>(k_tiles, dim3((unsigned)tile_count(c)), dim3(WAVE), 0, c->stream, t);
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

// the stage start's deposit and the exchange's particle sums, one launch
int launch_update_momentum_x0(Ctx *c) {
  if (c->np == 0) return EIF_OK;
  ProfScope ps(c, "ibm_apply");
  TileArgs t = tile_args(c, 1);
  go<TilesX0B>(k_tiles_x0, dim3((unsigned)(c->np + tile_count(c))), dim3(WAVE), 0, c->stream,
                     t, ibm_args(c));
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

int launch_materialise_du(Ctx *c) {
  const size_t bytes = (size_t)c->L.p_len() * sizeof(double);
  EIF_HIP(hipMemsetAsync(c->dux, 0, bytes, c->stream));
  EIF_HIP(hipMemsetAsync(c->duy, 0, bytes, c->stream));
  if (c->np > 0) {
    TileArgs t = tile_args(c, 0);
    go<TilesB>(k_tiles, dim3((unsigned)tile_count(c)), dim3(WAVE), 0, c->stream,
                       t);
    EIF_HIP(hipGetLastError());
  }
  int r = launch_bc_p(c, c->dux);
  if (r) return r;
  return launch_bc_p(c, c->duy);
}

// whether the collision broad phase uses the cell list
static bool coll_use_cells(const Ctx *c) {
  if (c->cl_ncy < 3 || c->coll_mode == 1) return false;
  return c->coll_mode == 2 || c->np >= COLL_CELLS_MIN;
}

int coll_cells_setup(Ctx *c, const double *rec) {
  double rmax = 0.;
  for (int n = 0; n < c->np; n++)
    rmax = fmax(rmax, fmax(rec[(size_t)n * R_N + R_A], rec[(size_t)n * R_N + R_B]));
  int ncx = 0, ncy = 0;
  if (rmax > 0.) {
    // cells at least the widest reach (with a margin above rounding), and
    // at most COLL_CELLS_CAP of them
    double h = fmax(2. * rmax * (1. + 1e-6), sqrt(c->lx * c->ly / COLL_CELLS_CAP));
    for (;;) {
      const double fx = fmax(floor(c->lx / h), 1.), fy = fmax(floor(c->ly / h), 1.);
      if (fx * fy <= COLL_CELLS_CAP) {
        ncx = (int)fx;
        ncy = (int)fy;
        break;
      }
      h *= 1.05;
    }
  }
  // sized for the most cells once: graphs keep the addresses.  The counts
  // start at zero and every build leaves them at zero; cells and places
  // start at zero, so that a build whose count was halted still places
  // within bounds
  if (!c->cl_start) {
    EIF_HIP(hipMalloc(&c->cl_start, (COLL_CELLS_CAP + 1) * sizeof(int)));
    EIF_HIP(hipMalloc(&c->cl_count, COLL_CELLS_CAP * sizeof(int)));
    const size_t n = (size_t)(c->np > 0 ? c->np : 1) * sizeof(int);
    EIF_HIP(hipMalloc(&c->cl_items, n));
    EIF_HIP(hipMalloc(&c->cl_cell, n));
    EIF_HIP(hipMalloc(&c->cl_slot, n));
    EIF_HIP(hipMemset(c->cl_start, 0, (COLL_CELLS_CAP + 1) * sizeof(int)));
    EIF_HIP(hipMemset(c->cl_count, 0, COLL_CELLS_CAP * sizeof(int)));
    EIF_HIP(hipMemset(c->cl_cell, 0, n));
    EIF_HIP(hipMemset(c->cl_slot, 0, n));
  }
  c->cl_ncx = ncx;
  c->cl_ncy = ncy;
  c->cl_hx = ncx > 0 ? c->lx / ncx : 0.;
  c->cl_hy = ncy > 0 ? c->ly / ncy : 0.;
  return EIF_OK;
}

int set_collision_search(Ctx *c, int mode) {
  if (mode < 0 || mode > 2) {
    set_error("collision search must be 0 (by particle count), 1 (all pairs) or 2 (cell list)");
    return EIF_ERR_ARG;
  }
  c->coll_mode = mode;
  return EIF_OK;
}

static CollArgs coll_args(Ctx *c, int cnstep) {
  CollArgs a;
  a.res = nullptr;
  a.sub = 0;
  a.np = c->np;
  a.lx = c->lx;
  a.ly = c->ly;
  a.prt = c->prt;
  a.cnstep = cnstep;
  a.rows = c->rows;
  a.row_cnt = c->row_cnt;
  a.wall_hit = c->wall_hit;
  a.flags = c->flags;
  a.halt = c->halt;
  a.use_cells = coll_use_cells(c) ? 1 : 0;
  a.ncx = c->cl_ncx;
  a.ncy = c->cl_ncy;
  a.hx = c->cl_hx;
  a.hy = c->cl_hy;
  a.cl_start = c->cl_start;
  a.cl_items = c->cl_items;
  a.cl_cell = c->cl_cell;
  a.cl_slot = c->cl_slot;
  a.cpos = c->cpos;
  return a;
}

// the cell list for a collision launch with these (gated) arguments
static void launch_cell_list(Ctx *c, const CollArgs &a, hipStream_t st) {
  if (!a.use_cells) return;
  const size_t lds = ((size_t)c->cl_ncx * c->cl_ncy + CELL_SCAN) * sizeof(int);
  if (c->np <= CELL_BUILD_MAX) {
    go<CellBuildB>(k_cell_build, dim3(1), dim3(CellBuildB::T), lds, st, a);
    return;
  }
  const dim3 g((c->np + 255) / 256);
  go<CellCountB>(k_cell_count, g, dim3(256), 0, st, a, c->cl_count);
  go<CellScanB>(k_cell_scan, dim3(1), dim3(1024), lds, st, a, c->cl_count);
  go<CellPlaceB>(k_cell_place, g, dim3(256), 0, st, a);
}

int launch_collision(Ctx *c, int cnstep, hipStream_t st, bool packed) {
  if (c->np == 0) return EIF_OK;
  if (!st) st = c->stream;
  ProfScope ps(c, "collision", st);
  const CollArgs a = coll_args(c, cnstep);
  if (!packed) go<CollPackB>(k_coll_pack, dim3((c->np + 255) / 256), dim3(256), 0, st, a);
  launch_cell_list(c, a, st);
  go<CollideB>(k_collide, dim3(c->np), dim3(WAVE), 0, st, a);
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

int launch_substep_forces(Ctx *c, int sub) {
  if (c->np == 0) return EIF_OK;
  IbmArgs a = ibm_args(c);
  a.res = c->res_slots;
  a.sub = sub;
  if (sub == 0) {
    // The first sub-iteration's positions are the stage start's (dx = 0
    // after the reset): collision(1) would repeat collision(0) operand for
    // operand, so the increment copies collision(0)'s forces instead
    ProfScope ps(c, "ibm_inertia");
    go_inertia(c, a, 1, c->stream);
    EIF_HIP(hipGetLastError());
    return EIF_OK;
  }
  CollArgs ca = coll_args(c, 1);
  ca.res = a.res;
  ca.sub = sub;
  launch_cell_list(c, ca, c->stream);
  hipEvent_t e0, e1;
  const bool timed = prof_kernel_events(c, "ibm_substep", &e0, &e1);
  by_slice(c, [&](auto u) {
    constexpr int U = decltype(u)::value;
    const dim3 grid(c->np + c->nslices), block(WAVE);
    if (timed)  // a sampled launch stamps its events
      hipExtLaunchKernelGGL(k_inertia_collide<U>, grid, block, 0, c->stream, e0, e1, 0, a, ca, 1);
    else
      go<InertiaCollideB<U>>(k_inertia_collide<U>, grid, block, 0, c->stream, a, ca, 1);
  });
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

int launch_increment(Ctx *c, int rk, int sub) {
  IbmArgs ia = ibm_args(c);
  double *res_out = c->dscal + S_RESIDUAL;
  if (sub < 0) {  // not gated: the residual starts from zero
    go<ZeroResidualB>(k_zero_residual, dim3(1), dim3(1), 0, c->stream, c->dscal);
  } else {  // the residual slot was cleared at the stage start
    ia.res = c->res_slots;
    ia.sub = sub;
    res_out = c->res_slots + sub;
  }
  const int waves = c->np >= INC_WIDE ? 16 : 4;
  if (c->np > 0)
    go<IncrementB>(k_increment, dim3((c->np + waves - 1) / waves), dim3(64 * waves), 0, c->stream,
                       c->prt, c->np, c->dscal, c->gamma[rk], c->cfg.Fr, res_out, ia,
                       sub >= 0 ? 1 : 0);
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

// one thread copies the state of the first `queued` sub-iterations into
// pinned host memory: how many ran, and the residual of the last one.  The
// record number is stored last with system-scope release, so a host that
// sees it sees the rest.
__global__ void k_status(const double *res, int queued, const int *flags,
                         const double *dscal, HostStatus *h, unsigned seq) {
  int done = 0;
  double r = 0.;
  for (int s = 0; s < queued && sub_open(res, s); s++) {
    done = s + 1;
    r = res[s];
  }
  h->residual = r;
  h->dt = dscal[S_DT];
  h->substeps = done;
  h->flags = flags[0];
  __hip_atomic_store(&h->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

int launch_status(Ctx *c, int queued) {
  hipLaunchKernelGGL(k_status, dim3(1), dim3(1), 0, c->stream, c->res_slots, queued,
                     c->flags, c->dscal, c->hstat, ++c->hstat_seq);
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

// Graph steps: the end of a stage's captured sub-iterations.  Records how
// many of the first K ran and the last residual; if the loop would go on
// (sub-iteration K is open), stops the rest of the step (halt = stage + 1)
// for the host to resume.
struct StageGateB {
  static constexpr int T = 1024, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, const double *res, int K, int stage, int *counts, double *resid,
                             int *halt) {
  if (*halt) return;
  int done = 0;
  double r = 0.;
  for (int s = 0; s < K && sub_open(res, s); s++) {
    done = s + 1;
    r = res[s];
  }
  counts[stage] = done;
  resid[stage] = r;
  if (sub_open(res, K)) *halt = stage + 1;
}
};
__global__ void k_stage_gate(const double *res, int K, int stage, int *counts, double *resid,
                             int *halt) {
  StageGateB::run(VB::here(), res, K, stage, counts, resid, halt);
}

int launch_stage_gate(Ctx *c, int stage, int K) {
  go<StageGateB>(k_stage_gate, dim3(1), dim3(1), 0, c->stream, c->res_slots, K, stage,
                     c->g_counts, c->g_resid, c->halt);
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

// Graph steps: the step's record for the host (two slots, by the parity of
// the device's step counter), the record number stored last with
// system-scope release.  Not gated: a stopped step reports its stop.
struct GraphStatusB {
  static constexpr int T = 1024, M = 0;
  static __device__ __forceinline__ void run(const VB &vb, const int *halt, const int *counts, const double *resid,
                               const double *dscal, const int *flags, unsigned *seq,
                               GraphStatus *h) {
  const unsigned s = *seq + 1;
  *seq = s;
  GraphStatus *o = h + (s & 1);
  o->dt = dscal[S_DT];
  for (int k = 0; k < 3; k++) {
    o->counts[k] = counts[k];
    o->resid[k] = resid[k];
  }
  o->halt = *halt;
  o->flags = flags[0];
  __hip_atomic_store(&o->seq, s, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
};
__global__ void k_graph_status(const int *halt, const int *counts, const double *resid,
                               const double *dscal, const int *flags, unsigned *seq,
                               GraphStatus *h) {
  GraphStatusB::run(VB::here(), halt, counts, resid, dscal, flags, seq, h);
}

int launch_graph_status(Ctx *c) {
  go<GraphStatusB>(k_graph_status, dim3(1), dim3(1), 0, c->stream, c->halt, c->g_counts,
                     c->g_resid, c->dscal, c->flags, c->g_seq, c->gstat);
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

int launch_update_particles(Ctx *c) {
  if (c->np == 0) return EIF_OK;
  go<UpdateParticlesB>(k_update_particles, dim3((c->np + 255) / 256), dim3(256), 0,
                     c->stream, c->prt, c->np, c->ly, c->halt);
  EIF_HIP(hipGetLastError());
  return EIF_OK;
}

}  // namespace eif
