// Per-cell and per-face work of one rate-of-change evaluation, written once
// for the gfx950 kernels (kernels.hip).  Everything is FP64.
//
// Reference semantics restated here:
//   reconstruction   include/zisa/reconstruction/local_reconstruction.hpp:69-156,
//                    src/zisa/reconstruction/{cweno_ao,weno_ao,hybrid_weno}.cpp,
//                    include/zisa/math/poly2d_impl.hpp:271-337
//   face flux        include/zisa/fvm_loops/flux_loop.hpp:126-193,
//                    include/zisa/flux/hllc.hpp:17-176
//   gravity source   include/zisa/fvm_loops/gravity_source_loop.hpp:32-148
//   equilibria       include/zisa/model/local_equilibrium_impl.hpp:41-93,
//                    include/zisa/model/isentropic_equilibrium.hpp:28-63
//   flux BC          include/zisa/boundary/flux_bc.hpp:25-42
//   RK stage         src/zisa/ode/runge_kutta.cpp:87-143
#pragma once

// Rounding: everything here is compiled with -ffp-contract=off, so no
// compiler decides where to fuse a multiply-add; the least-squares
// accumulation and the polynomial evaluation use explicit fma().  The same
// source therefore rounds identically in every kernel and in the host
// emulation, whatever the surrounding code.

#include <cstdint>
#include <type_traits>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define ZFV_HD __host__ __device__ __forceinline__
#else
#include <cmath>
#define ZFV_HD inline
#endif

namespace zfv {

// cell meta word: bits 0-2 index of the CWENO high-order stencil, 8 = first
// order (a ghost cell away from the interior), 16 = ghost cell
constexpr int32_t META_FAR_GHOST = 8 | 16;

constexpr int ROW_CELL_BITS = 27;
constexpr int32_t ROW_CELL_MASK = (1 << ROW_CELL_BITS) - 1;

// What the kernels read.  Pointers are device pointers (or host pointers in
// the CPU emulation used by the tests).
struct Img {
  int64_t n;   // cells
  int64_t ne;  // interior faces
  int64_t n_near;  // the first cells, those that are not ghosts away from the interior (META_FAR_GHOST)
  const double *P;
  const int32_t *rows;  // cell | shift_code << 27
  const int8_t *twin;   // (nrows - rc) * n: central row with the same member, or -1
  const double *crn;
  const double *xc;
  const double *len;
  const double *vol;
  const double *inr;
  const double *mom;
  const int32_t *meta;
  const int32_t *cface;  // per cell its face words, 4 int32 (one 16-byte load; 2D's fourth unused)
  const int32_t *fslot;  // ne pairs: cell-face slots of each interior face's left and right cell
  // the faces that an update wavefront evaluates for its tile of cells
  // (build_update_tiles): tile t's first 64 at uent + 64 t (l < 0: none), any
  // more in umore from uoff[t] to uoff[t + 1]; and per cell which of its tile's
  // entries its faces are.  Null in the host emulation.
  const int32_t *uent;
  const int32_t *uoff;
  const int32_t *umore;
  const uint32_t *ucell;
  const uint32_t *fperm;
  const double *steady;  // as the state (ghost cells only are read)
  const double *phim;    // n pairs: cell mean of phi and of (phi - mean)^2 (one 16-byte load), or null
  const double *pot;     // potential tables of the cell's own points (pot_index), or null
  const double *frm;     // normals and areas of the cells' local faces (load_face_frame)
  const double *ffr;     // per interior face its normal and area (face_table_frame)
  // 3D with an equilibrium: per cell its faces' outward normals times their
  // areas, n x (face 3 + d) (store_face_normals), or null
  const double *fan;
  // gravity: per cell vol sum_q vw_q b_alpha(x_q) d_d phi(x_q) over its volume
  // points, n x (alpha DIM + d), each cell's DOFC x DIM values contiguous
  // (store_source_moments), or null
  const double *smom;
  // the light set with an equilibrium, whose axial potential is affine, or
  // null; each cell's values contiguous (store_cell_phi).  3D: the potential
  // at its corners.  2D: the corners' mean and the sums of the squares and
  // cubes of their deviations from it.
  const double *cphi;
  // 2D light set: the equilibrium averages in series form (exp_average), used
  // while the exponents of a cell's stencil stay within its range: bounds over
  // the instance of |mean of a member - mean of the cell| and of the sums of
  // squares; 0: not available
  double es_dist, es_p2;
  double es[12];
  int phi_unshifted;  // 1: no translation changes the axial potential (shift_phi all zero)
  // stateful equilibria (steps_per_recompute > 1), or null: per cell theta
  // (2), found flag, EulerScaling (rho, a, E_int) and the equilibrium's own
  // cell average (rho, E) of the last recompute (8 x n), and calls since it
  // (n); launches that must leave them alone (autotuning, kernel timing) run
  // with eqc null and recompute
  double *eqc;
  int32_t *eqcnt;
  int spr;               // steps_per_recompute
  double eq_threshold;   // recompute_threshold
  // physics
  double gamma;
  double eps, exponent;
  double lw[5];  // normalized linear weights
  int mode;      // 0 CWENO-AO, 1 WENO-AO
  int scaling;   // 0 EulerScaling, 1 UnityScaling
  int vol_mean;  // 1: a reconstruction's volume-rule mean over its cell is its constant coefficient
  int flux;      // 0 HLLC, 1 Rusanov
  int eq;        // 0 none, 1 isentropic, 2 isothermal
  int gravity;   // 0 none, 1 axial, 2 radial, 3 polytrope
  double g, axis[3], rhoC, K, G;
  // isentropic equilibrium: 1/(gamma - 1) = eq_half / 2 + eq_db to the last
  // place, where it is a multiple of 1/2 up to rounding (eq_pow); eq_half 0: not
  int eq_half;
  double eq_db;
  int flux_bc;
  double shift[16][3];  // periodic translations addressed by the row shift code
  double shift_phi[16];  // axial potential of each translation (added to cphi's potentials)
  // normalized quadrature rules
  int qv;                   // points of the volume rule
  double fw[8], fx[8][3];   // face rule: weights, GL abscissa (2D) or barycentric (3D)
  double vw[16], vx[16][4]; // volume rule
};

template <int DIM>
struct Dims {
  static constexpr int NV = DIM + 2;
  static constexpr int NF = DIM + 1;
  static constexpr int DOFB = DIM + 1;
};

ZFV_HD double sqr(double x) { return x * x; }

ZFV_HD double dmin(double a, double b) { return a < b ? a : b; }
ZFV_HD double dmax(double a, double b) { return a > b ? a : b; }
// a / b where r = 1 / b is at hand, to the last place of a division
ZFV_HD double quotient(double a, double b, double r) {
  const double q = a * r;
  return fma(fma(-q, b, a), r, q);
}

// Where variable v of cell i stands in a state-shaped array (state, stage
// state, tendencies, source, steady state).  The kernels keep the NV values of
// a cell together (AOS): a stencil member's state is then one 32- or 40-byte
// piece that its group's lanes fetch side by side, where planes cost one cache
// line per variable and member.  The planes (v * n + i) are the layout of the
// host emulation.
template <bool AOS, int NV>
ZFV_HD int64_t state_at(int64_t n, int v, int64_t i) {
  return AOS ? i * NV + v : int64_t(v) * n + i;
}

// which of the two a lane exchange type's instances use: planes unless the
// type says otherwise (static constexpr bool kAos)
template <class X, class = void>
struct state_is_aos : std::false_type {};
template <class X>
struct state_is_aos<X, std::void_t<decltype(X::kAos)>> : std::bool_constant<X::kAos> {};

// a value that all lanes of a wavefront hold alike, where the compiler cannot
// see it (the host emulation's exchange has one lane at a time)
ZFV_HD int wave_uniform(int v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_readfirstlane(v);
#else
  return v;
#endif
}
// true on every active lane of the wavefront if it is on all of them
ZFV_HD bool wave_all(bool v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __all(v);
#else
  return v;
#endif
}
// no instruction is moved across (keeps later chunks' loads from being pulled
// forward into registers that the occupancy needs)
ZFV_HD void schedule_fence() {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_sched_barrier(0);
#endif
}

// the values are formed before this point (the compiler otherwise sinks
// accumulations to their last use and keeps their operands in registers)
template <int N>
ZFV_HD void computed_here(double *v) {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
  for (int k = 0; k < N; ++k) asm volatile("" : "+v"(v[k]));
#else
  (void)v;
#endif
}

// two adjacent doubles, one 16-byte load
struct alignas(16) PPair {
  double lo, hi;
};

// an interior face's two cell-face slots (left, right), one 8-byte load
struct alignas(8) SlotPair {
  int32_t l, r;
};

// a cell's four face words (face id << 2 | exterior << 1 | side), one load
struct alignas(16) FaceWords {
  int32_t w[4];
};
ZFV_HD FaceWords load_face_words(const Img &m, int64_t i) { return reinterpret_cast<const FaceWords *>(m.cface)[i]; }

// ---- gravity -----------------------------------------------------------------
// PH selects the physics a kernel is compiled for: PH_LIGHT covers no or axial
// gravity with no or isothermal equilibrium (exp only); PH_FULL adds radial
// and polytrope gravity and the isentropic equilibrium.  PH_LIN is PH_FULL
// restricted to the isentropic equilibrium of gamma = 2 with potential
// moments and no periodic images, where a member's equilibrium average needs
// only the member's two potential moments (linear_isentropic_avg), not its
// corners.  The transcendental functions of the full set and the member
// corners need many registers, so runs that do not need them use kernels
// without them.
constexpr int PH_LIGHT = 0;
constexpr int PH_FULL = 1;
constexpr int PH_LIN = 2;

// (an equilibrium of the light set has axial gravity)
template <int DIM>
ZFV_HD double axial_phi(const Img &m, const double *x) {
  double d = x[0] * m.axis[0] + x[1] * m.axis[1];
  if (DIM == 3) d += x[2] * m.axis[2];
  return m.g * d;
}

// the n = 1 polytrope's potential at radius r.  (A call on the device: the
// member averages' point loops are unrolled many times, and as many copies of
// the sine overflow the instruction cache.)
#if defined(__HIP_DEVICE_COMPILE__)
__device__ __attribute__((noinline))
#endif
inline double polytrope_phi(double rhoC, double K, double G, double r) {
  const double alpha = sqrt(2.0 * 3.14159265358979323846 * G / K);
  const double ce = alpha * (r + 2.2250738585072014e-308);
  return -2.0 * K * rhoC * sin(ce) / ce;
}

template <int DIM, int PH = PH_FULL>
ZFV_HD double phi(const Img &m, const double *x) {
  if (m.gravity == 1) return axial_phi<DIM>(m, x);
  if (PH == PH_LIGHT) return 0.0;
  double r2 = x[0] * x[0] + x[1] * x[1];
  if (DIM == 3) r2 += x[2] * x[2];
  double r = sqrt(r2);
  if (m.gravity == 2) return m.g * r;
  if (m.gravity == 3) return polytrope_phi(m.rhoC, m.K, m.G, r);
  return 0.0;
}

template <int DIM, int PH = PH_FULL>
ZFV_HD void grad_phi(const Img &m, const double *x, double *gp) {
  if (m.gravity == 1 || PH == PH_LIGHT) {
    for (int d = 0; d < DIM; ++d) gp[d] = m.gravity == 1 ? m.g * m.axis[d] : 0.0;
    return;
  }
  double r2 = x[0] * x[0] + x[1] * x[1];
  if (DIM == 3) r2 += x[2] * x[2];
  double r = sqrt(r2);
  double dd = 0.0;
  if (m.gravity == 2) {
    dd = m.g;
  } else if (m.gravity == 3) {
    double alpha = sqrt(2.0 * 3.14159265358979323846 * m.G / m.K);
    double ce = alpha * (r + 2.2250738585072014e-308);
    double dphi = (cos(ce) - sin(ce) / ce) / ce;
    dd = -2.0 * m.K * m.rhoC * dphi * alpha;
  }
  for (int d = 0; d < DIM; ++d) gp[d] = dd * (x[d] / (r + 1e-50));
}

// ---- local equilibrium: theta -> (rho, E) at x ------------------------------
// With the per-cell constants taken out of the point loops: isentropic (the
// reference's) a = (1/K)(gamma-1)/gamma and b = 1/(gamma-1); isothermal (an
// extension) a = -1/RT and b = RT/(gamma-1).
struct EqC {
  double th0, th1, phi_ref, a, b;
};

template <int PH>
ZFV_HD EqC eq_consts(const Img &m, const double *th, double phi_ref) {
  EqC c;
  c.th0 = th[0];
  c.th1 = th[1];
  c.phi_ref = phi_ref;
  if (PH == PH_LIN) {  // gamma = 2
    c.a = 1.0 / th[1] * 0.5;
    c.b = 1.0;
  } else if (PH != PH_LIGHT && m.eq == 1) {
    c.a = 1.0 / th[1] * (m.gamma - 1.0) / m.gamma;
    c.b = 1.0 / (m.gamma - 1.0);
  } else {
    c.a = -1.0 / th[1];
    c.b = th[1] / (m.gamma - 1.0);
  }
  return c;
}

// x^y with the exponents an ideal gas of gamma = 2 (the n = 1 polytrope)
// produces, 1 and 2, done exactly (x^1 = x; x^2 is one correctly rounded
// product); any other exponent goes to pow.  (A call: the equilibrium's point
// loops are unrolled many times, and as many copies of pow overflow the
// instruction cache.)
#if defined(__HIP_DEVICE_COMPILE__)
__device__ __attribute__((noinline)) inline double pow_call(double x, double y) { return pow(x, y); }
#else
inline double pow_call(double x, double y) { return pow(x, y); }
#endif
ZFV_HD double ipow(double x, double y) {
  if (y == 1.0) return x;
  if (y == 2.0) return x * x;
  return pow_call(x, y);
}

// x^(1/(gamma-1)).  For the common gases (gamma = 7/5, 5/3, 4/3, 3/2, 2 ...)
// the exponent is a half of a small whole number up to its last place: a
// product of a few factors and a square root, their rounding errors (e, fe)
// summed beside them, and the last place as a first order correction.  To half a
// place, as pow is (the bare products: up to 2.2 places).  The correction is
// below 1e-13 of the result, so that a single precision logarithm adds less than
// 1e-19 to the error.
ZFV_HD double eq_pow(const Img &m, double x, double b) {
  // (no factor or rounding error leaves the range of a double)
  if (m.eq_half > 0 && x > 1.0e-10 && x < 1.0e10) {
    int k = m.eq_half >> 1;
    double r = 1.0, e = 0.0;
    if (m.eq_half & 1) {
      r = sqrt(x);
      if (k > 0) {
        // sqrt(x) = r + (x - r^2) / (2 r), times x: x / r is r to first order
        const double t = r * x;
        e = fma(0.5 * r, fma(-r, r, x), fma(r, x, -t));
        r = t;
        k -= 1;
      }
    }
    if (k & 1) {
      const double t = r * x;
      e = fma(e, x, fma(r, x, -t));
      r = t;
    }
    double f = x, fe = 0.0;
    while ((k >>= 1) > 0) {
      const double s = f * f;
      fe = fma(f, f, -s) + 2.0 * (f * fe);
      f = s;
      if (k & 1) {
        const double t = r * f;
        e = fma(r, f, -t) + fma(r, fe, e * f);
        r = t;
      }
    }
#if defined(__HIP_DEVICE_COMPILE__)
    const double l = double(__logf(float(x)));
#else
    const double l = double(logf(float(x)));
#endif
    return r + fma(r, m.eq_db * l, e);
  }
  return ipow(x, b);
}

// eq_half and eq_db of a gas (host)
inline void eq_pow_constants(double gamma, int &half, double &db) {
  const double b = 1.0 / (gamma - 1.0);
  const double k = nearbyint(2.0 * b);
  half = 0;
  db = 0.0;
  if (k >= 1.0 && k <= 30.0 && fabs(b - 0.5 * k) <= 8.0 * 2.220446049250313e-16 * b) {
    half = int(k);
    db = b - 0.5 * k;
  }
}

// the equilibrium at a point of potential ph
template <int PH>
ZFV_HD void eq_at_phi(const Img &m, const EqC &c, double ph, double &rho, double &E) {
  if (PH != PH_LIGHT && m.eq == 1) {
    double h = c.th0 + c.phi_ref - ph;
    // PH_LIN has gamma = 2: the exponents are 1 and 2.  Else, with base =
    // a h and rho = base^b: p = K rho^gamma = K rho base, which is
    // (gamma - 1)/gamma rho h, so that E needs no power of its own
    rho = PH == PH_LIN ? c.a * h : eq_pow(m, c.a * h, c.b);
    E = PH == PH_LIN ? c.th1 * (rho * rho) : rho * h / m.gamma;
  } else {
    rho = c.th0 * exp((ph - c.phi_ref) * c.a);
    E = rho * c.b;
  }
}

template <int DIM, int PH>
ZFV_HD void eq_point(const Img &m, const EqC &c, const double *x, double &rho, double &E) {
  eq_at_phi<PH>(m, c, phi<DIM, PH>(m, x), rho, E);
}

// The isentropic equilibrium of an ideal gas with gamma = 2 is linear in the
// potential (rho = (h0 - phi) / (2K), E = K rho^2), so its average over a cell
// needs only the cell's quadrature mean of phi and of its squared deviation:
//   rho_avg = a (A - phim),  E_avg = th1 a^2 ((A - phim)^2 + phiv)
// with a = 1/(2K), A = th0 + phi_ref.  Exact in real arithmetic for the same
// quadrature rule; moments are per cell and time independent.
ZFV_HD bool linear_isentropic(const Img &m) { return m.eq == 1 && m.gamma == 2.0 && m.phim != nullptr; }

// the narrowest physics set whose kernel covers this instance
inline int physics_set(const Img &m) {
  if ((m.eq == 0 || m.eq == 2) && (m.gravity == 0 || m.gravity == 1)) return PH_LIGHT;
  if (linear_isentropic(m)) {
    bool shifted = false;  // a periodic image among the stencil members
    for (int c = 1; c < 16; ++c)
      for (int d = 0; d < 3; ++d) shifted = shifted || m.shift[c][d] != 0.0;
    if (!shifted) return PH_LIN;
  }
  return PH_FULL;
}

// the physics set of a kernel that runs instances of sets a and b
inline int physics_union(int a, int b) { return a == b ? a : PH_FULL; }

ZFV_HD void linear_isentropic_avg(const EqC &c, double phim, double phiv, double &ar, double &aE) {
  const double h = c.th0 + c.phi_ref - phim;
  ar = c.a * h;
  aE = c.th1 * (c.a * c.a) * (h * h + phiv);
}

// ---- geometry helpers ---------------------------------------------------------
// Corners are stored per cell, vertex by vertex, each vertex on 16 bytes:
// 2D (x, y), 3D (x, y, z, 0); corner_words doubles per cell
template <int DIM>
constexpr int corner_words() { return DIM == 2 ? 6 : 16; }

// vertex c of cell i
template <int DIM>
ZFV_HD void load_corner(const Img &m, int64_t i, int c, double *w) {
  const PPair *p = reinterpret_cast<const PPair *>(m.crn + i * corner_words<DIM>());
  if (DIM == 2) {
    const PPair a = p[c];
    w[0] = a.lo;
    w[1] = a.hi;
    w[2] = 0.0;
  } else {
    const PPair a = p[2 * c], b = p[2 * c + 1];
    w[0] = a.lo;
    w[1] = a.hi;
    w[2] = b.lo;
  }
}

// The centre (2D x y, 3D x y z 0) and the moments (indices 3 .. DOFC-1,
// padded to an even count) are stored per cell as well, in 16-byte pieces
template <int DIM>
constexpr int centre_words() { return DIM == 2 ? 2 : 4; }
template <int DOFC>
constexpr int moment_words() { return ((DOFC > 3 ? DOFC - 3 : 0) + 1) & ~1; }

template <int DIM>
ZFV_HD void load_centre(const Img &m, int64_t i, double *xc) {
  const PPair *p = reinterpret_cast<const PPair *>(m.xc + i * centre_words<DIM>());
  const PPair a = p[0];
  xc[0] = a.lo;
  xc[1] = a.hi;
  xc[2] = DIM == 3 ? p[1].lo : 0.0;
}

// cm[alpha] for alpha < DOFC: zero below 3, the cell's moments from 3 on
template <int DOFC>
ZFV_HD void load_moments(const Img &m, int64_t i, double *cm) {
  constexpr int MW = moment_words<DOFC>();
  for (int al = 0; al < DOFC && al < 3; ++al) cm[al] = 0.0;
  if (MW > 0) {
    const PPair *p = reinterpret_cast<const PPair *>(m.mom + i * MW);
    for (int k = 0; k < MW / 2; ++k) {
      const PPair v = p[k];
      if (3 + 2 * k < DOFC) cm[3 + 2 * k] = v.lo;
      if (4 + 2 * k < DOFC) cm[4 + 2 * k] = v.hi;
    }
  }
}

template <int DIM>
ZFV_HD void load_corners(const Img &m, int64_t i, double (*v)[3]) {
  for (int k = 0; k < DIM + 1; ++k) load_corner<DIM>(m, i, k, v[k]);
}

// vertices of local face f in the order of the face's left cell
template <int DIM>
ZFV_HD void face_vertices(uint32_t fperm, int f, const double (*v)[3], double (*w)[3]) {
  for (int r = 0; r < DIM; ++r) {
    int c = (fperm >> (2 * (f * 3 + r))) & 3u;
    w[r][0] = v[c][0];
    w[r][1] = v[c][1];
    w[r][2] = v[c][2];
  }
}

// Corner t of a cell's local face f, in the cell's own order (the GMSH tables;
// outward by the right-hand rule for the cells' standard vertex order)
template <int DIM>
ZFV_HD constexpr int face_corner(int f, int t) {
  if (DIM == 2) return (f + t) % 3;
  constexpr int tab[4][3] = {{0, 1, 3}, {0, 2, 1}, {0, 3, 2}, {1, 2, 3}};
  return tab[f][t];
}

// A face's quadrature points numbered along the cell's own vertex order of the
// face, and the number of the same point in the face's left cell's order
// (fperm): the rules are symmetric, so an edge's points run backwards in the
// other direction, and a triangle's points beyond the Q mod 3 central ones
// each belong to one vertex.
template <int DIM, int Q>
ZFV_HD int face_point_in_left_order(uint32_t fperm, int f, int q) {
  if (DIM == 2) return int((fperm >> (6 * f)) & 3u) == f ? q : Q - 1 - q;
  constexpr int C = Q % 3;
  if (q < C) return q;
  const int t = (q - C) % 3, own = face_corner<3>(f, t);
  const int pos = int((fperm >> (6 * f + 2)) & 3u) == own ? 1 : (int((fperm >> (6 * f + 4)) & 3u) == own ? 2 : 0);
  return q - t + pos;
}

// Face normal (src/zisa/math/face_factory.cpp:11-34) and measure (edge length /
// Heron area).  (The fluxes are formed in the global frame and need no
// tangents.)
template <int DIM>
ZFV_HD void face_frame(const double (*w)[3], double *n, double &area) {
  if (DIM == 2) {
    double dx = w[1][0] - w[0][0], dy = w[1][1] - w[0][1];
    double l = sqrt(dx * dx + dy * dy);
    area = l;
    n[0] = dy / l;
    n[1] = -(dx / l);
    n[2] = 0.0;
  } else {
    double a[3] = {w[1][0] - w[0][0], w[1][1] - w[0][1], w[1][2] - w[0][2]};
    double b[3] = {w[2][0] - w[0][0], w[2][1] - w[0][1], w[2][2] - w[0][2]};
    double c[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]};
    double lc = sqrt(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
    n[0] = c[0] / lc;
    n[1] = c[1] / lc;
    n[2] = c[2] / lc;
    // Heron on the side lengths (src/zisa/math/triangle.cpp:11-18)
    double e0[3] = {w[1][0] - w[2][0], w[1][1] - w[2][1], w[1][2] - w[2][2]};
    double e1[3] = {w[0][0] - w[2][0], w[0][1] - w[2][1], w[0][2] - w[2][2]};
    double sa = sqrt(e0[0] * e0[0] + e0[1] * e0[1] + e0[2] * e0[2]);
    double sb = sqrt(e1[0] * e1[0] + e1[1] * e1[1] + e1[2] * e1[2]);
    double sc = sqrt(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]);
    double s = 0.5 * (sa + sb + sc);
    area = sqrt(s * (s - sa) * (s - sb) * (s - sc));
  }
}

// Face normals are time independent: each cell's local faces keep theirs and
// the face measures in a table written once at setup (store_face_frames, with
// face_frame itself), DIM + 1 doubles per face, and the interior faces' (the
// left cell's view) are copied into a table in face order for the fluxes
// (store_face_table); the flux BC reads a cell's own.
template <int DIM>
constexpr int frame_words() { return DIM + 1; }
// doubles of one cell-face slot of face-point values: Q x NV rounded up to
// even, so that every slot starts on 16 bytes
template <int DIM, int Q>
constexpr int slot_doubles() { return (Q * (DIM + 2) + 1) & ~1; }

// writes the light set's potential values of cell i (Img::cphi; tab: (d + 1) n)
template <int DIM>
ZFV_HD void store_cell_phi(const Img &m, int64_t i, double *tab) {
  double v[DIM + 1][3], p[DIM + 1];
  load_corners<DIM>(m, i, v);
  for (int k = 0; k < DIM + 1; ++k) p[k] = phi<DIM, PH_LIGHT>(m, v[k]);
  if (DIM == 2) {
    const double mean = (p[0] + p[1] + p[2]) / 3.0;
    double p2 = 0.0, p3 = 0.0;
    for (int k = 0; k < 3; ++k) {
      const double d = p[k] - mean;
      p2 = fma(d, d, p2);
      p3 = fma(d * d, d, p3);
    }
    p[0] = mean;
    p[1] = p2;
    p[2] = p3;
  }
  for (int k = 0; k < DIM + 1; ++k) tab[i * (DIM + 1) + k] = p[k];
}
// (the emulation's name for it)
template <int DIM>
ZFV_HD void store_corner_phi(const Img &m, int64_t i, double *tab) { store_cell_phi<DIM>(m, i, tab); }

// ---- the isothermal average over a triangle as a series ----------------------
// With an affine potential the average of exp(a (phi - mean)) over a cell,
// sum_q w_q exp(a d_q), depends on the three corner deviations d_k (sum zero)
// only.  The rules' points come in classes (alpha, beta, beta) of three, at
// d = (alpha - beta) d_k, and single centroids at d = 0, so
//   sum_q w_q exp(a d_q) = W + sum_{k >= 2} C_k y_k,
//   C_k = sum_q w_q (alpha_q - beta_q)^k / (3 k!),   y_k = a^k sum_j d_j^k,
// and, the sum of the d_j being zero, Newton's identities give every power sum
// from y_2 and y_3: twelve multiply-adds up to the ninth order instead of an
// exponential a point.  For y_2 <= kSeriesMaxY2 (|a d| <= 0.125, of which the
// rules' points reach at most 0.73) the terms left out are below 1e-17.
constexpr double kSeriesMaxY2 = 0.0234;
// exp_near reaches full accuracy to this argument
constexpr double kSeriesMaxArg = 0.25;

// the constants (es) of the instance's volume rule; false: not of that form
inline bool exp_average_constants(const Img &m, double *es) {
  double W = 0.0, C[10] = {0};
  for (int q = 0; q < m.qv; ++q) {
    const double *x = m.vx[q];
    double s;
    if (x[0] == x[1] && x[1] == x[2]) s = 0.0;
    else if (x[1] == x[2]) s = x[0] - x[1];
    else if (x[0] == x[2]) s = x[1] - x[0];
    else if (x[0] == x[1]) s = x[2] - x[0];
    else return false;
    W = q == 0 ? m.vw[q] : W + m.vw[q];
    double t = m.vw[q] / 3.0;
    for (int k = 1; k < 10; ++k) {
      t = t * s / k;
      C[k] += t;
    }
  }
  const double v[12] = {W,        C[2],          C[3],          C[4] / 2,      5 * C[5] / 6, C[6] / 4,
                        C[6] / 3, 7 * C[7] / 12, C[8] / 8,      4 * C[8] / 9,  3 * C[9] / 8, C[9] / 9};
  for (int k = 0; k < 12; ++k) es[k] = v[k];
  return true;
}

ZFV_HD double exp_average(const Img &m, double y2, double y3) {
  const double *e = m.es;
  const double s0 = fma(y2, fma(y2, fma(y2, fma(y2, e[8], e[5]), e[3]), e[1]), e[0]);
  const double s2 = fma(y3, e[11], fma(y2, e[9], e[6]));
  const double s1 = fma(y3, s2, fma(y2, fma(y2, fma(y2, e[10], e[7]), e[4]), e[2]));
  return fma(y3, s1, s0);
}

// exp(z) for |z| <= kSeriesMaxArg, to the last place or so: its Taylor
// polynomial of degree 12 (the first term left out is below 3e-18)
ZFV_HD double exp_near(double z) {
  double r = 1.0 / 479001600;
  r = fma(r, z, 1.0 / 39916800);
  r = fma(r, z, 1.0 / 3628800);
  r = fma(r, z, 1.0 / 362880);
  r = fma(r, z, 1.0 / 40320);
  r = fma(r, z, 1.0 / 5040);
  r = fma(r, z, 1.0 / 720);
  r = fma(r, z, 1.0 / 120);
  r = fma(r, z, 1.0 / 24);
  r = fma(r, z, 1.0 / 6);
  r = fma(r, z, 0.5);
  r = fma(r, z, 1.0);
  return fma(r, z, 1.0);
}

// writes the normals of cell i's local faces (tab has frame_words (d+1) n entries)
template <int DIM>
ZFV_HD void store_face_frames(const Img &m, int64_t i, double *tab) {
  constexpr int W = frame_words<DIM>();
  double vtx[DIM + 1][3];
  load_corners<DIM>(m, i, vtx);
  const uint32_t fperm = m.fperm[i];
  for (int f = 0; f < DIM + 1; ++f) {
    double w3[3][3], n[3], area;
    face_vertices<DIM>(fperm, f, vtx, w3);
    face_frame<DIM>(w3, n, area);
    double *p = tab + int64_t(f * W) * m.n + i;
    for (int d = 0; d < DIM; ++d) p[int64_t(d) * m.n] = n[d];
    p[int64_t(DIM) * m.n] = area;
  }
}

template <int DIM>
ZFV_HD void load_face_frame(const Img &m, int64_t i, int f, double *n, double &area) {
  constexpr int W = frame_words<DIM>();
  const double *p = m.frm + int64_t(f * W) * m.n + i;
  for (int d = 0; d < DIM; ++d) n[d] = p[int64_t(d) * m.n];
  area = p[int64_t(DIM) * m.n];
}

// the outward normal of cell i's face f times its area (3D; the area and the
// normal of its frame table entry, so that the well-balanced source's face
// term and the fluxes see the same values)
ZFV_HD void face_normal_out(const Img &m, int64_t i, int f, double *an) {
  double n[3], area, c[4][3], xc[3] = {0.0, 0.0, 0.0};
  load_face_frame<3>(m, i, f, n, area);
  load_corners<3>(m, i, c);
  // (the sign against the vector from the cell's mean corner to the face's)
  for (int k = 0; k < 4; ++k)
    for (int d = 0; d < 3; ++d) xc[d] += 0.25 * c[k][d];
  double dd = 0.0;
  for (int d = 0; d < 3; ++d) {
    const double fc = (c[face_corner<3>(f, 0)][d] + c[face_corner<3>(f, 1)][d] + c[face_corner<3>(f, 2)][d]) / 3.0;
    dd += n[d] * (fc - xc[d]);
  }
  for (int d = 0; d < 3; ++d) an[d] = (dd < 0.0 ? -area : area) * n[d];
}

// writes the outward area normals of cell i's faces (tab: 12 n)
ZFV_HD void store_face_normals(const Img &m, int64_t i, double *tab) {
  for (int f = 0; f < 4; ++f) face_normal_out(m, i, f, tab + 12 * i + 3 * f);
}

// Per interior face its normal and area in face order, each face's values
// contiguous: written once at setup from the left cell's table entry
template <int DIM>
ZFV_HD void store_face_table(const Img &m, int64_t e, double *tab) {
  constexpr int NF = DIM + 1;
  const int64_t s = m.fslot[2 * e];
  double n[3], area;
  load_face_frame<DIM>(m, s / NF, int(s % NF), n, area);
  for (int d = 0; d < DIM; ++d) tab[e * (DIM + 1) + d] = n[d];
  tab[e * (DIM + 1) + DIM] = area;
}

template <int DIM>
ZFV_HD void face_table_frame(const Img &m, int64_t e, double *n, double &area) {
  const double *p = m.ffr + e * (DIM + 1);
  for (int d = 0; d < DIM; ++d) n[d] = p[d];
  area = p[DIM];
}

// quadrature point q of a face given its vertices in left-cell order
template <int DIM>
ZFV_HD void face_point(const Img &m, int q, const double (*w)[3], double *x) {
  if (DIM == 2) {
    double xi = m.fx[q][0];
    double a = 0.5 - 0.5 * xi, b = 0.5 + 0.5 * xi;
    x[0] = fma(b, w[1][0], a * w[0][0]);
    x[1] = fma(b, w[1][1], a * w[0][1]);
    x[2] = 0.0;
  } else {
    for (int d = 0; d < 3; ++d) x[d] = (m.fx[q][0] * w[0][d] + m.fx[q][1] * w[1][d]) + m.fx[q][2] * w[2][d];
  }
}

template <int DIM>
ZFV_HD void volume_point(const Img &m, int q, const double (*v)[3], double *x) {
  for (int d = 0; d < DIM; ++d) {
    double s = m.vx[q][0] * v[0][d];
    for (int k = 1; k < DIM + 1; ++k) s = fma(m.vx[q][k], v[k][d], s);
    x[d] = s;
  }
  if (DIM == 2) x[2] = 0.0;
}

// Quadrature mean of the potential over cell i and mean squared deviation
// from it (for linear_isentropic_avg)
template <int DIM>
ZFV_HD void phi_moments(const Img &m, int64_t i, double &mean, double &var) {
  double vtx[DIM + 1][3];
  load_corners<DIM>(m, i, vtx);
  double s = 0.0;
  for (int q = 0; q < m.qv; ++q) {
    double x[3];
    volume_point<DIM>(m, q, vtx, x);
    const double p = phi<DIM, PH_FULL>(m, x);
    s = (q == 0) ? m.vw[q] * p : s + m.vw[q] * p;
  }
  double v = 0.0;
  for (int q = 0; q < m.qv; ++q) {
    double x[3];
    volume_point<DIM>(m, q, vtx, x);
    const double d = phi<DIM, PH_FULL>(m, x) - s;
    v = (q == 0) ? m.vw[q] * (d * d) : v + m.vw[q] * (d * d);
  }
  mean = s;
  var = v;
}

// Potential tables.  Radial and polytrope gravity have no affine closed form,
// and the potential at a cell's own quadrature points does not change in time,
// so instances of the full physics sets with gravity keep it per cell,
// computed once with the functions above:
//   pot[i (DIM + 1) Q + f Q + q]         phi at point q of local face f (the
//                                        cell's own vertex order), each cell's
//                                        contiguous
//   pot[((DIM + 1) Q + q) n + i]         phi at volume point q (q < qv)
// The reconstruction then evaluates no transcendental function at its own
// points; the values are those the functions give at the same points.
template <int DIM>
ZFV_HD int64_t pot_index_vol(const Img &m, int nqf, int q) { return (int64_t(DIM + 1) * nqf + q) * m.n; }
// rows of the tables for nqf face points
template <int DIM>
ZFV_HD int pot_rows(int qv, int nqf) { return qv + (DIM + 1) * nqf; }

// fills the potential tables of cell i (tab has pot_rows * n entries)
template <int DIM>
ZFV_HD void potential_points(const Img &m, int nqf, int64_t i, double *tab) {
  double vtx[DIM + 1][3];
  load_corners<DIM>(m, i, vtx);
  for (int q = 0; q < m.qv; ++q) {
    double x[3];
    volume_point<DIM>(m, q, vtx, x);
    tab[pot_index_vol<DIM>(m, nqf, q) + i] = phi<DIM, PH_FULL>(m, x);
  }
  for (int f = 0; f < DIM + 1; ++f) {
    double w3[3][3];
    for (int t = 0; t < DIM; ++t)
      for (int d = 0; d < 3; ++d) w3[t][d] = vtx[face_corner<DIM>(f, t)][d];
    for (int q = 0; q < nqf; ++q) {
      double x[3];
      face_point<DIM>(m, q, w3, x);
      tab[i * int64_t((DIM + 1) * nqf) + f * nqf + q] = phi<DIM, PH_FULL>(m, x);
    }
  }
}

// ---- polynomial evaluation (include/zisa/math/poly2d_impl.hpp:271-323) -------
// a[alpha][v] for alpha < DOF, c = moments (0 for alpha < 3).  (The basis
// functions one by one, for setup and checks; the kernels use poly_nested.)
template <int DIM, int DEG, int NV>
ZFV_HD void poly_eval(const double (*a)[NV], const double *c, const double *X, double *px) {
  for (int v = 0; v < NV; ++v) px[v] = 0.0;
  double pxk = 1.0;
#pragma unroll
  for (int kx = 0; kx <= DEG; ++kx) {
    double pyk = 1.0;
#pragma unroll
    for (int ky = 0; ky <= DEG - kx; ++ky) {
      if (DIM == 2) {
        const int n = kx + ky;
        const int i = (n + 1) * n / 2 + ky;
        const double b = fma(pxk, pyk, -c[i]);
#pragma unroll
        for (int v = 0; v < NV; ++v) px[v] = fma(a[i][v], b, px[v]);
      } else {
        double pzk = 1.0;
#pragma unroll
        for (int kz = 0; kz <= DEG - kx - ky; ++kz) {
          const int n3 = kx + ky + kz - 1;
          const int d3 = n3 < 0 ? 0 : (n3 + 1) * (n3 + 2) * (n3 + 3) / 6;
          const int n2 = ky + kz;
          const int i = d3 + (n2 + 1) * n2 / 2 + kz;
          const double b = fma(pxk * pyk, pzk, -c[i]);
#pragma unroll
          for (int v = 0; v < NV; ++v) px[v] = fma(a[i][v], b, px[v]);
          pzk *= X[2];
        }
      }
      pyk *= X[1];
    }
    pxk *= X[0];
  }
}

// sum_alpha a[alpha] X^alpha in nested form (one multiply-add per
// coefficient past the first)
template <int DIM, int DEG>
ZFV_HD double poly_nested(const double *a, const double *X) {
  double rx = 0.0;
#pragma unroll
  for (int kx = DEG; kx >= 0; --kx) {
    double ry = 0.0;
#pragma unroll
    for (int ky = DEG - kx; ky >= 0; --ky) {
      if (DIM == 2) {
        const int n = kx + ky;
        const double c = a[(n + 1) * n / 2 + ky];
        ry = ky == DEG - kx ? c : fma(ry, X[1], c);
      } else {
        double rz = 0.0;
#pragma unroll
        for (int kz = DEG - kx - ky; kz >= 0; --kz) {
          const int n3 = kx + ky + kz - 1;
          const int d3 = n3 < 0 ? 0 : (n3 + 1) * (n3 + 2) * (n3 + 3) / 6;
          const int n2 = ky + kz;
          const double c = a[d3 + (n2 + 1) * n2 / 2 + kz];
          rz = kz == DEG - kx - ky ? c : fma(rz, X[2], c);
        }
        ry = ky == DEG - kx ? rz : fma(ry, X[1], rz);
      }
    }
    rx = kx == DEG ? ry : fma(rx, X[0], ry);
  }
  return rx;
}

// the basis of poly_eval at X, in its order: b[i] = X^alpha_i - c[i]
template <int DIM, int DEG>
ZFV_HD void poly_basis(const double *c, const double *X, double *b) {
  double pxk = 1.0;
#pragma unroll
  for (int kx = 0; kx <= DEG; ++kx) {
    double pyk = 1.0;
#pragma unroll
    for (int ky = 0; ky <= DEG - kx; ++ky) {
      if (DIM == 2) {
        const int n = kx + ky;
        b[(n + 1) * n / 2 + ky] = fma(pxk, pyk, -c[(n + 1) * n / 2 + ky]);
      } else {
        double pzk = 1.0;
#pragma unroll
        for (int kz = 0; kz <= DEG - kx - ky; ++kz) {
          const int n3 = kx + ky + kz - 1;
          const int d3 = n3 < 0 ? 0 : (n3 + 1) * (n3 + 2) * (n3 + 3) / 6;
          const int n2 = ky + kz;
          const int i = d3 + (n2 + 1) * n2 / 2 + kz;
          b[i] = fma(pxk * pyk, pzk, -c[i]);
          pzk *= X[2];
        }
      }
      pyk *= X[1];
    }
    pxk *= X[0];
  }
}

template <int DIM>
constexpr int dof_of(int deg) {
  return DIM == 2 ? (deg + 1) * (deg + 2) / 2 : (deg + 1) * (deg + 2) * (deg + 3) / 6;
}

template <int DIM>
constexpr int deg_of(int dof) {
  int d = 0;
  while (dof_of<DIM>(d + 1) <= dof) ++d;
  return d;
}

// The gravity source moments of cell i: M[alpha][d] = vol sum_q vw_q
// b_alpha(x_q) d_d phi(x_q) with the volume rule, the polynomial basis of the
// cell's reconstruction (poly_basis) and the potential's gradient at the
// points.  The volume terms of the source, sum_q w_q delta(x_q) d_d phi(x_q)
// for delta = scale sum_alpha a_alpha b_alpha, are then scale sum_alpha
// a_alpha M[alpha][d]: the same quadrature, summed over the points once at
// setup instead of per call.
template <int DIM, int DOFC>
ZFV_HD void store_source_moments(const Img &m, int64_t i, double *tab) {
  constexpr int DEG = deg_of<DIM>(DOFC);
  const int64_t n = m.n;
  double vtx[DIM + 1][3];
  load_corners<DIM>(m, i, vtx);
  double cm[DOFC];
  load_moments<DOFC>(m, i, cm);
  double xc[3];
  load_centre<DIM>(m, i, xc);
  const double inv_len = 1.0 / m.len[i];
  const double vol_i = m.vol[i];
  double acc[DOFC][DIM];
  for (int q = 0; q < m.qv; ++q) {
    double x[3], gp[3], b[DOFC];
    volume_point<DIM>(m, q, vtx, x);
    grad_phi<DIM, PH_FULL>(m, x, gp);
    const double Xs[3] = {(x[0] - xc[0]) * inv_len, (x[1] - xc[1]) * inv_len,
                          DIM == 3 ? (x[2] - xc[2]) * inv_len : 0.0};
    poly_basis<DIM, DEG>(cm, Xs, b);
    const double w = vol_i * m.vw[q];
    for (int al = 0; al < DOFC; ++al)
      for (int d = 0; d < DIM; ++d) acc[al][d] = (q == 0) ? w * (b[al] * gp[d]) : fma(w, b[al] * gp[d], acc[al][d]);
  }
  for (int al = 0; al < DOFC; ++al)
    for (int d = 0; d < DIM; ++d) tab[int64_t(i) * (DOFC * DIM) + al * DIM + d] = acc[al][d];
}

// ---- ideal gas / fluxes -------------------------------------------------------
// States (rho, momentum (DIM), E) in the global frame; n: the face's unit
// normal.  A flux in direction n needs the momentum's normal part and its
// length only, so no state is turned into a face frame and no flux back.

// What both fluxes need of a state: one division by the density serves the
// velocity, the pressure and the sound speed.  (The fluxes were bound by
// arithmetic, and a double precision division is some 14 instructions: 20 a
// point before, 5 now.)
template <int DIM>
struct FaceState {
  double r, mn, vn, p, a;  // 1/rho, momentum and velocity along n, pressure, sound speed
};
template <int DIM>
ZFV_HD FaceState<DIM> face_state(const double *u, const double *n, double gamma) {
  FaceState<DIM> s;
  s.r = 1.0 / u[0];
  s.mn = u[1] * n[0] + u[2] * n[1];
  double m2 = u[1] * u[1] + u[2] * u[2];
  if (DIM == 3) {
    s.mn += u[3] * n[2];
    m2 += u[3] * u[3];
  }
  s.vn = s.mn * s.r;
  s.p = (u[DIM + 1] - 0.5 * (m2 * s.r)) * (gamma - 1.0);
  s.a = sqrt(gamma * s.p * s.r);
  return s;
}

// the physical flux in direction n
template <int DIM>
ZFV_HD void euler_flux(const double *u, const FaceState<DIM> &s, const double *n, double *f) {
  f[0] = s.mn;
  for (int d = 0; d < DIM; ++d) f[1 + d] = s.vn * u[1 + d] + s.p * n[d];
  f[DIM + 1] = s.vn * (u[DIM + 1] + s.p);
}

template <int DIM>
ZFV_HD void hllc(const double *uL, const double *uR, const double *n, double gamma, double *nf) {
  constexpr int NV = DIM + 2;
  const FaceState<DIM> L = face_state<DIM>(uL, n, gamma), R = face_state<DIM>(uR, n, gamma);
  const double roe_ratio = sqrt(uR[0] * L.r);
  const double inv1 = 1.0 / (1.0 + roe_ratio);
  auto mean = [&](double x, double y) { return (x + y * roe_ratio) * inv1; };
  const double H = mean((uL[NV - 1] + L.p) * L.r, (uR[NV - 1] + R.p) * R.r);
  const double v = mean(L.vn, R.vn);
  double vroe = 0.0;
  for (int d = 0; d < DIM; ++d) {
    const double w = mean(uL[1 + d] * L.r, uR[1 + d] * R.r);
    vroe = d == 0 ? w * w : vroe + w * w;
  }
  const double a = sqrt((gamma - 1.0) * (H - 0.5 * vroe));
  const double sL = dmin(L.vn - L.a, v - a);
  const double sR = dmax(R.vn + R.a, v + a);
  const double s_star = (R.mn * (sR - R.vn) - L.mn * (sL - L.vn) + L.p - R.p) /
                        (uR[0] * (sR - R.vn) - uL[0] * (sL - L.vn));
  const bool left = 0.0 <= s_star;
  FaceState<DIM> K;
  K.mn = left ? L.mn : R.mn;
  K.vn = left ? L.vn : R.vn;
  K.p = left ? L.p : R.p;
  double uK[NV];
  for (int k = 0; k < NV; ++k) uK[k] = left ? uL[k] : uR[k];
  euler_flux<DIM>(uK, K, n, nf);
  if (sL < 0.0 && 0.0 <= sR) {
    // sK times the star state's difference from the cell's, with w = (s_star -
    // vK) / (sK - s_star): w (rho, m + rho (sK - vK) n, E + pK + rho (sK - vK)
    // s_star).  (The star state less the cell's, term by term, cancels.)
    const double sK = left ? sL : sR;
    const double w = sK * ((s_star - K.vn) / (sK - s_star)), r = uK[0] * (sK - K.vn);
    nf[0] += w * uK[0];
    for (int d = 0; d < DIM; ++d) nf[1 + d] += w * (uK[1 + d] + r * n[d]);
    nf[NV - 1] += w * (uK[NV - 1] + K.p + r * s_star);
  }
}

template <int DIM>
ZFV_HD void rusanov(const double *uL, const double *uR, const double *n, double gamma, double *f) {
  constexpr int NV = DIM + 2;
  const FaceState<DIM> L = face_state<DIM>(uL, n, gamma), R = face_state<DIM>(uR, n, gamma);
  const double s = dmax(fabs(L.vn) + L.a, fabs(R.vn) + R.a);
  double fL[NV], fR[NV];
  euler_flux<DIM>(uL, L, n, fL);
  euler_flux<DIM>(uR, R, n, fR);
  for (int k = 0; k < NV; ++k) f[k] = 0.5 * (fL[k] + fR[k]) - 0.5 * s * (uR[k] - uL[k]);
}

// ---- the per-cell reconstruction, one lane per conserved variable --------------
//
// Reads the cell's stencil, forms every stencil polynomial with the
// precomputed pseudo-inverses, applies the CWENO correction and the WENO
// weights, then evaluates the result at the quadrature points of the cell's
// interior faces (in the global frame) and, with gravity, computes the cell's
// source term.
//
// A group of NV lanes shares one cell: lane g owns conserved variable g (rho,
// momentum components, energy) and keeps only that variable's polynomial
// coefficients, so a lane needs a fraction of the registers of a whole cell.
// The lanes exchange values through X::bcast(v, k) / X::bcast_i(v, k) (value
// v of lane k of the same group) and through LDS (X::wave_lds(), X::lds()),
// ordered by X::sync():
//   - the equilibrium averages of the stencil members are computed by lane
//     (row mod NV) and read by the density and energy lanes,
//   - the smoothness indicator of a stencil is the maximum over the variables,
//   - the gravity source mixes momentum components.
// Every call of bcast sits in control flow that is uniform over the group.
//
// U: state (state_at).  fpv: per cell-face slot (i * NF + f) its Q x NV
// point values, written for interior faces (one group writes its cell's whole
// block, so cache lines fill within one XCD).  src: as the state, or null.
// LDS of one wavefront: first a row region of wave_lds_doubles holding each
// group's NV rows of row_doubles entries (the NC pseudo-inverse entries, then
// the member's equilibrium averages; group c at c NV row_doubles, an even
// stride that puts the groups' 16-byte reads on different banks; at least 6,
// which holds the exchange of the nonlinear weights), then per
// cell group the members' equilibrium averages: er and eE of each central row,
// for the one-sided rows that share their member, or in the light set er of
// every row (group_lds_doubles; at least the 4 + 3 x 3 rows of 2D second order).
template <int DOFC>
constexpr int row_doubles() { return ((DOFC + 1 + 1) & ~1) > 6 ? ((DOFC + 1 + 1) & ~1) : 6; }
template <int DIM, int DOFC>
constexpr int wave_lds_doubles() { return (64 / (DIM + 2)) * (DIM + 2) * row_doubles<DOFC>(); }
template <int RC>
constexpr int group_lds_doubles() { return 2 * RC > 14 ? 2 * RC : 14; }
template <int DIM, int DOFC, int RC>
constexpr int wave_block_doubles() { return wave_lds_doubles<DIM, DOFC>() + (64 / (DIM + 2)) * group_lds_doubles<RC>(); }

// The pseudo-inverses are stored in tiles of one wavefront's cells (gpw =
// 64 / nv consecutive cells; m gpw doubles a tile, m entries a cell), in the
// order the wavefront reads them: rows in chunks of nv (lane g of a group
// takes row g of the chunk), and within a chunk coefficient pairs (a, a + 1),
// each pair of all the tile's lanes contiguous, so that a load instruction
// reads one piece of 16 bytes a lane and a wavefront streams one contiguous
// tile.  Central rows come first (all pairs, then an odd last coefficient),
// then the one-sided stencils, whose rb rows form a chunk each.  These are
// the places inside a tile of coefficient a of central row r and of row rr of
// one-sided stencil kb, for the tile's cell grp.
ZFV_HD int p_central(int nv, int gpw, int nc, int rc, int a, int r, int grp) {
  const int c = r / nv, g = r - c * nv, np = nc / 2;
  const int vc = rc - c * nv < nv ? rc - c * nv : nv;  // rows of this chunk
  if (a < 2 * np) return 2 * ((c * nv * np + (a >> 1) * vc) * gpw + grp * vc + g) + (a & 1);
  return 2 * np * rc * gpw + c * nv * gpw + grp * vc + g;
}

ZFV_HD int p_onesided(int gpw, int nc, int rc, int nbc, int nb, int rb, int kb, int a, int rr, int grp) {
  const int base = nc * rc * gpw, np = nbc / 2;
  if (a < 2 * np) return base + 2 * ((kb * np + (a >> 1)) * rb * gpw + grp * rb + rr) + (a & 1);
  return base + 2 * np * nb * rb * gpw + (kb * gpw + grp) * rb + rr;
}

// linear isentropic equilibria: the part 4 v / r^2 up to which the solve starts
// from the root.  (Up to here the iteration from the guess leads to that root for
// 6e5 random states, the reference potential up to six standard deviations off
// its mean; from 0.032 on some do not converge.)
constexpr double kRootsApart = 0.02;

template <int DIM, int DOFC, int RC, int NB, int RB, int Q, int PH, class X>
ZFV_HD void reconstruct_lane(const Img &m, int64_t i, const int g, X &xch, const double *__restrict__ U,
                             double *__restrict__ fpv, double *__restrict__ src) {
  constexpr int NV = DIM + 2;
  constexpr int NF = DIM + 1;
  constexpr int NC = DOFC - 1;
  constexpr int NBC = DIM;
  constexpr int DEGC = deg_of<DIM>(DOFC);
  constexpr bool AOS = state_is_aos<X>::value;
  const int64_t n = m.n;
  const double gamma = PH == PH_LIN ? 2.0 : m.gamma;

  // own state and scale (include/zisa/model/characteristic_scale.hpp:23-32)
  double u0[NV];
  for (int v = 0; v < NV; ++v) u0[v] = U[state_at<AOS, NV>(n, v, i)];
  double msq = u0[1] * u0[1] + u0[2] * u0[2];
  if (DIM == 3) msq += u0[3] * u0[3];
  const double rho0 = u0[0];
  const double Eint0 = u0[NV - 1] - 0.5 * msq / rho0;
  // this call's scale (UnityScaling: all ones,
  // include/zisa/model/characteristic_scale.hpp:39-46); a stateful instance
  // may keep the last recompute's
  double sc_rho = rho0, sc_E = Eint0, sc_a = sqrt(gamma * (Eint0 * (gamma - 1.0)) / rho0);
  if (m.scaling == 1) sc_rho = sc_E = sc_a = 1.0;
  const bool is_rho = g == 0, is_E = g == NV - 1;
  // Stencil rows in chunks: lane g owns row c NV + g of central chunk c and
  // row g of each one-sided stencil's chunk.  All row entries and the first
  // chunk's member states are loaded before the equilibrium solve, whose
  // arithmetic then covers their latency (every row entry names a cell,
  // first-order cells included).
  static_assert(RB <= NV, "a one-sided stencil's rows form one chunk");
  constexpr int CCH = (RC + NV - 1) / NV;  // central chunks
  constexpr int NCH = CCH + NB;
  auto chunk_rows = [](int ch) { return ch < CCH ? (RC - ch * NV < NV ? RC - ch * NV : NV) : RB; };
  auto chunk_row0 = [](int ch) { return ch < CCH ? ch * NV : RC + (ch - CCH) * RB; };
  int32_t rw[NCH];
#pragma unroll
  for (int ch = 0; ch < NCH; ++ch) {
    // (a lane past the chunk's rows reads the chunk's last)
    const int rg = g < chunk_rows(ch) ? g : chunk_rows(ch) - 1;
    rw[ch] = m.rows[(chunk_row0(ch) + rg) * n + i];
  }
  // this lane's variable of the members of chunk ch.  (Byte offsets of 32
  // bits: the state of the largest instance that fits is under 4 GiB.)
  auto gather = [&](int ch, double *uk) {
    const int32_t j = rw[ch] & ROW_CELL_MASK;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      if (k >= chunk_rows(ch)) break;
      if (AOS) {
        const uint32_t at = uint32_t(xch.bcast_i(int32_t(uint32_t(j) * uint32_t(NV * 8)), k)) + uint32_t(g) * 8u;
        uk[k] = *reinterpret_cast<const double *>(reinterpret_cast<const char *>(U) + at);
      } else {
        uk[k] = U[state_at<AOS, NV>(n, g, xch.bcast_i(j, k))];
      }
    }
  };
  double uk[NV];
  gather(0, uk);

  // The 2D light set's averages in series form (exp_average) where the
  // exponents over every member of every cell of this wavefront are in range
  constexpr bool SERIES = DIM == 2 && PH == PH_LIGHT;
  const bool wb = PH == PH_LIN || m.eq != 0;

  // The potential at the cell's own quadrature points: from the instance's
  // tables in the full sets (always present in PH_LIN), else evaluated.
  const bool tab = PH == PH_LIN || (PH == PH_FULL && m.pot != nullptr);
  auto vol_phi = [&](int q, const double *x) {
    if (PH == PH_LIGHT) return axial_phi<DIM>(m, x);  // (asked for with an equilibrium only)
    return tab ? m.pot[pot_index_vol<DIM>(m, Q, q) + i] : phi<DIM, PH>(m, x);
  };

  // Average of an equilibrium over this cell with the quadrature points split
  // over the group's lanes: lane k sums the points q = k (mod NV) in order,
  // then every lane adds the NV partial sums in lane order, so all lanes hold
  // the same value.
  auto group_avg = [&](const EqC &tc, double &ar, double &aE) {
    if (PH == PH_LIN || (PH == PH_FULL && linear_isentropic(m))) {
      linear_isentropic_avg(tc, m.phim[2 * i], m.phim[2 * i + 1], ar, aE);
      return;
    }
    const double vol_i = m.vol[i];
    double vtx[DIM + 1][3];
    load_corners<DIM>(m, i, vtx);
    double pr = 0.0, pE = 0.0;
    for (int q = g; q < m.qv; q += NV) {
      double x[3];
      volume_point<DIM>(m, q, vtx, x);
      double r, E;
      eq_at_phi<PH>(m, tc, vol_phi(q, x), r, E);
      const double w = vol_i * m.vw[q];
      pr = pr + w * r;
      pE = pE + w * E;
    }
    double sr = xch.bcast(pr, 0), sE = xch.bcast(pE, 0);
    for (int k = 1; k < NV; ++k) {
      sr = sr + xch.bcast(pr, k);
      sE = sE + xch.bcast(pE, k);
    }
    ar = (1.0 * sr) / vol_i;
    aE = (1.0 * sE) / vol_i;
  };

  // local equilibrium of this cell: every lane solves it (identical results)
  double th[2] = {0.0, 0.0};
  double phi_ref = 0.0;
  // once solved, the equilibrium's average over the cell as the solve has it
  // (isothermal: in ar1 that of exp(a (phi - phi_ref)))
  double ar1 = -1.0, aE1 = 0.0;
  bool eq_found = false;
  double y_p2 = 0.0, y_p3 = 0.0;  // the cell's own power sums (SERIES)
  if (wb) {
    // The potential the equilibrium is written against: the corners' mean for
    // the 2D instances that run in the light set by themselves, else the first
    // volume point's.  (A property of the instance, not of the set it runs in: a
    // kept theta is read by another set when a member of another kind joins or
    // leaves its batch.)
    if (SERIES || (DIM == 2 && PH == PH_FULL && m.cphi != nullptr)) {
      phi_ref = m.cphi[3 * i];
      if (SERIES) {
        y_p2 = m.cphi[3 * i + 1];
        y_p3 = m.cphi[3 * i + 2];
      }
    } else {
      double xref[3], vtx[DIM + 1][3];
      load_corners<DIM>(m, i, vtx);
      volume_point<DIM>(m, 0, vtx, xref);
      phi_ref = vol_phi(0, xref);
    }
  }
  // Stateful equilibria (LocalReconstruction::recompute_equilibrium,
  // include/zisa/reconstruction/local_reconstruction.hpp:87-100): between
  // recomputes (every steps_per_recompute calls) the cell keeps the theta and
  // the scale of its last recompute, unless its (rho, E_int) has moved from
  // the kept equilibrium's own cell average by the threshold or more,
  // measured in the kept scale; a kept equilibrium that was not found
  // averages to zero there.
  int32_t calls = 0;
  bool reuse = false;
  if (m.eqc != nullptr) {
    calls = m.eqcnt[i];
    if (calls % m.spr != 0) {
      const bool kept_found = m.eqc[2 * n + i] != 0.0;
      const double kth[2] = {m.eqc[i], m.eqc[n + i]};
      const double c_rho = m.eqc[3 * n + i], c_a = m.eqc[4 * n + i], c_E = m.eqc[5 * n + i];
      const double er = m.eqc[6 * n + i], eE = m.eqc[7 * n + i];
      const double d0 = (rho0 - er) / c_rho, d1 = (Eint0 - eE) / c_E;
      reuse = !(sqrt(d0 * d0 + d1 * d1) >= m.eq_threshold);
      if (reuse) {
        th[0] = kth[0];
        th[1] = kth[1];
        eq_found = wb && kept_found;
        sc_rho = c_rho;
        sc_a = c_a;
        sc_E = c_E;
      }
    }
  }
  // the series is in range at temperature RT for every cell of the wavefront
  auto series_ok = [&](double RT) {
    const bool ok = m.es_dist > 0.0 && m.es_dist <= kSeriesMaxArg * RT && m.es_p2 <= kSeriesMaxY2 * (RT * RT);
    return wave_all(ok);
  };
  if (wb && !reuse) {
    // cell average of the equilibrium with parameters t over this cell
    auto cell_avg = [&](const double *t, double &ar, double &aE) {
      group_avg(eq_consts<PH>(m, t, phi_ref), ar, aE);
    };
    if (PH == PH_LIGHT || m.eq == 2) {
      double RT = (gamma - 1.0) * Eint0 / rho0;
      double t1[2] = {1.0, RT};
      double ar, aE;
      if (SERIES && series_ok(RT)) {
        const double a1 = -1.0 / RT;
        ar = exp_average(m, a1 * a1 * y_p2, a1 * a1 * a1 * y_p3);
      } else {
        cell_avg(t1, ar, aE);
      }
      ar1 = ar;
      th[0] = rho0 / ar;
      th[1] = RT;
      eq_found = true;
    } else {
      // The reference's quasi-Newton iteration (its guess, tolerance, limits
      // and convergence test: include/zisa/math/quasi_newton.hpp:12-50) with
      // the Jacobian in closed form instead of by central differences, one
      // evaluation an iteration instead of five.  With rho = (a h)^b, E = rho
      // h / gamma, averages R, Eavg and D = avg(rho / h):
      //   dR/dh = b D, dEavg/dh = b R, dR/dK = -b R / K, dEavg/dK = -b Eavg / K
      // (so a step is (E f0 - R f1, K (R f0 - D f1)) / (b (R^2 - D E))).
      const double p = Eint0 * (gamma - 1.0);
      const double guess[2] = {gamma / (gamma - 1.0) * p / rho0, p / (PH == PH_LIN ? rho0 * rho0 : ipow(rho0, gamma))};
      const double atol[2] = {1e-13 * guess[0], 1e-13 * guess[1]};
      double x0 = guess[0], x1 = guess[1];
      const double bexp = PH == PH_LIN ? 1.0 : 1.0 / (gamma - 1.0);
      const bool linear = PH == PH_LIN || linear_isentropic(m);
      // the potential at this lane's volume points q = g (mod NV)
      constexpr int QL = (16 + NV - 1) / NV;
      double phq[PH == PH_LIN ? 1 : QL];
      if (!linear) {
        double vtx[DIM + 1][3];
        load_corners<DIM>(m, i, vtx);
#pragma unroll
        for (int k = 0; k < (PH == PH_LIN ? 1 : QL); ++k) {
          phq[k] = 0.0;
          if (g + k * NV >= m.qv) continue;
          double x[3];
          volume_point<DIM>(m, g + k * NV, vtx, x);
          phq[k] = vol_phi(g + k * NV, x);
        }
      }
      double R, E, D;  // averages of the equilibrium of (x0, x1)
      auto average = [&]() {
        const double t[2] = {x0, x1};
        const EqC tc = eq_consts<PH>(m, t, phi_ref);
        if (linear) {
          linear_isentropic_avg(tc, m.phim[2 * i], m.phim[2 * i + 1], R, E);
          D = tc.a;
          return;
        }
        double pr = 0.0, pE = 0.0, pD = 0.0;
#pragma unroll
        for (int k = 0; k < (PH == PH_LIN ? 1 : QL); ++k) {
          if (g + k * NV >= m.qv) continue;
          double r, e;
          eq_at_phi<PH>(m, tc, phq[k], r, e);
          const double w = m.vw[g + k * NV];
          pr = fma(w, r, pr);
          pE = fma(w, e, pE);
          pD = fma(w, r / (tc.th0 + tc.phi_ref - phq[k]), pD);
        }
        R = xch.bcast(pr, 0);
        E = xch.bcast(pE, 0);
        D = xch.bcast(pD, 0);
#pragma unroll
        for (int k = 1; k < NV; ++k) {
          R = R + xch.bcast(pr, k);
          E = E + xch.bcast(pE, k);
          D = D + xch.bcast(pD, k);
        }
      };
      // For the linear isentropic gas R = u / (2 K), E = R (u + v / u) / 2 with
      // u the enthalpy at the potential's mean and v the potential's variance:
      // u is the larger root of u^2 - (2 E / R) u + v.  Where the roots are well
      // apart the iteration from the guess leads there; it starts from the root
      // instead and ends after the step that confirms it, one step for about
      // four (7,000 of the 66,000 cycles a wavefront of the polytrope n = 40
      // spends; reconstruction 119 -> 113 us a launch).  Near a double root and
      // without one it starts from the guess.
      if (PH == PH_LIN) {
        const double v = m.phim[2 * i + 1], r = guess[0], disc = r * r - 4.0 * v;
        if (r > 0.0 && 4.0 * v <= kRootsApart * (r * r)) {
          const double u = 0.5 * (r + sqrt(disc));
          x0 = u + (m.phim[2 * i] - phi_ref);
          x1 = 0.5 * u / rho0;
        }
      }
      average();
      double fx0 = rho0 - R, fx1 = Eint0 - E;
      double dx0 = 2.0 * atol[0] + 1.0, dx1 = 2.0 * atol[1] + 1.0;
      double h00 = 0, h01 = 0, h10 = 0, h11 = 0;  // previous two steps
      bool ok = true;
      int iter = 0;
      while (!(fabs(dx0) <= atol[0] && fabs(dx1) <= atol[1]) && iter < 20) {
        const double inv_det = 1.0 / (bexp * (R * R - D * E));
        dx0 = inv_det * (E * fx0 - R * fx1);
        dx1 = inv_det * x1 * (R * fx0 - D * fx1);
        x0 -= dx0;
        x1 -= dx1;
        average();
        fx0 = rho0 - R;
        fx1 = Eint0 - E;
        if (iter >= 4 && !(dx0 <= atol[0] && dx1 <= atol[1])) {
          double rate0 = log(fabs(dx0) / fabs(h10)) / log(fabs(h10) / fabs(h00));
          double rate1 = log(fabs(dx1) / fabs(h11)) / log(fabs(h11) / fabs(h01));
          if (!(rate0 >= 0.0) || !(rate1 >= 0.0)) ok = false;
        }
        h00 = h10;
        h01 = h11;
        h10 = dx0;
        h11 = dx1;
        if (!ok) break;
        ++iter;
      }
      if (ok && !(iter == 20 && !(fabs(dx0) <= 1000.0 * atol[0] && fabs(dx1) <= 1000.0 * atol[1]))) {
        th[0] = x0;
        th[1] = x1;
        eq_found = true;
        ar1 = R;
        aE1 = E;
      }
    }
  }
  if (m.eqc != nullptr) {
    xch.sync();  // every lane of the group has read the kept state
  }
  if (m.eqc != nullptr && g == 0) {
    if (!reuse) {
      m.eqc[i] = th[0];
      m.eqc[n + i] = th[1];
      m.eqc[2 * n + i] = eq_found ? 1.0 : 0.0;
      m.eqc[3 * n + i] = sc_rho;
      m.eqc[4 * n + i] = sc_a;
      m.eqc[5 * n + i] = sc_E;
    }
    m.eqcnt[i] = reuse ? calls + 1 : 1;
  }
  const double scale_g = g == 0 ? sc_rho : (g == NV - 1 ? sc_E : sc_a);
  const double inv_g = 1.0 / scale_g;

  // (without an equilibrium, constants that evaluate to zero everywhere, so
  // that its evaluations need no branch)
  const bool eq_sub = wb && eq_found;
  EqC thc = eq_consts<PH>(m, th, phi_ref);
  if (!eq_sub) {
    thc.th0 = thc.th1 = thc.phi_ref = thc.a = 0.0;
    if (!(PH != PH_LIGHT && m.eq == 1)) thc.b = 0.0;  // (isentropic: the exponent)
  }

  const bool series = SERIES && wb && series_ok(eq_sub ? th[1] : 1.0e300);
  const double aa = thc.a * thc.a;
  // equilibrium average of this cell's equilibrium over a member cell given
  // its (translated) corners and volume
  auto member_avg = [&](const double (*w3)[3], double vol_j, double &er, double &eE) {
    if (PH == PH_LIGHT) {
      // axial gravity: phi is affine, so its point values follow from the
      // corner potentials load_member left in w3[k][0]; rho_eq = th0
      // exp(a (phi - phi_ref)) and E_eq = b rho_eq (b constant), so both
      // averages come from one weighted sum
      double pv[DIM + 1];
      for (int k = 0; k < DIM + 1; ++k) pv[k] = w3[k][0];
      // two points per iteration: independent exponentials interleave; the
      // sum still runs in point order.  An odd last point pairs with itself
      // at weight zero (adding +0 leaves the sum unchanged), so the loop body
      // is the only copy of the exponential.
      auto point = [&](int q) {
        double ph = m.vx[q][0] * pv[0];
        for (int k = 1; k < DIM + 1; ++k) ph = fma(m.vx[q][k], pv[k], ph);
        return exp((ph - thc.phi_ref) * thc.a);
      };
      double se = 0.0;
      for (int q = 0; q < m.qv; q += 2) {
        const bool pair = q + 1 < m.qv;
        const double e0 = point(q), e1 = point(pair ? q + 1 : q);
        const double w1 = pair ? m.vw[q + 1] : 0.0;
        se = (q == 0) ? m.vw[q] * e0 : fma(m.vw[q], e0, se);
        se = fma(w1, e1, se);
      }
      er = thc.th0 * se;
      eE = er * thc.b;
      return;
    }
    double sr = 0.0, sE = 0.0;
    for (int q = 0; q < m.qv; ++q) {
      double x[3];
      volume_point<DIM>(m, q, w3, x);
      double r, E;
      eq_point<DIM, PH>(m, thc, x, r, E);
      double w = vol_j * m.vw[q];
      if (q == 0) {
        sr = w * r;
        sE = w * E;
      } else {
        sr = sr + w * r;
        sE = sE + w * E;
      }
    }
    er = (1.0 * sr) / vol_j;
    eE = (1.0 * sE) / vol_j;
  };
  // this cell's equilibrium averaged over the cell itself, the points split
  // over the group's lanes
  auto own_eq = [&](double &er, double &eE) { group_avg(thc, er, eE); };
  double q0;
  {
    double er = 0.0, eE = 0.0;
    if (eq_sub) {
      // isothermal: the equilibrium is th0 times the function the solve just
      // averaged over this cell (same points, weights and order), so its own
      // average is th0 ar1 (to rounding), with E = b rho pointwise
      if (ar1 > 0.0 && PH != PH_LIGHT && m.eq == 1) {
        er = ar1;
        eE = aE1;
      } else if (ar1 > 0.0) {
        er = th[0] * ar1;
        eE = er * thc.b;
      } else if (series) {
        er = th[0] * exp_average(m, aa * y_p2, aa * thc.a * y_p3);
        eE = er * thc.b;
      } else {
        own_eq(er, eE);
      }
    }
    if (m.eqc != nullptr && !reuse && g == 0) {
      // the recomputed equilibrium's own average (zero if none), which the
      // next calls measure the threshold against
      m.eqc[6 * n + i] = er;
      m.eqc[7 * n + i] = eE;
    }
    q0 = u0[g];
    if (is_rho) q0 -= er;
    if (is_E) q0 -= eE;
    q0 = q0 * inv_g;
  }

  const int32_t meta = m.meta[i];
  const bool first_order = (meta & 8) != 0;
  const int kh = meta & 7;

  // this variable's coefficients: central c[alpha] (alpha = 1..DOFC-1),
  // one-sided b[k][alpha] (alpha = 1..DIM)
  double c[NC];
  double b[NB > 0 ? NB : 1][NBC];
  for (int a = 0; a < NC; ++a) c[a] = 0.0;

  if (!first_order) {
    // Per chunk each lane computes its row's member equilibrium average, and
    // its row of the pseudo-inverse and that average reach the group's lanes
    // through LDS.  The next chunk's pseudo-inverse rows, member states and
    // member data are loaded as soon as this chunk's have left their
    // registers, so that they are in flight during its arithmetic.
    constexpr int ROWW = row_doubles<DOFC>();
    double *pl = xch.wave_lds() + xch.lane0() * ROWW;  // this group's NV rows
    // the members' averages: (er, eE) of every central row; in the light set
    // er of every row (eE is er times the cell constant b)
    double *ceq = xch.lds();
    static_assert(RC + NB * RB <= group_lds_doubles<RC>(), "every row's average fits the group's scratch");
    constexpr int NCP = NC / 2;                        // coefficient pairs of a central row
    constexpr int GPW = 64 / NV;
    // the tile of pseudo-inverses of this wavefront's cells
    const int64_t tile = wave_uniform(int(uint32_t(i) / uint32_t(GPW)));
    const int grp = int(i - tile * GPW);
    const double *Pt = m.P + tile * (int64_t(NC) * RC + NB * RB * NBC) * GPW;
    // this lane's row of chunk ch: NC entries (central) or NBC (one-sided);
    // lanes past the chunk's rows read its last
    auto load_P = [&](int ch, double *pr) {
      const PPair *pp = reinterpret_cast<const PPair *>(Pt);
      const int gr = g < chunk_rows(ch) ? g : chunk_rows(ch) - 1;
      if (ch < CCH) {
#pragma unroll
        for (int p = 0; p < NCP; ++p) {
          const PPair v = pp[uint32_t(p_central(NV, GPW, NC, RC, 2 * p, ch * NV, 0) / 2) +
                             uint32_t(grp * chunk_rows(ch) + gr)];
          pr[2 * p] = v.lo;
          pr[2 * p + 1] = v.hi;
        }
        if (NC & 1)
          pr[NC - 1] = Pt[uint32_t(p_central(NV, GPW, NC, RC, NC - 1, ch * NV, 0)) + uint32_t(grp * chunk_rows(ch) + gr)];
      } else {
#pragma unroll
        for (int p = 0; p < NBC / 2; ++p) {
          const PPair v = pp[uint32_t(p_onesided(GPW, NC, RC, NBC, NB, RB, ch - CCH, 2 * p, 0, 0) / 2) +
                             uint32_t(grp * RB + gr)];
          pr[2 * p] = v.lo;
          pr[2 * p + 1] = v.hi;
        }
        if (NBC & 1)
          pr[NBC - 1] = Pt[uint32_t(p_onesided(GPW, NC, RC, NBC, NB, RB, ch - CCH, NBC - 1, 0, 0)) + uint32_t(grp * RB + gr)];
      }
    };
    // scaled deviation of row k of the chunk in this lane's variable
    // (the equilibrium parts enter with factors 1 or 0: u - 1 er = u - er
    // and x - 0 eE = x exactly, so this equals the branchy form bit for bit)
    // In the light set the energy average is the density average times the
    // cell constant b, so one factor serves each lane.
    const double f_rho = (wb && is_rho) ? 1.0 : ((PH == PH_LIGHT && wb && is_E) ? thc.b : 0.0);
    const double f_E = (PH != PH_LIGHT && wb && is_E) ? 1.0 : 0.0;
    auto deviation = [&](double u, double er, double eE) {
      double d = fma(-f_rho, er, u);
      if (PH != PH_LIGHT) d = fma(-f_E, eE, d);
      return fma(d, inv_g, -q0);
    };
    // what the equilibrium average over a member (row entry rw) needs: its potential
    // moments (linear isentropic equilibrium, untranslated member) or its
    // translated corners and volume
    struct Member {
      double w3[DIM + 1][3];
      double vol;
      double pm, pv;
      double sphi;  // light set: the translation's potential, added at use
      int lin;
      int32_t cell;  // 2D light set: the member, for averages out of the series' range
    };
    auto load_member = [&](int32_t entry, Member &mb) {
      const int64_t j = entry & ROW_CELL_MASK;
      const int code = entry >> ROW_CELL_BITS;
      if (PH == PH_LIGHT) {
        mb.sphi = m.phi_unshifted ? 0.0 : m.shift_phi[code];
        mb.cell = int32_t(j);
        if (SERIES) return;  // (averages out of the series' range)
        // the member's potential values (cphi) in w3[k][0] and its
        // translation's potential, added where they are used (so that the
        // loads stay in flight until then)
        const double *cp = m.cphi + uint32_t(j) * uint32_t(DIM + 1);
        for (int k = 0; k < DIM + 1; ++k) mb.w3[k][0] = cp[k];
        return;
      }
      mb.lin = PH == PH_LIN || (PH == PH_FULL && linear_isentropic(m) && code == 0) ? 1 : 0;
      if (PH == PH_LIN || mb.lin) {
        const PPair pv2 = reinterpret_cast<const PPair *>(m.phim)[j];
        mb.pm = pv2.lo;
        mb.pv = pv2.hi;
        return;
      }
      load_corners<DIM>(m, j, mb.w3);
      for (int k = 0; k < DIM + 1; ++k)
        for (int d = 0; d < DIM; ++d) mb.w3[k][d] += m.shift[code][d];
      mb.vol = m.vol[j];
    };
    auto member_avg_of = [&](const Member &mb, double &er, double &eE) {
      if (PH == PH_LIN || (PH == PH_FULL && mb.lin)) {
        linear_isentropic_avg(thc, mb.pm, mb.pv, er, eE);
      } else if (PH == PH_LIGHT) {
        double w3[DIM + 1][3];
        if (SERIES) {
          // out of the series' range: the rule's points one by one
          load_corners<DIM>(m, mb.cell, w3);
          for (int k = 0; k < DIM + 1; ++k) w3[k][0] = axial_phi<DIM>(m, w3[k]) + (mb.sphi - thc.phi_ref);
          double se = 0.0;
#pragma unroll 1
          for (int q = 0; q < m.qv; ++q) {
            double ph = m.vx[q][0] * w3[0][0];
            for (int k = 1; k < DIM + 1; ++k) ph = fma(m.vx[q][k], w3[k][0], ph);
            se = fma(m.vw[q], exp(ph * thc.a), se);
          }
          er = thc.th0 * se;
          eE = er * thc.b;
          return;
        }
        for (int k = 0; k < DIM + 1; ++k) w3[k][0] = mb.w3[k][0] + mb.sphi;
        member_avg(w3, mb.vol, er, eE);
      } else {
        member_avg(mb.w3, mb.vol, er, eE);
      }
    };
    // a one-sided row whose member is also a central row takes that row's
    // averages from LDS (the same values: same member, same function)
    // instead of loading the member and averaging again; not in PH_LIN and
    // in series form, where a member average costs less than the lookup
    auto twin_of = [&](int ch) {
      if (PH == PH_LIN || series || !eq_sub || ch < CCH || g >= RB) return -1;
      return int(m.twin[(chunk_row0(ch) + g - RC) * n + i]);
    };
    for (int k = 0; k < NB; ++k)
      for (int a = 0; a < NBC; ++a) b[k][a] = 0.0;
    double pr[NC];
    for (int a = 0; a < NC; ++a) pr[a] = 0.0;
    Member mb{};
    int tw = -1;
    load_P(0, pr);
    if (series) {
      // In series form all rows' averages come first: the chains of the
      // chunks are independent, so one lane's chunks overlap, and the members'
      // data are loaded together.
      double z[NCH], p2[NCH], p3[NCH];
#pragma unroll
      for (int ch = 0; ch < NCH; ++ch) {
        const int32_t j = rw[ch] & ROW_CELL_MASK;
        const double *cp = m.cphi + uint32_t(j) * 3u;
        z[ch] = cp[0];
        p2[ch] = cp[1];
        p3[ch] = cp[2];
        if (!m.phi_unshifted) z[ch] += m.shift_phi[rw[ch] >> ROW_CELL_BITS];
      }
#pragma unroll
      for (int ch = 0; ch < NCH; ++ch) {
        // th0 exp(a (mean - phi_ref)) times the average about the mean
        const double er = thc.th0 * (exp_near((z[ch] - thc.phi_ref) * thc.a) *
                                     exp_average(m, aa * p2[ch], aa * thc.a * p3[ch]));
        if (g < chunk_rows(ch)) ceq[chunk_row0(ch) + g] = er;
      }
    } else if (wb) {
      load_member(rw[0], mb);
    }
#pragma unroll
    for (int ch = 0; ch < NCH; ++ch) {
      const int cnt = chunk_rows(ch);
      xch.sync();  // the previous chunk's reads are done
#pragma unroll
      for (int a = 0; a < (ch < CCH ? NC : NBC); ++a) pl[g * ROWW + a] = pr[a];
      const Member mc = mb;
      const int tc = tw;
      double uc[NV];
#pragma unroll
      for (int k = 0; k < NV; ++k) uc[k] = uk[k];
      if (ch + 1 < NCH) {
        load_P(ch + 1, pr);
        gather(ch + 1, uk);
        tw = twin_of(ch + 1);
        if (wb && !series && tw < 0) load_member(rw[ch + 1], mb);
      }
      if (wb && !series) {
        double er = 0.0, eE = 0.0;
        if (PH == PH_LIGHT) {
          if (tc >= 0) er = ceq[tc];
          else member_avg_of(mc, er, eE);
          if (g < cnt) ceq[chunk_row0(ch) + g] = er;
        } else {
          if (tc >= 0) {
            er = ceq[2 * tc];
            eE = ceq[2 * tc + 1];
          } else {
            member_avg_of(mc, er, eE);
          }
          if (PH != PH_LIN && ch < CCH && g < cnt) {
            ceq[2 * (ch * NV + g)] = er;
            ceq[2 * (ch * NV + g) + 1] = eE;
          }
          pl[g * ROWW + NC] = er;
          pl[g * ROWW + NC + 1] = eE;
        }
      }
      xch.sync();
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        if (k >= cnt) break;
        const double *row = pl + k * ROWW;
        double er = 0.0, eE = 0.0;
        if (wb) {
          er = PH == PH_LIGHT ? ceq[chunk_row0(ch) + k] : row[NC];
          if (PH != PH_LIGHT) eE = row[NC + 1];
        }
        const double d = deviation(uc[k], er, eE);
        if (ch < CCH) {
#pragma unroll
          for (int a = 0; a < NC; ++a) c[a] = fma(row[a], d, c[a]);
        } else {
#pragma unroll
          for (int a = 0; a < NBC; ++a) b[ch < CCH ? 0 : ch - CCH][a] = fma(row[a], d, b[ch < CCH ? 0 : ch - CCH][a]);
        }
        // one row's entries in registers at a time
        if (ch < CCH) computed_here<NC>(c);
        else computed_here<NBC>(b[ch < CCH ? 0 : ch - CCH]);
        schedule_fence();
      }
    }
  }

  // final polynomial of this variable
  double a[DOFC];
  if (first_order) {
    a[0] = 0.0 + 1.0 * q0;
    for (int al = 1; al < DOFC; ++al) a[al] = 0.0;
  } else {
    double a0[NB + 1];
    for (int k = 0; k <= NB; ++k) a0[k] = q0;
    if (m.mode == 0) {
      // CWENO: p_hi <- (p_hi - sum_{k != hi} c_k p_k) * (1 / c_hi)
      if (kh == 0) {
#pragma unroll
        for (int k = 1; k <= NB; ++k) {
          const double w = m.lw[k];
          a0[0] = a0[0] - w * a0[k];
          for (int al = 0; al < NBC; ++al) c[al] = c[al] - w * b[k - 1][al];
        }
        const double iw = 1.0 / m.lw[0];
        a0[0] = iw * a0[0];
        for (int al = 0; al < NC; ++al) c[al] = iw * c[al];
      } else if (NB > 0) {
        // the corrected polynomial is a one-sided one (central stencil reduced
        // to order 1); compile-time indices keep b in registers
#pragma unroll
        for (int hb = 0; hb < NB; ++hb) {
          if (hb != kh - 1) continue;
#pragma unroll
          for (int k = 0; k <= NB; ++k) {
            if (k == hb + 1) continue;
            const double w = m.lw[k];
            a0[hb + 1] = a0[hb + 1] - w * a0[k];
            for (int al = 0; al < NBC; ++al) {
              double o = (k == 0) ? c[al] : b[k > 0 ? k - 1 : 0][al];
              b[hb][al] = b[hb][al] - w * o;
            }
          }
          const double iw = 1.0 / m.lw[hb + 1];
          a0[hb + 1] = iw * a0[hb + 1];
          for (int al = 0; al < NBC; ++al) b[hb][al] = iw * b[hb][al];
        }
      }
    }
    // Smoothness indicators (maximum over the variables, in variable order) and
    // nonlinear weights (src/zisa/reconstruction/hybrid_weno.cpp:110-127).  The
    // lanes exchange their sums of squares through LDS; lane k then forms
    // stencil k's weight, so that its power and division run once a cell
    // instead of once a lane.
    static_assert(NB + 1 <= NV, "one lane per stencil");
    static_assert((NB + 1) * (NV + 1) <= NV * row_doubles<DOFC>(), "the exchange fits the group's rows");
    double *sq = xch.wave_lds() + xch.lane0() * row_doubles<DOFC>();  // [stencil][variable], then the weights
    double *wk = sq + (NB + 1) * NV;
    xch.sync();
#pragma unroll
    for (int k = 0; k <= NB; ++k) {
      double t = 0.0;
      if (k == 0) {
        for (int al = 0; al < NC; ++al) t += c[al] * c[al];
      } else {
        for (int al = 0; al < NBC; ++al) t += b[k - 1][al] * b[k - 1][al];
      }
      sq[k * NV + g] = t;
    }
    xch.sync();
    const int my_k = g <= NB ? g : NB;
    double IS = sq[my_k * NV];
#pragma unroll
    for (int v = 1; v < NV; ++v) IS = dmax(IS, sq[my_k * NV + v]);
    const double isp = m.exponent == 4.0 ? sqr(sqr(IS)) : pow(IS, m.exponent);
    wk[my_k] = m.lw[my_k] / (m.eps + isp);
    xch.sync();
    double alpha[NB + 1];
    double al_tot = 0.0;
#pragma unroll
    for (int k = 0; k <= NB; ++k) {
      alpha[k] = wk[k];
      al_tot += alpha[k];
    }
    const double inv_tot = 1.0 / al_tot;
    const double w0 = quotient(alpha[0], al_tot, inv_tot);
    a[0] = 0.0 + w0 * a0[0];
    for (int al = 1; al < DOFC; ++al) a[al] = 0.0 + w0 * c[al - 1];
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const double w = quotient(alpha[k + 1], al_tot, inv_tot);
      a[0] = a[0] + w * a0[k + 1];
      for (int al = 1; al <= NBC; ++al) a[al] = a[al] + w * b[k][al - 1];
    }
  }

  // moments: zero for alpha < 3
  double cm[DOFC];
  load_moments<DOFC>(m, i, cm);
  double xc[3];
  load_centre<DIM>(m, i, xc);
  const double len = m.len[i];
  const uint32_t fperm = m.fperm[i];
  const double inv_len = 1.0 / len;

  // The deviation of this variable, sum_alpha a_alpha (X^alpha - c_alpha): the
  // variable's scale goes into the coefficients and the moments into the
  // constant one, so that a point costs one nested evaluation.  The mean (the
  // coefficient of the basis function 1) is added last: the rest is a difference
  // from it, small where the state varies little, and keeps its own last places.
  for (int al = 0; al < DOFC; ++al) a[al] = scale_g * a[al];
  const double mean = a[0];
  a[0] = 0.0;
  for (int al = 3; al < DOFC; ++al) a[0] = fma(-a[al], cm[al], a[0]);

  double s_acc = 0.0;
  const bool gravity_src = (m.gravity != 0) && (src != nullptr);
  // EquilibriumFluxBC (flux_bc 2, include/zisa/boundary/equilibrium_flux_bc.hpp:36-62):
  // at the cell's boundary faces, the flux of its isentropic equilibrium
  // (this cell's own, solved above: the same solve_exact from the same
  // average) as a state at rest, (0, p_eq n, 0), integrated with the face
  // rule and subtracted.  It has the form of the well-balanced source's face
  // term, w p_eq n out of the cell, and cancels it there.  An equilibrium that
  // was not found gives NaN, as the reference's zero extrapolation does.
  // (Isentropic only: never in the light physics set.)
  const bool eq_flux_bc = PH != PH_LIGHT && m.flux_bc == 2 && gravity_src;

  // The face points along the cell's own vertex order, so that every corner
  // index is known at compile time; a point's values go to the place of the
  // same point in the left cell's order, in which the fluxes read them.
  const FaceWords cfw = load_face_words(m, i);
  double V[DIM + 1][3];
  load_corners<DIM>(m, i, V);
  // this lane's component of a face's outward normal times the area (momentum
  // lanes; zero for the others): 2D the turned edge, 3D from the table
  const bool mom_lane = g >= 1 && g <= DIM;
  double an2[DIM == 2 ? NF : 1];
  if (DIM == 2) {
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const double *p0 = V[face_corner<DIM>(f, 0)], *p1 = V[face_corner<DIM>(f, 1)];
      an2[DIM == 2 ? f : 0] = g == 1 ? p1[1] - p0[1] : p0[0] - p1[0];
    }
  }
  auto face_normal = [&](int f) -> double {
    if (!mom_lane || (eq_flux_bc && cfw.w[f] == 2)) return 0.0;
    if (DIM == 2) return an2[DIM == 2 ? f : 0];
#if defined(__HIP_DEVICE_COMPILE__)
    return m.fan[uint32_t(i) * 12u + uint32_t(3 * f + g - 1)];
#else
    double v[3];
    face_normal_out(m, i, f, v);
    return v[g - 1];
#endif
  };
  // in series form: the exponents a (phi - phi_ref) at the corners
  double zc[DIM + 1];
  for (int k = 0; k < DIM + 1; ++k) zc[k] = 0.0;
  if (series) {
#pragma unroll
    for (int k = 0; k < DIM + 1; ++k) zc[k] = (axial_phi<DIM>(m, V[k]) - thc.phi_ref) * thc.a;
  }
#pragma unroll
  for (int k = 0; k < DIM + 1; ++k)
    for (int d = 0; d < DIM; ++d) V[k][d] = (V[k][d] - xc[d]) * inv_len;
  const double eq_rho = is_rho ? 1.0 : 0.0, eq_E = is_E ? 1.0 : 0.0;
  // The source's face term is summed of the equilibrium energies' differences
  // from one of them, where the face normals, the turned edges, sum to zero (not
  // where the flux BC has a boundary face's left out): the differences are exact
  // and small, the full terms would cancel to their last places.  (3D: the
  // tables' normals sum to zero only as far as the fluxes' do.)
  const bool closed = DIM == 2 && !(eq_flux_bc && (cfw.w[0] == 2 || cfw.w[1] == 2 || cfw.w[2] == 2));
  double E0 = 0.0;
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int32_t cf = cfw.w[f];
    const bool exterior = (cf & 2) != 0;
    // the face's corners in scaled coordinates, then its points
    double w3[3][3];
#pragma unroll
    for (int t = 0; t < DIM; ++t)
      for (int d = 0; d < 3; ++d) w3[t][d] = d < DIM ? V[face_corner<DIM>(f, t)][d] : 0.0;
    // equilibrium point values: every lane forms all of them where that is
    // cheap (PH_LIN); else lane k evaluates point k (mod NV) and every lane
    // receives them
    double eqr[Q], eqE[Q];
    for (int q = 0; q < Q; ++q) eqr[q] = eqE[q] = 0.0;
    const double *pf = m.pot + i * int64_t(NF * Q) + f * Q;
    if (PH == PH_LIN) {
      double ph[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) ph[q] = pf[q];
#pragma unroll
      for (int q = 0; q < Q; ++q) eq_at_phi<PH>(m, thc, ph[q], eqr[q], eqE[q]);
    } else if (series) {
      // (within an exponent of 0.125: exp_near)
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const double xi = m.fx[q][0], z0 = zc[face_corner<DIM>(f, 0)], z1 = zc[face_corner<DIM>(f, 1)];
        eqr[q] = thc.th0 * exp_near(fma(0.5 + 0.5 * xi, z1, (0.5 - 0.5 * xi) * z0));
        eqE[q] = eqr[q] * thc.b;
      }
    } else if (wb) {
#pragma unroll
      for (int q0 = 0; q0 < Q; q0 += NV) {
        double my_r = 0.0, my_E = 0.0;
        if (q0 + g < Q) {
          double ph;
          if (tab) {
            ph = pf[q0 + g];
          } else {
            double x[3];
            face_point<DIM>(m, q0 + g, w3, x);
            for (int d = 0; d < DIM; ++d) x[d] = fma(x[d], len, xc[d]);
            ph = PH == PH_LIGHT ? axial_phi<DIM>(m, x) : phi<DIM, PH>(m, x);
          }
          eq_at_phi<PH>(m, thc, ph, my_r, my_E);
        }
#pragma unroll
        for (int k = 0; k < NV; ++k) {
          const double r = xch.bcast(my_r, k), E = xch.bcast(my_E, k);
          if (q0 + k < Q) {
            eqr[q0 + k] = r;
            eqE[q0 + k] = E;
          }
        }
      }
    }
    if (closed && f == 0) E0 = eqE[0];
    double fs = 0.0, u[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      double Xs[3];
      face_point<DIM>(m, q, w3, Xs);
      u[q] = mean + poly_nested<DIM, DEGC>(a, Xs);
      if (wb) {
        u[q] = fma(eq_rho, eqr[q], fma(eq_E, eqE[q], u[q]));
        fs = fma(m.fw[q], eqE[q] - E0, fs);
      }
    }
    computed_here<Q>(u);
    // in the global frame, as the fluxes take them
    if (!exterior) {
      double *slot = fpv + (int64_t(i) * NF + f) * slot_doubles<DIM, Q>() + g;
#pragma unroll
      for (int q = 0; q < Q; ++q) slot[face_point_in_left_order<DIM, Q>(fperm, f, q) * NV] = u[q];
    }
    if (gravity_src && wb) s_acc = fma((gamma - 1.0) * fs, face_normal(f), s_acc);
    if (eq_flux_bc && cf == 2 && !eq_sub) s_acc = __builtin_nan("");
    schedule_fence();
  }

  if (gravity_src) {
    const double vol_i = m.vol[i];
    // The volume terms, -(rho - rho_eq) grad phi for the momentum and
    // -m . grad phi for the energy, need only the lanes' own deviations (the
    // equilibrium is at rest and differs from the state only in rho and E;
    // without one the deviation is the state): every lane forms -sum_q w_q
    // delta(x_q) d_d phi(x_q) for every d; the density lane's sums feed the
    // momentum lanes, momentum lane d's d-th sum the energy lane.
    double acc[DIM];
    if (PH == PH_LIGHT && m.vol_mean) {
      // constant gradient (axial gravity): sum_q w_q delta(x_q) grad phi is
      // vol grad phi times the rule's mean of delta over the cell, which is
      // its constant coefficient (the rule and the moments integrate every
      // other basis function, X^alpha - c_alpha, to zero)
      double gp[3];
      grad_phi<DIM, PH>(m, xc, gp);
      const double s0 = vol_i * mean;
#pragma unroll
      for (int d = 0; d < DIM; ++d) acc[d] = -s0 * gp[d];
    } else if (PH == PH_LIGHT) {
      // constant gradient, rules that do not integrate the basis exactly:
      // the quadrature over the points
      double vtx[DIM + 1][3];
      load_corners<DIM>(m, i, vtx);
#pragma unroll 1
      for (int q = 0; q < m.qv; ++q) {
        double x[3], Xs[3] = {0.0, 0.0, 0.0};
        volume_point<DIM>(m, q, vtx, x);
        for (int d = 0; d < DIM; ++d) Xs[d] = (x[d] - xc[d]) * inv_len;
        const double dl = mean + poly_nested<DIM, DEGC>(a, Xs);
        double gp[3];
        grad_phi<DIM, PH>(m, x, gp);
        const double w = vol_i * m.vw[q];
#pragma unroll
        for (int d = 0; d < DIM; ++d) acc[d] = (q == 0) ? w * (-dl * gp[d]) : fma(w, -dl * gp[d], acc[d]);
      }
    } else {
      // from the polynomial and the cell's source moments (store_source_moments)
#pragma unroll
      for (int d = 0; d < DIM; ++d) acc[d] = 0.0;
      // (the cell's DOFC x DIM moments are contiguous: 16-byte loads)
      double sm[DOFC * DIM];
      {
        const PPair *sp = reinterpret_cast<const PPair *>(m.smom + int64_t(i) * (DOFC * DIM));
#pragma unroll
        for (int k = 0; k < DOFC * DIM / 2; ++k) {
          const PPair v = sp[k];
          sm[2 * k] = v.lo;
          sm[2 * k + 1] = v.hi;
        }
      }
      // (a[0] holds the nested form's moments; the basis function 1 has mean)
#pragma unroll
      for (int al = 0; al < DOFC; ++al)
#pragma unroll
        for (int d = 0; d < DIM; ++d) acc[d] = fma(al == 0 ? -mean : -a[al], sm[al * DIM + d], acc[d]);
    }
    double cs_ = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      const double rs = xch.bcast(acc[d], 0);      // the density lane's sum for direction d
      const double bm = xch.bcast(acc[d], 1 + d);  // momentum lane d's sum for its own direction
      if (g == 1 + d) cs_ = rs;
      if (is_E) cs_ = (d == 0) ? bm : cs_ + bm;
    }
    double sum = wb ? (s_acc + 1.0 * cs_) : 1.0 * cs_;
    src[state_at<AOS, NV>(n, g, i)] = sum / vol_i;
  }
}

// LocalCFL's candidate of a cell of inradius inr: inradius / (|v| + a); 0 for a
// NaN or non-physical state, which surfaces as dt = 0
// (include/zisa/model/local_cfl_condition_impl.hpp:25-40)
template <int DIM>
ZFV_HD double cfl_of_cell(const double *u, double inr, double gamma) {
  double m2 = u[1] * u[1] + u[2] * u[2];
  if (DIM == 3) m2 += u[3] * u[3];
  const double v2 = m2 / (u[0] * u[0]);
  const double p = (u[DIM + 1] - 0.5 * m2 / u[0]) * (gamma - 1.0);
  const double a = sqrt(gamma * p / u[0]);
  const double r = inr / (sqrt(v2) + a);
  return r > 0.0 ? r : 0.0;
}

// ---- the per-face flux ----------------------------------------------------------
// the flux through interior face e from its left to its right cell (global
// frame, times the face's measure), which the left cell loses and the right
// cell gains, from the two cells' point values (slot layout)
template <int DIM, int Q>
ZFV_HD void flux_between(const Img &m, int64_t e, const double *bL, const double *bR, double *flux) {
  constexpr int NV = DIM + 2;
  double nn[3], area;
  face_table_frame<DIM>(m, e, nn, area);
  for (int v = 0; v < NV; ++v) flux[v] = 0.0;
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    double f[NV];
    if (m.flux == 0) hllc<DIM>(bL + q * NV, bR + q * NV, nn, m.gamma, f);
    else rusanov<DIM>(bL + q * NV, bR + q * NV, nn, m.gamma, f);
    for (int v = 0; v < NV; ++v) flux[v] = flux[v] + m.fw[q] * f[v];
  }
  for (int v = 0; v < NV; ++v) flux[v] = area * flux[v];
}

// the point values of one cell-face slot, in 16-byte loads
template <int DIM, int Q>
ZFV_HD void load_slot(const double *__restrict__ fpv, int64_t slot, double *b) {
  constexpr int SQ = slot_doubles<DIM, Q>();
  const PPair *p = reinterpret_cast<const PPair *>(fpv + slot * SQ);
#pragma unroll
  for (int k = 0; k < SQ / 2; ++k) {
    const PPair v = p[k];
    b[2 * k] = v.lo;
    b[2 * k + 1] = v.hi;
  }
}

// every interior face's flux stored once per face (the host emulation's form;
// the kernels form a cell's fluxes where the cell is updated)
template <int DIM, int Q>
ZFV_HD void face_flux(const Img &m, int64_t e, const double *__restrict__ fpv, double *__restrict__ G) {
  constexpr int NV = DIM + 2;
  constexpr int SQ = slot_doubles<DIM, Q>();
  double bL[SQ], bR[SQ], flux[NV];
  const SlotPair sl = reinterpret_cast<const SlotPair *>(m.fslot)[e];
  load_slot<DIM, Q>(fpv, sl.l, bL);
  load_slot<DIM, Q>(fpv, sl.r, bR);
  flux_between<DIM, Q>(m, e, bL, bR, flux);
  for (int v = 0; v < NV; ++v) G[v * m.ne + e] = flux[v];
}

// One face of an update tile: an interior face e with the slots of its left and
// right cell, or (r < 0) the boundary face f of cell e
struct alignas(16) UpdateFace {
  int32_t l, r, e, f;
};
// a cell's word: 8 bits per face, the entry's place in the tile (7 bits; 127:
// no contribution) and whether the cell is on the face's right side
constexpr uint32_t UPDATE_NO_FACE = 127u;

// FluxBC at a boundary face f of cell i: the physical flux of the cell average
// out of the cell (global frame, times the face measure; the weights sum to one)
template <int DIM, bool AOS>
ZFV_HD void boundary_flux(const Img &m, int64_t i, int f, const double *__restrict__ U, double *flux) {
  constexpr int NV = DIM + 2;
  double nn[3], area, u[NV];
  load_face_frame<DIM>(m, i, f, nn, area);
  for (int v = 0; v < NV; ++v) u[v] = U[state_at<AOS, NV>(m.n, v, i)];
  euler_flux<DIM>(u, face_state<DIM>(u, nn, m.gamma), nn, flux);
  for (int v = 0; v < NV; ++v) flux[v] = area * flux[v];
}

// the flux of one face of an update tile
template <int DIM, int Q>
ZFV_HD void update_face_flux(const Img &m, const UpdateFace &u, const double *__restrict__ U,
                             const double *__restrict__ fpv, double *flux) {
  constexpr int SQ = slot_doubles<DIM, Q>();
  if (u.r < 0) {
    boundary_flux<DIM, true>(m, u.e, u.f, U, flux);
    return;
  }
  double bL[SQ], bR[SQ];
  load_slot<DIM, Q>(fpv, u.l, bL);
  load_slot<DIM, Q>(fpv, u.r, bR);
  flux_between<DIM, Q>(m, u.e, bL, bR, flux);
}

// ---- the per-cell rate of change -------------------------------------------------
// (emulation) L = -(1/vol) sum of the cell's fluxes (+ source) (+ flux BC), over
// planes and stored fluxes
template <int DIM>
ZFV_HD void cell_rate(const Img &m, int64_t i, const double *__restrict__ U, const double *__restrict__ G,
                      const double *__restrict__ src, double *L) {
  constexpr int NV = DIM + 2;
  constexpr int NF = DIM + 1;
  const int64_t n = m.n;
  double acc[NV];
  for (int v = 0; v < NV; ++v) acc[v] = 0.0;
  const FaceWords cfw = load_face_words(m, i);
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int32_t cf = cfw.w[f];
    const bool exterior = (cf & 2) != 0;
    // ghost-pair faces (cf == 3) carry neither a flux nor the flux BC; the
    // equilibrium flux BC (flux_bc 2) is part of the source term
    if (exterior && (m.flux_bc != 1 || (cf & 1))) continue;
    double g[NV];
    if (!exterior) {
      // the flux through the face (global frame, times area)
      const double sgn = (cf & 1) ? 1.0 : -1.0;
      for (int v = 0; v < NV; ++v) g[v] = sgn * G[v * m.ne + (cf >> 2)];
    } else {
      boundary_flux<DIM, false>(m, i, f, U, g);
      for (int v = 0; v < NV; ++v) g[v] = -1.0 * g[v];
    }
    for (int v = 0; v < NV; ++v) acc[v] += g[v];
  }
  const double vol = m.vol[i];
  for (int v = 0; v < NV; ++v) L[v] = acc[v] / vol;
  if (m.gravity != 0 && src != nullptr)
    for (int v = 0; v < NV; ++v) L[v] += src[state_at<false, NV>(n, v, i)];
}

}  // namespace zfv
