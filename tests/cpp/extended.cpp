// TEST-ONLY: the 2D rate of change of the kernels' math (stage_math.hpp) in
// 80-bit arithmetic on the tables that the library's setup computes in double
// precision: what the double precision evaluation is rounded from.  Built by
// tests/test_rounding.py.
#include <math.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

#include "../../zisafvm_amd/csrc/common.hpp"
#include "../../zisafvm_amd/csrc/setup.hpp"

// (in a namespace of its own: the setup has the same header in double)
typedef long double real;
#define double real
#define zfv zfv_extended
#include "../../zisafvm_amd/csrc/stage_math.hpp"
#undef zfv
#undef double

using namespace zfv_extended;
using zfv::HostImage;
using zfv::Shape;

namespace {

// the lanes of a cell's group as threads in lockstep
struct Lanes {
  int n;
  std::atomic<int> in{0};
  std::atomic<long> turn{0};
  real slot[8] = {0}, lds[128] = {0}, wave[640] = {0};
  void wait() {
    const long t = turn.load();
    if (in.fetch_add(1) + 1 == n) {
      in = 0;
      turn.fetch_add(1);
    } else {
      while (turn.load() == t) std::this_thread::yield();
    }
  }
};

struct Exchange {
  Lanes *l;
  int g;
  real bcast(real v, int k) {
    l->slot[g] = v;
    l->wait();
    const real r = l->slot[k];
    l->wait();
    return r;
  }
  int32_t bcast_i(int32_t v, int k) { return int32_t(bcast(real(v), k)); }
  real *lds() { return l->lds; }
  real *wave_lds() { return l->wave; }
  int lane0() const { return 0; }
  void sync() { l->wait(); }
};

template <int DOFC, int RC, int Q>
void run(const Img &m, int ph, const real *U, real *fpv, real *src, real *L) {
  Lanes lanes{4};
  std::vector<std::thread> t;
  for (int g = 0; g < 4; ++g)
    t.emplace_back([&, g] {
      Exchange x{&lanes, g};
      for (int64_t i = 0; i < m.n; ++i) {
        if (ph == PH_LIGHT) reconstruct_lane<2, DOFC, RC, 3, 3, Q, PH_LIGHT>(m, i, g, x, U, fpv, src);
        else reconstruct_lane<2, DOFC, RC, 3, 3, Q, PH_FULL>(m, i, g, x, U, fpv, src);
      }
    });
  for (auto &x : t) x.join();
  std::fill(L, L + 4 * m.n, real(0));
  for (int64_t e = 0; e < m.ne; ++e) {
    constexpr int SQ = slot_doubles<2, Q>();
    const int32_t *s = m.fslot + 2 * e;
    real f[4];
    flux_between<2, Q>(m, e, fpv + int64_t(s[0]) * SQ, fpv + int64_t(s[1]) * SQ, f);
    for (int v = 0; v < 4; ++v) {
      L[v * m.n + s[0] / 3] -= f[v];
      L[v * m.n + s[1] / 3] += f[v];
    }
  }
  for (int64_t i = 0; i < m.n; ++i)
    for (int v = 0; v < 4; ++v) L[v * m.n + i] = L[v * m.n + i] / m.vol[i] + (src ? src[v * m.n + i] : real(0));
}

}  // namespace

extern "C" {

// dudt (n x 5, caller order) = L(u); -1: no such kernel shape or parameters.
// series: the isothermal averages in series form, as the device has them, where
// the cell's exponents are in range (else an exponential per point throughout);
// the least and the largest part of the range that a cell's need go to range.
int ext_rate(const zfv_mesh *mesh, const zfv_params *p, const double *u, long double *dudt, int series, double *range) {
  HostImage im;
  zfv::build_image(*mesh, *p, im);
  const Shape &s = im.s;
  const int64_t n = im.n;
  if (s.dim != 2 || p->flux_bc == 1 || p->gamma == 2.0) return -1;
  std::vector<std::vector<real>> kept;
  auto wide = [&](const std::vector<double> &v) {
    kept.emplace_back(v.begin(), v.end());
    return kept.back().data();
  };
  auto room = [&](size_t k) {
    kept.emplace_back(k, real(0));
    return kept.back().data();
  };
  kept.reserve(32);
  Img m{};
  m.n = n;
  m.ne = im.ne;
  m.P = wide(im.P);
  m.rows = im.rows.data();
  m.twin = im.twin.data();
  m.crn = wide(im.crn);
  m.xc = wide(im.xc);
  m.len = wide(im.len);
  m.vol = wide(im.vol);
  m.inr = wide(im.inr);
  m.mom = wide(im.mom);
  m.meta = im.meta.data();
  m.cface = im.cface.data();
  m.fslot = im.fslot.data();
  m.fperm = im.fperm.data();
  m.gamma = p->gamma;
  m.eps = p->epsilon;
  m.exponent = p->exponent;
  for (int k = 0; k < 5; ++k) m.lw[k] = im.linear_weights[k];
  m.mode = p->reconstruction;
  m.scaling = p->scaling;
  m.vol_mean = zfv::volume_mean_is_constant_term(*p, s) ? 1 : 0;
  m.flux = p->flux;
  m.eq = p->equilibrium;
  m.gravity = p->gravity;
  m.g = p->gravity_g;
  for (int d = 0; d < 3; ++d) m.axis[d] = p->gravity_axis[d];
  m.flux_bc = p->flux_bc;
  m.spr = 1;
  for (int q = 0; q < 16; ++q)
    for (int d = 0; d < 3; ++d) m.shift[q][d] = im.shift[3 * q + d];
  for (size_t q = 0; q < im.face_w.size(); ++q) {
    m.fw[q] = im.face_w[q];
    m.fx[q][0] = im.face_x[q];
  }
  m.qv = int(im.vol_w.size());
  for (int q = 0; q < m.qv; ++q) {
    m.vw[q] = im.vol_w[q];
    for (int d = 0; d < 3; ++d) m.vx[q][d] = im.vol_x[3 * q + d];
  }
  real *frm = room(size_t(3) * frame_words<2>() * n);
  for (int64_t i = 0; i < n; ++i) store_face_frames<2>(m, i, frm);
  m.frm = frm;
  real *ffr = room(size_t(frame_words<2>()) * std::max<int64_t>(im.ne, 1));
  for (int64_t e = 0; e < im.ne; ++e) store_face_table<2>(m, e, ffr);
  m.ffr = ffr;
  for (int c = 0; c < 16; ++c) m.shift_phi[c] = phi<2, PH_LIGHT>(m, m.shift[c]);
  const int ph = physics_set(m);
  if (ph == PH_LIGHT && m.eq != 0) {
    real *cphi = room(size_t(3) * n);
    for (int64_t i = 0; i < n; ++i) store_cell_phi<2>(m, i, cphi);
    m.cphi = cphi;
    if (series && exp_average_constants(m, m.es)) {
      m.phi_unshifted = 1;
      for (real v : m.shift_phi) m.phi_unshifted &= v == 0;
      for (int64_t i = 0; i < n; ++i) {
        m.es_p2 = std::max(m.es_p2, m.cphi[3 * i + 1]);
        for (int r = 0; r < s.nrows; ++r) {
          const int32_t e = m.rows[r * n + i];
          m.es_dist = std::max(m.es_dist, std::fabs(m.cphi[3 * int64_t(e & ROW_CELL_MASK)] +
                                                    m.shift_phi[e >> ROW_CELL_BITS] - m.cphi[3 * i]));
        }
      }
      range[0] = 1e300;
      range[1] = 0.0;
      for (int64_t i = 0; i < n; ++i) {
        const double *a = u + 5 * int64_t(im.perm[i]);
        const real RT = (p->gamma - 1.0) * (a[4] - 0.5 * (a[1] * a[1] + a[2] * a[2]) / a[0]) / a[0];
        const double part = double(std::max(m.es_dist / (kSeriesMaxArg * RT), std::sqrt(m.es_p2 / (kSeriesMaxY2 * RT * RT))));
        range[0] = std::min(range[0], part);
        range[1] = std::max(range[1], part);
      }
    }
  }
  real *src = nullptr;
  if (m.gravity != 0) {
    real *smom = room(size_t(s.dofc) * 2 * n);
    for (int64_t i = 0; i < n; ++i) {
      if (s.dofc == 10) store_source_moments<2, 10>(m, i, smom);
      else if (s.dofc == 6) store_source_moments<2, 6>(m, i, smom);
      else store_source_moments<2, 3>(m, i, smom);
    }
    m.smom = smom;
    src = room(size_t(4) * n);
  }
  std::vector<real> U(4 * n), L(4 * n), fpv(size_t(3) * ((s.q * 4 + 1) & ~1) * n);
  for (int64_t ip = 0; ip < n; ++ip) {
    const double *a = u + 5 * int64_t(im.perm[ip]);
    for (int v = 0; v < 4; ++v) U[v * n + ip] = a[v == 3 ? 4 : v];
  }
  if (s.dofc == 6 && s.q == 2) run<6, 10, 2>(m, ph, U.data(), fpv.data(), src, L.data());
  else if (s.dofc == 10 && s.q == 3) run<10, 18, 3>(m, ph, U.data(), fpv.data(), src, L.data());
  else return -1;
  for (int64_t ip = 0; ip < n; ++ip) {
    long double *a = dudt + 5 * int64_t(im.perm[ip]);
    for (int v = 0; v < 5; ++v) a[v] = v == 3 ? 0 : L[(v == 4 ? 3 : v) * n + ip];
  }
  return 0;
}

}  // extern "C"
