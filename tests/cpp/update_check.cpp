// TEST-ONLY: the update of the gfx950 kernels (update.hpp) run on the host over
// the tables that the library's setup builds, one wavefront's lanes after another
// in a shuffled order, against loops over the faces and the cells.  Built with
// AddressSanitizer by tests/test_update_host.py: every array, the wavefront's LDS
// among them, has exactly its size.  What a step reconstructs is not of interest
// here: point values are made up from the state they belong to.
//
//   update_check <dims> <n> <mesh> <flux> <flux_bc> <edge_deg> <seed>
//   mesh: periodic, bounded, ghosts (bounded with frozen ghost layers), pairs
//   (disjoint pairs of triangles, most of them ghosts: tiles of many faces)
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <memory>
#include <numeric>
#include <random>
#include <string>
#include <vector>

#include "../../zisafvm_amd/csrc/common.hpp"
#include "../../zisafvm_amd/csrc/setup.hpp"
#include "../../zisafvm_amd/csrc/stage_math.hpp"
#include "../../zisafvm_amd/csrc/update.hpp"

using namespace zfv;

namespace {

constexpr double kNaN = std::numeric_limits<double>::quiet_NaN();
std::mt19937_64 rng;

#define CHECK(cond)                                                       \
  do {                                                                    \
    if (!(cond)) {                                                        \
      std::fprintf(stderr, "line %d: " #cond " does not hold\n", __LINE__); \
      std::exit(1);                                                       \
    }                                                                     \
  } while (0)

bool same(double a, double b) { return std::memcmp(&a, &b, sizeof(a)) == 0; }

struct HostWave {
  template <class R>
  struct Lanes {
    R r[64];
  };
  template <class R, class F>
  void each(Lanes<R> &regs, F &&f) {
    int order[64];
    std::iota(order, order + 64, 0);
    std::shuffle(order, order + 64, rng);
    for (int lane : order) f(lane, regs.r[lane]);
  }
  void sync() {}
  template <class F>
  double least(F &&f) {
    double r = f(0);
    for (int lane = 1; lane < 64; ++lane) r = std::min(r, f(lane));
    return r;
  }
  template <class F>
  void lower(unsigned long long *word, F &&f) {
    const double r = least(f);
    unsigned long long bits;
    std::memcpy(&bits, &r, sizeof(bits));
    *word = std::min(*word, bits);
  }
  void flag(int *word) { *word |= 1; }
};

// an instance's tables and arrays, all of exactly their sizes
struct Instance {
  HostImage im;
  Img m{};
  std::vector<int32_t> off, entries, more;
  std::vector<uint32_t> words;
  std::vector<double> frm, ffr, U, X, K, fpv, src, steady;
};

zfv_params params(int dims, int flux, int flux_bc, int edge_deg) {
  zfv_params p{};
  p.n_dims = dims;
  p.n_stencils = dims + 2;
  for (int k = 0; k < p.n_stencils; ++k) {
    p.orders[k] = k == 0 ? (edge_deg == 1 ? 2 : 3) : 2;
    p.biases[k] = k > 0;
    p.overfit[k] = k == 0 ? 2.0 : 1.5;
    p.linear_weights[k] = k == 0 ? 100.0 : 1.0;
  }
  p.epsilon = 1e-6;
  p.exponent = 4.0;
  p.gamma = 1.4;
  p.gas_constant = 1.0;
  p.flux = flux;
  p.flux_bc = flux_bc;
  p.gravity = ZFV_GRAVITY_AXIAL;  // with a source
  p.gravity_g = 1.0;
  p.gravity_axis[1] = 1.0;
  p.edge_deg = edge_deg;
  p.volume_deg = dims == 2 ? 4 : 2;
  p.moments_deg = -1;
  p.steps_per_recompute = 1;
  p.recompute_threshold = 1e300;
  return p;
}

MeshBuf pairs_mesh(int n) {
  MeshBuf b;
  const double a[4][2] = {{0, 0}, {1, 0}, {0, 1}, {1, 1}};
  const int tri[2][3] = {{0, 1, 2}, {1, 3, 2}};
  for (int k = 0; k < n; ++k)
    for (auto &t : tri) {
      for (int v : t) {
        const double s = 0.1 * (1.0 + 0.3 * std::sin(k));
        b.vertex_ids.push_back(4 * k + v);
        b.corners.insert(b.corners.end(), {0.3 * (k % 7) + s * a[v][0], 0.3 * (k / 7) + s * a[v][1], 0.0});
      }
      b.ghost.push_back(k > 0);
      ++b.n_cells;
    }
  return b;
}

template <int DIM>
double conserved(int v, double s) {  // a state with pressure
  if (v == 0) return 1.0 + 0.3 * s;
  return v == DIM + 1 ? 3.0 + s : 0.4 * s;
}

template <int DIM>
std::unique_ptr<Instance> instance(const std::string &kind, int n, const zfv_params &p, uint64_t seed) {
  auto I = std::make_unique<Instance>();
  std::unique_ptr<MeshBuf> b;
  if (kind == "pairs") b = std::make_unique<MeshBuf>(pairs_mesh(n));
  else if (DIM == 3) b.reset(mesh_ball3d(n, 1.0, kind == "ghosts" ? 0.6 : 1.0, 0.1, seed));
  else b.reset(mesh_lattice2d(n, 0.2, seed, kind == "periodic", kind == "periodic", kind == "ghosts" ? 3 : 0));
  const zfv_mesh mesh{DIM, b->n_cells, b->vertex_ids.data(), b->corners.data(), b->ghost.data()};
  build_image(mesh, p, I->im);
  const HostImage &im = I->im;
  Img &m = I->m;
  m.n = im.n;
  m.ne = im.ne;
  m.n_near = im.n_near;
  m.crn = im.crn.data();
  m.vol = im.vol.data();
  m.inr = im.inr.data();
  m.meta = im.meta.data();
  m.cface = im.cface.data();
  m.fslot = im.fslot.data();
  m.fperm = im.fperm.data();
  m.gamma = p.gamma;
  m.flux = p.flux;
  m.flux_bc = p.flux_bc;
  m.gravity = p.gravity;
  for (size_t q = 0; q < im.face_w.size(); ++q) m.fw[q] = im.face_w[q];
  I->frm.assign(size_t(DIM + 1) * frame_words<DIM>() * im.n, kNaN);
  for (int64_t i = 0; i < im.n; ++i) store_face_frames<DIM>(m, i, I->frm.data());
  m.frm = I->frm.data();
  I->ffr.assign(size_t(frame_words<DIM>()) * im.ne, kNaN);
  for (int64_t e = 0; e < im.ne; ++e) store_face_table<DIM>(m, e, I->ffr.data());
  m.ffr = I->ffr.data();
  build_update_tiles(im, update_cells_of_wave(DIM), p.flux_bc == ZFV_FLUX_BC_CONSTANT, I->entries, I->off, I->more,
                     I->words);
  m.uent = I->entries.data();
  m.uoff = I->off.data();
  m.umore = I->more.data();
  m.ucell = I->words.data();
  const int nv = DIM + 2;
  std::uniform_real_distribution<double> r(-1.0, 1.0);
  I->U.resize(nv * im.n);
  for (size_t k = 0; k < I->U.size(); ++k) I->U[k] = conserved<DIM>(int(k % nv), r(rng));
  I->X.assign(nv * im.n, kNaN);
  I->K.assign(2 * nv * im.n, kNaN);
  I->src.resize(nv * im.n);
  for (double &s : I->src) s = r(rng);
  I->fpv.assign(size_t(DIM + 1) * ((im.s.q * nv + 1) & ~1) * im.n, kNaN);
  if (kind == "ghosts" || kind == "pairs") {
    I->steady.resize(nv * im.n);
    for (size_t k = 0; k < I->steady.size(); ++k) I->steady[k] = conserved<DIM>(int(k % nv), r(rng));
    m.steady = I->steady.data();
    for (size_t k = 0; k < I->U.size(); ++k)
      if (m.meta[k / nv] & META_GHOST) I->U[k] = I->steady[k];
  }
  return I;
}

// made-up point values of a state; only interior faces' slots hold any
template <int DIM, int Q>
void point_values(Instance &I, const std::vector<double> &U) {
  constexpr int NV = DIM + 2, NF = DIM + 1, SQ = slot_doubles<DIM, Q>();
  std::fill(I.fpv.begin(), I.fpv.end(), kNaN);
  for (int64_t s = 0; s < 2 * I.im.ne; ++s) {
    const int64_t slot = I.im.fslot[s], i = slot / NF;
    for (int q = 0; q < Q; ++q)
      for (int v = 0; v < NV; ++v)
        I.fpv[slot * SQ + q * NV + v] = U[i * NV + v] * (1.0 + 0.02 * std::sin(double(slot + 3 * q + v)));
    if (SQ > Q * NV) I.fpv[slot * SQ + Q * NV] = 0.0;
  }
}

// every face of every cell is where the cell's word says, once per tile
template <int DIM>
void check_tables(const Instance &I, bool flux_bc) {
  constexpr int NF = DIM + 1, CW = update_cells_of_wave(DIM);
  const HostImage &im = I.im;
  const int64_t tiles = (im.n + CW - 1) / CW;
  auto *first = reinterpret_cast<const UpdateFace *>(I.entries.data());
  auto *rest = reinterpret_cast<const UpdateFace *>(I.more.data());
  CHECK(int64_t(I.entries.size()) == 4 * 64 * tiles && int64_t(I.off.size()) == tiles + 1 && I.off[0] == 0);
  CHECK(int64_t(I.words.size()) == im.n && int64_t(I.more.size()) >= 4 * int64_t(I.off[tiles]));
  for (int64_t t = 0; t < tiles; ++t) {
    const int more = I.off[t + 1] - I.off[t];
    int count = 0;
    while (count < 64 && first[64 * t + count].l >= 0) ++count;
    for (int k = count; k < 64; ++k) CHECK(first[64 * t + k].l < 0);
    CHECK(more >= 0 && (more == 0 || count == 64) && count + more <= CW * NF);
    count += more;
    std::vector<int> uses(count, 0);
    auto entry = [&](int k) { return k < 64 ? first[64 * t + k] : rest[I.off[t] + k - 64]; };
    for (int64_t i = t * CW; i < std::min<int64_t>(im.n, (t + 1) * CW); ++i)
      for (int f = 0; f < NF; ++f) {
        const int32_t cf = im.cface[4 * i + f];
        const uint32_t at = (I.words[i] >> (8 * f)) & 0xFFu;
        const bool interior = !(cf & CFACE_EXTERIOR), boundary = !interior && flux_bc && !(cf & CFACE_SIDE_R);
        if (!interior && !boundary) {
          CHECK((at & 127u) == UPDATE_NO_FACE);
          continue;
        }
        CHECK(int(at & 127u) < count);
        const UpdateFace u = entry(at & 127u);
        uses[at & 127u] += 1;
        if (interior) {
          CHECK(u.r >= 0 && u.e == cf >> 2 && u.l == im.fslot[2 * u.e] && u.r == im.fslot[2 * u.e + 1]);
          CHECK(((at & 128u) != 0) == ((cf & CFACE_SIDE_R) != 0));
          CHECK((at & 128u ? u.r : u.l) == i * NF + f);
        } else {
          CHECK(u.r < 0 && u.e == i && u.f == f && !(at & 128u));
        }
      }
    for (int c : uses) CHECK(c == 1 || c == 2);
  }
}

// L of a state from its point values: all fluxes, then all cells
template <int DIM, int Q>
std::vector<double> rate(const Instance &I, const std::vector<double> &U) {
  constexpr int NV = DIM + 2;
  const int64_t n = I.m.n;
  std::vector<double> planes(NV * n), src(NV * n), G(NV * std::max<int64_t>(I.m.ne, 1)), L(NV * n);
  for (int64_t i = 0; i < n; ++i)
    for (int v = 0; v < NV; ++v) {
      planes[v * n + i] = U[i * NV + v];
      src[v * n + i] = I.src[i * NV + v];
    }
  for (int64_t e = 0; e < I.m.ne; ++e) face_flux<DIM, Q>(I.m, e, I.fpv.data(), G.data());
  for (int64_t i = 0; i < n; ++i) {
    double l[NV];
    cell_rate<DIM>(I.m, i, planes.data(), G.data(), src.data(), l);
    for (int v = 0; v < NV; ++v) L[i * NV + v] = l[v];
  }
  return L;
}

// one SSP3 step under the frozen BC, by the formulas
template <int DIM, int Q>
std::vector<double> step(Instance &I, const std::vector<double> &U, double dt) {
  const double c[3][3] = {{1.0, 0.0, 0.0}, {0.25, 0.25, 0.0}, {1.0 / 6, 1.0 / 6, 2.0 / 3}};
  std::vector<double> K[3], X = U;
  for (int s = 0; s < 3; ++s) {
    point_values<DIM, Q>(I, X);
    K[s] = rate<DIM, Q>(I, X);
    for (size_t k = 0; k < X.size(); ++k) {
      double sum = 0.0;
      for (int j = 0; j <= s; ++j) sum += c[s][j] * K[j][k];
      X[k] = U[k] + dt * sum;
      if (I.m.steady && (I.m.meta[k / (DIM + 2)] & META_GHOST)) X[k] = I.m.steady[k];
    }
  }
  return X;
}

template <int DIM>
double cfl_minimum(const Instance &I, const std::vector<double> &U) {
  double r = 1.0e300;
  for (int64_t i = 0; i < I.m.n; ++i) r = std::min(r, cfl_of_cell<DIM>(&U[i * (DIM + 2)], I.m.inr[i], I.m.gamma));
  return r;
}

// the tiles of one launch, in any order; work(tile, lds)
template <int DIM, class F>
void launch(int64_t cells, F &&work) {
  constexpr int CW = update_cells_of_wave(DIM);
  std::vector<int64_t> tiles((cells + CW - 1) / CW);
  std::iota(tiles.begin(), tiles.end(), 0);
  std::shuffle(tiles.begin(), tiles.end(), rng);
  for (int64_t t : tiles) {
    std::vector<double> lds(CW * (DIM + 1) * (DIM + 2), kNaN);
    work(t, lds.data());
  }
}

void expect(const std::vector<double> &a, const std::vector<double> &b) {
  CHECK(a.size() == b.size());
  for (size_t k = 0; k < a.size(); ++k) CHECK(same(a[k], b[k]));
}

template <int DIM, int Q>
void check_rate_and_steps(Instance &I) {
  const Img &m = I.m;
  HostWave w;
  const UpdateChecks none{nullptr, 0.0, nullptr};
  point_values<DIM, Q>(I, I.U);
  StageCoeffs only{};
  only.write_rate_only = 1;
  std::vector<double> L(I.U.size(), kNaN);
  const UpdateArgs ra{only, 0, 0.0, I.U.data(), I.fpv.data(), I.src.data(), I.U.data(), L.data(), nullptr};
  launch<DIM>(update_cells_of_stage(m, ra), [&](int64_t t, double *lds) { update_cells<DIM, Q>(m, ra, 0.0, none, t, lds, w); });
  expect(L, rate<DIM, Q>(I, I.U));
  // two steps of fixed dt
  const double dt = 0.1 * cfl_minimum<DIM>(I, I.U);
  std::vector<double> ref = I.U;
  for (int k = 0; k < 2; ++k) {
    ref = step<DIM, Q>(I, ref, dt);
    for (int s = 0; s < 3; ++s) {
      const std::vector<double> &from = s == 0 ? I.U : I.X;
      point_values<DIM, Q>(I, from);
      const UpdateArgs a{ssp3_coeffs(s), s, dt, from.data(), I.fpv.data(), I.src.data(), I.U.data(), I.K.data(),
                         s == 2 ? I.U.data() : I.X.data()};
      launch<DIM>(update_cells_of_stage(m, a), [&](int64_t t, double *lds) { update_cells<DIM, Q>(m, a, dt, none, t, lds, w); });
    }
    expect(I.U, ref);
  }
}

// the time loop of zfv_advance, with and without step rejection
template <int DIM, int Q>
void check_advance(Instance &I, double crit, double t_end_in_steps) {
  const Img &m = I.m;
  HostWave w;
  std::vector<double> ref = I.U;
  const double cfl = 0.4, t_end = t_end_in_steps * cfl * cfl_minimum<DIM>(I, ref), min_factor = 0.125;
  const int max_steps = 5, kAttempts = 30;
  // by the rules (TimeLoop, RejectLargeDensityChange)
  double t = 0.0, factor = 1.0, retry = 0.0;
  int steps = 0, rejected = 0;
  bool good = true;
  for (int k = 0; k < kAttempts && t < t_end && steps < max_steps; ++k) {
    double dt = retry > 0.0 ? retry : factor * (cfl * cfl_minimum<DIM>(I, ref));
    dt = std::min(dt, t_end - t);
    const std::vector<double> next = step<DIM, Q>(I, ref, dt);
    bool bad = false;
    if (crit > 0.0)
      for (int64_t i = 0; i < m.n; ++i) bad |= std::fabs(ref[i * (DIM + 2)] - next[i * (DIM + 2)]) > crit * ref[i * (DIM + 2)];
    retry = 0.0;
    if (bad) {
      good = false;
      factor = std::max(min_factor, std::min(factor / 2.0, 1.0));
      retry = factor * dt;
      ++rejected;
      continue;
    }
    if (crit > 0.0) {
      factor = std::max(min_factor, std::min(good ? factor * 2.0 : factor, 1.0));
      good = true;
    }
    ref = next;
    t += dt;
    ++steps;
  }
  AdvState a{};
  a.t_end = t_end;
  a.cfl = cfl;
  a.max_steps = max_steps;
  a.active = 1;
  a.drho_crit = crit;
  a.factor = 1.0;
  a.min_factor = crit > 0.0 ? min_factor : 1.0;
  a.prev_good = 1;
  std::vector<unsigned long long> slots(kAdvSlots * kAdvSlotStride, adv_no_bound());
  const double first = cfl_minimum<DIM>(I, I.U);
  std::memcpy(&slots[5 * kAdvSlotStride], &first, sizeof(first));
  for (int k = 0; k < kAttempts; ++k) {  // (steps past the end leave everything as it is)
    for (int s = 0; s < 3; ++s) {
      const std::vector<double> &from = s == 0 ? I.U : I.X;
      point_values<DIM, Q>(I, from);
      const UpdateArgs u{ssp3_coeffs(s), s, 0.0, from.data(), I.fpv.data(), I.src.data(), I.U.data(), I.K.data(),
                         s == 2 && !(crit > 0.0) ? I.U.data() : I.X.data()};
      launch<DIM>(update_cells_of_stage(m, u), [&](int64_t tile, double *lds) {
        update_cells_adv<DIM, Q>(m, u, &a, slots.data(), tile, lds, w);
      });
    }
    if (crit > 0.0) {  // the commit
      if (!a.bad && a.active) I.U = I.X;
      adv_end(&a);
    }
  }
  CHECK(bool(a.active) == (t < t_end && steps < max_steps));
  CHECK(same(a.t, t) && a.steps == steps && a.rejections == rejected);
  expect(I.U, ref);
}

// members of a batch, one of them ending by its step limit, one by its end time
template <int DIM, int Q>
void check_batch(const std::vector<Instance *> &members, bool xcd) {
  const int k_members = int(members.size());
  std::vector<DevInst> d(k_members);
  std::vector<std::vector<double>> ref(k_members);
  std::vector<double> t_ref(k_members, 0.0), dt_ref(k_members, 0.0);
  std::vector<int> n_ref(k_members, 0);
  std::vector<int64_t> cells(k_members);
  for (int k = 0; k < k_members; ++k) {
    Instance &I = *members[k];
    cells[k] = I.m.n;
    DevInst &x = d[k];
    x = DevInst{};
    x.m = I.m;
    x.U = I.U.data();
    x.X = I.X.data();
    x.K = I.K.data();
    x.fpv = I.fpv.data();
    x.src = I.src.data();
    x.cfl = 0.4;
    x.t_end = k == 0 ? 1.0 : 2.5 * 0.4 * cfl_minimum<DIM>(I, I.U);
    x.active = 1;
    x.max_steps = k == 0 ? 3 : 0x7fffffff;
    const double c = cfl_minimum<DIM>(I, I.U);
    std::memcpy(&x.dt_bits, &c, sizeof(c));
    ref[k] = I.U;
    while (t_ref[k] < x.t_end && n_ref[k] < x.max_steps) {
      const double dt = std::min(0.4 * cfl_minimum<DIM>(I, ref[k]), x.t_end - t_ref[k]);
      ref[k] = step<DIM, Q>(I, ref[k], dt);
      t_ref[k] += dt;
      dt_ref[k] = dt;
      ++n_ref[k];
    }
  }
  HostWave w;
  constexpr int CW = update_cells_of_wave(DIM);
  for (int k = 0; k < 6; ++k)
    for (int s = 0; s < 3; ++s) {
      for (int j = 0; j < k_members; ++j) {
        Instance &I = *members[j];
        if (d[j].active && (s == 0 ? kb_step_dt(d[j]) > 0.0 : d[j].running)) point_values<DIM, Q>(I, s == 0 ? I.U : I.X);
      }
      auto blocks = block_table(cells, update_cells_of_block(DIM), int64_t(1) << 30, xcd);
      std::shuffle(blocks.begin(), blocks.end(), rng);
      for (const BlockRef &b : blocks) {
        if (b.inst < 0) continue;
        int waves[4] = {0, 1, 2, 3};
        std::shuffle(waves, waves + 4, rng);
        for (int wave : waves) {
          DevInst &x = d[b.inst];
          double dt;
          if (!kb_update_begin(x, s, b.local == 0 && wave == 0, dt)) continue;
          const int64_t tile = int64_t(b.local) * 4 + wave;
          if (tile * CW >= x.m.n) continue;
          std::vector<double> lds(CW * (DIM + 1) * (DIM + 2), kNaN);
          update_cells<DIM, Q>(x.m, kb_update_args(x, ssp3_coeffs(s), s), dt, kb_update_checks(x, s), tile, lds.data(), w);
        }
      }
    }
  for (int k = 0; k < k_members; ++k) {
    CHECK(!d[k].active && same(d[k].t, t_ref[k]) && same(d[k].dt, dt_ref[k]) && d[k].steps_done == n_ref[k]);
    expect(members[k]->U, ref[k]);
  }
}

template <int DIM, int Q>
void run(const std::string &kind, int n, const zfv_params &p, uint64_t seed) {
  auto fresh = [&](int size) { return instance<DIM>(kind, size, p, seed); };
  auto I = fresh(n);
  check_tables<DIM>(*I, p.flux_bc == ZFV_FLUX_BC_CONSTANT);
  check_rate_and_steps<DIM, Q>(*I);
  for (double crit : {0.0, 0.02, 1e-9})
    for (double steps : {2.5, 100.0}) check_advance<DIM, Q>(*fresh(n), crit, steps);
  for (bool xcd : {false, true}) {
    auto a = fresh(n), b = fresh(n + 1);
    check_batch<DIM, Q>({a.get(), b.get()}, xcd);
  }
}

}  // namespace

int main(int argc, char **argv) {
  CHECK(argc == 8);
  const int dims = std::atoi(argv[1]), n = std::atoi(argv[2]);
  const std::string kind = argv[3];
  const zfv_params p = params(dims, std::atoi(argv[4]), std::atoi(argv[5]), std::atoi(argv[6]));
  const uint64_t seed = std::strtoull(argv[7], nullptr, 10);
  rng.seed(seed);
  const int q = shape_for(p).q;
  if (dims == 2 && q == 1) run<2, 1>(kind, n, p, seed);
  else if (dims == 2 && q == 2) run<2, 2>(kind, n, p, seed);
  else if (dims == 2 && q == 3) run<2, 3>(kind, n, p, seed);
  else if (dims == 3 && q == 3) run<3, 3>(kind, n, p, seed);
  else if (dims == 3 && q == 4) run<3, 4>(kind, n, p, seed);
  else CHECK(!"no such shape");
  std::printf("update_check: OK\n");
  return 0;
}
