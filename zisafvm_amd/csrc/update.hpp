// A stage's update: the face fluxes and the sum of every cell's, over tiles of
// cells (build_update_tiles), with what a time loop keeps up inside it.  Written
// once, for the gfx950 kernels (kernels.hip) and for checks on the host that run
// it over the library's own tables (tests/cpp/update_check.cpp).
#pragma once

#include <cstdint>
#include <cstring>

#include "batch.hpp"

namespace zfv {

struct StageCoeffs {
  double c[2];  // coefficients of the earlier stages' tendencies in the next state's sum
  double cl;    // and of this stage's own
  int write_rate_only;  // 1: store L in K[stage] (pinned host memory) and stop (zfv_rate)
};

inline StageCoeffs ssp3_coeffs(int stage) {
  // next-state coefficients after stage s: a[s+1][:] and b for the last stage
  // (src/zisa/ode/runge_kutta.cpp:154-165)
  if (stage == 0) return StageCoeffs{{0.0, 0.0}, 1.0, 0};
  if (stage == 1) return StageCoeffs{{0.25, 0.0}, 0.25, 0};
  return StageCoeffs{{1.0 / 6, 1.0 / 6}, 2.0 / 3, 0};
}

// A single instance's time loop on the device (zfv_advance): TimeLoop's
// step with LocalCFL (src/zisa/fvm_loops/time_loop.cpp:36-81,
// include/zisa/model/local_cfl_condition_impl.hpp:25-40), dt clamped to the
// end time as the simulation clock does (its library is not vendored in the
// reference), with no host round trip per step.
struct AdvState {
  double t, t_end, cfl, dt;
  int steps, max_steps, active;
  unsigned blocks_done;  // of k_adv_commit
  // RejectLargeDensityChange (src/zisa/ode/step_rejection.cpp:17-57; off
  // when drho_crit <= 0): factor scales the CFL step, halves on a rejected
  // step (which is retried with factor * its dt, TimeLoop::reject_step,
  // src/zisa/fvm_loops/time_loop.cpp:182-196) and doubles after two good
  // steps in a row, within [min_factor, 1]
  double drho_crit, factor, min_factor, retry_dt;
  int bad, prev_good, retry, rejections;
};

// The step's CFL minimum is reduced into kAdvSlots words of 128 bytes (one word
// would serialise thousands of atomics): the last stage's update leaves the new
// state's minimum there, the next step's first update picks dt from it, and the
// second stage's update sets the words back.
constexpr int kAdvSlots = 64, kAdvSlotStride = 16;
constexpr size_t kAdvSlotBytes = size_t(kAdvSlots) * kAdvSlotStride * sizeof(unsigned long long);

// start value of the CFL reduction (bits of 1e300)
ZFV_HD unsigned long long adv_no_bound() { return kb_no_bound(); }

// StepRejection::pick_time_step: factor * the CFL step, or the retry step;
// zero when finished, when the CFL gives no positive step (a non-physical
// state) or when the step no longer advances the time
ZFV_HD double adv_pick(const AdvState &a, double cfl_min) {
  double dt = a.retry ? a.retry_dt : a.factor * (a.cfl * cfl_min);
  const double rest = a.t_end - a.t;
  if (dt > rest) dt = rest;
  if (!a.active || !(dt > 0.0) || a.t + dt == a.t) dt = 0.0;  // the stages leave U as it is (U + 0 * dudt)
  return dt;
}

// the end of a step: the time advances, or the step is to be retried
ZFV_HD void adv_end(AdvState *a) {
  if (!a->active) return;
  const int bad = a->bad;
  a->bad = 0;
  a->retry = 0;
  if (a->drho_crit > 0.0) {
    const double f = a->factor;
    if (bad) {
      a->prev_good = 0;
      a->factor = fmax(a->min_factor, fmin(f / 2.0, 1.0));
      a->retry = 1;
      a->retry_dt = a->factor * a->dt;
      a->rejections += 1;
      return;  // the time does not advance; the state was kept
    }
    a->factor = fmax(a->min_factor, fmin(a->prev_good ? f * 2.0 : f, 1.0));
    a->prev_good = 1;
  }
  a->t += a->dt;
  a->steps += 1;
  if (a->t >= a->t_end || a->steps >= a->max_steps) a->active = 0;
}

// What the last stage's update also does in a time loop that chooses its steps:
// the new state's CFL minimum goes to cfl[slot] (null: not wanted), a density
// change of more than crit times its old value in any cell sets *bad (crit 0:
// not asked)
struct UpdateChecks {
  unsigned long long *cfl;
  double crit;
  int *bad;
};

// What a stage's update reads and writes: K[stage] = L(Ustage); Unext = U0 +
// dt * sum_j c_j K[j] (src/zisa/ode/runge_kutta.cpp:122-143), then FrozenBC for
// ghost cells.  Ustage, U0 and Unext may name the same buffer (stages 1 and 2
// read and write the stage state X; a wavefront reads only its own cells'
// entries, before it writes them), so none of them is declared __restrict__.
struct UpdateArgs {
  StageCoeffs sc;
  int stage;
  double dt;  // (zfv_advance: chosen on the device)
  const double *Ustage, *fpv, *src, *U0;
  double *K, *Unext;
};

// Cells of an update wavefront: as many as have about 64 faces between them
// along the cells' Hilbert order (32 triangles 58 on average and 66 at most on
// the jittered lattices, 20 tetrahedra 62 and 68 in the ball), and of a block
constexpr int update_cells_of_wave(int dim) { return dim == 2 ? 32 : 20; }
constexpr int update_cells_of_block(int dim) { return 4 * update_cells_of_wave(dim); }

// The update of a wavefront's tile of cells.  First each lane forms the flux
// through one of the tile's faces (build_update_tiles; a face between two tiles
// is evaluated by both, with the same operands in the same order: conservation
// holds bit for bit), then one lane per cell and variable sums its cell's
// fluxes, which it reads from LDS (lds: NF CW NV doubles).  Bound by latency:
// a wavefront is one chain of entry, point values, flux, sum, so everything
// the sum needs is loaded first.  Against a kernel over faces and one over
// cells it does without a flux array in memory and takes one launch less:
// 263,520 triangles (3 points a face) 44 -> 34 us, 201,196 tetrahedra 42 -> 38,
// 1,152 triangles 9.4 -> 4.8.  (One lane per cell face, every face evaluated
// twice: 48, 50 and 5.0 us; four wavefronts per SIMD spill in 3D: 54 us.)
//
// W is the wavefront: each() runs a part of the work once per lane, with the
// lane's registers, and what one part leaves in LDS the next may read after
// sync().  (The host's checks run the lanes one after another.)
template <int DIM>
struct UpdateRegs {
  static constexpr int NP = (update_cells_of_wave(DIM) * (DIM + 2) + 63) / 64;  // passes over the tile's cells and variables
  double part[NP], base[NP], src[NP], vol[NP];
  uint32_t word[NP];
  bool inside[NP], frozen_cell[NP];
};

template <int DIM, int Q, class W>
ZFV_HD void update_cells(const Img &m, const UpdateArgs &a, double dt, const UpdateChecks &chk, int64_t tile, double *lds,
                         W &w) {
  constexpr int NV = DIM + 2;
  constexpr int NF = DIM + 1;
  constexpr int CW = update_cells_of_wave(DIM);
  constexpr int NP = UpdateRegs<DIM>::NP;
  const int64_t n = m.n;
  const int64_t i0 = tile * CW;
  typename W::template Lanes<UpdateRegs<DIM>> regs;
  w.each(regs, [&](int lane, UpdateRegs<DIM> &r) {
    const UpdateFace mine = reinterpret_cast<const UpdateFace *>(m.uent)[tile * 64 + lane];
    const int more0 = m.uoff[tile], more1 = m.uoff[tile + 1];
    // What the second part needs besides the fluxes is loaded first, to be in
    // flight with the faces' entries and point values
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int e = p * 64 + lane, c = e / NV;
      int64_t i = i0 + c;
      r.inside[p] = e < CW * NV && i < n;
      i = r.inside[p] ? i : i0;
      const int64_t at = i * NV + (e - c * NV);
      const int32_t meta = m.meta[i];
      r.word[p] = m.ucell[i];
      r.vol[p] = m.vol[i];
      r.src[p] = m.gravity != 0 && a.src != nullptr ? a.src[at] : 0.0;
      r.part[p] = r.base[p] = 0.0;
      if (!a.sc.write_rate_only) {
        r.base[p] = a.U0[at];
#pragma unroll
        for (int j = 0; j < 2; ++j)
          if (j < a.stage && a.sc.c[j] != 0.0) r.part[p] += a.sc.c[j] * a.K[int64_t(j) * NV * n + at];
      }
      // frozen ghost cells keep the steady state whatever their fluxes
      r.frozen_cell[p] = !a.sc.write_rate_only && (meta & 16) != 0 && m.steady != nullptr;
      if (r.frozen_cell[p]) r.base[p] = m.steady[at];
    }
    UpdateFace face = mine;
    for (int k = lane; face.l >= 0;) {
      double g[NV];
      update_face_flux<DIM, Q>(m, face, a.Ustage, a.fpv, g);
#pragma unroll
      for (int v = 0; v < NV; ++v) lds[k * NV + v] = g[v];
      k += 64;  // (tiles of more than 64 faces)
      if (k >= 64 + more1 - more0) break;
      face = reinterpret_cast<const UpdateFace *>(m.umore)[more0 + k - 64];
    }
  });
  w.sync();
  w.each(regs, [&](int lane, UpdateRegs<DIM> &r) {
    bool bad = false;
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      if (!r.inside[p]) continue;
      const int e = p * 64 + lane, v = e % NV;
      const int64_t at = i0 * NV + e;
      // RejectLargeDensityChange::check: |rho1 - rho0| > crit rho0
      auto check = [&](double r0, double r1) {
        bad |= v == 0 && fabs(r0 - r1) > chk.crit * r0;
      };
      if (r.frozen_cell[p]) {
        if (chk.crit > 0.0) check(a.U0[at], r.base[p]);
        a.Unext[at] = r.base[p];
        continue;
      }
      double L = 0.0;
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const uint32_t k = (r.word[p] >> (8 * f)) & 127u;
        const bool right = (r.word[p] >> (8 * f)) & 128u;
        if (k != UPDATE_NO_FACE) {
          const double g = lds[k * NV + v];
          L += right ? g : -g;
        }
      }
      L = L / r.vol[p];
      if (m.gravity != 0 && a.src != nullptr) L += r.src[p];
      // the last stage's tendency enters only its own sum (no later stage reads it)
      if (a.sc.write_rate_only || a.stage < 2) a.K[int64_t(a.stage) * NV * n + at] = L;
      if (a.sc.write_rate_only) continue;
      const double un = r.base[p] + dt * (r.part[p] + a.sc.cl * L);
      if (chk.crit > 0.0) check(r.base[p], un);
      r.base[p] = un;
      a.Unext[at] = un;
    }
    if (bad) w.flag(chk.bad);
  });
  if (chk.cfl == nullptr) return;
  // the CFL minimum of the new state: its values go through LDS to one lane a cell
  w.sync();
  w.each(regs, [&](int lane, UpdateRegs<DIM> &r) {
#pragma unroll
    for (int p = 0; p < NP; ++p)
      if (p * 64 + lane < CW * NV) lds[p * 64 + lane] = r.base[p];
  });
  w.sync();
  w.lower(chk.cfl, [&](int lane) {
    return lane < CW && i0 + lane < n ? cfl_of_cell<DIM>(lds + lane * NV, m.inr[i0 + lane], m.gamma) : 1.0e300;
  });
}

// The cells that a stage's update covers: under the frozen BC the second leaves
// out the ghosts away from the interior, whose X the first has set (the third
// sets U)
ZFV_HD int64_t update_cells_of_stage(const Img &m, const UpdateArgs &a) {
  return !a.sc.write_rate_only && m.steady != nullptr && a.stage == 1 && m.n_near > 0 ? m.n_near : m.n;
}

// The update inside the time loop of zfv_advance, with its bookkeeping: the
// first stage picks the step's dt (every wavefront for itself, the first one
// for the record), the second sets the CFL words back and, without step
// rejection, advances the time, the third reduces the next step's CFL minimum.
template <int DIM, int Q, class W>
ZFV_HD void update_cells_adv(const Img &m, const UpdateArgs &a, AdvState *adv, unsigned long long *slots, int64_t tile,
                             double *lds, W &w) {
  double dt;
  struct None {};
  typename W::template Lanes<None> none;
  if (a.stage == 0) {
    dt = adv_pick(*adv, w.least([&](int lane) {
      double r;
      memcpy(&r, &slots[lane * kAdvSlotStride], sizeof(r));
      return r;
    }));
    if (tile == 0)
      w.each(none, [&](int lane, None &) {
        if (lane != 0) return;
        adv->dt = dt;
        if (!(dt > 0.0)) adv->active = 0;
      });
  } else {
    dt = adv->dt;
    if (a.stage == 1 && tile == 0)
      w.each(none, [&](int lane, None &) {
        slots[lane * kAdvSlotStride] = adv_no_bound();
        if (lane == 0 && !(adv->drho_crit > 0.0)) adv_end(adv);
      });
  }
  UpdateChecks chk{nullptr, 0.0, nullptr};
  if (a.stage == 2) chk = UpdateChecks{slots + (tile & (kAdvSlots - 1)) * kAdvSlotStride, adv->drho_crit, &adv->bad};
  update_cells<DIM, Q>(m, a, dt, chk, tile, lds, w);
}

// ---- a batch's update -----------------------------------------------------------
// A thread's part of its member's bookkeeping in a stage's update (first: the
// member's first thread): its dt; false: the member makes no step.  The step's
// dt comes from the CFL minimum of the member's state: every thread forms the
// same value, and the first records it for the later stages (and stops a member
// that cannot advance or has finished, whose threads all leave).  The time and
// the CFL minimum are not read before the next step's first stage but by the
// last stage's reduction, so the second stage ends the step.
ZFV_HD bool kb_update_begin(DevInst &d, int stage, bool first, double &dt) {
  if (!d.active) return false;
  dt = d.dt;
  if (stage == 0) {
    dt = kb_step_dt(d);
    if (first) kb_begin_instance(d, dt);
    return dt > 0.0;
  }
  if (!d.running) return false;
  if (stage == 1 && first) kb_end_instance(d);
  return true;
}

ZFV_HD UpdateArgs kb_update_args(const DevInst &c, const StageCoeffs &sc, int stage) {
  return UpdateArgs{sc, stage, 0.0, stage == 0 ? c.U : c.X, c.fpv, c.src, c.U, c.K, stage == 2 ? c.U : c.X};
}

ZFV_HD UpdateChecks kb_update_checks(DevInst &d, int stage) {
  return UpdateChecks{stage == 2 ? &d.dt_bits : nullptr, 0.0, nullptr};
}

}  // namespace zfv
