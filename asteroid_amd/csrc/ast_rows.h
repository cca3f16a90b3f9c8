// ast_rows.h -- the evaluator with several lanes per model.
//
// With one lane per model a launch of few models leaves the chip idle: 4096
// models are 64 wavefronts on 1024 SIMDs, and a wavefront alone on its SIMD
// issues one FP64 instruction every 4.3 cycles whatever its lanes hold, so
// its time is its instruction count (600 per point of the torque form: 1.35
// RK4 steps of 248 and 263 of brightness, 1.3 us).  Here LP = 16 or 4
// neighbouring lanes (a DPP row or quad) share one model and the count per
// point falls to about 300 or 350 (0.70 and 0.90 us):
//
//   * the two sine/cosine pairs of an RK4 stage (theta and psi; without
//     torque theta and 2 psi) are one call, even lanes taking the first angle
//     and odd lanes the second, the results handed round by DPP moves (a step
//     is then 197 instructions);
//   * the brightness, which needs only the Euler angles at its point, runs
//     once per LP points, lane j doing point j of the batch;
//   * the chi^2 sums then take the batch's residuals in the points' order.
//
// Where SIMDs are still free, a team of wavefronts walks the models of one:
// the Euler angles are a serial chain that nothing else has to wait in.  Their
// wavefront is left 153 instructions a step (132 without torque); with torque
// a second one integrates the angular velocity, which does not depend on the
// angles, ahead of it, and another one follows with the brightness and the
// sums (0.61 us per point; a 57-point chi^2 call of one model 93 -> 76 us).
//
// Every value comes from the same operations on the same operands as in
// chi2_model, in the same order where order matters (the integration and the
// sums), so the results are bitwise those of one lane per model.  The
// lanes of a model hold equal values of everything but the shared angle and
// the brightness.
#pragma once
#include "ast_device.h"

namespace ast {

// The intrinsic behind the DPP builtins, which take 32-bit values only: a
// 64-bit row broadcast is one v_mov_b64 on gfx950.
__device__ long long dpp_mov_b64(long long old, long long src, int ctrl, int row_mask, int bank_mask,
                                 bool bound_ctrl) __asm("llvm.amdgcn.update.dpp.i64");

// The table as vector loads read it (a generic pointer would make them FLAT
// loads, which the table reads in LDS have to wait for).
typedef __attribute__((address_space(1))) const PointRec* LanePtr;

// A team's exchange buffers: 64 / LP models, each a row of LP lanes in every
// one of its wavefronts.
typedef double double2x __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) double2x* SpinPtr;
template <bool TQ, int LP>
struct TeamLds {
  static constexpr int STEPS = LP == 16 ? 4 : 8;  // RK4 steps between two barriers
  double2x spin[TQ ? 2 : 1][STEPS][64 / LP][6];   // angular velocities of a step's later stages and its end
  double angle[2][LP][64];                        // of a point: theta, psi and phi in lanes 0, 1, 2 of a row
};
template <int VC, int LP>
using TeamPtr = __attribute__((address_space(3))) TeamLds<VarF<VC>::TQ, LP>*;
enum { ROLE_ALL, ROLE_ANGLES, ROLE_SPIN, ROLE_LIGHT };

// As pin_sgpr, for a value a vector load gives: what was loaded before this
// point is waited for here and not, over and over, at its uses in a loop.
template <class T> __device__ inline void pin_vgpr(T& v) { asm volatile("" : "+v"(v)); }

// Value of lane K of the caller's LP-lane group.
template <int LP, int K>
AST_AI double lane_of(double x) {
  static_assert(LP == 16 || LP == 4, "a DPP row or a quad");
  const long long b = __builtin_bit_cast(long long, x);
  if constexpr (LP == 16) {
    return __builtin_bit_cast(double, dpp_mov_b64(0, b, 0x150 + K, 0xf, 0xf, true));  // row_newbcast:K
  } else {
    constexpr int ctrl = K * 0x55;  // quad_perm:[K,K,K,K]
    const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)b, ctrl, 0xf, 0xf, true);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(b >> 32), ctrl, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
  }
}

// f(integral_constant<int, 0>), ..., f(integral_constant<int, N - 1>).
template <int K>
struct IntC {
  static constexpr int value = K;
};
template <int N, int K = 0, class F>
AST_AI void unroll_lanes(const F& f) {
  if constexpr (K < N) {
    f(IntC<K>{});
    unroll_lanes<N, K + 1>(f);
  }
}

// One RK4 step of the shared integration (cuda.c:348-372).  w holds the
// angular velocity (torque form only), phi the first Euler angle and p the
// lane's angle (theta on even lanes, psi on odd ones); sc the sine/cosine
// pairs at the step's start (theta and psi, without torque theta and 2 psi),
// replaced by those at its end.  The same operations as
// rk4_step's; their order puts the next stage's table read as early as
// its angle is known (the barrier keeps it there) and the angular velocity's
// part of the stage behind it, so that a wavefront alone on its SIMD does not
// wait for the read.  With FED the angular velocities at the later stages and
// the step's end are read from rec, where another wavefront left them.
template <bool TQ, int LP, bool FED = false>
AST_AI void rk4_shared(double* w, double& phi, double& p, double* sc, const double* mu, double mu02, bool odd,
                       double h, double hh, double h6, SpinPtr rec = nullptr) {
  const double twice = odd ? 2.0 : 1.0;  // without torque the odd lanes' argument is 2 psi
  double sw[3] = {0, 0, 0}, fw[3] = {w[0], w[1], w[2]}, sphi, sp;
  double2x fed[6];
  if constexpr (FED) {
#pragma unroll
    for (int k = 0; k < 6; ++k) fed[k] = rec[k];
  }
#pragma unroll
  for (int stage = 0; stage < 4; ++stage) {
    double kphi, kp;
    if (TQ) {
      kphi = astm::div_rn(__builtin_fma(fw[1], sc[3], fw[0] * sc[2]), sc[0]);
      const double kth = __builtin_fma(-fw[1], sc[2], fw[0] * sc[3]);
      const double kps = __builtin_fma(-kphi, sc[1], fw[2]);
      kp = odd ? kps : kth;
    } else {
      kphi = mu[0] * __builtin_fma(-mu[2], sc[3], mu[1]);
      const double kth = (mu02 * sc[0]) * sc[2];
      const double kps = sc[1] * (mu[0] - kphi);
      kp = odd ? kps : kth;
    }
    const double hs = stage < 2 ? hh : h;
    double a;
    if (stage < 3) {
      a = __builtin_fma(hs, kp, p);
    } else {
      p = __builtin_fma(h6, sp + kp, p);
      a = p;
    }
    if (!TQ) a = twice * a;
    const double kb = astm::sincos_t_k(a);
    double ts, tc, s, c;
    astm::sctab_get(astm::sctab_index(kb), &ts, &tc);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (FED) {
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const int k = 3 * stage + j;
        if (stage < 3) fw[j] = fed[k / 2][k % 2];
        else w[j] = fed[k / 2][k % 2];
      }
    } else if (TQ) {
      spin_stage(stage, w, fw, sw, mu, hs, h6);
    }
    if (stage == 0) {
      sphi = kphi;
      sp = kp;
    } else if (stage < 3) {
      sphi = __builtin_fma(2.0, kphi, sphi);
      sp = __builtin_fma(2.0, kp, sp);
    } else {
      phi = __builtin_fma(h6, sphi + kphi, phi);
    }
    astm::sincos_t_end(a, kb, ts, tc, &s, &c);
    sc[0] = lane_of<LP, 0>(s);
    sc[1] = lane_of<LP, 0>(c);
    sc[2] = lane_of<LP, 1>(s);
    sc[3] = lane_of<LP, 1>(c);
  }
}

// The angular velocity's part of an RK4 step alone, its values at the later
// stages and the end left in rec for rk4_shared.
AST_AI void rk4_spin(double* w, const double* mu, double h, double hh, double h6, SpinPtr rec) {
  double sw[3], fw[3] = {w[0], w[1], w[2]}, out[12];
#pragma unroll
  for (int stage = 0; stage < 4; ++stage) {
    spin_stage(stage, w, fw, sw, mu, stage < 2 ? hh : h, h6);
#pragma unroll
    for (int j = 0; j < 3; ++j) out[3 * stage + j] = stage < 3 ? fw[j] : w[j];
  }
#pragma unroll
  for (int k = 0; k < 6; ++k) rec[k] = double2x{out[2 * k], out[2 * k + 1]};
}

// chi2_model with LP lanes per model (same arguments, same results in every
// lane of a model).  All lanes of a model must be active together.  With
// FORM_PLOT vplot is the model's own curve (stride 1).
//
// ROLE other than ROLE_ALL is one wavefront's part of a team of two (without
// torque) or three that walks the curve together, exchanging through `team`:
//   ROLE_SPIN    the angular velocities, a chunk of TEAM_STEPS steps ahead,
//   ROLE_ANGLES  the Euler angles, from those,
//   ROLE_LIGHT   brightness and sums of the batch of points before.
// All three run the same loops over the curve's steps and meet at a barrier
// where ROLE_ANGLES starts a chunk (a batch's last chunk may be short, and a
// batch without steps has one too) and once more at the end.  Both buffers
// are used in turn: while chunk k is read chunk k + 1 is written; a batch's
// angles are read between the next batch's first barrier and its second, and
// written again from the first barrier after that on.
template <class CF, int VC, int NF, bool MX, int FORM, int LP, int ROLE = ROLE_ALL>
__device__ CF chi2_model_rows(const double* params, PointPtr pts, LanePtr pts_g, int n_data, int n_filters, int dof,
                              const double* sum_w, CF* dV, double* vplot = nullptr, double dv0 = 0.0,
                              TeamPtr<VC, LP> team = nullptr) {
  using P = Pos<VC>;
  AST_VFLAGS(VC);
  static_assert(ROLE == ROLE_ALL || !T2, "a team's models share their step counts");
  constexpr int TEAM_STEPS = TeamLds<TQ, LP>::STEPS;
  static_assert(!(TR && (T2 || NU)), "PointRec.aux is the phase angle under TREND and the time otherwise");
  const int lane = (int)__lane_id() & (LP - 1);
  const bool odd = lane & 1;
  // With several filters a lane keeps the sums of filter lane (and lane + LP
  // where there are more filters than lanes); with one, every lane keeps them.
  constexpr int SLOTS = NF == 1 ? 1 : (NF + LP - 1) / LP;
  double sy2[SLOTS], sy[SLOTS];
#pragma unroll
  for (int m = 0; m < SLOTS; ++m) { sy2[m] = 0.0; sy[m] = 0.0; }
  const double bt = params[P::b_tumb], ct = params[P::c_tumb];
  const double den = __builtin_fma(ct, ct, bt * bt);
  const double Is = __builtin_fma(bt, bt, 1.0) / den;
  const double Ii = __builtin_fma(ct, ct, 1.0) / den;
  const double Is_inv = 1.0 / Is;
  const double Ii_inv = 1.0 / Ii;
  SpinFrame<double> Fd;
  double mu[6];
  double mu02 = 0.0;
  double w[3] = {0, 0, 0}, phi, p, sc[4];
  // The rotation's start (or a segment's): the state as begin_rotation gives
  // it, the lane's angle picked out, and without torque the sine and cosine
  // of 2 psi beside those of theta.
  auto begin = [&](int k) {
    double y[6];
    begin_rotation<VC>(params, k, Is_inv, Ii_inv, Is, Ii, Fd, y, mu, mu02, sc);
    if (TQ) {
      w[0] = y[0]; w[1] = y[1]; w[2] = y[2];
      phi = y[3];
      p = odd ? y[5] : y[4];
    } else {
      phi = y[0];
      p = odd ? y[2] : y[1];
      astm::sincos_t(2.0 * y[2], &sc[2], &sc[3]);
    }
  };
  begin(0);
  ModelConsts K{0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  if constexpr (RO) {
    astm::sincos_t(params[P::phi_R], &K.sR, &K.cR);
    astm::sincos_t(params[P::theta_R], &K.stR, &K.ctR);
    astm::sincos_t(params[P::psi_R], &K.sPR, &K.cPR);
  }
  if (BW) {
    astm::sincos_t(params[P::phi_R], &K.sR, &K.cR);
    astm::sincos_t(params[P::theta_R], &K.stR, &K.ctR);
    K.kappa = params[P::kappa];
  } else {
    const double b = BC ? params[P::b] : bt;
    const double c = BC ? params[P::c] : ct;
    K.ib = 1.0 / b;
    K.ic = 1.0 / c;
    K.bcp = b * c;
  }
  const float bcpf = (float)K.bcp;  // mixed form
  float nu_t[NU ? NU_M_MAX : 1], nu_V[NU ? NU_M_MAX : 1];
  NudgeState nu;
  nu.t_mod = nu_t;
  nu.V_mod = nu_V;
  TailPtr mr = (TailPtr)(pts + n_data);
  double trendA = 0.0, t_split = 0.0;
  if constexpr (TR) trendA = params[P::A];
  bool switched = false;
  if constexpr (T2)  // cuda.c:291
    t_split = __builtin_fma(params[P::Tt], pts[n_data - 1].aux - pts[0].aux, pts[0].aux);
  // Each lane reads the record of its own point of a batch (the curve's last
  // one, for lanes beyond it, whose results are left out) with vector loads:
  // the step count and size a batch ahead, handed out point by point with
  // readlane, the rest while the batch is integrated.  Scalar loads of the
  // records one point ahead were waited for at every point, since they share
  // their counter with the table reads: 0.62 us per point of a one-model
  // plot.
  const int row0 = __builtin_amdgcn_readfirstlane((int)__lane_id()) & ~(LP - 1);
  int nx_steps = pts_g[lane < n_data ? lane : n_data - 1].nsteps;
  double nx_h = pts_g[lane < n_data ? lane : n_data - 1].h;
  pin_vgpr(nx_steps);
  pin_vgpr(nx_h);
  int left = 0;  // a team's: steps until the next barrier
  int spin_buf = 0, angle_buf = 0;
  const int row = (int)__lane_id() / LP;
  if constexpr (ROLE == ROLE_ANGLES) spin_buf = 1;
  if constexpr (ROLE == ROLE_LIGHT) __syncthreads();
  for (int i0 = 0; i0 < n_data; i0 += LP) {
    if constexpr (ROLE == ROLE_ANGLES) {
      __syncthreads();
      spin_buf ^= 1;
    }
    left = TEAM_STEPS;
    const int m = n_data - i0 < LP ? n_data - i0 : LP;
    const int lane_steps = nx_steps;
    const uint64_t lane_h = astm::bits_of(nx_h);
    {
      const int nx = i0 + LP + lane;
      nx_steps = pts_g[nx < n_data ? nx : n_data - 1].nsteps;
      nx_h = pts_g[nx < n_data ? nx : n_data - 1].h;
    }
    const LanePtr pr = pts_g + (i0 + (lane < m ? lane : m - 1));
    const double E[3] = {pr->E[0], pr->E[1], pr->E[2]};
    const double S[3] = {pr->S[0], pr->S[1], pr->S[2]};
    const float pV = pr->V, pw = pr->w;
    double aux = 0.0;
    if constexpr (TR) aux = pr->aux;
    int lane_filter = 0;
    if constexpr (NF > 1) lane_filter = pr->filter;
    double cphi = 0.0, cth = 0.0, cps = 0.0;  // the Euler angles at the lane's point
    SpinFrame<double> Fl = Fd;                // and, with segments, its spin frame
    for (int j = 0; j < m; ++j) {
      const int i = i0 + j;
      int nsteps = __builtin_amdgcn_readlane(lane_steps, row0 + j);
      const uint32_t h_lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)lane_h, row0 + j);
      const uint32_t h_hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(lane_h >> 32), row0 + j);
      double h = astm::of_bits(((uint64_t)h_hi << 32) | h_lo);
      double hh = 0.5 * h, h6 = 1 / 6.0 * h;  // as the table's
      if constexpr (SG) {
        if (nsteps < 0) begin(-1 - nsteps);
      }
      if constexpr (ROLE == ROLE_LIGHT) {
        for (left -= nsteps > 0 ? nsteps : 0; left < 0; left += TEAM_STEPS) __syncthreads();
        if constexpr (SG) {
          if (lane == j) Fl = Fd;
        }
        continue;
      }
      if constexpr (ROLE == ROLE_ANGLES || ROLE == ROLE_SPIN) {
        for (int l = 0; l < nsteps; ++l) {
          if (left == 0) {
            __syncthreads();
            spin_buf ^= 1;
            left = TEAM_STEPS;
          }
          const SpinPtr rec = team->spin[TQ ? spin_buf : 0][TEAM_STEPS - left][row];
          if constexpr (ROLE == ROLE_ANGLES) rk4_shared<TQ, LP, TQ>(w, phi, p, sc, mu, mu02, odd, h, hh, h6, rec);
          else rk4_spin(w, mu, h, hh, h6, rec);
          --left;
        }
        if constexpr (ROLE == ROLE_ANGLES) team->angle[angle_buf][j][__lane_id()] = lane == 2 ? phi : p;
        continue;
      }
      int nsub = 1;
      double t2_end = 0.0;
      if constexpr (T2) {  // cuda.c:288-317
        if (i > 0 && !switched && t_split >= pts[i - 1].aux && t_split < pts[i].aux) {
          const double t1 = pts[i - 1].aux;
          nsub = 2;
          t2_end = pts[i].aux;
          nsteps = (int)((t_split - t1) / mr->ts + 1);
          h = (t_split - t1) / nsteps;
          hh = 0.5 * h;
          h6 = 1 / 6.0 * h;
        }
      }
      for (int isub = 0; isub < nsub; ++isub) {
        if constexpr (T2) {
          if (isub == 1) {
            nsteps = (int)((t2_end - t_split) / mr->ts + 1);
            h = (t2_end - t_split) / nsteps;
            hh = 0.5 * h;
            h6 = 1 / 6.0 * h;
            mu[3] = params[P::T2i];
            mu[4] = params[P::T2s];
            mu[5] = params[P::T2l];
            switched = true;
          }
        }
        for (int l = 0; l < nsteps; ++l) rk4_shared<TQ, LP>(w, phi, p, sc, mu, mu02, odd, h, hh, h6);
      }
      const double th = lane_of<LP, 0>(p), ps = lane_of<LP, 1>(p);
      const bool mine = lane == j;
      cphi = mine ? phi : cphi;
      cth = mine ? th : cth;
      cps = mine ? ps : cps;
      if constexpr (SG) {
        if (mine) Fl = Fd;
      }
    }
    pin_vgpr(nx_steps);
    pin_vgpr(nx_h);
    if constexpr (ROLE == ROLE_ANGLES) {
      angle_buf ^= 1;
      continue;
    }
    if constexpr (ROLE == ROLE_SPIN || ROLE == ROLE_LIGHT) __syncthreads();
    if constexpr (ROLE == ROLE_SPIN) {
      spin_buf ^= 1;
      continue;
    }
    if constexpr (ROLE == ROLE_LIGHT) {
      const auto angle = &team->angle[angle_buf][lane][row * LP];
      cth = lane < m ? angle[0] : 0.0;
      cps = lane < m ? angle[1] : 0.0;
      cphi = lane < m ? angle[2] : 0.0;
      angle_buf ^= 1;
    }
    // Brightness of the lane's point.
    double asc[4], a[3], b[3], c[3];
    astm::sincos_t(cth, &asc[0], &asc[1]);
    if (TQ) astm::sincos_t(cps, &asc[2], &asc[3]);
    axes_at<TQ>(SG ? Fl : Fd, cphi, cps, asc, a, b, c);
    if constexpr (RO) rotate_axes(a, b, c, K);
    double Vmod;
    if constexpr (RC) {
      Vmod = rect_mag(a, b, c, E, params[P::b], params[P::c]);
    } else if (BW) {
      const double arg = bw_arg_f64(a, b, c, E, K);
      Vmod = MX ? M2P5_LOG10_2 * log2_f32x((float)arg) : -2.5 * astm::log10(arg);
    } else {
      const ScaledDirs u = scaled_dirs(a, b, c, E, S, K);
      if (MX) Vmod = ls_tail_mx(u, bcpf);
      else Vmod = ls_tail_f64(u, K.bcp);
    }
    if constexpr (TR) Vmod = __builtin_fma(-trendA, aux, Vmod);  // cuda.c:692-697
    if constexpr (NU) {
      // The minima are found point by point, by every lane alike.
      const int base = (int)__lane_id() & ~(LP - 1);
      for (int j = 0; j < m; ++j) {
        const double Vj = __shfl(Vmod, base + j);
        if constexpr (FORM == FORM_PLOT)
          if (lane == j) vplot[i0 + j] = nu.failed ? __builtin_nan("") : Vj + dv0;
        nu.point(i0 + j, pts[i0 + j].aux, Vj, mr);
      }
    }
    if constexpr (FORM == FORM_PLOT) {
      if constexpr (!NU)
        if (lane < m) vplot[i0 + lane] = Vmod + dv0;
      continue;
    }
    // The sums, in the points' order.  Lanes past the curve's end give a
    // residual and a weight of 0, which leave the sums as they are (a sum
    // that is an exact zero is +0).
    const bool in = lane < m;
    const double wl = in ? (double)pw : 0.0;
    const double yv = in ? (double)pV - Vmod : 0.0;
    const double yq = yv * yv;
    unroll_lanes<LP>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      const double yj = lane_of<LP, j>(yv), qj = lane_of<LP, j>(yq), wj = lane_of<LP, j>(wl);
      if constexpr (NF == 1) {
        sy2[0] = __builtin_fma(qj, wj, sy2[0]);
        sy[0] = __builtin_fma(yj, wj, sy[0]);
      } else {
        const int f = __builtin_amdgcn_readlane(lane_filter, row0 + j);
#pragma unroll
        for (int k = 0; k < SLOTS; ++k)
          if (lane + k * LP == f) {
            sy2[k] = __builtin_fma(qj, wj, sy2[k]);
            sy[k] = __builtin_fma(yj, wj, sy[k]);
          }
      }
    });
  }
  if constexpr (ROLE == ROLE_ANGLES || ROLE == ROLE_SPIN) {
    __syncthreads();
    return CF(0.0);
  }
  if constexpr (FORM == FORM_PLOT) return CF(0.0);
  if constexpr (NU)
    if (nu.failed) return CF(1e30);
  double all2[NF], all1[NF];
  unroll_lanes<NF>([&](auto mc) {
    constexpr int m = decltype(mc)::value;
    all2[m] = NF == 1 ? sy2[0] : lane_of<LP, m % LP>(sy2[m / LP]);
    all1[m] = NF == 1 ? sy[0] : lane_of<LP, m % LP>(sy[m / LP]);
  });
  return model_score<CF, VC, NF, FORM>(all2, all1, n_filters, dof, sum_w, dV, NU ? &nu : nullptr, mr);
}

// The parts of a team that do not depend on the form, the filters or the type
// of the score: one copy for all kernels of a build.
template <int VC, int LP, int ROLE>
__device__ __attribute__((noinline)) void team_walk(const double* params, size_t stride, const PointRec* pts_g,
                                                    int n_data, TeamPtr<VC, LP> team) {
  constexpr int N = Pos<VC>::N;
  const uint64_t pu = (uint64_t)(uintptr_t)pts_g;
  const uint64_t plo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)pu);
  const uint64_t phi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(pu >> 32));
  const uintptr_t pa = (uintptr_t)((phi << 32) | plo);
  n_data = __builtin_amdgcn_readfirstlane(n_data);
  double prm[N];
#pragma unroll
  for (int i = 0; i < N; ++i) prm[i] = params[(size_t)i * stride];
  chi2_model_rows<double, VC, 1, false, FORM_CHI2, LP, ROLE>(prm, (PointPtr)pa, (LanePtr)pa, n_data, 1, 0, nullptr,
                                                             nullptr, nullptr, 0.0, team);
}

// What the wavefronts of a team other than its first do: wave 1 the Euler
// angles, wave 2 (with torque) the angular velocities.
template <int VC, int LP>
__device__ inline void team_helper(int wave, const double* params, size_t stride, const PointRec* pts_g, int n_data,
                                   TeamPtr<VC, LP> team) {
  if (wave == 1) team_walk<VC, LP, ROLE_ANGLES>(params, stride, pts_g, n_data, team);
  if constexpr (VarF<VC>::TQ)
    if (wave == 2) team_walk<VC, LP, ROLE_SPIN>(params, stride, pts_g, n_data, team);
}

}  // namespace ast
