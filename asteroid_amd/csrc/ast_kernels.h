// ast_kernels.h -- the fitting kernels (template definitions; each variant
// is instantiated in its own translation unit, ast_k_*.hip).
//
// The simplex of chi2_gpu (cuda.c:1424-1807) calls chi2one from five places
// (initial vertices, reflection, expansion, contraction, shrink), so the
// lanes of a wavefront diverge across the most expensive call in the
// program.  Here the Nelder-Mead control flow is a per-lane state machine:
// every "tick" each lane holds at most one pending point, all lanes
// evaluate their points through ONE call of the evaluator (divergence-free,
// since every model walks the same observation loop), and each lane then
// advances its own state machine with the result until it needs the next
// point.  The sequence of points a lane evaluates, the comparisons it makes
// and every stored value are those of the reference control flow, so a
// lane's trajectory is the oracle's trajectory.
//
// Simplex state lives in HBM in lane-fastest (structure-of-arrays) layout,
// so every access of a wavefront is one contiguous, coalesced segment.  A
// workgroup is one reseed group (the reference's block): after every tick
// it votes on whether all of its simplexes finished the stage; if so the
// block argmin, stage reseed or best-per-group write of cuda.c:1739-1823 run
// in place.  Kernel launches are chunks of ticks; all state persists in
// HBM between launches.
#pragma once
#include "ast_device.h"
#include "ast_rows.h"

namespace ast {

enum Phase : int {
  PH_START = 0,     // begin a stage: draw the start point and the simplex
  PH_INIT = 1,      // pending/complete: chi^2 of initial vertex j
  PH_BEGIN = 2,     // internal: top of the simplex loop (sort, centroid, tests)
  PH_REFLECT = 3,   // pending/complete: reflected point
  PH_EXPAND = 4,    // pending/complete: expanded point
  PH_CONTRACT = 5,  // pending/complete: contracted point
  PH_SHRINK = 6,    // pending/complete: shrunk vertex ind[j]
  PH_SHRINK_NEXT = 7,  // internal: shrink the next vertex
  PH_STAGE_DONE = 8,
  PH_FIT_DONE = 9
};

__device__ inline bool phase_pending(int ph) {
  return ph == PH_INIT || ph == PH_REFLECT || ph == PH_EXPAND || ph == PH_CONTRACT || ph == PH_SHRINK;
}

// Simplex state of the resident simplexes ("slots"), lane-fastest.  A group
// of G simplexes owns slot fits [slot*G, slot*G + G) while it runs; nf is the
// slot capacity.  Element (row, fit) of an array of fixed type (IND, PRM and
// the int32 counters) lives at row * nf + fit.  The arrays of simplex floats
// (CF) are made of 8-byte cells so that float and double groups can share the
// pool side by side: with KC = 8 / sizeof(CF), element (row, fit = slot*G + t)
// lives at CF index row * (KC*nf) + KC*slot*G + t, i.e. a float group packs
// its G values into the first half of its slot's cells of the row.  Every
// access of a wavefront stays one contiguous segment.
template <class CF>
struct SlotBufs {
  CF* X;        // [(N+1)*N]  simplex vertices
  CF* F;        // [N+1]      chi^2 at the vertices
  uint8_t* IND; // [N+1]      sorted vertex indices
  CF* X0;       // [N]        centroid
  CF* XR;       // [N]        reflected point
  CF* XP;       // [N]        expanded / contracted point
  double* PRM;  // [N]        the thread's params[] buffer (cuda.c:1344)
  CF* DV;       // [MAXF]     delta_V of the last evaluation
  int32_t* ctl;       // phase | j<<4 | failed<<10 | bad<<11 (j <= N <= 63)
  int32_t* lstep;     // simplex steps in this stage (l, cuda.c:1436)
  int32_t* nev;       // chi^2 evaluations in this stage
  int32_t* nev_tot;   // evaluations, all stages of this job
  int32_t* steps_tot; // steps, all stages of this job
  CF* fr;             // f_r kept for the expansion test
  CF* sf;             // stage-final best chi^2 (s_f, cuda.c:1739-1742)
  int32_t* fitid;     // the job's index of the fit the lane runs (its random stream)
  int32_t* work;      // evaluations the lane did since its group started (all fits)
  int32_t* g_reopt;   // per group slot: s_x2_params.reopt
  int32_t* g_stage;   // per group slot: current stage
  int32_t* g_done;    // per group slot: all stages finished
  size_t nf;          // slot capacity (fits)
};

// One group of one job, as a launch sees it (read once per workgroup,
// wave-uniform).  The job's curve, model space, start model, random streams
// and per-group best arrays are the job's own, so where a group runs (its
// slot, its neighbours in the launch) does not change its results.
template <class CF>
struct GroupDesc {
  const PointRec* pts;
  const double* sum_w;
  const Space<CF>* sp;
  const double* params0;
  uint32_t* rng;          // the job's stream counters, by job fit index
  CF* best_f;             // d_f of the job, by group
  double* best_params;    // d_params, [group][N]
  double* best_dV;        // d_dV, [group][n_filters]
  int32_t* job_done;      // groups of the job that finished
  uint64_t seed;
  CF size2_min;
  int n_data, n_filters, dof;
  int nstages, n_steps, eval_budget, reopt;
  int slot;               // group slot
  int group_in_job;       // the group (with refill: the worker) index within the job
  int ticks;              // evaluation rounds in this launch
  // Per-fit results of the job, written by each fit when it ends: its
  // stage-final best chi^2 (1e30 if it failed), evaluations and simplex steps
  // over all its stages.
  CF* fit_f;
  int32_t* fit_nev;
  int32_t* fit_steps;
  // Refill (single-stage jobs run by fewer workgroups than the job has
  // groups): a lane whose fit ended takes the next unstarted fit of the job
  // from queue[0] (queue[1] counts finished fits) and keeps the ended fit's
  // best point (x2params of its best vertex) and its last delta_V, from which
  // group_best_kernel forms each group's result once every fit has ended.
  int refill;
  int n_fits;
  int32_t* queue;
  double* fit_params;     // [n_fits][N]
  double* fit_dV;         // [n_fits][n_filters]
};

template <class CF>
struct LaneRegs {
  int phase, j, failed, bad, l, nev, nev_tot, steps_tot, work;
  uint32_t rng;
  CF fr, sf;
};

// Per-stage settings a lane needs while advancing (copied out of the descriptor).
template <class CF>
struct StageCfg {
  uint64_t seed;
  CF size2_min;
  int n_steps, eval_budget;
};

// A wave-uniform value (pointer or 64-bit size) that arrived in vector
// registers or memory, moved to scalar registers.
__device__ inline uint64_t uniform64(uint64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}
// Pointers into device memory by global (not FLAT) accesses.
template <class T>
using GlobalPtr = __attribute__((address_space(1))) T*;
template <class T>
using GlobalRef = __attribute__((address_space(1))) T&;

// One lane's simplex and its control flow.  Uniform members are the same for
// the wavefront; the lane's own are its slot fit index and offsets.
template <class CF, int VC>
struct Machine {
  using P = Pos<VC>;
  static constexpr int N = P::N;
  static constexpr bool BC = VarF<VC>::BC;
  // uniform
  SpacePtr<CF> sp;
  GlobalPtr<CF> bX, bF, bX0, bXR, bXP, bDV;
  GlobalPtr<uint8_t> bIND;
  GlobalPtr<double> bPRM;
  StageCfg<CF> C;
  uint64_t nf, rs;  // row strides: fixed-type arrays and CF arrays
  // the lane's
  uint32_t fit;     // slot fit index
  uint32_t fo;      // the same element in the CF arrays
  uint64_t jfit;    // fit index within the job (random stream)
  int reopt;

  __device__ static Machine of(const GroupDesc<CF>& D, const SlotBufs<CF>& B, size_t fit, size_t fo, uint64_t jfit,
                               int reopt) {
    Machine m;
    m.sp = (SpacePtr<CF>)(uintptr_t)D.sp;
    m.bX = (GlobalPtr<CF>)B.X;
    m.bF = (GlobalPtr<CF>)B.F;
    m.bX0 = (GlobalPtr<CF>)B.X0;
    m.bXR = (GlobalPtr<CF>)B.XR;
    m.bXP = (GlobalPtr<CF>)B.XP;
    m.bDV = (GlobalPtr<CF>)B.DV;
    m.bIND = (GlobalPtr<uint8_t>)B.IND;
    m.bPRM = (GlobalPtr<double>)B.PRM;
    m.C = StageCfg<CF>{D.seed, D.size2_min, D.n_steps, D.eval_budget};
    m.nf = B.nf;
    m.rs = (8 / sizeof(CF)) * B.nf;
    m.fit = (uint32_t)fit;
    m.fo = (uint32_t)fo;
    m.jfit = jfit;
    m.reopt = reopt;
    return m;
  }
  // The uniform members in scalar registers.
  __device__ void to_scalar() {
    sp = (SpacePtr<CF>)(uintptr_t)uniform64((uint64_t)(uintptr_t)sp);
    bX = (GlobalPtr<CF>)uniform64((uint64_t)bX);
    bF = (GlobalPtr<CF>)uniform64((uint64_t)bF);
    bX0 = (GlobalPtr<CF>)uniform64((uint64_t)bX0);
    bXR = (GlobalPtr<CF>)uniform64((uint64_t)bXR);
    bXP = (GlobalPtr<CF>)uniform64((uint64_t)bXP);
    bDV = (GlobalPtr<CF>)uniform64((uint64_t)bDV);
    bIND = (GlobalPtr<uint8_t>)uniform64((uint64_t)bIND);
    bPRM = (GlobalPtr<double>)uniform64((uint64_t)bPRM);
    nf = uniform64(nf);
    rs = uniform64(rs);
    C.seed = uniform64(C.seed);
    C.n_steps = __builtin_amdgcn_readfirstlane(C.n_steps);
    C.eval_budget = __builtin_amdgcn_readfirstlane(C.eval_budget);
    reopt = __builtin_amdgcn_readfirstlane(reopt);
  }

  // Makes the row addresses and the model space unknown to the compiler at
  // this point.  Else it computes the addresses of every row of every array,
  // and loads every limit, once, ahead of the loop they are used in, and keeps
  // the 200 of them in scratch memory.
  __device__ void renew() {
    pin_sgpr(sp);
    pin_sgpr(bX);
    pin_sgpr(bF);
    pin_sgpr(bX0);
    pin_sgpr(bXR);
    pin_sgpr(bXP);
    pin_sgpr(bIND);
    pin_sgpr(bPRM);
  }

  // Element of a row: a scalar row address and the lane's 32-bit byte offset
  // (at least 1 KB of state per fit keeps 8 * nf far below 2^32).
  template <class T>
  __device__ static GlobalRef<T> at(GlobalPtr<T> base, uint64_t row_stride, int row, uint32_t lane_index) {
    return *(GlobalPtr<T>)((GlobalPtr<char>)(base + (uint64_t)row * row_stride) + lane_index * (uint32_t)sizeof(T));
  }
  __device__ GlobalRef<CF> X(int v, int i) const { return at(bX, rs, v * N + i, fo); }
  __device__ GlobalRef<CF> F(int v) const { return at(bF, rs, v, fo); }
  __device__ GlobalRef<uint8_t> IND(int v) const { return at(bIND, nf, v, fit); }
  __device__ GlobalRef<CF> X0(int i) const { return at(bX0, rs, i, fo); }
  __device__ GlobalRef<CF> XR(int i) const { return at(bXR, rs, i, fo); }
  __device__ GlobalRef<CF> XP(int i) const { return at(bXP, rs, i, fo); }
  __device__ GlobalRef<CF> DVL(int m) const { return at(bDV, rs, m, fo); }
  __device__ GlobalRef<double> PRM(int i) const { return at(bPRM, nf, i, fit); }

  // x2params on a point, through the persistent params[] buffer.
  __device__ bool propose(const CF* xv) const {
    double prm[N];
#pragma unroll
    for (int i = 0; i < N; ++i) prm[i] = PRM(i);
    int rc = x2params_at<CF, VC>(xv, prm, *sp, reopt);
#pragma unroll
    for (int i = 0; i < N; ++i) PRM(i) = prm[i];
    return rc == 0;
  }

  __device__ float rnd(LaneRegs<CF>& R) const { return astrng::uniform01(C.seed, jfit, R.rng++); }

  // Stage start (cuda.c:1456-1546): x[0] random or around the reoptimised
  // point, then the N displaced vertices.
  __device__ void start(LaneRegs<CF>& R, CF* x0v) const {
    const CF DX_INI = (CF)0.001, D2X_INI = (CF)-1.2, DX_RAND = (CF)0.0001;  // asteroid.h:205-209
    int LAM = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) x0v[i] = X(0, i);
    for (int i = 0; i < N; ++i) {
      float r = rnd(R);
      if (BC && !reopt) {
        if (i == P::c) { x0v[i] = x0v[P::c_tumb]; continue; }
        if (i == P::b) { x0v[i] = x0v[P::b_tumb]; continue; }
      }
      int per = sp->periodic[i];
      CF xi;
      if (!reopt || (reopt && sp->frozen[i] == -1)) {
        xi = DX_INI + SMALL + r * (1.0 - 2 * (SMALL + DX_INI));
      } else {
        CF xmin = x0v[i] - DX_RAND;
        CF xmax = x0v[i] + DX_RAND;
        if (xmin < SMALL && hard_left(per, LAM)) xmin = SMALL;
        if (xmax > 1.0 - SMALL && hard_right(per, LAM)) xmax = 1.0 - SMALL;
        xi = xmin + r * (xmax - xmin);
      }
      x0v[i] = xi;
      if (P::is_Es(i)) LAM = xi >= 0.5;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) X(0, i) = x0v[i];
    for (int jj = 1; jj < N + 1; ++jj) {
      for (int i = 0; i < N; ++i) {
        if (i == jj - 1) {
          int per = sp->periodic[i];
          float d2x = rnd(R);
          CF dx = DX_INI * cf_exp((CF)(D2X_INI * d2x));
          if (rnd(R) < 0.5) {
            dx = -dx;
            if (x0v[i] + dx < SMALL && hard_left(per, LAM)) dx = -dx;
          } else {
            if (x0v[i] + dx > 1.0 - SMALL && hard_right(per, LAM)) dx = -dx;
          }
          X(jj, i) = x0v[i] + dx;
        } else {
          X(jj, i) = x0v[i];
        }
      }
    }
  }

  __device__ void finish(LaneRegs<CF>& R) const {
    R.sf = R.failed ? (CF)1e30 : F(IND(0));
    R.steps_tot += R.l;
    R.phase = PH_STAGE_DONE;
  }

  // A fit's own results, when it ends (refill): stage-final best chi^2,
  // counts, the physical parameters of its best vertex (x2params through the
  // lane's params[] buffer, as the group's writer does at cuda.c:1810-1823)
  // and the delta_V of its last evaluation (cuda.c:1816-1822).
  __device__ void end_fit(const LaneRegs<CF>& R, const GroupDesc<CF>& D) const {
    D.fit_f[jfit] = R.sf;
    D.fit_nev[jfit] = R.nev_tot;
    D.fit_steps[jfit] = R.steps_tot;
    D.rng[jfit] = R.rng;
    if (!R.failed) {
      CF xb[N];
      double prm[N];
      const int b = IND(0);
#pragma unroll
      for (int i = 0; i < N; ++i) { xb[i] = X(b, i); prm[i] = PRM(i); }
      x2params_at<CF, VC>(xb, prm, *sp, reopt);
#pragma unroll
      for (int i = 0; i < N; ++i) D.fit_params[jfit * N + i] = prm[i];
    }
    for (int m = 0; m < D.n_filters; ++m) D.fit_dV[jfit * D.n_filters + m] = DVL(m);
  }

  // The lane's state for a new fit (as fit_init_kernel leaves a group's
  // lanes): PH_START.
  __device__ void begin_fit(LaneRegs<CF>& R, const GroupDesc<CF>& D) const {
#pragma unroll
    for (int v = 0; v <= N; ++v) IND(v) = (uint8_t)v;
    double prm[N];
#pragma unroll
    for (int i = 0; i < N; ++i) prm[i] = reopt ? D.params0[i] : 0.0;
#pragma unroll
    for (int i = 0; i < N; ++i) PRM(i) = prm[i];
    CF x[N];
    if (reopt) params2x<CF, VC>(x, prm, *sp);
    else
      for (int i = 0; i < N; ++i) x[i] = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) X(0, i) = x[i];
    for (int m = 0; m < MAXF; ++m) DVL(m) = 0;
    R.phase = PH_START;
    R.nev_tot = 0;
    R.steps_tot = 0;
    R.rng = D.rng[jfit];
    R.fr = 0;
    R.sf = (CF)1e30;
  }

  __device__ void replace_worst(GlobalPtr<CF> point, CF fv) const {
    const int w = IND(N);
    CF xn[N];
#pragma unroll
    for (int i = 0; i < N; ++i) xn[i] = at(point, rs, i, fo);
#pragma unroll
    for (int i = 0; i < N; ++i) X(w, i) = xn[i];
    F(w) = fv;
  }

  // The vertices in order of chi^2 (cuda.c:1570-1600), and the worst one: the
  // reference takes the lowest value left, the last vertex of equal ones, so
  // a vertex's place is the number of those before it.
  __device__ int sort_vertices() const {
    CF f[N + 1];
#pragma unroll
    for (int v = 0; v <= N; ++v) f[v] = F(v);
    bool plain = true;  // every value can be taken (none is NaN or above 1e30)
#pragma unroll
    for (int v = 0; v <= N; ++v) plain = plain & (f[v] <= (CF)1e30);
    int w = 0;
    if (plain) {
      if constexpr (N <= 16) {  // one comparison per pair
        int place[N + 1];
#pragma unroll
        for (int v = 0; v <= N; ++v) place[v] = v;
#pragma unroll
        for (int v = 1; v <= N; ++v)
#pragma unroll
          for (int u = 0; u < v; ++u) {
            const int before = f[v] <= f[u] ? 1 : 0;  // v comes before u
            place[u] += before;
            place[v] -= before;
          }
#pragma unroll
        for (int v = 0; v <= N; ++v) {
          IND(place[v]) = (uint8_t)v;
          w = place[v] == N ? v : w;
        }
      } else {
#pragma unroll 1
        for (int v = 0; v <= N; ++v) {
          const CF fv = F(v);
          int place = 0;
#pragma unroll
          for (int u = 0; u <= N; ++u) place += (f[u] < fv ? 1 : 0) + ((u > v) & (f[u] == fv) ? 1 : 0);
          IND(place) = (uint8_t)v;
          w = place == N ? v : w;
        }
      }
    } else {
      uint64_t taken = 0;
      int jmin = 0;
#pragma unroll 1
      for (int v = 0; v <= N && jmin >= 0; ++v) {
        CF fmin = 1e30;
        jmin = -1;
#pragma unroll 1
        for (int u = 0; u <= N; ++u) {
          const CF fu = F(u);
          if (!((taken >> u) & 1) && fu <= fmin) { fmin = fu; jmin = u; }
        }
        if (jmin >= 0) {
          IND(v) = (uint8_t)jmin;
          taken |= 1ull << jmin;
        } else {  // NaN values left (cuda.c:1592-1598)
          IND(0) = 0;
          F(0) = 1e30;
        }
      }
      w = IND(N);
    }
    return w;
  }

  // K elements of the simplex, from row `first` on every `stride` rows.
  template <int K>
  __device__ void fetch(CF* out, int first, int stride) const {
    const uint64_t step = (uint64_t)stride * rs * sizeof(CF);
    uint64_t p = (uint64_t)bX + (uint64_t)first * rs * sizeof(CF);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      pin_sgpr(p);
      out[k] = *(GlobalPtr<CF>)((GlobalPtr<char>)p + fo * (uint32_t)sizeof(CF));
      p += step;
    }
  }

  // The top of the simplex loop (cuda.c:1568-1645): sort, centroid, size and
  // the stopping tests; false if the stage is over, else the reflected point
  // in xv.
  __device__ bool begin_step(LaneRegs<CF>& R, CF* xv) const {
    const CF ALPHA = 1.0;  // asteroid.h:239
    constexpr int UN = N <= 16 ? N : 1;  // whole rows in registers for the smaller simplexes
    R.l++;
    const int w = sort_vertices();
    // One pass over the simplex, column by column, each fetched while the one
    // before it is worked on: the centroid's coordinate, then every vertex's
    // share of the size (each vertex's sum takes the coordinates in their
    // order, as a pass row by row would).
    CF x0[N], dist2[N + 1], cur[N + 1], nxt[N + 1];
#pragma unroll
    for (int v = 0; v < N + 1; ++v) dist2[v] = 0.0;
    fetch<N + 1>(cur, 0, N);
#pragma unroll UN
    for (int i = 0; i < N; ++i) {
      if (i + 1 < N) fetch<N + 1>(nxt, i + 1, N);
      __builtin_amdgcn_sched_barrier(0);
      CF sum = 0.0;
#pragma unroll
      for (int v = 0; v < N + 1; ++v) sum = sum + cur[v];
      x0[i] = sum / (N + 1);
#pragma unroll
      for (int v = 0; v < N + 1; ++v) {
        CF dx = cur[v] - x0[i];
        dist2[v] = dist2[v] + dx * dx;
      }
#pragma unroll
      for (int v = 0; v < N + 1; ++v) cur[v] = nxt[v];
      __builtin_amdgcn_sched_barrier(0);
    }
    CF size2 = 0.0;
#pragma unroll
    for (int v = 0; v < N + 1; ++v) size2 = size2 + dist2[v];
    size2 = size2 / N;
    if (size2 < C.size2_min || R.l > C.n_steps || (C.eval_budget > 0 && R.nev >= C.eval_budget)) return false;
    CF xw[N];
#pragma unroll
    for (int i = 0; i < N; ++i) xw[i] = X(w, i);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      xv[i] = (sp->frozen[i] != 1) ? (CF)(x0[i] + ALPHA * (x0[i] - xw[i])) : xw[i];
      X0(i) = x0[i];
      XR(i) = xv[i];
    }
    return true;
  }

  // Advance the lane until it has a pending point or its stage is over.
  // `val` is the chi^2 of the pending point when has_result.  The lanes of a
  // wavefront are in different phases, so each part of the control flow
  // stands once in a pass and what follows from it behind it: the decision
  // about the value, the next vertex of a shrink, the top of the simplex
  // loop, and one proposal for whatever point came out of them.  (With a
  // proposal per phase a pass ran the parameter map up to four times, and
  // with pointers read through memory every load of the simplex was waited
  // for by itself: 110 us per round of 64-lane FP64 fits of 11 parameters,
  // 370 us with the chip full, of 580 and 2900 us.)
  //
  // The loop has one exit, and in the SEGMENT builds `more` goes through a
  // register the compiler cannot see through, so that it does not make several
  // again from what it knows of `more`.  With several it keeps, per exit, the
  // mask of the lanes that took it in a lane of a spill register; and ROCm 7.2's
  // hipcc declares that register without a value at the head of the block that
  // adds to the mask, inside the loop, so that it may give it to other spills
  // for the rest of a pass.  It did in the FP64 build of four segments with
  // torque and BC (40 parameters), whose fits then never ended; in ten other
  // SEGMENT builds the register happened to stay free.  (In every build the
  // register costs 0.5% of 2^18 mixed fits and 0.9% of re-optimised BC fits.)
  __device__ void advance(LaneRegs<CF>& R, CF val, bool has_result) {
    const CF GAMMA = 2.0, RHO = 0.5, SIGMA = 0.5;  // asteroid.h:240-242
    int more = has_result || R.phase == PH_START;
    CF xv[N];
    while (more) {
      renew();
      more = 0;
      bool over = false;
      if (R.phase == PH_START) {
        start(R, xv);
        R.l = 0;
        R.nev = 0;
        R.failed = 0;
        R.bad = 0;
        R.j = 0;
        R.phase = PH_INIT;
      } else if (R.phase == PH_INIT) {  // cuda.c:1550-1559
        F(R.j) = val;
        R.j++;
        if (R.j <= N) {
#pragma unroll
          for (int i = 0; i < N; ++i) xv[i] = X(R.j, i);
        } else {
          R.phase = PH_BEGIN;
        }
      } else if (R.phase == PH_REFLECT) {  // cuda.c:1646-1712 (decisions after the reflection)
        R.fr = val;
        const CF fb = F(IND(0));
        if (val >= fb && val < F(IND(N - 1))) {
          replace_worst(bXR, val);
          R.phase = PH_BEGIN;
        } else {
          // expansion (from the reflected point) or contraction (from the worst)
          const bool expand = val < fb;
          const CF k = expand ? GAMMA : RHO;
          const int w = IND(N);
          CF xf[N], x0[N];
#pragma unroll
          for (int i = 0; i < N; ++i) {
            xf[i] = expand ? XR(i) : X(w, i);
            x0[i] = X0(i);
          }
#pragma unroll
          for (int i = 0; i < N; ++i) {
            xv[i] = (sp->frozen[i] != 1) ? (CF)(x0[i] + k * (xf[i] - x0[i])) : xf[i];
            XP(i) = xv[i];
          }
          R.phase = expand ? PH_EXPAND : PH_CONTRACT;
        }
      } else if (R.phase == PH_EXPAND) {  // cuda.c:1671-1689
        const bool better = val < R.fr;
        replace_worst(better ? bXP : bXR, better ? val : R.fr);
        R.phase = PH_BEGIN;
      } else if (R.phase == PH_CONTRACT) {  // cuda.c:1703-1712
        if (val < F(IND(N))) {
          replace_worst(bXP, val);
          R.phase = PH_BEGIN;
        } else {
          R.bad = 0;
          R.j = 1;
          R.phase = PH_SHRINK_NEXT;
        }
      } else if (R.phase == PH_SHRINK) {  // cuda.c:1726
        F(IND(R.j)) = val;
        R.j++;
        R.phase = PH_SHRINK_NEXT;
      }
      if (R.phase == PH_SHRINK_NEXT) {  // cuda.c:1716-1733
        if (R.j <= N) {
          const int v = IND(R.j), b = IND(0);
          CF xb[N];
#pragma unroll
          for (int i = 0; i < N; ++i) {
            xv[i] = X(v, i);
            xb[i] = X(b, i);
          }
#pragma unroll
          for (int i = 0; i < N; ++i) {
            if (sp->frozen[i] != 1) xv[i] = xb[i] + SIGMA * (xv[i] - xb[i]);
            X(v, i) = xv[i];
          }
        } else {
          if (R.bad) R.failed = 1;
          R.phase = PH_BEGIN;
        }
      }
      if (R.phase == PH_BEGIN) {
        over = R.failed || !begin_step(R, xv);
        if (over) finish(R);
        else R.phase = PH_REFLECT;
      }
      if (!over) {
        if (propose(xv)) {
          if (R.phase == PH_SHRINK_NEXT) R.phase = PH_SHRINK;
        } else {  // outside the hard limits
          more = 1;
          if (R.phase == PH_INIT) {
            R.failed = 1;
            R.phase = PH_BEGIN;
          } else if (R.phase == PH_SHRINK_NEXT) {
            R.bad = 1;
            R.j++;
          } else {
            val = 1e30;
          }
        }
      }
      if constexpr (VarF<VC>::SG) pin_vgpr(more);
    }
  }
};

// advance() out of line, one copy for the kernels of a simplex type: its
// registers do not compete with the evaluator's.
template <class CF, int VC>
__device__ __attribute__((noinline)) void advance_lane(const Machine<CF, VC>& machine, LaneRegs<CF>& regs, CF val,
                                                       bool has_result) {
  Machine<CF, VC> m = machine;
  m.to_scalar();
  LaneRegs<CF> R = regs;
  m.advance(R, val, has_result);
  regs = R;
}

// --------------------------------------------------------------- init kernel
// A group's start (one workgroup of G threads per new group): identity sort
// order, stage-0 start point (params2x of the reoptimisation model,
// cuda.c:1409-1416), counters, group flags.
template <class CF, int VC>
__global__ void fit_init_kernel(const GroupDesc<CF>* descs, SlotBufs<CF> B) {
  using P = Pos<VC>;
  AST_VFLAGS(VC);
  constexpr int N = P::N;
  constexpr int KC = 8 / sizeof(CF);
  const GroupDesc<CF>& D = descs[blockIdx.x];
  const size_t nf = B.nf, rs = KC * nf;
  const size_t fit = (size_t)D.slot * blockDim.x + threadIdx.x;
  const size_t fo = (size_t)D.slot * blockDim.x * KC + threadIdx.x;
  for (int v = 0; v <= N; ++v) B.IND[v * nf + fit] = (uint8_t)v;
  double prm[N];
  for (int i = 0; i < N; ++i) prm[i] = D.reopt ? D.params0[i] : 0.0;
  for (int i = 0; i < N; ++i) B.PRM[i * nf + fit] = prm[i];
  CF x[N];
  if (D.reopt) params2x<CF, VC>(x, prm, *D.sp);
  else
    for (int i = 0; i < N; ++i) x[i] = 0;
  for (int i = 0; i < N; ++i) B.X[(size_t)i * rs + fo] = x[i];
  for (int m = 0; m < MAXF; ++m) B.DV[m * rs + fo] = 0;
  B.ctl[fit] = PH_START;
  B.lstep[fit] = 0;
  B.nev[fit] = 0;
  B.nev_tot[fit] = 0;
  B.steps_tot[fit] = 0;
  B.fitid[fit] = D.group_in_job * (int)blockDim.x + (int)threadIdx.x;
  B.work[fit] = 0;
  B.fr[fo] = 0;
  B.sf[fo] = (CF)1e30;
  if (threadIdx.x == 0) {
    B.g_reopt[D.slot] = D.reopt;
    B.g_stage[D.slot] = 0;
    B.g_done[D.slot] = 0;
  }
}

// One lane's evaluation inside the fitting kernel: parameters from the
// lane's params[] buffer, delta_V to its last-dV slot.  Kept out of line so
// the evaluator's register allocation does not compete with the simplex
// bookkeeping live across it.  W (the calling kernel's waves per SIMD) makes
// one copy per register budget: a function shared by kernels of different
// budgets is compiled for the smallest, 128 VGPRs, where the FP64 evaluator
// spills.  The mixed form keeps the one 128-VGPR copy, which measured faster
// than copies given more registers.
template <class CF, int VC, int NF, bool MX, int W>
__device__ __attribute__((noinline)) CF eval_lane(const double* PRM, CF* DV, size_t nf, size_t fit, size_t rs,
                                                   size_t fo, const PointRec* pts_g, int n_data, int n_filters, int dof,
                                                   const double* sum_w) {
  constexpr int N = Pos<VC>::N;
  // Arguments of a device function arrive in vector registers; the table
  // pointer and the sizes are wave-uniform, so move them to scalar registers
  // to keep the observation loop on scalar loads and scalar branches.
  const uint64_t pu = (uint64_t)(uintptr_t)pts_g;
  const uint64_t plo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)pu);
  const uint64_t phi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(pu >> 32));
  PointPtr pts = (PointPtr)(uintptr_t)((phi << 32) | plo);
  n_data = __builtin_amdgcn_readfirstlane(n_data);
  n_filters = __builtin_amdgcn_readfirstlane(n_filters);
  dof = __builtin_amdgcn_readfirstlane(dof);
  double prm[N];
#pragma unroll
  for (int i = 0; i < N; ++i) prm[i] = PRM[(size_t)i * nf + fit];
  CF dv[NF];
  if constexpr (VarF<VC>::NU) {
    // a failed NUDGE model leaves delta_V as the lane's last evaluation left it
#pragma unroll
    for (int m = 0; m < NF; ++m) dv[m] = m < n_filters ? DV[(size_t)m * rs + fo] : CF(0);
  }
  CF fv = chi2_model<CF, VC, NF, MX>(prm, pts, n_data, n_filters, dof, sum_w, dv);
#pragma unroll
  for (int m = 0; m < NF; ++m)
    if (m < n_filters) DV[(size_t)m * rs + fo] = dv[m];
  return fv;
}

// The next `1` from a counter shared by many lanes: one atomic per
// wavefront for all of its lanes that ask in this pass, each getting its own
// value in lane order.  queue[1] counts the requests (each follows a fit's
// end), queue[0] hands out the fit indices.
__device__ inline int take_fit(int32_t* queue) {
  const uint64_t mask = __ballot(1);
  const int lane = (int)__lane_id();
  const int leader = __ffsll((unsigned long long)mask) - 1;
  const int rank = __popcll(mask & ((1ull << lane) - 1ull));
  int base = 0;
  if (lane == leader) {
    const int cnt = __popcll(mask);
    base = atomicAdd(&queue[0], cnt);
    atomicAdd(&queue[1], cnt);
  }
  base = __shfl(base, leader);
  return base + rank;
}

// Each group's result from its fits' own results, once every fit of the job
// has ended (refill): the block argmin and the best-per-group write of
// cuda.c:1739-1742, 1810-1823 -- the lowest chi^2 of the group's fits, the
// first one on ties, replaces the stored best only when strictly lower.
template <class CF>
__global__ __launch_bounds__(64) void group_best_kernel(const CF* fit_f, const double* fit_params,
                                                        const double* fit_dV, int G, int N, int n_filters,
                                                        int n_groups, CF* best_f, double* best_params,
                                                        double* best_dV) {
  const int g = blockIdx.x;
  if (threadIdx.x != 0 || g >= n_groups) return;
  int tm = 0;
  CF smin = (CF)1e30;
  for (int k = 0; k < G; ++k) {
    const CF f = fit_f[(size_t)g * G + k];
    if (f < smin) { smin = f; tm = k; }
  }
  if (smin < best_f[g]) {
    const size_t j = (size_t)g * G + tm;
    best_f[g] = smin;
    for (int i = 0; i < N; ++i) best_params[(size_t)g * N + i] = fit_params[j * N + i];
    for (int m = 0; m < n_filters; ++m) best_dV[(size_t)g * n_filters + m] = fit_dV[j * n_filters + m];
  }
}

// ----------------------------------------------------------------- stage end
// The end of a stage, by the whole workgroup (one thread per simplex of the
// group, all of which finished the stage; cuda.c:1739-1823): the block argmin,
// then either the next stage's reseed (the lanes are left at PH_START, true)
// or the best-per-group write and the fits' own results (false).  s_f: one
// value per simplex in LDS.
template <class CF, int VC>
__device__ bool group_stage_end(const GroupDesc<CF>& D, const Machine<CF, VC>& M, LaneRegs<CF>& R, int t, int G,
                                int& stage, int& reopt, CF* s_f) {
  constexpr int N = Pos<VC>::N;
  __shared__ CF s_x0[MAXP];
  __shared__ int s_tm;
  __shared__ CF s_smin;
  const SpacePtr<CF> sp = M.sp;
  s_f[t] = R.sf;
  __syncthreads();
  if (t == 0) {
    int tm = 0;
    CF smin = (CF)1e30;
    for (int k = 0; k < G; ++k)
      if (s_f[k] < smin) { smin = s_f[k]; tm = k; }
    s_tm = tm;
    s_smin = smin;
  }
  __syncthreads();
  const int tm = s_tm;
  const CF smin = s_smin;
  if (D.nstages > 1 && stage < D.nstages - 1) {
    if (t == tm) {
      CF xb[N];
      const int b = M.IND(0);
#pragma unroll
      for (int i = 0; i < N; ++i) xb[i] = M.X(b, i);
      if (sp->p_psi && reopt == 0) {  // cuda.c:1791-1798
        double prm[N];
#pragma unroll
        for (int i = 0; i < N; ++i) prm[i] = M.PRM(i);
        x2params_at<CF, VC>(xb, prm, *sp, reopt);
        params2x<CF, VC>(xb, prm, *sp);
#pragma unroll
        for (int i = 0; i < N; ++i) { M.PRM(i) = prm[i]; M.X(b, i) = xb[i]; }
      }
#pragma unroll
      for (int i = 0; i < N; ++i) s_x0[i] = xb[i];
    }
    __syncthreads();
    reopt = 1;
    stage++;
#pragma unroll
    for (int i = 0; i < N; ++i) M.X(0, i) = s_x0[i];
    R.phase = PH_START;
    return true;
  }
  const int g = D.group_in_job;
  if (t == tm && smin < D.best_f[g]) {  // cuda.c:1810-1823
    D.best_f[g] = smin;
    CF xb[N];
    double prm[N];
    const int b = M.IND(0);
#pragma unroll
    for (int i = 0; i < N; ++i) { xb[i] = M.X(b, i); prm[i] = M.PRM(i); }
    x2params_at<CF, VC>(xb, prm, *sp, reopt);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      M.PRM(i) = prm[i];
      D.best_params[(size_t)g * N + i] = prm[i];
    }
    for (int m = 0; m < D.n_filters; ++m)
      D.best_dV[(size_t)g * D.n_filters + m] = M.DVL(m);
  }
  D.fit_f[M.jfit] = R.sf;
  D.fit_nev[M.jfit] = R.nev_tot;
  D.fit_steps[M.jfit] = R.steps_tot;
  stage++;
  R.phase = PH_FIT_DONE;
  return false;
}

// A lane's machine state, from and to its slot.
template <class CF>
__device__ inline LaneRegs<CF> load_lane(const SlotBufs<CF>& B, size_t fit, size_t fo, uint32_t rng) {
  LaneRegs<CF> R;
  const int ctl = B.ctl[fit];
  R.phase = ctl & 15;
  R.j = (ctl >> 4) & 63;
  R.failed = (ctl >> 10) & 1;
  R.bad = (ctl >> 11) & 1;
  R.l = B.lstep[fit];
  R.nev = B.nev[fit];
  R.nev_tot = B.nev_tot[fit];
  R.steps_tot = B.steps_tot[fit];
  R.work = B.work[fit];
  R.rng = rng;
  R.fr = B.fr[fo];
  R.sf = B.sf[fo];
  return R;
}
template <class CF>
__device__ inline void store_lane(const SlotBufs<CF>& B, size_t fit, size_t fo, const LaneRegs<CF>& R, uint64_t jfit) {
  B.ctl[fit] = R.phase | (R.j << 4) | (R.failed << 10) | (R.bad << 11);
  B.lstep[fit] = R.l;
  B.nev[fit] = R.nev;
  B.nev_tot[fit] = R.nev_tot;
  B.steps_tot[fit] = R.steps_tot;
  B.work[fit] = R.work;
  B.fitid[fit] = (int32_t)jfit;
  B.fr[fo] = R.fr;
  B.sf[fo] = R.sf;
}

// One evaluation with LP lanes per model (chi2_model_rows), for the kernels
// below: parameters at PRM[i * stride], delta_V to DV[m * dv_stride].  Out of
// line, so that a kernel class has one copy of it for its kernels.  Being
// called by fit_kernel too, the copies without a team are compiled for 128
// registers; copies of their own budget for the other kernels measured the same
// (256 to 16384 models, with and without torque and torque2: chi^2 between 3%
// less and 2% more time, fits within 2%).
template <class CF, int VC, int NF, bool MX, int LP, int ROLE = ROLE_ALL>
__device__ __attribute__((noinline)) CF eval_rows(const double* PRM, size_t stride, CF* DV, size_t dv_stride,
                                                   const PointRec* pts_g, int n_data, int n_filters, int dof,
                                                   const double* sum_w, TeamPtr<VC, LP> team = nullptr) {
  constexpr int N = Pos<VC>::N;
  const uint64_t pu = (uint64_t)(uintptr_t)pts_g;
  const uint64_t plo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)pu);
  const uint64_t phi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(pu >> 32));
  const uintptr_t pa = (uintptr_t)((phi << 32) | plo);
  n_data = __builtin_amdgcn_readfirstlane(n_data);
  n_filters = __builtin_amdgcn_readfirstlane(n_filters);
  dof = __builtin_amdgcn_readfirstlane(dof);
  double prm[N];
#pragma unroll
  for (int i = 0; i < N; ++i) prm[i] = PRM[(size_t)i * stride];
  CF dv[NF];
#pragma unroll
  for (int m = 0; m < NF; ++m)  // a failed NUDGE model leaves delta_V as it was
    dv[m] = VarF<VC>::NU && m < n_filters ? DV[(size_t)m * dv_stride] : CF(0);
  CF fv = chi2_model_rows<CF, VC, NF, MX, FORM_CHI2, LP, ROLE>(prm, (PointPtr)pa, (LanePtr)pa, n_data, n_filters,
                                                               dof, sum_w, dv, nullptr, 0.0, team);
#pragma unroll
  for (int m = 0; m < NF; ++m)
    if (m < n_filters) DV[(size_t)m * dv_stride] = dv[m];
  return fv;
}

// ---------------------------------------------------------------- fit kernel
// One workgroup = one group (the reference's block); it runs D.ticks rounds
// of "evaluate the pending points, advance every lane", then saves its state.
// W is the register budget as waves per SIMD: 4 (128 VGPRs, groups of up to
// 1024 simplexes), 3 (168 VGPRs) or 2 (256 VGPRs), both for groups of up to
// 256.  The arithmetic is the same for every W; only speed differs, and the
// autotuner picks W per kernel class by measurement.
template <class CF, int VC, int NF, bool MX, int W>
__global__ __launch_bounds__(W == 4 ? 1024 : 256) __attribute__((amdgpu_waves_per_eu(W, W)))
void fit_kernel(const GroupDesc<CF>* descs, SlotBufs<CF> B) {
  astm::sincos_table_load();  // the evaluator's sin/cos table into LDS (whole workgroup)
  using P = Pos<VC>;
  AST_VFLAGS(VC);
  constexpr int N = P::N;
  constexpr int KC = 8 / sizeof(CF);
  const GroupDesc<CF>& D = descs[blockIdx.x];
  const int t = threadIdx.x;
  const int G = blockDim.x;
  const int slot = D.slot;
  const size_t nf = B.nf, rs = KC * nf;
  const size_t fit = (size_t)slot * G + t;
  const size_t fo = (size_t)slot * G * KC + t;
  if (B.g_done[slot]) return;  // same value for every thread of the group
  // group_in_job * G + t unless the lane has refilled
  Machine<CF, VC> M = Machine<CF, VC>::of(D, B, fit, fo, (uint64_t)B.fitid[fit], B.g_reopt[slot]);
  const int ticks = D.ticks;
  int stage = B.g_stage[slot];
  LaneRegs<CF> R = load_lane(B, fit, fo, D.rng[M.jfit]);
  const bool refill = D.refill != 0;
  bool done = false;
  // Fits waiting for an evaluation, packed to the front of the workgroup when
  // that frees a wavefront, and their chi^2 (at a stage's end, its argmin's).
  __shared__ uint16_t s_fit[1024];
  __shared__ CF s_val[1024];
  __shared__ int s_packed;
  CF fv = 0;
  bool have = false;
  for (int tick = 0;;) {
    advance_lane<CF, VC>(M, R, fv, have);  // a lane at a stage start draws its simplex
    int pending;
    if (refill) {
      // A lane whose fit ended keeps its results and starts the job's next
      // unstarted fit (one that fails at its start ends at once and the lane
      // takes another); with the queue empty it idles.  The group is done
      // when every lane idles.
      while (R.phase == PH_STAGE_DONE) {
        M.end_fit(R, D);
        const int nj = take_fit(D.queue);
        if (nj >= D.n_fits) {
          R.phase = PH_FIT_DONE;
          break;
        }
        M.jfit = (uint64_t)nj;
        M.begin_fit(R, D);
        advance_lane<CF, VC>(M, R, (CF)0, false);
      }
      pending = __syncthreads_count(R.phase != PH_FIT_DONE);
      if (pending == 0) done = true;
    } else {
      pending = __syncthreads_count(phase_pending(R.phase));
      if (pending == 0) {
        // Every simplex of the group finished the stage.
        if (group_stage_end<CF, VC>(D, M, R, t, G, stage, M.reopt, s_val)) {
          have = false;
          continue;
        }
        done = true;
      }
    }
    if (done || tick == ticks) break;
    ++tick;
    have = phase_pending(R.phase);
    // An evaluation costs a wavefront the same for one fit as for 64.  Once
    // enough of the group's fits have ended to leave a wavefront without one,
    // the others' points are dealt to the first lanes, whichever fit they
    // belong to (a fit's values do not depend on the lane), and the chi^2 goes
    // back through LDS.  Fits that stop at an evaluation budget end within
    // about N + 1 rounds of each other (12 with LS and torque: the last step's
    // shrink is finished); those that converge or fail end earlier, and with
    // refill each at its own time.  224 groups, two stages of 50 evaluations
    // 74.4 -> 69.3 ms; 2^18 fits of 100, mixed, 212 -> 202; of 4800 the same.
    // With the chip's SIMDs not shared (groups of 65536 fits at most), few enough
    // points take 4 or 16 lanes each: the two-stage search 69.3 -> 64.4 ms, 260
    // groups of 64 fits and 60 evaluations 41.7 -> 36.1.
    const bool spread = (size_t)gridDim.x * G <= 65536;
    const int lp = spread && pending * 16 <= G ? 16 : spread && pending * 4 <= G ? 4 : 1;
    const bool pack = pending <= G - 64 || lp > 1;
    int e = t;
    bool eval = have;
    if (pack) {
      if (t == 0) s_packed = 0;
      __syncthreads();
      const uint64_t mask = __ballot(have);
      const int lane = (int)__lane_id();
      int base = 0;
      if (lane == 0) base = atomicAdd(&s_packed, __popcll(mask));
      base = __builtin_amdgcn_readfirstlane(base);
      if (have) s_fit[base + __popcll(mask & ((1ull << lane) - 1ull))] = (uint16_t)t;
      __syncthreads();
      eval = t / lp < pending;
      if (eval) e = s_fit[t / lp];
    }
    const size_t efit = (size_t)slot * G + e, efo = (size_t)slot * G * KC + e;
    if (lp == 16) {
      if (eval)
        fv = eval_rows<CF, VC, NF, MX, 16>(B.PRM + efit, nf, B.DV + efo, rs, D.pts, D.n_data, D.n_filters, D.dof,
                                           D.sum_w);
    } else if (lp == 4) {
      if (eval)
        fv = eval_rows<CF, VC, NF, MX, 4>(B.PRM + efit, nf, B.DV + efo, rs, D.pts, D.n_data, D.n_filters, D.dof,
                                          D.sum_w);
    } else if (eval)
      fv = eval_lane<CF, VC, NF, MX, MX ? 4 : W>(B.PRM, B.DV, nf, efit, rs, efo, D.pts, D.n_data, D.n_filters, D.dof,
                                                 D.sum_w);
    if (pack) {
      if (eval) s_val[e] = fv;
      __syncthreads();
      if (have) fv = s_val[t];
    }
    if (have) {
      R.nev++;
      R.nev_tot++;
      R.work++;
    }
  }
  const uint64_t jfit = M.jfit;
  const int reopt = M.reopt;
  store_lane(B, fit, fo, R, jfit);
  D.rng[jfit] = R.rng;
  if (t == 0) {
    B.g_reopt[slot] = reopt;
    B.g_stage[slot] = stage;
    B.g_done[slot] = done ? 1 : 0;
    if (done) atomicAdd(D.job_done, 1);
  }
}

// ---------------------------------------------------- several lanes per model
// Registers for one or two waves per SIMD for what is inlined (the simplex's
// set-up): these kernels run where the chip is not full.
#define AST_ROWS_BOUNDS __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 2)))

// chi2_batch_kernel with LP lanes per model, 64 / LP models per workgroup (of
// one wavefront, so that few models spread over the CUs).
template <class CF, int VC, int NF, bool MX, int LP>
__global__ AST_ROWS_BOUNDS void chi2_rows_kernel(const PointRec* pts_g, const double* sum_w, int n_data,
                                                 int n_filters, int dof, const double* params, int n, double* chi2,
                                                 double* dV) {
  astm::sincos_table_load();
  constexpr int N = Pos<VC>::N, M = 64 / LP;
  __shared__ CF s_dv[M][NF];
  const int row = threadIdx.x / LP;
  const int k = blockIdx.x * M + row;
  if (k >= n) return;
  for (int m = 0; m < NF; ++m) s_dv[row][m] = VarF<VC>::NU ? CF(__builtin_nan("")) : CF(0);
  const CF c = eval_rows<CF, VC, NF, MX, LP>(params + (size_t)k * N, 1, s_dv[row], 1, pts_g, n_data, n_filters, dof,
                                             sum_w);
  chi2[k] = c;
  for (int m = 0; m < n_filters; ++m) dV[(size_t)k * n_filters + m] = s_dv[row][m];
}

// The grid walk of model_curve_kernel with LP lanes per model: delta_V of the
// first filter from dV, written by chi2_rows_kernel before it.
template <class CF, int VC, int NF, bool MX, int LP>
__global__ AST_ROWS_BOUNDS void curve_rows_kernel(const double* sum_w, int n_filters, int dof,
                                                  const PointRec* grid_g, int n_plot, const double* params, int n,
                                                  const double* dV, double* vmod) {
  astm::sincos_table_load();
  constexpr int N = Pos<VC>::N, M = 64 / LP;
  const int k = blockIdx.x * M + threadIdx.x / LP;
  if (k >= n) return;
  double prm[N];
#pragma unroll
  for (int i = 0; i < N; ++i) prm[i] = params[(size_t)k * N + i];
  CF dv[NF];
  chi2_model_rows<CF, VC, NF, MX, FORM_PLOT, LP>(prm, (PointPtr)(uintptr_t)grid_g, (LanePtr)(uintptr_t)grid_g, n_plot, n_filters, dof,
                                                 sum_w, dv, vmod + (size_t)k * n_plot, dV[(size_t)k * n_filters]);
}

// The two kernels above with a team of wavefronts for 64 / LP models (rows past
// the last model repeat it).
#define AST_TEAM_BOUNDS __launch_bounds__(192) __attribute__((amdgpu_waves_per_eu(1, 3)))
template <int VC>
constexpr int TEAM_THREADS = VarF<VC>::TQ ? 192 : 128;

template <class CF, int VC, int NF, bool MX, int LP>
__global__ AST_TEAM_BOUNDS void chi2_team_kernel(const PointRec* pts_g, const double* sum_w, int n_data, int n_filters,
                                                 int dof, const double* params, int n, double* chi2, double* dV) {
  astm::sincos_table_load();
  constexpr int N = Pos<VC>::N, M = 64 / LP;
  __shared__ TeamLds<VarF<VC>::TQ, LP> s_team;
  __shared__ CF s_dv[M][NF];
  const TeamPtr<VC, LP> team = (TeamPtr<VC, LP>)&s_team;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  const int row = (int)threadIdx.x % 64 / LP;
  const int k = (int)blockIdx.x * M + row < n ? (int)blockIdx.x * M + row : n - 1;
  const double* prm = params + (size_t)k * N;
  if (wave > 0) return team_helper<VC, LP>(wave, prm, 1, pts_g, n_data, team);
  for (int m = 0; m < NF; ++m) s_dv[row][m] = VarF<VC>::NU ? CF(__builtin_nan("")) : CF(0);
  const CF c = eval_rows<CF, VC, NF, MX, LP, ROLE_LIGHT>(prm, 1, s_dv[row], 1, pts_g, n_data, n_filters, dof, sum_w,
                                                         team);
  chi2[k] = c;
  for (int m = 0; m < n_filters; ++m) dV[(size_t)k * n_filters + m] = s_dv[row][m];
}

template <class CF, int VC, int NF, bool MX, int LP>
__global__ AST_TEAM_BOUNDS void curve_team_kernel(const double* sum_w, int n_filters, int dof, const PointRec* grid_g,
                                                  int n_plot, const double* params, int n, const double* dV,
                                                  double* vmod) {
  astm::sincos_table_load();
  constexpr int N = Pos<VC>::N, M = 64 / LP;
  __shared__ TeamLds<VarF<VC>::TQ, LP> s_team;
  const TeamPtr<VC, LP> team = (TeamPtr<VC, LP>)&s_team;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  const int row = (int)threadIdx.x % 64 / LP;
  const int k = (int)blockIdx.x * M + row < n ? (int)blockIdx.x * M + row : n - 1;
  const double* pk = params + (size_t)k * N;
  if (wave > 0) return team_helper<VC, LP>(wave, pk, 1, grid_g, n_plot, team);
  double prm[N];
#pragma unroll
  for (int i = 0; i < N; ++i) prm[i] = pk[i];
  CF dv[NF];
  chi2_model_rows<CF, VC, NF, MX, FORM_PLOT, LP, ROLE_LIGHT>(prm, (PointPtr)(uintptr_t)grid_g,
                                                             (LanePtr)(uintptr_t)grid_g, n_plot, n_filters, dof, sum_w,
                                                             dv, vmod + (size_t)k * n_plot,
                                                             dV[(size_t)k * n_filters], team);
}

// take_fit for LP lanes per model: one fit per asking model.
template <int LP>
__device__ inline int take_fit_rows(int32_t* queue) {
  constexpr uint64_t firsts = LP == 16 ? 0x0001000100010001ull : 0x1111111111111111ull;
  const uint64_t mask = __ballot(1) & firsts;
  const int lane = (int)__lane_id();
  const int leader = __ffsll((unsigned long long)mask) - 1;
  const int rank = __popcll(mask & ((1ull << (lane & ~(LP - 1))) - 1ull));
  int base = 0;
  if (lane == leader) {
    const int cnt = __popcll(mask);
    base = atomicAdd(&queue[0], cnt);
    atomicAdd(&queue[1], cnt);
  }
  base = __shfl(base, leader);
  return base + rank;
}

// The fitting kernel with LP lanes per model: a workgroup is one wavefront
// that runs 64 / LP of a group's simplexes, so that the simplexes of a few
// groups spread over the whole chip.  Every lane of a model holds and stores
// the model's state (equal values to the same addresses).  A wavefront ends
// its launch when none of its simplexes has a pending point; the end of the
// group's stage, which needs them all, is group_step_kernel's, launched
// after it.  With TEAM the wavefront is the first of a team, whose others
// take their parts of its evaluations.
template <class CF, int VC, int NF, bool MX, int LP, bool TEAM>
__device__ inline void fit_rows(const GroupDesc<CF>* descs, const SlotBufs<CF>& B, int G) {
  astm::sincos_table_load();
  constexpr int KC = 8 / sizeof(CF), MODELS = 64 / LP;
  const int per_group = G / MODELS;
  const GroupDesc<CF>& D = descs[blockIdx.x / per_group];
  const int t = (int)(blockIdx.x % per_group) * MODELS + (int)threadIdx.x % 64 / LP;
  const int slot = D.slot;
  const size_t nf = B.nf, rs = KC * nf;
  const size_t fit = (size_t)slot * G + t;
  const size_t fo = (size_t)slot * G * KC + t;
  if (B.g_done[slot]) return;
  TeamPtr<VC, LP> team = nullptr;
  uint64_t* pending = nullptr;  // the lanes to evaluate; 0 ends the launch
  if constexpr (TEAM) {
    __shared__ TeamLds<VarF<VC>::TQ, LP> s_team;
    __shared__ uint64_t s_pending;
    team = (TeamPtr<VC, LP>)&s_team;
    pending = &s_pending;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
    if (wave > 0) {
      for (;;) {
        __syncthreads();
        const uint64_t lanes = s_pending;
        if (lanes == 0) return;
        if (lanes >> __lane_id() & 1) team_helper<VC, LP>(wave, B.PRM + fit, nf, D.pts, D.n_data, team);
      }
    }
  }
  Machine<CF, VC> M = Machine<CF, VC>::of(D, B, fit, fo, (uint64_t)B.fitid[fit], B.g_reopt[slot]);
  const int ticks = D.ticks;
  LaneRegs<CF> R = load_lane(B, fit, fo, D.rng[M.jfit]);
  const bool refill = D.refill != 0;
  CF fv = 0;
  bool have = false;
  for (int tick = 0;; ++tick) {
    advance_lane<CF, VC>(M, R, fv, have);
    if (refill) {  // as in fit_kernel
      while (R.phase == PH_STAGE_DONE) {
        M.end_fit(R, D);
        const int nj = take_fit_rows<LP>(D.queue);
        if (nj >= D.n_fits) {
          R.phase = PH_FIT_DONE;
          break;
        }
        M.jfit = (uint64_t)nj;
        M.begin_fit(R, D);
        advance_lane<CF, VC>(M, R, (CF)0, false);
      }
    }
    have = phase_pending(R.phase);
    const uint64_t lanes = tick == ticks ? 0 : __ballot(have);
    if constexpr (TEAM) {
      *pending = lanes;
      __syncthreads();
    }
    if (lanes == 0) break;
    if (have) {
      fv = eval_rows<CF, VC, NF, MX, LP, TEAM ? ROLE_LIGHT : ROLE_ALL>(B.PRM + fit, nf, B.DV + fo, rs, D.pts, D.n_data,
                                                                       D.n_filters, D.dof, D.sum_w, team);
      R.nev++;
      R.nev_tot++;
      R.work++;
    }
  }
  const uint64_t jfit = M.jfit;
  store_lane(B, fit, fo, R, jfit);
  D.rng[jfit] = R.rng;
}

template <class CF, int VC, int NF, bool MX, int LP>
__global__ AST_ROWS_BOUNDS void fit_rows_kernel(const GroupDesc<CF>* descs, SlotBufs<CF> B, int G) {
  fit_rows<CF, VC, NF, MX, LP, false>(descs, B, G);
}
template <class CF, int VC, int NF, bool MX, int LP>
__global__ AST_TEAM_BOUNDS void fit_team_kernel(const GroupDesc<CF>* descs, SlotBufs<CF> B, int G) {
  fit_rows<CF, VC, NF, MX, LP, true>(descs, B, G);
}

// After fit_rows_kernel: one workgroup per group ends the group's stage once
// all of its simplexes have (fit_kernel does this in place).
template <class CF, int VC>
__global__ __launch_bounds__(1024) void group_step_kernel(const GroupDesc<CF>* descs, SlotBufs<CF> B) {
  constexpr int KC = 8 / sizeof(CF);
  const GroupDesc<CF>& D = descs[blockIdx.x];
  const int t = threadIdx.x, G = blockDim.x, slot = D.slot;
  if (B.g_done[slot]) return;
  const size_t nf = B.nf, rs = KC * nf;
  const size_t fit = (size_t)slot * G + t, fo = (size_t)slot * G * KC + t;
  const int phase = B.ctl[fit] & 15;
  if (__syncthreads_count(phase != (D.refill ? PH_FIT_DONE : PH_STAGE_DONE))) return;
  bool done = true;
  int stage = B.g_stage[slot], reopt = B.g_reopt[slot];
  if (!D.refill) {
    const uint64_t jfit = (uint64_t)B.fitid[fit];
    LaneRegs<CF> R = load_lane(B, fit, fo, D.rng[jfit]);
    const Machine<CF, VC> M = Machine<CF, VC>::of(D, B, fit, fo, jfit, reopt);
    __shared__ CF s_f[1024];
    done = !group_stage_end<CF, VC>(D, M, R, t, G, stage, reopt, s_f);
    store_lane(B, fit, fo, R, jfit);
  }
  if (t == 0) {
    B.g_reopt[slot] = reopt;
    B.g_stage[slot] = stage;
    B.g_done[slot] = done ? 1 : 0;
    if (done) atomicAdd(D.job_done, 1);
  }
}

// ------------------------------------------------------------- chi2 batch
template <class CF, int VC, int NF, bool MX>
__global__ __launch_bounds__(256) void chi2_batch_kernel(const PointRec* pts_g, const double* sum_w, int n_data,
                                                        int n_filters, int dof, const double* params, int n,
                                                        double* chi2, double* dV) {
  astm::sincos_table_load();  // the evaluator's sin/cos table into LDS (whole workgroup)
  using P = Pos<VC>;
  AST_VFLAGS(VC);
  constexpr int N = P::N;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  PointPtr pts = (PointPtr)(uintptr_t)pts_g;
  double prm[N];
#pragma unroll
  for (int i = 0; i < N; ++i) prm[i] = params[(size_t)k * N + i];
  CF dv[NF];
#pragma unroll
  for (int m = 0; m < NF; ++m) dv[m] = NU ? CF(__builtin_nan("")) : CF(0);  // NaN: a failed NUDGE model
  CF c = chi2_model<CF, VC, NF, MX>(prm, pts, n_data, n_filters, dof, sum_w, dv);
  chi2[k] = c;
  for (int m = 0; m < n_filters; ++m) dV[(size_t)k * n_filters + m] = dv[m];
}

// ------------------------------------------------------------ model curve
// The -plot evaluation (chi2_plot, cuda.c:1865-1966, without PROFILES and
// ANIMATE), one model per lane: chi^2 and delta_V of the model against the
// observations (step one, cuda.c:1939-1942), then the model magnitude plus
// delta_V[0] at each point of the plotting grid (step two, cuda.c:1949-1950),
// integrated along the grid from its first time.  vmod is model-major: lane
// k writes vmod[k * n_plot + i].
template <class CF, int VC, int NF, bool MX>
__global__ __launch_bounds__(256) void model_curve_kernel(const PointRec* pts_g, const double* sum_w, int n_data,
                                                         int n_filters, int dof, const PointRec* grid_g, int n_plot,
                                                         const double* params, int n, double* chi2, double* dV,
                                                         double* vmod) {
  astm::sincos_table_load();  // the evaluator's sin/cos table into LDS (whole workgroup)
  using P = Pos<VC>;
  AST_VFLAGS(VC);
  constexpr int N = P::N;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  double prm[N];
#pragma unroll
  for (int i = 0; i < N; ++i) prm[i] = params[(size_t)k * N + i];
  CF dv[NF];
#pragma unroll
  for (int m = 0; m < NF; ++m) dv[m] = NU ? CF(__builtin_nan("")) : CF(0);  // NaN: a failed NUDGE model
  CF c = chi2_model<CF, VC, NF, MX>(prm, (PointPtr)(uintptr_t)pts_g, n_data, n_filters, dof, sum_w, dv);
  chi2[k] = c;
  for (int m = 0; m < n_filters; ++m) dV[(size_t)k * n_filters + m] = dv[m];
  chi2_model<CF, VC, NF, MX, FORM_PLOT>(prm, (PointPtr)(uintptr_t)grid_g, n_plot, n_filters, dof, sum_w,
                                               dv, vmod + (size_t)k * n_plot, 1, (double)dv[0]);
}

// ------------------------------------------------------------------- RMSD
// Confidence intervals by random shifts around an input model
// (chi2_gpu_rms, cuda.c:2148-2389, the RMSD build).  RmsdRef holds what
// every thread of the reference computes first (cuda.c:2217-2247): the
// input model in scale-free coordinates, its RMSD f0 and the acceptance
// threshold f1 = f0 + f0/sqrt(N_data - N_PARAMS - N_filters).
template <class CF>
struct RmsdRef {
  CF x0[MAXP];
  CF f0, f1;
  double phi_M0, phi_00, phi_K0;  // the input model's phi_M, phi_0 and torque azimuth
};

template <class CF>
struct RmsdArgs {
  const PointRec* pts;
  const double* sum_w;
  int n_data, n_filters, dof;
  const Space<CF>* sp;
  int reopt;
  const double* params0;  // d_params0
  RmsdRef<CF>* ref;
  uint32_t* rng;          // per-lane stream counters (the curandState array)
  uint64_t seed;
  int n_samples;          // Nstages: random points per lane
  float dx;               // dx_rand
  int spherical_k;        // SPHERICAL_K
  float* par_min;         // [group][N_PARAMS] (dpar_min)
  float* par_max;
  int32_t* counts;        // [group][2]: Ntot, Nbad
};

template <class CF, int VC, int NF, bool MX>
__global__ AST_ROWS_BOUNDS void rmsd_ref_kernel(RmsdArgs<CF> A) {
  astm::sincos_table_load();  // the evaluator's sin/cos table into LDS (whole workgroup)
  using P = Pos<VC>;
  AST_VFLAGS(VC);
  constexpr int N = P::N;
  if (threadIdx.x >= 16) return;  // one model, a row of lanes
  double prm[N];
  for (int i = 0; i < N; ++i) prm[i] = A.params0[i];
  CF x[N];
  params2x<CF, VC>(x, prm, *A.sp);
  CF dv[NF];
  const CF f0 = chi2_model_rows<CF, VC, NF, MX, FORM_RMSD, 16>(prm, (PointPtr)(uintptr_t)A.pts, (LanePtr)(uintptr_t)A.pts, A.n_data,
                                                               A.n_filters, A.dof, A.sum_w, dv);
  if (threadIdx.x != 0) return;
  RmsdRef<CF>& R = *A.ref;
  for (int i = 0; i < N; ++i) R.x0[i] = x[i];
  R.f0 = f0;
  R.f1 = f0 + f0 / (CF)__builtin_sqrt((double)(CF)A.dof);
  R.phi_M0 = prm[P::phi_M];
  R.phi_00 = prm[P::phi_0];
  R.phi_K0 = 0.0;
  if (TQ) {
    const double bt = prm[P::b_tumb], ct = prm[P::c_tumb];
    const double Is = (1.0 + bt * bt) / (bt * bt + ct * ct);
    const double Ii = (1.0 + ct * ct) / (bt * bt + ct * ct);
    R.phi_K0 = astm::atan2(Is * prm[P::Ts], Ii * prm[P::Ti]);
  }
}

// One lane per thread of the reference: n_samples shifted models each,
// the range of the accepted ones per parameter, reduced per group in lane
// order by the group's first thread (cuda.c:2356-2381).
template <class CF, int VC, int NF, bool MX, int W>
__global__ __launch_bounds__(W == 4 ? 1024 : 256) __attribute__((amdgpu_waves_per_eu(W, W))) void rmsd_kernel(
    RmsdArgs<CF> A) {
  astm::sincos_table_load();  // the evaluator's sin/cos table into LDS (whole workgroup)
  using P = Pos<VC>;
  AST_VFLAGS(VC);
  constexpr int N = P::N;
  constexpr double PI = 3.141592653589793238;
  constexpr double SMALL = 1e-8;  // cuda.c:2258
  __shared__ float s_min[1024], s_max[1024];
  __shared__ int32_t s_cnt[2][1024];
  const int t = threadIdx.x;
  const uint64_t id = (uint64_t)blockIdx.x * blockDim.x + t;
  const auto& sp = *(SpacePtr<CF>)(uintptr_t)A.sp;
  const RmsdRef<CF>& R = *A.ref;
  CF pmin[N], pmax[N];
  for (int i = 0; i < N; ++i) { pmin[i] = (CF)1e30; pmax[i] = (CF)-1e30; }
  int32_t ntot = 0, nbad = 0;
  uint32_t ctr = A.rng[id];
  double prm[N];
  for (int s = 0; s < A.n_samples; ++s) {
    int LAM = 0;
    CF x1[N];
    for (int i = 0; i < N; ++i) {  // cuda.c:2276-2287
      const float z = astrng::normal01(A.seed, id, ctr);
      ctr += 2;
      CF xx = R.x0[i] + (CF)(A.dx * z);
      const int per = sp.periodic[i];
      if (xx < SMALL && hard_left(per, LAM)) xx = (CF)SMALL;
      else if (xx > 1.0 - SMALL && hard_right(per, LAM)) xx = (CF)(1.0 - SMALL);
      x1[i] = xx;
      if (P::is_Es(i)) LAM = x1[i] >= (CF)0.5;
    }
    if (x2params_at<CF, VC>(x1, prm, sp, A.reopt)) continue;
    CF dv[NF];
    const CF f = chi2_model<CF, VC, NF, MX, FORM_RMSD>(prm, (PointPtr)(uintptr_t)A.pts, A.n_data,
                                                               A.n_filters, A.dof, A.sum_w, dv);
    ntot++;
    if (f < R.f1) {
      // cuda.c:2304-2311, as written: an angle beyond +-pi of the input's is
      // set to the input's value -2 pi, which the second test then moves to
      // the input's value +2 pi
      if (prm[P::phi_M] > R.phi_M0 + PI) prm[P::phi_M] = R.phi_M0 - 2 * PI;
      if (prm[P::phi_M] < R.phi_M0 - PI) prm[P::phi_M] = R.phi_M0 + 2 * PI;
      if (prm[P::phi_0] > R.phi_00 + PI) prm[P::phi_0] = R.phi_00 - 2 * PI;
      if (prm[P::phi_0] < R.phi_00 - PI) prm[P::phi_0] = R.phi_00 + 2 * PI;
      if (TQ && A.spherical_k) {  // cuda.c:2312-2333
        const double bt = prm[P::b_tumb], ct = prm[P::c_tumb];
        const double Is = (1.0 + bt * bt) / (bt * bt + ct * ct);
        const double Ii = (1.0 + ct * ct) / (bt * bt + ct * ct);
        const double Ki = Ii * prm[P::Ti], Ks = Is * prm[P::Ts], Kl = prm[P::Tl];
        const double K = __builtin_sqrt(Ki * Ki + Ks * Ks + Kl * Kl);
        prm[P::Ti] = K;
        prm[P::Ts] = astm::acos(Kl / K);
        double phi = astm::atan2(Ks, Ki);
        if (phi > R.phi_K0 + PI) phi = phi - 2 * PI;
        if (phi < R.phi_K0 - PI) phi = phi + 2 * PI;
        prm[P::Tl] = phi;
      }
      for (int i = 0; i < N; ++i) {
        if (prm[i] < pmin[i]) pmin[i] = (CF)prm[i];
        if (prm[i] > pmax[i]) pmax[i] = (CF)prm[i];
      }
    } else {
      nbad++;
    }
  }
  A.rng[id] = ctr;
  s_cnt[0][t] = ntot;
  s_cnt[1][t] = nbad;
  for (int i = 0; i < N; ++i) {
    s_min[t] = (float)pmin[i];
    s_max[t] = (float)pmax[i];
    __syncthreads();
    if (t == 0) {
      float fmin = 1e30f, fmax = -1e30f;
      for (int j = 0; j < (int)blockDim.x; ++j) {
        if (s_min[j] < fmin) fmin = s_min[j];
        if (s_max[j] > fmax) fmax = s_max[j];
      }
      A.par_min[(size_t)blockIdx.x * N + i] = fmin;
      A.par_max[(size_t)blockIdx.x * N + i] = fmax;
    }
    __syncthreads();
  }
  if (t == 0) {
    int32_t a = 0, b = 0;
    for (int j = 0; j < (int)blockDim.x; ++j) { a += s_cnt[0][j]; b += s_cnt[1][j]; }
    A.counts[(size_t)blockIdx.x * 2] = a;
    A.counts[(size_t)blockIdx.x * 2 + 1] = b;
  }
}

// --------------------------------------------------------- launch interface
struct LaunchArgs {
  int op;  // 0 init groups, 1 fit ticks, 2 chi2 batch, 3 model curve, 4 and 5 RMSD,
           // 6 the grid of a model curve (several lanes per model, after its chi2 batch)
  int precision;
  hipStream_t stream;
  // fit: descriptors of the groups of this launch (device), their count, G
  const void* descs;   // GroupDesc<CF>*
  const void* bufs;    // SlotBufs<CF>*
  int n_groups, group_size, n_filters;
  int waves;           // fit kernel register budget: 4, 3 or 2 waves per SIMD
  int64_t fits;        // fit: fits evaluated side by side (fit_shape)
  // batch
  const PointRec* pts;
  const double* sum_w;
  int n_data, dof;
  const double* params;
  int n;
  double* chi2;
  double* dV;
  // model curve: the plotting grid and the magnitudes on it
  const PointRec* grid;
  int n_plot;
  double* vmod;
  // RMSD: RmsdArgs<CF> (op 4: the input model, op 5: the shifted models)
  const void* rmsd;
};

// Lanes per model, and whether a team of wavefronts walks the models of a
// wavefront, for n models (fits, in a cycle) evaluated side by side: as many
// lanes as leave each of the 1024 SIMDs one wavefront, since a wavefront alone
// takes its own time whatever its lanes hold, and teams where their two
// wavefronts (three with torque, of which the first is idle half the time)
// find a SIMD each; the model cut in two parts (torque2) has no teams, its
// step counts being the model's own.
// Kernel time with 16-lane teams / 16 lanes / 4-lane teams / 4 lanes / one lane
// (LS, 400 points over 3 days, FP64; the form taken in brackets):
//   chi^2, torque, us        fits of 30 evaluations, torque, ms
//     64 [244] 277 257 341 511    256 [11.1] 12.1 12.3 14.6 19.5
//   1024 [261] 292 264 345 515   1024 [11.6] 12.9 12.7 15.9 20.1
//   2048 342 307 [267] 346 515   2048 21.3 13.6 [12.8] 16.0 20.1
//   4096 431 326 [272] 346 512   4096 41.0 16.1 [13.3] 16.1 20.1
//   6144 775 549 332 [348] 515   6144 58.2 24.2 23.2 [18.9] 20.1
//  12288 - 811 369 [365] 520    12288 - - 35.4 [21.8] 20.2
//  16384 - 1037 599 [375] 524   16384 - - 46.3 [22.8] 20.3
//  24576 - - 827 636 [538]      24576 - - 67.4 33.6 [20.6]
//   chi^2, no torque, us     fits, no torque, ms
//   1024 [207] 216 212 281 461   1024 8.1 [8.4] 9.1 11.6 16.2
//   2048 244 229 [214] 287 462   2048 8.5 [8.9] 9.2 11.7 16.3
//   4096 265 243 [215] 293 459   4096 16.0 [9.5] 9.5 12.0 16.2
//   8192 695 409 [245] 296 464   8192 30.6 17.5 [10.3] 13.2 16.3
//  12288 927 576 255 [302] 465  12288 - - 17.1 [14.1] 16.4
//  16384 - 731 302 [309] 468    16384 - - 18.8 [14.9] 16.3
//  24576 - - 551 491 [475]      24576 - - 26.3 23.1 [16.6]
// The lines are the fits' with torque, and are taken for chi^2 too: its 4-lane
// teams would still be 4% ahead at 6144 and 8192.  Without torque, where only
// the brightness is taken off, chi^2 teams end with the fits' although they are
// ahead up to 16384 (16% at 12288), and 16-lane teams are not built for the
// fits: ahead by 4% up to 2048 only (a BC search by 4 to 6%).  From 12288 fits on
// one lane is ahead in the table since its last fits share wavefronts, which is
// much of 30 evaluations; of 200, fits with torque take 81 and 84 ms on 4 lanes
// at 12288 and 16384, 111 and 112 on one, and 153 and 113 at 20480.
struct RowShape {
  int lanes;
  bool team;
};
constexpr RowShape chi2_shape(bool torque, bool torque2, int64_t n) {
  if (torque2) return {n <= 4096 ? 16 : n <= 16384 ? 4 : 1, false};
  const bool team = n <= (torque ? 4096 : 8192);
  return {n <= 1024 ? 16 : n <= 16384 ? 4 : 1, team};
}
constexpr RowShape fit_shape(bool torque, bool torque2, int64_t n) {
  if (torque && !torque2) return chi2_shape(torque, torque2, n);
  return {n <= 4096 ? 16 : n <= 16384 ? 4 : 1, !torque2 && n > 4096 && n <= 8192};
}
constexpr int64_t ROWS_MAX = 16384;  // more models take a lane each
// More model curves take a lane each.  The line is where 4-lane teams with
// torque still find a SIMD for each wavefront; curves of 2000 points take 1.29
// ms up to there and 2.75 beyond (4-lane teams 1.65 for 4097, 1.71 for 8192, 1.85
// for 12288 and 2.87 against 2.83 for 16384; without torque 1.24, 1.33, 1.68 and
// 1.98 against 2.63 to 2.71), as before there were several lanes per model.
constexpr int CURVE_ROWS_MAX = 4096;

template <class CF, int VC, int NF, bool MX, int LP, bool TEAM>
void launch_chi2_rows(const LaunchArgs& a) {
  const dim3 grid((a.n + 64 / LP - 1) / (64 / LP));
  if constexpr (TEAM)
    hipLaunchKernelGGL((chi2_team_kernel<CF, VC, NF, MX, LP>), grid, dim3(TEAM_THREADS<VC>), 0, a.stream, a.pts,
                       a.sum_w, a.n_data, a.n_filters, a.dof, a.params, a.n, a.chi2, a.dV);
  else
    hipLaunchKernelGGL((chi2_rows_kernel<CF, VC, NF, MX, LP>), grid, dim3(64), 0, a.stream, a.pts, a.sum_w, a.n_data,
                       a.n_filters, a.dof, a.params, a.n, a.chi2, a.dV);
}
template <class CF, int VC, int NF, bool MX, int LP>
void launch_curve_rows(const LaunchArgs& a) {
  const dim3 grid((a.n + 64 / LP - 1) / (64 / LP));
  if constexpr (VarF<VC>::T2)
    hipLaunchKernelGGL((curve_rows_kernel<CF, VC, NF, MX, LP>), grid, dim3(64), 0, a.stream, a.sum_w, a.n_filters,
                       a.dof, a.grid, a.n_plot, a.params, a.n, a.dV, a.vmod);
  else
    hipLaunchKernelGGL((curve_team_kernel<CF, VC, NF, MX, LP>), grid, dim3(TEAM_THREADS<VC>), 0, a.stream, a.sum_w,
                       a.n_filters, a.dof, a.grid, a.n_plot, a.params, a.n, a.dV, a.vmod);
}
template <class CF, int VC, int NF, bool MX, int LP, bool TEAM>
void launch_fit_rows(const LaunchArgs& a) {
  const GroupDesc<CF>* d = (const GroupDesc<CF>*)a.descs;
  const SlotBufs<CF>& B = *(const SlotBufs<CF>*)a.bufs;
  const dim3 grid(a.n_groups * (a.group_size / (64 / LP)));
  if constexpr (TEAM)
    hipLaunchKernelGGL((fit_team_kernel<CF, VC, NF, MX, LP>), grid, dim3(TEAM_THREADS<VC>), 0, a.stream, d, B,
                       a.group_size);
  else
    hipLaunchKernelGGL((fit_rows_kernel<CF, VC, NF, MX, LP>), grid, dim3(64), 0, a.stream, d, B, a.group_size);
  hipLaunchKernelGGL((group_step_kernel<CF, VC>), dim3(a.n_groups), dim3(a.group_size), 0, a.stream, d, B);
}

template <class CF, int VC, int NF, bool MX>
hipError_t launch_nf(const LaunchArgs& a) {
  constexpr bool TQ = VarF<VC>::TQ, T2 = VarF<VC>::T2;
  const RowShape fit = fit_shape(TQ, T2, a.fits), chi2 = chi2_shape(TQ, T2, a.n);
  if (a.op == 0) {
    hipLaunchKernelGGL((fit_init_kernel<CF, VC>), dim3(a.n_groups), dim3(a.group_size), 0, a.stream,
                       (const GroupDesc<CF>*)a.descs, *(const SlotBufs<CF>*)a.bufs);
  } else if (a.op == 1 && fit.lanes == 16) {
    launch_fit_rows<CF, VC, NF, MX, 16, TQ && !T2>(a);
  } else if (a.op == 1 && fit.lanes == 4 && fit.team) {
    launch_fit_rows<CF, VC, NF, MX, 4, !T2>(a);
  } else if (a.op == 1 && fit.lanes == 4) {
    launch_fit_rows<CF, VC, NF, MX, 4, false>(a);
  } else if (a.op == 1) {
    const GroupDesc<CF>* d = (const GroupDesc<CF>*)a.descs;
    const SlotBufs<CF>& B = *(const SlotBufs<CF>*)a.bufs;
    const int w = a.group_size > 256 ? 4 : a.waves;  // W < 4 kernels take groups of up to 256
    if (w == 2)
      hipLaunchKernelGGL((fit_kernel<CF, VC, NF, MX, 2>), dim3(a.n_groups), dim3(a.group_size), 0, a.stream,
                         d, B);
    else if (w == 3)
      hipLaunchKernelGGL((fit_kernel<CF, VC, NF, MX, 3>), dim3(a.n_groups), dim3(a.group_size), 0, a.stream,
                         d, B);
    else
      hipLaunchKernelGGL((fit_kernel<CF, VC, NF, MX, 4>), dim3(a.n_groups), dim3(a.group_size), 0, a.stream,
                         d, B);
  } else if (a.op == 2 && chi2.lanes == 16) {
    launch_chi2_rows<CF, VC, NF, MX, 16, !T2>(a);
  } else if (a.op == 2 && chi2.lanes == 4 && chi2.team) {
    launch_chi2_rows<CF, VC, NF, MX, 4, !T2>(a);
  } else if (a.op == 2 && chi2.lanes == 4) {
    launch_chi2_rows<CF, VC, NF, MX, 4, false>(a);
  } else if (a.op == 2) {
    int blocks = (a.n + 255) / 256;
    hipLaunchKernelGGL((chi2_batch_kernel<CF, VC, NF, MX>), dim3(blocks), dim3(256), 0, a.stream, a.pts,
                       a.sum_w, a.n_data, a.n_filters, a.dof, a.params, a.n, a.chi2, a.dV);
  } else if (a.op == 6 && chi2.lanes == 16) {
    launch_curve_rows<CF, VC, NF, MX, 16>(a);
  } else if (a.op == 6) {
    if constexpr (!T2) launch_curve_rows<CF, VC, NF, MX, 4>(a);  // torque2: CURVE_ROWS_MAX models take 16
  } else if (a.op == 3) {
    int blocks = (a.n + 255) / 256;
    hipLaunchKernelGGL((model_curve_kernel<CF, VC, NF, MX>), dim3(blocks), dim3(256), 0, a.stream, a.pts,
                       a.sum_w, a.n_data, a.n_filters, a.dof, a.grid, a.n_plot, a.params, a.n, a.chi2, a.dV,
                       a.vmod);
  } else if (a.op == 4) {
    hipLaunchKernelGGL((rmsd_ref_kernel<CF, VC, NF, MX>), dim3(1), dim3(64), 0, a.stream,
                       *(const RmsdArgs<CF>*)a.rmsd);
  } else if (a.group_size > 256) {  // groups of up to 1024: 128 registers
    hipLaunchKernelGGL((rmsd_kernel<CF, VC, NF, MX, 4>), dim3(a.n_groups), dim3(a.group_size), 0, a.stream,
                       *(const RmsdArgs<CF>*)a.rmsd);
  } else {
    hipLaunchKernelGGL((rmsd_kernel<CF, VC, NF, MX, 2>), dim3(a.n_groups), dim3(a.group_size), 0, a.stream,
                       *(const RmsdArgs<CF>*)a.rmsd);
  }
  return hipGetLastError();
}

template <class CF, int VC, bool MX>
hipError_t launch_cf(const LaunchArgs& a) {
  if (a.n_filters <= 1) return launch_nf<CF, VC, 1, MX>(a);
  if (a.n_filters <= 4) return launch_nf<CF, VC, 4, MX>(a);
  return launch_nf<CF, VC, MAXF, MX>(a);
}

// Simplex float and evaluator form by precision: FP64 (double simplex, FP64
// evaluator), F32SIMPLEX (float simplex, FP64 evaluator: the reference's
// default CHI_FLOAT), MIXED (float simplex, mixed-precision evaluator).
template <int VC>
hipError_t launch_variant(const LaunchArgs& a) {
  if (a.precision == AST_PREC_FP64) return launch_cf<double, VC, false>(a);
  if (a.precision == AST_PREC_MIXED) return launch_cf<float, VC, true>(a);
  return launch_cf<float, VC, false>(a);
}

}  // namespace ast
