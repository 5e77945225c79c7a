// nbg_split.h -- device code of the two-wave launches (nbg_run_split): the
// state of a system, or of two, on one wave and its Jacobian on another.
//
// The state of AHL21 never reads the Jacobian, so a workgroup divides every
// step between two waves:
//  * the state wave takes the drifts, the Kepler levels, the force-gradient
//    velocities, the transit tests and Newton's iterations; it runs ahead;
//  * the Jacobian wave follows: the pairs' analytic Jacobians, the row
//    updates, Phi and its product, the drifts of J, dq/dt, and the transits'
//    gradients.
// Alone on a compute unit the two run on different SIMDs and a step takes the
// longer of the two instead of their sum; with four workgroups a compute unit
// each SIMD holds two waves, so that one issues while the other waits (a lone
// wave issues vector instructions about 40 % of the time).  The half of the
// code that each wave runs also keeps registers within the 256 that two waves
// per SIMD leave each.
//
// The waves talk through LDS: a ring of pair slots (22 doubles each; the rest
// of a pair's drift is formed again from them, with the same operations) and
// three messages a step (PRE: the step's kind, size and velocities; MID: the
// positions between the sweeps; POST: the final state), each buffer with one
// writer and one reader, published by workgroup-scope release of a counter.
// Waits are bounded like those of nbg_run_coop: a failure ends both waves and
// is reported, it never hangs.
//
// Systems with Kepler pairs only and no massless pair (their schedule of
// levels is the same for every system of a body count); every operation is the
// one-wave step's, so results are the same bits.
#pragma once

#include "nbg_device.h"

namespace nbg {

// The level schedule of both sweeps of NB bodies, every pair a Kepler pair.
template <int NB> struct Schedule {
  static constexpr int NP = NB * (NB - 1) / 2, NL = 2 * NB - 3;
  uint8_t pairs[2][2 * NP];
  uint8_t width[2][NL];
};
template <int NB> constexpr Schedule<NB> make_schedule() {
  Schedule<NB> s{};
  constexpr int NP = Schedule<NB>::NP;
  for (int dir = 0; dir < 2; ++dir) {
    int pi[NP] = {}, pj[NP] = {}, lv[NP] = {}, last[NB] = {};
    int np = 0;
    if (dir == 0) {
      for (int i = 0; i < NB - 1; ++i)
        for (int j = i + 1; j < NB; ++j) { pi[np] = i; pj[np] = j; ++np; }
    } else {
      for (int i = NB - 2; i >= 0; --i)
        for (int j = NB - 1; j >= i + 1; --j) { pi[np] = i; pj[np] = j; ++np; }
    }
    for (int p = 0; p < NP; ++p) {
      const int a = last[pi[p]], b = last[pj[p]];
      lv[p] = (a > b ? a : b) + 1;
      last[pi[p]] = last[pj[p]] = lv[p];
    }
    int w = 0;
    for (int l = 0; l < Schedule<NB>::NL; ++l)
      for (int p = 0; p < NP; ++p)
        if (lv[p] == l + 1) {
          s.pairs[dir][2 * w] = (uint8_t)pi[p];
          s.pairs[dir][2 * w + 1] = (uint8_t)pj[p];
          ++w;
          s.width[dir][l] += 1;
        }
  }
  return s;
}
template <int NB> __device__ constexpr Schedule<NB> kSchedule = make_schedule<NB>();

// What the state wave hands over of a pair's drift; the other quantities of
// KParams and the drift itself follow from these.
struct RingSlot {
  double x0[3], v0[3];
  double gamma, g1, g2, g3, h1, h2, r0, r, r0inv, rinv, beta, betainv, eta, sqb;
  double mijinv;
  int i, j;
};
// A pair's Jacobian as the row updates read it.
struct JacSlot {
  double kep[48];
  double mc[24];
  double mi, mj;
  int i, j;
};

// The state wave's record of a system.
template <int NB> struct StateRec {
  static constexpr int N3 = 3 * NB, NP = NB * (NB - 1) / 2;
  double x[N3], v[N3], xe[N3], ve[N3], m[NB];  // in this order (pair_state)
  double px[N3], pv[N3], pxe[N3], pve[N3];     // s_prior
  double a[N3];
  double fac[3 * NP];  // the force-gradient stage's pair factors
  double gsave[NB];
  double t, pt;
  int64_t count[NB];
};

// The Jacobian wave's record.  mv, mx, qx, qv: the messages' buffers.
template <int NB, bool G> struct JacRec {
  static constexpr int N3 = 3 * NB, N6 = 6 * NB, N7 = 7 * NB;
  static constexpr int JOFF = N6 * N7;
  static constexpr bool JG = G;
  double JJ[JG ? 1 : 2 * N6 * N7];
  double* jg;
  double dqij[14];
  double x[N3], v[N3], m[NB], a[N3];
  double dqdt[N7], dqdt_phi[N7], dqdt_kick[N7];
  double run_dqdt[N7];  // dq/dt as the run leaves it (searches use dqdt)
  double mv[N3], mx[N3], qx[N3], qv[N3];
};

// The Jacobian wave's work area: the force-gradient stage, or pair Jacobians.
template <int NB> struct JacWork {
  static constexpr int N3 = 3 * NB, N4 = 4 * NB, NP = NB * (NB - 1) / 2, PQ = 13;
  struct F {
    double phi[N3 * N4];
    double dadq[N3 * N4];
    double pq[NP * PQ];
  };
  static constexpr int FIT = (int)(sizeof(F) / sizeof(JacSlot));
  static constexpr int CH = FIT < 1 ? 1 : (FIT < NP ? FIT : NP);
  union {
    F f;
    JacSlot slot[CH];
  };
};

// Steps of a system as the Jacobian wave sees them (RunCursor's act).
enum : int { SPLIT_J = 4, SPLIT_Q = 8, SPLIT_SAVE = 16 };
struct SplitCtl {
  int tail, head;     // pairs published / released, per system
  int sent, seen;     // messages published / copied
  int answered;       // steps whose dq/dt is complete
  int quit;           // the state wave is done, or a wait ran out
  int act[2];         // PRE: what the step is
  int body[2];        // PRE: a gradient step's body ...
  int64_t index[2];   // ... and transit
  double h[2];
};

template <int NB, bool G, bool TWO, int LIMIT> struct SplitLds {
  static constexpr int NS = TWO ? 2 : 1;
  static constexpr bool HALF = TWO && 7 * NB <= 32 && !G;  // every stage on half-waves
  static constexpr size_t FIXED = NS * (sizeof(StateRec<NB>) + sizeof(JacRec<NB, G>)) + sizeof(SplitCtl) +
                                  sizeof(Schedule<NB>) + 64;
  static constexpr int NP = NB * (NB - 1) / 2;
  static constexpr int RMIN = NB / 2 < 1 ? 1 : NB / 2;
  // two work areas where they fit: both systems' force gradients at once
  static constexpr bool PHI2 = TWO && 4 * NB <= 32 && NP <= 32 &&
                               FIXED + 2 * sizeof(JacWork<NB>) + 2 * RMIN * sizeof(RingSlot) <= (size_t)LIMIT;
  static constexpr int NW = PHI2 ? 2 : 1;
  static constexpr long LEFT = (long)LIMIT - (long)(FIXED + NW * sizeof(JacWork<NB>));
  static constexpr int RFIT = LEFT > 0 ? (int)(LEFT / (long)(NS * sizeof(RingSlot))) : 0;
  static constexpr int R = RFIT < NP ? RFIT : NP;  // ring slots per system
  static constexpr bool fits = RFIT >= RMIN;
  // pairs per chunk of the Jacobian wave (a chunk is a run of whole levels)
  static constexpr int CHW = TWO && !PHI2 ? JacWork<NB>::CH / 2 : JacWork<NB>::CH;
  static constexpr int CHL = TWO ? 32 : 64;
  static constexpr int CH0 = CHW < CHL ? CHW : CHL;
  static constexpr int RR = R < 1 ? 1 : R;
  static constexpr int CH = CH0 < RR ? CH0 : RR;
  static constexpr bool ok = fits && CH >= RMIN;
  StateRec<NB> t[NS];
  JacRec<NB, G> j[NS];
  JacWork<NB> w[NW];
  RingSlot ring[NS][RR];
  SplitCtl ctl;
  Schedule<NB> sched;
};

__device__ __forceinline__ void publish(int* counter, int v, int lane) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  if (lane == 0) ring_store(counter, v);
}
// Waits until *counter >= v (as a difference); false when the other wave has
// quit or the bound runs out.
__device__ __forceinline__ bool wait_for(const int* counter, int v, SplitCtl* ctl, int64_t bound, unsigned long long* err,
                                         int lane) {
  int64_t spins = 0;
  while (ring_load(counter) - v < 0) {
    if (ring_load(&ctl->quit) == 2) return false;
    if (++spins > bound) {
      if (lane == 0) {
        atomicOr(err, 4ull);
        ring_store(&ctl->quit, 2);
      }
      return false;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  return true;
}

// ---------------------------------------------------------------------------
// State wave
// ---------------------------------------------------------------------------
// A sweep of one system or two of equal body count (act: which have a step):
// lanes [0, w) the first's pairs of a level, [w, 2w) the second's.  keep: the
// Jacobian wave follows, so each level's pairs go to the ring once it has room.
// One out-of-line copy per direction for every body count.
struct SplitSweep {
  uint32_t x0, x1, ring0, ring1, pairs, width, ctl;
  int n3, levels, act0, act1, keep, slots, pos, made;
  double hh0, hh1;
  int64_t bound;
  unsigned long long* err;
};
template <bool DF> static __device__ __attribute__((noinline)) bool split_levels(SplitSweep R) {
  const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  auto uni = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  const int levels = uni(R.levels), n3 = uni(R.n3), slots = uni(R.slots);
  const bool a0 = uni(R.act0) != 0, a1 = uni(R.act1) != 0, keep = uni(R.keep) != 0;
  int pos = uni(R.pos), made = uni(R.made);
  const uint8_t* lw = lds_at<uint8_t>(uni(R.width));
  const uint8_t* pl = lds_at<uint8_t>(uni(R.pairs));
  SplitCtl* ctl = lds_at<SplitCtl>(uni(R.ctl));
  // the next level's width and pairs are read while this one is solved
  int q0 = 0, w = uni((int)lw[0]);
  bool second = lane >= w;
  int q = lane - (second ? w : 0);
  bool on = lane < 2 * w && (second ? a1 : a0);
  uint32_t ij = 0;
  if (on) ij = pl[2 * q] | ((uint32_t)pl[2 * q + 1] << 8);
#pragma unroll 1
  for (int L = 0; L < levels; ++L) {
    const int w1 = L + 1 < levels ? (int)lw[L + 1] : 0;
    if (keep && !wait_for(&ctl->head, made + w - slots, ctl, R.bound, R.err, lane)) return false;
    if (on) {
      const int i = ij & 0xff, j = ij >> 8;
      double x0[3], v0[3], d[6], m_i, m_j, mijinv;
      KParams P;
      pair_state<DF>(lds_at<double>(second ? R.x1 : R.x0), n3, i, j, second ? R.hh1 : R.hh0, x0, v0, P, d, m_i, m_j,
                     mijinv);
      if (keep) {
        int at = pos + q;
        if (at >= slots) at -= slots;
        RingSlot* o = lds_at<RingSlot>((second ? R.ring1 : R.ring0) + (uint32_t)(at * sizeof(RingSlot)));
        for (int k = 0; k < 3; ++k) {
          o->x0[k] = x0[k];
          o->v0[k] = v0[k];
        }
        o->gamma = P.gamma; o->g1 = P.g1; o->g2 = P.g2; o->g3 = P.g3; o->h1 = P.h1; o->h2 = P.h2;
        o->r0 = P.r0; o->r = P.r; o->r0inv = P.r0inv; o->rinv = P.rinv;
        o->beta = P.beta; o->betainv = P.betainv; o->eta = P.eta; o->sqb = P.sqb;
        o->mijinv = mijinv;
        o->i = i; o->j = j;
      }
    }
    q0 += w;
    made += w;
    pos += w;
    if (pos >= slots) pos -= slots;
    w = uni(w1);
    second = lane >= w;
    q = lane - (second ? w : 0);
    on = lane < 2 * w && (second ? a1 : a0);
    if (on) ij = pl[2 * (q0 + q)] | ((uint32_t)pl[2 * (q0 + q) + 1] << 8);
    wsync();
    if (keep) publish(&ctl->tail, made, lane);
  }
  return true;
}

// Lexicographic pair index of (i, j), i < j, and back, without branches.
template <int NB> __device__ __forceinline__ int pair_index(int i, int j) { return i * (2 * NB - i - 1) / 2 + (j - i - 1); }
template <int NB> __device__ __forceinline__ void pair_at(int p, int& i, int& j) {
  int r = 0, start = 0;
#pragma unroll
  for (int b = 1; b < NB - 1; ++b) {
    const int first = b * (2 * NB - b - 1) / 2;
    const bool past = p >= first;
    r += past ? 1 : 0;
    start = past ? first : start;
  }
  i = r;
  j = r + 1 + (p - start);
}

// phisalpha! (ahl21.jl:558-700, alpha = 2) on the state alone: one lane per
// pair for the factors, one per body and coordinate for the accelerations and
// velocities, whose sums run over the partners in increasing order like the
// reference's pair loop.  STEP lanes.
template <int NB, int STEP> __device__ __attribute__((always_inline)) inline void phi_state(StateRec<NB>& S, double h, int col) {
  constexpr int N3 = 3 * NB, NP = StateRec<NB>::NP, PP = (NP + STEP - 1) / STEP, EE = (N3 + STEP - 1) / STEP;
  const double coeff = (((2.0 * (h * h * h)) / 96.0) * 2.0) * NBG_GNEWT;
  double r2s[PP], r1s[PP];
#pragma unroll
  for (int u = 0; u < PP; ++u) {
    const int p = col + u * STEP;
    if (p >= NP) continue;
    int i, j;
    pair_at<NB>(p, i, j);
    double rij[3];
    for (int k = 0; k < 3; ++k) rij[k] = S.x[3 * i + k] - S.x[3 * j + k];
    r2s[u] = dot3(rij);
    r1s[u] = __builtin_sqrt(r2s[u]);
    const double fac2 = NBG_GNEWT / (r2s[u] * r1s[u]);
    for (int k = 0; k < 3; ++k) S.fac[3 * p + k] = fac2 * rij[k];
  }
  wsync();
#pragma unroll
  for (int u = 0; u < EE; ++u) {
    const int e = col + u * STEP;
    if (e >= N3) continue;
    const int b = e / 3, k = e - 3 * b;
    double ab = 0.0;
#pragma unroll
    for (int q = 0; q < NB - 1; ++q) {
      const bool bi = q >= b;  // the partner c comes after b
      const int c = bi ? q + 1 : q;
      const double mf = S.m[c] * S.fac[3 * (bi ? pair_index<NB>(b, c) : pair_index<NB>(c, b)) + k];
      ab += bi ? -mf : mf;
    }
    S.a[e] = ab;
  }
  wsync();
#pragma unroll
  for (int u = 0; u < PP; ++u) {
    const int p = col + u * STEP;
    if (p >= NP) continue;
    int i, j;
    pair_at<NB>(p, i, j);
    double rij[3], aij[3];
    for (int k = 0; k < 3; ++k) {
      aij[k] = S.a[3 * i + k] - S.a[3 * j + k];
      rij[k] = S.x[3 * i + k] - S.x[3 * j + k];
    }
    const double r2 = r2s[u], r1 = r1s[u];
    const double ardot = dot3(aij, rij);
    const double fac1 = coeff / ((r2 * r2) * r1);
    const double fac2 = ((2.0 * NBG_GNEWT) * (S.m[i] + S.m[j])) / r1 + 3.0 * ardot;
    for (int k = 0; k < 3; ++k) S.fac[3 * p + k] = fac1 * (rij[k] * fac2 - r2 * aij[k]);
  }
  wsync();
#pragma unroll
  for (int u = 0; u < EE; ++u) {
    const int e = col + u * STEP;
    if (e >= N3) continue;
    const int b = e / 3, k = e - 3 * b;
    double vb = S.v[e], veb = S.ve[e];
#pragma unroll
    for (int q = 0; q < NB - 1; ++q) {
      const bool bi = q >= b;
      const int c = bi ? q + 1 : q;
      const double mf = S.m[c] * S.fac[3 * (bi ? pair_index<NB>(b, c) : pair_index<NB>(c, b)) + k];
      kahan(vb, veb, bi ? mf : -mf);
    }
    S.v[e] = vb;
    S.ve[e] = veb;
  }
  wsync();
}

template <int NB> __device__ inline void split_save_prior(StateRec<NB>& S, int lane) {
  for (int q = lane; q < 3 * NB; q += WAVE) {
    S.px[q] = S.x[q]; S.pv[q] = S.v[q]; S.pxe[q] = S.xe[q]; S.pve[q] = S.ve[q];
  }
  if (lane == 0) S.pt = S.t;
  wsync();
}
template <int NB> __device__ inline void split_restore_prior(StateRec<NB>& S, int lane) {
  for (int q = lane; q < 3 * NB; q += WAVE) {
    S.x[q] = S.px[q]; S.v[q] = S.pv[q]; S.xe[q] = S.pxe[q]; S.ve[q] = S.pve[q];
  }
  if (lane == 0) S.t = S.pt;
  wsync();
}

// detect_transits! from body c.body on (cursor_detect).
template <int NB> __device__ void split_detect(StateRec<NB>& S, const SysDesc& D, RunCursor& c, int lane) {
  const int ti = D.ti;
  int act = c.is < c.iend ? ACT_MAIN : ACT_DONE;
  int body = NB;
#pragma unroll 1
  for (int i = c.body; i < NB; ++i) {
    if (i == ti) continue;
    const double gi = gsky<NB>(S, i, ti);
    const double ri = __builtin_sqrt((S.x[3 * i] * S.x[3 * i] + S.x[3 * i + 1] * S.x[3 * i + 1]) + S.x[3 * i + 2] * S.x[3 * i + 2]);
    if (gi > 0.0 && S.gsave[i] < 0.0 && -S.x[3 * i + 2] > 0.25 * ri && ri < 1e12) {
      const int64_t cnt = S.count[i] + 1;
      wsync();
      if (lane == 0) S.count[i] = cnt;
      wsync();
      if (cnt >= 1 && cnt <= D.ntt) {
        if (!c.saved) {
          split_save_prior<NB>(S, lane);
          c.saved = 1;
        }
        c.dt0 = ((-gi) * D.hstep) / (gi - S.gsave[i]);
        c.gi = gi;
        c.jb = i;
        c.iter = 0;
        c.stmp = 0.0;
        c.tt1 = c.dt0 + 1.0;
        c.tt2 = c.dt0 + 2.0;
        act = ACT_NEWTON;
        body = i;  // gsave[i] is written when the search ends
        break;
      }
    }
    wsync();
    if (lane == 0) S.gsave[i] = gi;
    wsync();
  }
  c.act = __builtin_amdgcn_readfirstlane(act);
  c.body = __builtin_amdgcn_readfirstlane(body);
}

// The step of the cursor's next action (cursor_prepare): its size, and what
// it needs of the Jacobian wave (SPLIT_*).
template <int NB> __device__ void split_prepare(StateRec<NB>& S, const SysDesc& D, RunCursor& c, double& h, int& need, int lane) {
  const bool grad = D.grad != 0;
  if (c.act == ACT_MAIN) {
    const bool land = c.is == D.nsteps;  // MODE_STEPS: the extra step onto the time
    const bool last = c.is + 1 == D.nsteps + (D.mode == MODE_STEPS && D.hlast != 0.0 ? 1 : 0);
    h = land ? D.hlast : D.h;
    need = ACT_MAIN | (grad ? SPLIT_J : 0) | (grad && last ? SPLIT_Q : 0);
    return;
  }
  split_restore_prior<NB>(S, lane);
  h = c.dt0;
  need = c.act | SPLIT_Q;
  if (c.act == ACT_NEWTON) {
    c.tt2 = c.tt1;
    c.tt1 = c.dt0;
    return;
  }
  need |= SPLIT_J | SPLIT_SAVE;
}

// A found transit's time (and sky velocity, impact parameter) and counters.
template <int NB> __device__ void split_record(StateRec<NB>& S, const SysDesc& D, const SysBufs& B, const RunCursor& c, int lane) {
  const int n = NB, ti = D.ti, jb = c.jb, nb = D.ntbv;
  const int64_t cc = S.count[jb] - 1;
  if (lane == 0) {
    double* tt = B.tt + D.off_tt + nb * (jb + n * cc);
    tt[0] = S.t + c.dt0;
    if (nb == 3) {
      const double dx = S.x[3 * jb] - S.x[3 * ti], dy = S.x[3 * jb + 1] - S.x[3 * ti + 1];
      const double dvx = S.v[3 * jb] - S.v[3 * ti], dvy = S.v[3 * jb + 1] - S.v[3 * ti + 1];
      tt[1] = __builtin_sqrt(dvx * dvx + dvy * dvy);
      tt[2] = dx * dx + dy * dy;
    }
    int64_t* ints = B.ints + D.off_int;
    ints[NB + 1] += 1;
    ints[NB + 2] += c.iter;
  }
}

// After the cursor's step (cursor_finish).  J: the Jacobian wave's record,
// whose dq/dt is complete for a Newton step.
template <int NB, class R>
__device__ void split_finish(StateRec<NB>& S, R& J, const SysDesc& D, const SysBufs& B, RunCursor& c, int lane) {
  if (c.act == ACT_MAIN) {
    if (D.mode == MODE_TRANSITS && lane == 0) S.t = D.t0 + ((double)(c.is + 1) * D.h);
    wsync();
    c.is += 1;
    c.saved = 0;
    c.body = 0;
    if (D.mode == MODE_TRANSITS) split_detect<NB>(S, D, c, lane);
    else c.act = c.is < c.iend ? ACT_MAIN : ACT_DONE;
    return;
  }
  if (c.act == ACT_NEWTON) {
    const double gs = gsky<NB>(S, D.ti, c.jb);
    // gdot with this record's x and v and the other's dq/dt
    const int i = D.ti, j = c.jb;
    const double* q = J.dqdt;
    const double gd = (((S.x[3 * j] - S.x[3 * i]) * (q[7 * j + 3] - q[7 * i + 3]) +
                        (S.x[3 * j + 1] - S.x[3 * i + 1]) * (q[7 * j + 4] - q[7 * i + 4])) +
                       (S.v[3 * j] - S.v[3 * i]) * (q[7 * j + 0] - q[7 * i + 0])) +
                      (S.v[3 * j + 1] - S.v[3 * i + 1]) * (q[7 * j + 1] - q[7 * i + 1]);
    const double dt = -gs / gd;
    kahan(c.dt0, c.stmp, dt);
    c.iter += 1;
    if (!(c.iter >= 20 || c.dt0 == c.tt1 || c.dt0 == c.tt2)) return;  // another iteration
    if (D.grad) {
      c.act = ACT_JSTEP;
      return;
    }
  }
  split_record<NB>(S, D, B, c, lane);
  split_restore_prior<NB>(S, lane);
  wsync();
  if (lane == 0) S.gsave[c.jb] = c.gi;
  wsync();
  c.body = c.jb + 1;
  split_detect<NB>(S, D, c, lane);
}

template <int NB> __device__ void split_load_state(StateRec<NB>& S, const SysDesc& D, const SysBufs& B, int lane) {
  const double* st = B.state + D.off_state;
  for (int q = lane; q < 3 * NB; q += WAVE) {
    S.x[q] = st[off_x(NB) + q];
    S.v[q] = st[off_v(NB) + q];
    S.xe[q] = st[off_xe(NB) + q];
    S.ve[q] = st[off_ve(NB) + q];
  }
  for (int q = lane; q < NB; q += WAVE) {
    S.m[q] = st[off_m(NB) + q];
    S.gsave[q] = st[off_gsave(NB) + q];
    S.count[q] = B.ints[D.off_int + q];
  }
  if (lane == 0) S.t = st[off_t(NB)];
  wsync();
  // gsave[i] = g!(i, ti, x, v) before the loop (Transits.jl:146-149)
  if (D.mode == MODE_TRANSITS && B.ints[D.off_int + NB] == 0) {
    if (lane == 0)
      for (int i = 0; i < NB; ++i)
        if (i != D.ti) S.gsave[i] = gsky<NB>(S, i, D.ti);
    wsync();
  }
}
template <int NB> __device__ void split_store_state(StateRec<NB>& S, const SysDesc& D, const SysBufs& B, int64_t istep, int lane) {
  wsync();
  double* st = B.state + D.off_state;
  for (int q = lane; q < 3 * NB; q += WAVE) {
    st[off_x(NB) + q] = S.x[q];
    st[off_v(NB) + q] = S.v[q];
    st[off_xe(NB) + q] = S.xe[q];
    st[off_ve(NB) + q] = S.ve[q];
  }
  for (int q = lane; q < NB; q += WAVE) {
    st[off_gsave(NB) + q] = S.gsave[q];
    B.ints[D.off_int + q] = S.count[q];
  }
  if (lane == 0) {
    st[off_t(NB)] = S.t;
    B.ints[D.off_int + NB] = istep;
  }
}

// The visit of a system: steps [begin, end) of its run (MODE_STEPS counts the
// step onto the time as one more); begin > the run's steps: finished earlier.
struct Visit {
  int64_t begin, end, total;
};
__device__ inline Visit visit_of(const SysDesc& D, const SysBufs& B, int64_t chunk) {
  Visit v;
  v.begin = B.ints[D.off_int + D.n];
  v.total = D.nsteps + (D.mode == MODE_STEPS && D.hlast != 0.0 ? 1 : 0);
  v.end = v.begin > D.nsteps ? v.begin : (chunk > 0 && v.begin + chunk < D.nsteps) ? v.begin + chunk : v.total;
  return v;
}

template <int NB, bool G, bool TWO, int LIMIT>
__device__ void split_state(SplitLds<NB, G, TWO, LIMIT>& P, const SysDesc& D0, const SysDesc& D1, const SysBufs& B,
                            const Visit& v0, const Visit& v1, int lane, int64_t bound, unsigned long long* err) {
  using L = SplitLds<NB, G, TWO, LIMIT>;
  constexpr int N3 = 3 * NB, NP = L::NP, K = TWO ? 1 : 0;
  constexpr int STEP = TWO && N3 <= 32 ? 32 : WAVE;
  SplitCtl* ctl = &P.ctl;
  RunCursor c[2];
  const Visit* vs[2] = {&v0, &v1};
  for (int k = 0; k < 2; ++k) {
    const Visit& v = *vs[k];
    const bool any = (k == 0 || TWO) && v.begin < v.end;
    c[k].is = v.begin; c[k].iend = v.end; c[k].act = any ? ACT_MAIN : ACT_DONE; c[k].body = NB; c[k].saved = 0;
  }
  SplitSweep R;
  R.x0 = lds_off(P.t[0].x); R.x1 = lds_off(P.t[K].x);
  R.ring0 = lds_off(P.ring[0]); R.ring1 = lds_off(P.ring[K]);
  R.ctl = lds_off(ctl);
  R.n3 = N3; R.levels = Schedule<NB>::NL; R.slots = L::RR;
  R.pos = 0; R.made = 0;
  R.bound = bound; R.err = err;
  int sent = 0, asked = 0;
  const int half = STEP == 32 ? lane >> 5 : 0, col = STEP == 32 ? lane & 31 : lane;
#pragma unroll 1
  while (c[0].act != ACT_DONE || c[1].act != ACT_DONE) {
    const bool a0 = c[0].act != ACT_DONE, a1 = TWO && c[1].act != ACT_DONE;
    double h0 = 0.0, h1 = 0.0;
    int n0 = ACT_DONE, n1 = ACT_DONE;
    if (a0) split_prepare<NB>(P.t[0], D0, c[0], h0, n0, lane);
    if (a1) split_prepare<NB>(P.t[K], D1, c[1], h1, n1, lane);
    const bool keep = ((n0 | n1) & (SPLIT_J | SPLIT_Q)) != 0;
    if (keep) {
      // PRE; its buffers are free once the message three before it is copied
      if (!wait_for(&ctl->seen, sent - 2, ctl, bound, err, lane)) return;
      for (int q = lane; q < N3; q += WAVE) {
        if (n0 & SPLIT_Q) P.j[0].mv[q] = P.t[0].v[q];
        if (n1 & SPLIT_Q) P.j[K].mv[q] = P.t[K].v[q];
      }
      if (lane == 0) {
        ctl->act[0] = n0; ctl->h[0] = h0; ctl->body[0] = c[0].jb; ctl->index[0] = n0 & SPLIT_SAVE ? P.t[0].count[c[0].jb] - 1 : 0;
        ctl->act[1] = n1; ctl->h[1] = h1; ctl->body[1] = c[1].jb; ctl->index[1] = n1 & SPLIT_SAVE ? P.t[K].count[c[1].jb] - 1 : 0;
      }
      wsync();
      publish(&ctl->sent, ++sent, lane);
    }
    R.act0 = a0; R.act1 = a1; R.keep = keep;
    R.hh0 = 0.5 * h0; R.hh1 = 0.5 * h1;
    const bool mine = STEP == 32 ? (half ? a1 : a0) : true;
    auto drift = [&]() {
      if constexpr (STEP == 32) {
        if (mine) drift_state<NB, 32>(half ? P.t[K] : P.t[0], 0.5 * (half ? h1 : h0), col);
      } else {
        if (a0) drift_state<NB, WAVE>(P.t[0], 0.5 * h0, lane);
        if (a1) drift_state<NB, WAVE>(P.t[K], 0.5 * h1, lane);
      }
      wsync();
    };
    drift();
    R.pairs = lds_off(P.sched.pairs[0]); R.width = lds_off(P.sched.width[0]);
    if (!split_levels<true>(R)) return;
    if (keep) {
      R.made += NP; R.pos = (R.pos + NP) % L::RR;
      if (!wait_for(&ctl->seen, sent - 2, ctl, bound, err, lane)) return;
      for (int q = lane; q < N3; q += WAVE) {
        if (a0) P.j[0].mx[q] = P.t[0].x[q];
        if (a1) P.j[K].mx[q] = P.t[K].x[q];
      }
      wsync();
      publish(&ctl->sent, ++sent, lane);
    }
    if constexpr (STEP == 32) {
      if (mine) phi_state<NB, 32>(half ? P.t[K] : P.t[0], half ? h1 : h0, col);
    } else {
      if (a0) phi_state<NB, WAVE>(P.t[0], h0, lane);
      if (a1) phi_state<NB, WAVE>(P.t[K], h1, lane);
    }
    wsync();
    R.pairs = lds_off(P.sched.pairs[1]); R.width = lds_off(P.sched.width[1]);
    if (!split_levels<false>(R)) return;
    drift();
    if (keep) {
      R.made += NP; R.pos = (R.pos + NP) % L::RR;
      if (!wait_for(&ctl->seen, sent - 2, ctl, bound, err, lane)) return;
      for (int q = lane; q < N3; q += WAVE) {
        if (n0 & SPLIT_Q) { P.j[0].qx[q] = P.t[0].x[q]; P.j[0].qv[q] = P.t[0].v[q]; }
        if (n1 & SPLIT_Q) { P.j[K].qx[q] = P.t[K].x[q]; P.j[K].qv[q] = P.t[K].v[q]; }
      }
      wsync();
      publish(&ctl->sent, ++sent, lane);
      ++asked;
    }
    if ((a0 && c[0].act == ACT_NEWTON) || (a1 && c[1].act == ACT_NEWTON))
      if (!wait_for(&ctl->answered, asked, ctl, bound, err, lane)) return;
    if (a0) split_finish<NB>(P.t[0], P.j[0], D0, B, c[0], lane);
    if (a1) split_finish<NB>(P.t[K], P.j[K], D1, B, c[1], lane);
  }
  for (int k = 0; k < L::NS; ++k) {
    const Visit& v = *vs[k];
    const SysDesc& D = k ? D1 : D0;
    if (v.begin <= D.nsteps) split_store_state<NB>(P.t[k], D, B, v.end == v.total ? D.nsteps + 1 : v.end, lane);
  }
  // quit: the Jacobian wave finishes what it was sent and ends (a run that
  // never needs it has it at the barrier already)
  if (!wait_for(&ctl->seen, sent - 2, ctl, bound, err, lane)) return;
  if (lane == 0) ctl->act[0] = -1;
  wsync();
  publish(&ctl->sent, ++sent, lane);
}

// ---------------------------------------------------------------------------
// Jacobian wave
// ---------------------------------------------------------------------------
// One pair's Jacobian (pair_jacobian) from its ring slot: the drift's other
// quantities by the formulas of jac_delxv_gamma!.
template <bool DF>
static __device__ __attribute__((noinline)) void split_pair_jacobian(uint32_t ring, uint32_t slot, double m_i, double m_j, double h) {
  const RingSlot* a = lds_at<RingSlot>(ring);
  JacSlot* o = lds_at<JacSlot>(slot);
  KParams P;
  double x0[3], v0[3], kep[48], jm[6], dl[6];
  for (int k = 0; k < 3; ++k) {
    x0[k] = a->x0[k];
    v0[k] = a->v0[k];
  }
  P.gamma = a->gamma; P.g1 = a->g1; P.g2 = a->g2; P.g3 = a->g3; P.h1 = a->h1; P.h2 = a->h2;
  P.r0 = a->r0; P.r = a->r; P.r0inv = a->r0inv; P.rinv = a->rinv;
  P.beta = a->beta; P.betainv = a->betainv; P.eta = a->eta; P.sqb = a->sqb;
  const double mijinv = a->mijinv, mi = m_i * mijinv, mj = m_j * mijinv;
  const double k = NBG_GNEWT * (m_i + m_j);
  P.k = k;
  P.h = h;
  P.iters = 0;
  P.zeta = k - P.r0 * P.beta;
  P.g0 = 1.0 - P.beta * P.g2;
  P.dfdt = (((-k) * P.g1) * P.rinv) * P.r0inv;
  if (DF) {
    P.fm1 = ((-k) * P.r0inv) * P.g2;
    P.gmh = (k * P.r0inv) * (h * P.g2 - P.r0 * P.g3);
    P.dgdtm1 = ((k * P.r0inv) * P.rinv) * (h * P.g1 - P.r0 * P.g2);
  } else {
    P.fm1 = (k * P.rinv) * (P.g2 - (k * P.r0inv) * P.h1);
    P.gmh = (k * P.rinv) * (P.r0 * P.h2 + P.eta * P.h1);
    P.dgdtm1 = ((-k) * P.rinv) * P.g2;
  }
  for (int q = 0; q < 3; ++q) {
    dl[q] = P.fm1 * x0[q] + P.gmh * v0[q];
    dl[3 + q] = P.dfdt * x0[q] + P.dgdtm1 * v0[q];
  }
  for (int q = 0; q < 48; ++q) kep[q] = 0.0;
  for (int q = 0; q < 6; ++q) jm[q] = 0.0;
  compute_jacobian_gamma(P, x0, v0, kep, jm, DF);
  for (int rk = 0; rk < 6; ++rk) {
    o->mc[rk] = jm[rk] * m_j;
    o->mc[6 + rk] = (((-mj) * dl[rk]) * mijinv) - ((NBG_GNEWT * mi) * kep[rk + 36]);
    o->mc[12 + rk] = ((mi * dl[rk]) * mijinv) + ((NBG_GNEWT * mj) * kep[rk + 36]);
    o->mc[18 + rk] = (-jm[rk]) * m_i;
  }
  for (int q = 0; q < 48; ++q) o->kep[q] = kep[q];
  o->mi = mi; o->mj = mj;
  o->i = a->i; o->j = a->j;
}

// jij_coef from a JacSlot (the mass columns as pair_cols takes them).
__device__ inline double split_coef(const JacSlot& sl, bool rowi, int rk, int k) {
  if (k == 6) return sl.mc[(rowi ? 0 : 6) + rk];
  if (k == 13) return sl.mc[(rowi ? 12 : 18) + rk];
  const double kv = sl.kep[rk + 6 * (k < 7 ? k : k - 7)];
  if (rowi == (k < 7)) return 0.0 + (rowi ? sl.mj : sl.mi) * kv;
  return 0.0 - (rowi ? sl.mj : sl.mi) * kv;
}

// Phase C of a chunk (sweep_rows).
template <int NB, bool G, int STEP, bool FACT, class R>
__device__ __attribute__((always_inline)) inline void split_rows(R& S, const JacSlot* slots, int cnt, bool needJ, bool needQ, int col) {
#pragma unroll 1
  for (int q = 0; q < cnt; ++q) {
    const JacSlot& sl = slots[q];
    const int i = sl.i, j = sl.j;
    if (needJ)
      for (int c = col; c < 7 * NB; c += STEP) pair_cols<NB, G, FACT>(S, sl, i, j, c);
    if (needQ) {
      // dqdt_ij (ahl21.jl:743-748) and dq/dt's rows
      if (col < 14) {
        const bool rowi = col < 7;
        const int rk = rowi ? col : col - 7;
        double q1[14];
        for (int k = 0; k < 7; ++k) {
          q1[k] = S.dqdt[7 * i + k];
          q1[7 + k] = S.dqdt[7 * j + k];
        }
        double s2 = 0.0, dq = S.dqij[col];
        const double mine = S.dqdt[rowi ? 7 * i + rk : 7 * j + rk];
        if (rk < 6) {
          dq = (rowi ? sl.mj : -sl.mi) * sl.kep[rk + 42];
          for (int k = 0; k < 14; ++k) s2 = fmad(split_coef(sl, rowi, rk, k), q1[k], s2);
        } else {
          for (int k = 0; k < 14; ++k) s2 = fmad(0.0, q1[k], s2);
        }
        const double nd = (dq * 0.5) + (mine + s2);
        S.dqij[col] = nd;
        S.dqdt[rowi ? 7 * i + rk : 7 * j + rk] = nd;
      }
    }
    wsync();
  }
}

template <int NB, bool G, bool TWO, int LIMIT> struct SplitFollow {
  int head, pos;
  int64_t bound;
  unsigned long long* err;
};

// A sweep on the Jacobian wave: chunks of whole levels as the ring delivers
// them -- the pair Jacobians of both systems at once, then each system's rows.
template <int NB, bool G, bool TWO, int LIMIT, bool FACT>
__device__ __attribute__((always_inline)) inline bool split_sweep(SplitLds<NB, G, TWO, LIMIT>& P,
                                                                  SplitFollow<NB, G, TWO, LIMIT>& F, int dir, double hh0,
                                                                  double hh1, int n0, int n1, int lane) {
  using L = SplitLds<NB, G, TWO, LIMIT>;
  constexpr int K = TWO ? 1 : 0, NL = Schedule<NB>::NL;
  const uint8_t* lw = P.sched.width[dir];
  const bool p0 = (n0 & (SPLIT_J | SPLIT_Q)) != 0, p1 = TWO && (n1 & (SPLIT_J | SPLIT_Q)) != 0;
  JacSlot* s0 = P.w[0].slot;
  JacSlot* s1 = L::PHI2 ? P.w[L::NW - 1].slot : P.w[0].slot + L::CH;
  int lev = 0;
  while (lev < NL) {
    int cnt = 0;
    while (lev < NL && cnt + lw[lev] <= L::CH) cnt += lw[lev++];
    if (!wait_for(&P.ctl.tail, F.head + cnt, &P.ctl, F.bound, F.err, lane)) return false;
    if (lane < (TWO ? 2 : 1) * cnt) {
      const bool second = lane >= cnt;
      const int q = lane - (second ? cnt : 0);
      if (second ? p1 : p0) {
        int at = F.pos + q;
        if (at >= L::RR) at -= L::RR;
        const RingSlot* a = &P.ring[second ? K : 0][at];
        const double* m = second ? P.j[K].m : P.j[0].m;
        JacSlot* o = (second ? s1 : s0) + q;
        const double hh = second ? hh1 : hh0;
        if (dir == 0) split_pair_jacobian<true>(lds_off(a), lds_off(o), m[a->i], m[a->j], hh);
        else split_pair_jacobian<false>(lds_off(a), lds_off(o), m[a->i], m[a->j], hh);
      }
    }
    wsync();
    F.head += cnt;
    F.pos += cnt;
    if (F.pos >= L::RR) F.pos -= L::RR;
    publish(&P.ctl.head, F.head, lane);
    if constexpr (L::HALF) {
      const bool sys = lane >= 32;
      if (sys ? p1 : p0)
        split_rows<NB, G, 32, FACT>(sys ? P.j[K] : P.j[0], sys ? s1 : s0, cnt, ((sys ? n1 : n0) & SPLIT_J) != 0,
                                    ((sys ? n1 : n0) & SPLIT_Q) != 0, lane & 31);
      wsync();
    } else {
      if (p0) split_rows<NB, G, WAVE, FACT>(P.j[0], s0, cnt, (n0 & SPLIT_J) != 0, (n0 & SPLIT_Q) != 0, lane);
      if (p1) split_rows<NB, G, WAVE, FACT>(P.j[K], s1, cnt, (n1 & SPLIT_J) != 0, (n1 & SPLIT_Q) != 0, lane);
    }
  }
  return true;
}

// The Jacobian kept for (or back from) a transit's gradient step.
template <int NB, class R> __device__ void split_keep_jac(R& S, double* ws, bool back, int lane) {
  const auto J_ = jj<NB>(S);
  constexpr int N6 = 6 * NB, N7 = 7 * NB;
  for (int col = lane; col < N7; col += WAVE)
#pragma unroll 4
    for (int r = 0; r < 2 * N6; ++r) {
      if (back) J_[(unsigned)(r * N7 + col)] = ws[r * N7 + col];
      else ws[r * N7 + col] = J_[(unsigned)(r * N7 + col)];
    }
}

// The dt/dq rows of a transit (cursor_record), from the final state of its
// gradient step in the record.
template <int NB, class R>
__device__ void split_gradient(R& S, const SysDesc& D, const SysBufs& B, int jb, int64_t cc, int lane) {
  constexpr int N7 = 7 * NB;
  const int n = NB, ti = D.ti, nb = D.ntbv;
  const auto J_ = jj<NB>(S);
  const double gd = gdot<NB>(S, ti, jb);
  const double dx = S.x[3 * jb] - S.x[3 * ti], dy = S.x[3 * jb + 1] - S.x[3 * ti + 1];
  const double dvx = S.v[3 * jb] - S.v[3 * ti], dvy = S.v[3 * jb + 1] - S.v[3 * ti + 1];
  double* dq = B.dq + D.off_dq;
  const int64_t ntt = D.ntt;
  for (int col = lane; col < N7; col += WAVE) {
    const int rj = 6 * jb, ri = 6 * ti;
    auto dJ = [&](int k) { return J_[(unsigned)((rj + k) * N7 + col)] - J_[(unsigned)((ri + k) * N7 + col)]; };
    const double jx = dJ(0), jy = dJ(1), jvx = dJ(3), jvy = dJ(4);
    const double d0 = -(((jx * dvx + jy * dvy) + jvx * dx) + jvy * dy) / gd;
    const int64_t base = (int64_t)jb + n * (cc + ntt * (int64_t)col);
    dq[0 + nb * base] = d0;
    if (nb == 3) {
      const double vsky = __builtin_sqrt(dvx * dvx + dvy * dvy);
      const double dvdt = (dvx * (S.dqdt[7 * jb + 3] - S.dqdt[7 * ti + 3]) +
                           dvy * (S.dqdt[7 * jb + 4] - S.dqdt[7 * ti + 4])) / vsky;
      dq[1 + nb * base] = (jvx * dvx + jvy * dvy) / vsky + dvdt * d0;
      dq[2 + nb * base] = 2.0 * (jx * dx + jy * dy);
    }
  }
}

template <int NB, bool G> __device__ void split_load_jac(JacRec<NB, G>& S, const SysDesc& D, const SysBufs& B, int lane) {
  constexpr int N7 = 7 * NB;
  if constexpr (G) {
    if (lane == 0) S.jg = B.ws + D.off_ws + 2 * (int64_t)(6 * NB) * N7;  // after the transit-step copy
    wsync();
  }
  const double* st = B.state + D.off_state;
  for (int q = lane; q < NB; q += WAVE) S.m[q] = st[off_m(NB) + q];
  for (int q = lane; q < N7; q += WAVE) S.run_dqdt[q] = st[off_dqdt(NB) + q];
  if (D.grad) {
    const auto J_ = jj<NB>(S);
    const double* J = B.jac + D.off_jac;
    const double* JE = J + (int64_t)N7 * N7;
    for (int c = lane; c < N7; c += WAVE)
      for (int b = 0; b < NB; ++b)
        for (int k = 0; k < 6; ++k) {
          J_[(unsigned)((6 * b + k) * N7 + c)] = J[(7 * b + k) + (int64_t)N7 * c];
          J_[(unsigned)(JacRec<NB, G>::JOFF + (6 * b + k) * N7 + c)] = JE[(7 * b + k) + (int64_t)N7 * c];
        }
  }
  wsync();
}
template <int NB, bool G> __device__ void split_store_jac(JacRec<NB, G>& S, const SysDesc& D, const SysBufs& B, int lane) {
  constexpr int N7 = 7 * NB;
  double* st = B.state + D.off_state;
  for (int q = lane; q < N7; q += WAVE) st[off_dqdt(NB) + q] = S.run_dqdt[q];
  if (D.grad) {
    const auto J_ = jj<NB>(S);
    double* J = B.jac + D.off_jac;
    double* JE = J + (int64_t)N7 * N7;
    for (int c = lane; c < N7; c += WAVE)
      for (int b = 0; b < NB; ++b)
        for (int k = 0; k < 6; ++k) {
          J[(7 * b + k) + (int64_t)N7 * c] = J_[(unsigned)((6 * b + k) * N7 + c)];
          JE[(7 * b + k) + (int64_t)N7 * c] = J_[(unsigned)(JacRec<NB, G>::JOFF + (6 * b + k) * N7 + c)];
        }
  }
  wsync();
}

template <int NB, bool G, bool TWO, int LIMIT, bool FACT>
__device__ void split_jacobian(SplitLds<NB, G, TWO, LIMIT>& P, const SysDesc& D0, const SysDesc& D1, const SysBufs& B,
                               const Visit& v0, const Visit& v1, int lane, int64_t bound, int64_t bound_job,
                               unsigned long long* err) {
  using L = SplitLds<NB, G, TWO, LIMIT>;
  constexpr int N3 = 3 * NB, N7 = 7 * NB, K = TWO ? 1 : 0;
  constexpr int STEP = L::HALF ? 32 : WAVE;
  SplitCtl* ctl = &P.ctl;
  SplitFollow<NB, G, TWO, LIMIT> F{0, 0, bound, err};
  JacRec<NB, G>& J0 = P.j[0];
  JacRec<NB, G>& J1 = P.j[K];
  JacWork<NB>& W0 = P.w[0];
  JacWork<NB>& W1 = P.w[L::NW - 1];
  const bool sys = L::HALF && lane >= 32;
  const int col = L::HALF ? lane & 31 : lane;
  int seen = 0, answered = 0;
#pragma unroll 1
  while (true) {
    if (!wait_for(&ctl->sent, seen + 1, ctl, bound_job, err, lane)) return;
    const int n0 = __builtin_amdgcn_readfirstlane(ctl->act[0]);
    if (n0 < 0) break;
    const int n1 = TWO ? __builtin_amdgcn_readfirstlane(ctl->act[1]) : (int)ACT_DONE;
    const double h0 = ctl->h[0], h1 = ctl->h[1];
    const int b0 = ctl->body[0], b1 = ctl->body[1];
    const int64_t i0 = ctl->index[0], i1 = ctl->index[1];
    const bool j0 = (n0 & SPLIT_J) != 0, q0 = (n0 & SPLIT_Q) != 0, j1 = (n1 & SPLIT_J) != 0, q1 = (n1 & SPLIT_Q) != 0;
    for (int q = lane; q < N3; q += WAVE) {
      if (q0) J0.v[q] = J0.mv[q];
      if (q1) J1.v[q] = J1.mv[q];
    }
    wsync();
    publish(&ctl->seen, ++seen, lane);
    if (n0 & SPLIT_SAVE) split_keep_jac<NB>(J0, B.ws + D0.off_ws, false, lane);
    if (n1 & SPLIT_SAVE) split_keep_jac<NB>(J1, B.ws + D1.off_ws, false, lane);
    if constexpr (L::HALF) {
      step_pre<NB, G, 32, FACT, false>(sys ? J1 : J0, W0, sys ? h1 : h0, sys ? j1 : j0, sys ? q1 : q0, false, col);
    } else {
      step_pre<NB, G, STEP, FACT, false>(J0, W0, h0, j0, q0, false, lane);
      if constexpr (TWO) step_pre<NB, G, STEP, FACT, false>(J1, W0, h1, j1, q1, false, lane);
    }
    if (!split_sweep<NB, G, TWO, LIMIT, FACT>(P, F, 0, 0.5 * h0, 0.5 * h1, n0, n1, lane)) return;
    if (!wait_for(&ctl->sent, seen + 1, ctl, bound, err, lane)) return;
    for (int q = lane; q < N3; q += WAVE) {
      J0.x[q] = J0.mx[q];
      if (TWO) J1.x[q] = J1.mx[q];
    }
    wsync();
    publish(&ctl->seen, ++seen, lane);
    if constexpr (L::PHI2) {
      {
        const bool hi = lane >= 32;
        if (hi ? (j1 || q1) : (j0 || q0))
          phisalpha_cols<NB, G, 32, FACT, false>(hi ? J1 : J0, hi ? W1 : W0, hi ? h1 : h0, false, hi ? q1 : q0, lane & 31);
      }
      wsync();
      if constexpr (L::HALF) {
        step_mid_rest<NB, G, 32, FACT>(sys ? J1 : J0, sys ? W1 : W0, sys ? j1 : j0, sys ? q1 : q0, col);
      } else {
        step_mid_rest<NB, G, WAVE, FACT>(J0, W0, j0, q0, lane);
        step_mid_rest<NB, G, WAVE, FACT>(J1, W1, j1, q1, lane);
      }
    } else {
      if (j0 || q0) {
        phisalpha_cols<NB, G, WAVE, FACT, false>(J0, W0, h0, false, q0, lane);
        wsync();
        step_mid_rest<NB, G, WAVE, FACT>(J0, W0, j0, q0, lane);
      }
      if (TWO && (j1 || q1)) {
        phisalpha_cols<NB, G, WAVE, FACT, false>(J1, W0, h1, false, q1, lane);
        wsync();
        step_mid_rest<NB, G, WAVE, FACT>(J1, W0, j1, q1, lane);
      }
    }
    if (!split_sweep<NB, G, TWO, LIMIT, FACT>(P, F, 1, 0.5 * h0, 0.5 * h1, n0, n1, lane)) return;
    if (!wait_for(&ctl->sent, seen + 1, ctl, bound, err, lane)) return;
    for (int q = lane; q < N3; q += WAVE) {
      if (q0) { J0.x[q] = J0.qx[q]; J0.v[q] = J0.qv[q]; }
      if (q1) { J1.x[q] = J1.qx[q]; J1.v[q] = J1.qv[q]; }
    }
    wsync();
    publish(&ctl->seen, ++seen, lane);
    if constexpr (L::HALF) {
      step_post<NB, G, 32, FACT, false>(sys ? J1 : J0, W0, sys ? h1 : h0, sys ? j1 : j0, sys ? q1 : q0, false, col);
    } else {
      step_post<NB, G, STEP, FACT, false>(J0, W0, h0, j0, q0, false, lane);
      if constexpr (TWO) step_post<NB, G, STEP, FACT, false>(J1, W0, h1, j1, q1, false, lane);
    }
    publish(&ctl->answered, ++answered, lane);
    auto end = [&](JacRec<NB, G>& S, const SysDesc& D, int need, int body, int64_t index) {
      if (need & SPLIT_SAVE) {
        split_gradient<NB>(S, D, B, body, index, lane);
        split_keep_jac<NB>(S, B.ws + D.off_ws, true, lane);
      } else if ((need & 3) == ACT_MAIN && (need & SPLIT_Q)) {
        for (int q = lane; q < N7; q += WAVE) S.run_dqdt[q] = S.dqdt[q];
        wsync();
      }
    };
    end(J0, D0, n0, b0, i0);
    if (TWO) end(J1, D1, n1, b1, i1);
  }
  for (int k = 0; k < L::NS; ++k) {
    const SysDesc& D = k ? D1 : D0;
    const Visit& v = k ? v1 : v0;
    if (v.begin > D.nsteps) continue;
    split_store_jac<NB, G>(P.j[k], D, B, lane);
  }
}

// calc_dtdelements! (dtdelements) of a finished system, both waves at work:
// wave w takes the transits w, w + 2, ...; jac_init staged transposed in the
// Jacobian's store (the Jacobian is already stored).
template <int NB, class L> __device__ void split_elements(L& P, int k, const SysDesc& D, const SysBufs& B, int wave, int lane) {
  constexpr int N7 = 7 * NB;
  const int n = NB, nb = D.ntbv;
  const auto jt = jj<NB>(P.j[k]);
  const double* jinit = B.jac + D.off_jac + 2 * (int64_t)N7 * N7;
  for (int col = lane; col < N7; col += WAVE)
    for (int cp = wave; cp < N7; cp += 2) jt[(unsigned)(col + N7 * cp)] = jinit[cp + (int64_t)N7 * col];
  __syncthreads();
  const double* dq = B.dq + D.off_dq;
  double* del = B.del + D.off_del;
  const int64_t ntt = D.ntt;
  int turn = 0;
  for (int b = 0; b < nb; ++b)
    for (int i = 0; i < n; ++i) {
      const int64_t cnt = P.t[k].count[i] < ntt ? P.t[k].count[i] : ntt;
      for (int64_t t = 0; t < cnt; ++t, turn ^= 1) {
        if (turn != wave) continue;
        for (int col = lane; col < N7; col += WAVE) {
          double acc = 0.0;
          for (int cp = 0; cp < N7; ++cp)
            acc = acc + dq[b + nb * ((int64_t)i + n * (t + ntt * cp))] * jt[(unsigned)(col + N7 * cp)];
          del[b + nb * ((int64_t)i + n * (t + ntt * col))] = acc;
        }
      }
    }
}

// One visit of a system, or of two of equal body count, by a workgroup of two
// waves.
template <int NB, bool G, bool TWO, int LIMIT>
__device__ void split_run(unsigned char* raw, int wave, const SysDesc& D0, const SysDesc& D1, const SysBufs& B, int64_t chunk0,
                          int64_t chunk1, bool pair, int64_t bound, int64_t bound_job, unsigned long long* err, int lane) {
  using L = SplitLds<NB, G, TWO, LIMIT>;
  L& P = *reinterpret_cast<L*>(raw);
  const Visit v0 = visit_of(D0, B, chunk0);
  Visit v1 = visit_of(D1, B, chunk1);
  if (!pair) v1.begin = v1.end = v1.total + 1;  // no second system: as one that finished earlier
  if (wave == 0) {
    split_load_state<NB>(P.t[0], D0, B, lane);
    if (TWO) split_load_state<NB>(P.t[L::NS - 1], D1, B, lane);
    for (int w = lane; w < (int)sizeof(SplitCtl) / 4; w += WAVE) reinterpret_cast<int*>(&P.ctl)[w] = 0;
    for (int w = lane; w < (int)sizeof(Schedule<NB>); w += WAVE)
      reinterpret_cast<uint8_t*>(&P.sched)[w] = reinterpret_cast<const uint8_t*>(&kSchedule<NB>)[w];
  } else {
    split_load_jac<NB, G>(P.j[0], D0, B, lane);
    if (TWO) split_load_jac<NB, G>(P.j[L::NS - 1], D1, B, lane);
  }
  __syncthreads();
  if (wave == 0) {
    split_state<NB, G, TWO, LIMIT>(P, D0, D1, B, v0, v1, lane, bound, err);
  } else if (D0.grad || D0.mode == MODE_TRANSITS || (pair && (D1.grad || D1.mode == MODE_TRANSITS))) {
    if (D0.rowupd) split_jacobian<NB, G, TWO, LIMIT, true>(P, D0, D1, B, v0, v1, lane, bound, bound_job, err);
    else split_jacobian<NB, G, TWO, LIMIT, false>(P, D0, D1, B, v0, v1, lane, bound, bound_job, err);
  }
  __syncthreads();  // every row is written
  if (D0.mode == MODE_TRANSITS && D0.grad && v0.begin <= D0.nsteps && v0.end == v0.total)
    split_elements<NB>(P, 0, D0, B, wave, lane);
  if (TWO && D1.mode == MODE_TRANSITS && D1.grad && v1.begin <= D1.nsteps && v1.end == v1.total)
    split_elements<NB>(P, L::NS - 1, D1, B, wave, lane);
  __syncthreads();
}

// Systems keep J in LDS where a workgroup of LIMIT bytes holds it.
template <int NB, bool TWO, int LIMIT> constexpr bool split_global() {
  if constexpr (TWO) return !(7 * NB <= 32 && SplitLds<NB, false, true, LIMIT>::ok);
  else return !SplitLds<NB, false, false, LIMIT>::ok;
}
template <int NB, int LIMIT> constexpr bool split_pairs() {
  return SplitLds<NB, split_global<NB, true, LIMIT>(), true, LIMIT>::ok;
}
template <int N, int HI, bool TWO, int LIMIT>
__device__ __forceinline__ void split_dispatch(unsigned char* raw, int wave, const SysDesc& D0, const SysDesc& D1,
                                               const SysBufs& B, int64_t c0, int64_t c1, bool pair, int64_t bound, int64_t bound_job,
                                               unsigned long long* err, int lane) {
  if constexpr (N <= HI) {
    if (D0.n == N) {
      split_run<N, split_global<N, TWO, LIMIT>(), TWO, LIMIT>(raw, wave, D0, D1, B, c0, c1, pair, bound, bound_job, err, lane);
      return;
    }
    split_dispatch<N + 1, HI, TWO, LIMIT>(raw, wave, D0, D1, B, c0, c1, pair, bound, bound_job, err, lane);
  }
}

// Persistent two-wave launch of bodies up to HI: like nbg_run (TWO: like
// nbg_run_duo, one unit of one or two systems at a time).  LIMIT: the
// workgroup's LDS.  units[13] collects wait failures.
template <int HI, bool TWO, int LIMIT>
__device__ __forceinline__ void split_body(unsigned char* raw, int* share, const GroupList& gl, const SysBufs& B, int64_t chunk,
                                           int64_t bound, int64_t bound_job, unsigned long long* units,
                                           unsigned long long* err) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lane = threadIdx.x % WAVE;
  int g = 0;
#pragma unroll 1
  while (g < gl.ng) {
    if (threadIdx.x == 0) *share = atomicAdd(gl.queue[g], 1);
    __syncthreads();
    const int u = __builtin_amdgcn_readfirstlane(*share);
    __syncthreads();  // thread 0 writes it again
    if (u >= (TWO ? gl.nunits[g] : gl.nsys[g])) {
      ++g;
      continue;
    }
    int idx = u;
    bool two = false;
    if constexpr (TWO) {
      idx = __builtin_amdgcn_readfirstlane(gl.ustart[g][u]);
      two = __builtin_amdgcn_readfirstlane(gl.ustart[g][u + 1]) - idx == 2;
    }
    SysDesc D0 = gl.descs[g][idx];
    SysDesc D1 = gl.descs[g][two ? idx + 1 : idx];
    D0.rowupd = gl.rowupd;
    D1.rowupd = gl.rowupd;
    const int64_t* ints0 = B.ints + D0.off_int;
    const int64_t* ints1 = B.ints + D1.off_int;
    const int64_t before0 = ints0[D0.n], tr00 = ints0[D0.n + 1], it00 = ints0[D0.n + 2];
    const int64_t before1 = ints1[D1.n], tr01 = ints1[D1.n + 1], it01 = ints1[D1.n + 2];
    const int64_t c0 = D0.chunk > 0 ? D0.chunk : chunk, c1 = D1.chunk > 0 ? D1.chunk : chunk;
    __syncthreads();  // both waves have read the counters
    split_dispatch<2, HI, TWO, LIMIT>(raw, wave, D0, D1, B, c0, c1, two, bound, bound_job, err, lane);
    if (threadIdx.x == 0) {
      visit_done(D0, ints0, before0, tr00, it00, B, units);
      if (two) visit_done(D1, ints1, before1, tr01, it01, B, units);
    }
  }
}

}  // namespace nbg
