// nbg_split.h -- device code of the two- and three-wave launches
// (nbg_run_split, nbg_run_split_duo, nbg_run_split_wide): the state of a
// system, or of two, on one wave and its Jacobian on another, or on two.
//
// The state of AHL21 never reads the Jacobian, so a workgroup divides every
// step between two waves:
//  * the state wave takes the drifts, the Kepler levels, the force-gradient
//    velocities, the transit tests and Newton's iterations; it runs ahead;
//  * the Jacobian wave follows: the pairs' analytic Jacobians, the row
//    updates, Phi and its product, the drifts of J, dq/dt, and the transits'
//    gradients.
// With four workgroups a compute unit each SIMD holds two waves, so that one
// issues while the other waits (a lone wave issues vector instructions about
// 40 % of the time); the half of the code that each wave runs also keeps
// registers within the 256 that two waves per SIMD leave each.  Few systems
// have a compute unit each: there the waves run on different SIMDs, a step
// takes the longest of them instead of their sum, and the Jacobian wave's work
// is divided between two (a pair wave and a row wave, at SplitLds3 below).
//
// The waves talk through LDS: a ring of pair slots (22 doubles each; the rest
// of a pair's drift is formed again from them, with the same operations) and
// three messages a step (PRE: the step's kind, size and velocities; MID: the
// positions between the sweeps; POST: the final state), each buffer with one
// writer and one reader, published by workgroup-scope release of a counter.
// Waits are bounded (wait_for, wait_next): one that has polled about a second
// without an answer, or without a new step of the state wave, ends the
// workgroup's waves and is reported as an error.
//
// Systems with Kepler pairs only and no massless pair (the levels of their
// sweeps are the same for every system of a body count); every operation is the
// one-wave step's, so results are the same bits.
#pragma once

#include <type_traits>

#include "nbg_device.h"

namespace nbg {

// The levels of a sweep over nb bodies whose pairs are all Kepler pairs.  In
// lexicographic order pair (i, j) waits for (i, j - 1) and (i - 1, j) and no
// others that are not already behind those, so level L has the pairs with
// i + j = L + 1; the second sweep's order is the reverse, its levels too.
// Widths read the same from either end.
__host__ __device__ constexpr int level_count(int nb) { return 2 * nb - 3; }
__host__ __device__ constexpr int level_first(int nb, int sum) { return sum - nb + 1 > 0 ? sum - nb + 1 : 0; }  // the smallest i
__host__ __device__ constexpr int level_width(int nb, int level) { return level / 2 - level_first(nb, level + 1) + 1; }
// Pairs of the levels before `level` (the sum of their widths).
__host__ __device__ constexpr int level_start(int nb, int level) {
  const int left = level_count(nb) - level;
  return level < nb ? (level + 1) * (level + 1) / 4 : nb * (nb - 1) / 2 - (left + 1) * (left + 1) / 4;
}

// What the state wave hands over of a pair's drift; the other quantities of
// KParams and the drift itself follow from these.
struct RingSlot {
  double x0[3], v0[3];  // first
  double gamma, g1, g2, g3, h1, h2, r0, r, r0inv, rinv, beta, betainv, eta, sqb;
  double mijinv;
  int i, j;
};
// A pair's Jacobian as the row updates read it: their coefficients in the
// order of use -- in the reference's order mj * kep (36), mi * kep (36) and the
// mass columns mc (24); factored kep (36) and mc (24) -- and kep's h column.
// The kep block is column-major, rk + 6 k.
struct JacSlot {
  double c[96];
  double kh[6];
  double mi, mj;
  int i, j;
};

// acc[r] = fma(+-coefficient I + r, x, acc[r]), r = 0..5, the coefficients held
// one per lane: lane l of every row of 16 lanes has coefficients l, 16 + l, ...
// in cf, and each multiply-add broadcasts its own along the row (DPP
// row_newbcast).  Read from LDS instead, a coefficient costs every lane its
// bytes -- 16 cycles of the compute unit's LDS per pair of coefficients -- and a wait:
// an update of 9 bodies' rows took 2,850 cycles of which its arithmetic
// issues 1,000.  Every lane of the row must be active.  The leading wait keeps
// a coefficient that was just copied between registers readable by DPP.  The
// accumulators are written before the last inputs are read ("&"), so none may
// share a register with an input of the same value.
template <int I, bool NEG = false> __device__ __forceinline__ void fmac6(double* acc, const double* cf, double x) {
#define NBG_FMAC6(SIGN)                                                                              \
  asm("s_nop 1\n\t"                                                                                  \
      "v_fmac_f64_dpp %0, %6, " SIGN "%12 row_newbcast:%13 row_mask:0xf bank_mask:0xf\n\t"           \
      "v_fmac_f64_dpp %1, %7, " SIGN "%12 row_newbcast:%14 row_mask:0xf bank_mask:0xf\n\t"           \
      "v_fmac_f64_dpp %2, %8, " SIGN "%12 row_newbcast:%15 row_mask:0xf bank_mask:0xf\n\t"           \
      "v_fmac_f64_dpp %3, %9, " SIGN "%12 row_newbcast:%16 row_mask:0xf bank_mask:0xf\n\t"           \
      "v_fmac_f64_dpp %4, %10, " SIGN "%12 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"          \
      "v_fmac_f64_dpp %5, %11, " SIGN "%12 row_newbcast:%18 row_mask:0xf bank_mask:0xf"              \
      : "+&v"(acc[0]), "+&v"(acc[1]), "+&v"(acc[2]), "+&v"(acc[3]), "+&v"(acc[4]), "+&v"(acc[5])     \
      : "v"(cf[I / 16]), "v"(cf[(I + 1) / 16]), "v"(cf[(I + 2) / 16]), "v"(cf[(I + 3) / 16]),        \
        "v"(cf[(I + 4) / 16]), "v"(cf[(I + 5) / 16]), "v"(x), "n"(I % 16), "n"((I + 1) % 16),        \
        "n"((I + 2) % 16), "n"((I + 3) % 16), "n"((I + 4) % 16), "n"((I + 5) % 16))
  if constexpr (NEG) NBG_FMAC6("-");
  else NBG_FMAC6("");
#undef NBG_FMAC6
}
// s = fma(coefficient I + r, x[r], s) for r = 0..2, then coefficient M with u.
template <int I, int M> __device__ __forceinline__ double fmac_body(double s, const double* cf, const double* x, double u) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %1, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %2, %6 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %3, %7 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %4, %8 row_newbcast:%12 row_mask:0xf bank_mask:0xf"
      : "+&v"(s)
      : "v"(cf[I / 16]), "v"(cf[(I + 1) / 16]), "v"(cf[(I + 2) / 16]), "v"(cf[M / 16]), "v"(x[0]), "v"(x[1]), "v"(x[2]),
        "v"(u), "n"(I % 16), "n"((I + 1) % 16), "n"((I + 2) % 16), "n"(M % 16));
  return s;
}

template <int NB, int D> __device__ __forceinline__ double split_row_product(double s, const double* cf, const double* P, const double* u) {
  if constexpr (D < NB) {
    s = fmac_body<3 * D, 3 * NB + D>(s, cf, P + 3 * D, u[D]);
    return split_row_product<NB, D + 1>(s, cf, P, u);
  }
  return s;
}

// A column of J and its error: rows at whole distances from one 32-bit
// offset, so that an access is a base, an offset register and an immediate
// (global: the scalar base of the record's store).
template <int NB, class R> struct Column {
  static constexpr int N7 = 7 * NB;
  static constexpr uint32_t ERR = 8u * R::JOFF;
  typename std::conditional<R::JG, __attribute__((address_space(1))) char*, char*>::type base;
  uint32_t off;
  __device__ __forceinline__ Column(R& S, int row, int c) : off(8u * (uint32_t)(row * N7 + c)) {
    if constexpr (R::JG) base = (__attribute__((address_space(1))) char*)uniform_global(S.jg);
    else base = (char*)S.JJ;
  }
  __device__ __forceinline__ auto& j(int k) const { return at(off + 8u * (uint32_t)(k * N7)); }
  __device__ __forceinline__ auto& e(int k) const { return at(off + ERR + 8u * (uint32_t)(k * N7)); }
  __device__ __forceinline__ auto& at(uint32_t o) const {
    if constexpr (R::JG) return *(gdouble*)(base + o);
    else return *(double*)(base + o);
  }
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

// The Jacobian wave's work area: the force-gradient stage, or pair Jacobians
// -- as many as fit beside it, and at least CHMIN (a call that forms pair
// Jacobians takes the same time for one pair as for a wave of them).
template <int NB, int CHMIN> struct JacWork {
  static constexpr int N3 = 3 * NB, N4 = 4 * NB, NP = NB * (NB - 1) / 2, PQ = 13;
  struct F {
    double phi[N3 * N4];
    double dadq[N3 * N4];
    double pq[NP * PQ];
  };
  static constexpr int FIT = (int)(sizeof(F) / sizeof(JacSlot));
  static constexpr int CH1 = FIT < CHMIN ? CHMIN : FIT;
  static constexpr int CH = CH1 < NP ? CH1 : NP;
  union {
    F f;
    JacSlot slot[CH];
  };
};

// Steps of a system as the Jacobian wave sees them (RunCursor's act).
enum : int { SPLIT_J = 4, SPLIT_Q = 8, SPLIT_SAVE = 16 };
struct SplitCtl {
  // counters (counter_reached), from COUNTER_START on
  uint32_t tail, head;  // pairs published / released, per system
  uint32_t sent, seen;  // messages published / copied
  uint32_t answered;    // steps whose dq/dt is complete
  uint32_t begun;       // steps the state wave has begun, followed or not (wait_next)
  int quit;           // the state wave is done, or a wait ran out
  int act[2];         // PRE: what the step is
  int body[2];        // PRE: a gradient step's body ...
  int64_t index[2];   // ... and transit (else the step's number)
  double h[2];
};

template <int NB, bool G, bool TWO, int LIMIT> struct SplitLds {
  static constexpr int NS = TWO ? 2 : 1;
  static constexpr bool HALF = TWO && 7 * NB <= 32 && !G;  // every stage on half-waves
  static constexpr size_t FIXED = NS * (sizeof(StateRec<NB>) + sizeof(JacRec<NB, G>)) + sizeof(SplitCtl) + 64;
  static constexpr int NP = NB * (NB - 1) / 2;
  static constexpr int RMIN = NB / 2 < 1 ? 1 : NB / 2;
  using Work = JacWork<NB, (NB <= 4 ? 6 : 1)>;
  // two work areas where they fit: both systems' force gradients at once
  static constexpr bool PHI2 = TWO && 4 * NB <= 32 && NP <= 32 &&
                               FIXED + 2 * sizeof(Work) + 2 * RMIN * sizeof(RingSlot) <= (size_t)LIMIT;
  static constexpr int NW = PHI2 ? 2 : 1;
  static constexpr long LEFT = (long)LIMIT - (long)(FIXED + NW * sizeof(Work));
  static constexpr int RFIT = LEFT > 0 ? (int)(LEFT / (long)(NS * sizeof(RingSlot))) : 0;
  static constexpr int R = RFIT < NP ? RFIT : NP;  // ring slots per system
  static constexpr bool fits = RFIT >= RMIN;
  // pairs per chunk of the Jacobian wave (a chunk is a run of whole levels)
  static constexpr int CHW = TWO && !PHI2 ? Work::CH / 2 : Work::CH;
  static constexpr int CHL = TWO ? 32 : 64;
  static constexpr int CH0 = CHW < CHL ? CHW : CHL;
  static constexpr int RR = R < 1 ? 1 : R;
  static constexpr int CH = CH0 < RR ? CH0 : RR;
  static constexpr bool ok = fits && CH >= RMIN;
  StateRec<NB> t[NS];
  JacRec<NB, G> j[NS];
  Work w[NW];
  RingSlot ring[NS][RR];
  SplitCtl ctl;
};

__device__ __forceinline__ void start_counters(SplitCtl& c, int lane) {
  if (lane != 0) return;
  c.tail = c.head = c.sent = c.seen = c.answered = c.begun = COUNTER_START;
  c.quit = 0;
}
__device__ __forceinline__ void publish(uint32_t* counter, uint32_t v, int lane) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  if (lane == 0) ring_store(counter, v);
}
// Ends a wait that found nothing in `bound` polls.
__device__ __forceinline__ void wait_failed(SplitCtl* ctl, unsigned long long* err, int lane) {
  if (lane == 0) {
    atomicOr(err, 4ull);
    ring_store(&ctl->quit, 2);
  }
}
// Waits until the counter has reached v; false when another wave has quit or
// the bound runs out.
__device__ __forceinline__ bool wait_for(const uint32_t* counter, uint32_t v, SplitCtl* ctl, int64_t bound,
                                         unsigned long long* err, int lane) {
  int64_t spins = 0;
  while (!counter_reached(ring_load(counter), v)) {
    if (ring_load(&ctl->quit) == 2) return false;
    if (++spins > bound) {
      wait_failed(ctl, err, lane);
      return false;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  return true;
}
// The same for the next step that needs the waiting wave, which may be a whole
// run away: the bound counts polls since the state wave last began a step.
__device__ __forceinline__ bool wait_next(const uint32_t* counter, uint32_t v, SplitCtl* ctl, int64_t bound,
                                          unsigned long long* err, int lane) {
  int64_t spins = 0;
  uint32_t begun = ring_load(&ctl->begun);
  while (!counter_reached(ring_load(counter), v)) {
    if (ring_load(&ctl->quit) == 2) return false;
    const uint32_t b = ring_load(&ctl->begun);
    if (b != begun) {
      begun = b;
      spins = 0;
    } else if (++spins > bound) {
      wait_failed(ctl, err, lane);
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
// A sweep of one system or two of equal body count (act: which have a step).
// A pair takes eight lanes: the first w groups of eight are the first system's
// pairs of a level, the next w the second's.  All eight solve the pair's
// Kepler problem alike (a wave pays for an instruction, not for its lanes);
// then lane r < 6 moves coordinate r of the two bodies -- the positions' three,
// the velocities' three -- in 20 instructions where one lane for all of them
// took 110 and twice the LDS accesses (lanes 6 and 7 repeat 0 and 1).  keep:
// the Jacobian wave follows, so each level's pairs go to the ring once it has
// room.  One out-of-line copy per direction for every body count.
constexpr int PAIR_LANES = 8;
struct SplitSweep {
  uint32_t x0, x1, ring0, ring1, ctl;
  int n, act0, act1, keep, slots, pos;
  uint32_t made;
  double hh0, hh1;
  int64_t bound;
  unsigned long long* err;
};
template <bool DF> static __device__ __attribute__((noinline)) bool split_levels(SplitSweep R) {
  const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  auto uni = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
  const int n = uni(R.n), slots = uni(R.slots), n3 = 3 * n, levels = level_count(n);
  const bool a0 = uni(R.act0) != 0, a1 = uni(R.act1) != 0, keep = uni(R.keep) != 0;
  int pos = uni(R.pos);
  uint32_t made = uni(R.made);
  SplitCtl* ctl = lds_at<SplitCtl>(uni(R.ctl));
  const int group = lane / PAIR_LANES, role = lane % PAIR_LANES < 6 ? lane % PAIR_LANES : lane % PAIR_LANES - 6;
  const bool vel = role >= 3;
  const int c = vel ? role - 3 : role, mine = vel ? n3 + c : c;
#pragma unroll 1
  for (int L = 0; L < levels; ++L) {
    const int sum = DF ? L + 1 : levels - L, w = level_width(n, sum - 1);
    if (keep && !wait_for(&ctl->head, made + w - slots, ctl, R.bound, R.err, lane)) return false;
    const bool second = group >= w;
    const int q = second ? group - w : group;
    if (q < w && (second ? a1 : a0)) {
      const int i = level_first(n, sum) + q, j = sum - i;
      double* x = lds_at<double>(second ? R.x1 : R.x0);
      const double *bi = x + 3 * i, *bj = x + 3 * j;
      const double hh = second ? R.hh1 : R.hh0;
      // every LDS operand is read before anything is written back
      double x0[3], v0[3];
      for (int k = 0; k < 3; ++k) {
        x0[k] = bi[k] - bj[k];
        v0[k] = bi[n3 + k] - bj[n3 + k];
      }
      const double m_i = x[4 * n3 + i], m_j = x[4 * n3 + j];
      const double x0c = bi[c] - bj[c], v0c = bi[n3 + c] - bj[n3 + c];
      double si = bi[mine], sj = bj[mine], ei = bi[2 * n3 + mine], ej = bj[2 * n3 + mine];
      const double gm = NBG_GNEWT * (m_i + m_j);  // not 0: no pair is massless
      double d[6], mijinv;
      KParams P;
      if (jac_delxv_gamma_fast<DF>(x0, v0, d, gm, hh, P)) {
        mijinv = fdiv(1.0, m_i + m_j);  // gm is in the plain range
      } else {
        DriftOut o;
        pair_drift_general(x0[0], x0[1], x0[2], v0[0], v0[1], v0[2], gm, hh, DF, &o);
        P = o.P;
        mijinv = 1.0 / (m_i + m_j);
      }
      const double delta = (vel ? P.dfdt : P.fm1) * x0c + (vel ? P.dgdtm1 : P.gmh) * v0c;
      kahan(si, ei, (m_j * mijinv) * delta);
      kahan(sj, ej, (-(m_i * mijinv)) * delta);
      x[3 * i + mine] = si;
      x[3 * j + mine] = sj;
      x[2 * n3 + 3 * i + mine] = ei;
      x[2 * n3 + 3 * j + mine] = ej;
      if (keep) {
        int at = pos + q;
        if (at >= slots) at -= slots;
        RingSlot* o = lds_at<RingSlot>((second ? R.ring1 : R.ring0) + (uint32_t)(at * sizeof(RingSlot)));
        reinterpret_cast<double*>(o)[role] = vel ? v0c : x0c;  // x0, then v0
        if (lane % PAIR_LANES == 0) {
          o->gamma = P.gamma; o->g1 = P.g1; o->g2 = P.g2; o->g3 = P.g3; o->h1 = P.h1; o->h2 = P.h2;
          o->r0 = P.r0; o->r = P.r; o->r0inv = P.r0inv; o->rinv = P.rinv;
          o->beta = P.beta; o->betainv = P.betainv; o->eta = P.eta; o->sqb = P.sqb;
          o->mijinv = mijinv;
          o->i = i; o->j = j;
        }
      }
    }
    made += w;
    pos += w;
    if (pos >= slots) pos -= slots;
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

// detect_transits! from body c.body on (cursor_detect), a lane a body: the
// first that transits starts a search, those before it keep their g; the ones
// after it are looked at again when the search has ended.  One body after the
// other, each took its own chain of LDS reads and a square root.
template <int NB> __device__ void split_detect(StateRec<NB>& S, const SysDesc& D, RunCursor& c, int lane) {
  const int ti = D.ti;
  int act = c.is < c.iend ? ACT_MAIN : ACT_DONE;
  int body = NB, from = c.body;
#pragma unroll 1
  while (from < NB) {
    const bool mine = lane >= from && lane < NB && lane != ti;
    double g = 0.0;
    bool hit = false;
    if (mine) {
      const double *x = S.x + 3 * lane;
      g = gsky<NB>(S, lane, ti);
      const double r = __builtin_sqrt((x[0] * x[0] + x[1] * x[1]) + x[2] * x[2]);
      hit = g > 0.0 && S.gsave[lane] < 0.0 && -x[2] > 0.25 * r && r < 1e12;
    }
    const uint64_t hits = __builtin_amdgcn_ballot_w64(hit);
    const int i = hits ? __builtin_ctzll(hits) : NB;
    wsync();
    if (mine && lane < i) S.gsave[lane] = g;
    wsync();
    if (i == NB) break;
    const int64_t cnt = S.count[i] + 1;
    wsync();
    if (lane == 0) S.count[i] = cnt;
    wsync();
    if (cnt >= 1 && cnt <= D.ntt) {
      if (!c.saved) {
        split_save_prior<NB>(S, lane);
        c.saved = 1;
      }
      const double gi = gsky<NB>(S, i, ti);
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
    if (lane == i) S.gsave[i] = g;
    wsync();
    from = i + 1;
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

// The state before step k of a MODE_CARTESIAN run (write_snapshot's part
// without the Jacobian).
template <int NB> __device__ void split_write_state(const StateRec<NB>& S, const SysDesc& D, const SysBufs& B, int64_t k, int lane) {
  constexpr int N3 = 3 * NB;
  const int64_t ns = D.nsteps;
  double* base = B.traj + D.off_traj;
  if (lane == 0) base[k] = (k == 0) ? D.t0 : D.t0 + (D.h * (double)k);  // s.t[1] = t0 + (h * i)
  for (int q = lane; q < N3; q += WAVE) {
    base[traj_off_x(NB, ns) + N3 * k + q] = S.x[q];
    base[traj_off_v(NB, ns) + N3 * k + q] = S.v[q];
    if (D.traj & TRAJ_ERR) {
      base[traj_off_xe(NB, ns) + N3 * k + q] = S.xe[q];
      base[traj_off_ve(NB, ns) + N3 * k + q] = S.ve[q];
    }
  }
}
// ... and the Jacobian's part: column-major matrices, an element a lane; the
// mass rows are unit rows of jac_step and zero rows of jac_error.
template <int NB, class R> __device__ void split_write_jac(R& S, const SysDesc& D, const SysBufs& B, int64_t k, int lane) {
  constexpr int N7 = 7 * NB, NN = N7 * N7;
  const auto J_ = jj<NB>(S);
  double* base = B.traj + D.off_traj;
  for (int w = 0; w < 2; ++w) {
    if (!(D.traj & (w ? TRAJ_JACERR : TRAJ_JAC))) continue;
    double* o = base + (w ? traj_off_jacerr(NB, D.nsteps, D.traj) : traj_off_jac(NB, D.nsteps, D.traj)) + (int64_t)NN * k;
#pragma unroll 4
    for (int e = lane; e < NN; e += WAVE) {
      const int c = e / N7, r = e - N7 * c, b = r / 7, kk = r - 7 * b;
      double v = w == 0 && c == r ? 1.0 : 0.0;
      if (kk < 6) v = J_[(unsigned)((w ? R::JOFF : 0) + (6 * b + kk) * N7 + c)];
      o[e] = v;
    }
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

template <int NB, bool TWO, class L>
__device__ void split_state(L& P, const SysDesc& D0, const SysDesc& D1, const SysBufs& B,
                            const Visit& v0, const Visit& v1, int lane, int64_t bound, unsigned long long* err) {
  constexpr int N3 = 3 * NB, NP = L::NP, K = TWO ? 1 : 0;
  constexpr int STEP = TWO && N3 <= 32 ? 32 : WAVE;
  static_assert(L::NS * (NB / 2) * PAIR_LANES <= WAVE, "a level's pairs must fit the wave");
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
  R.n = NB; R.slots = L::RR;
  R.pos = 0; R.made = COUNTER_START;
  R.bound = bound; R.err = err;
  uint32_t sent = COUNTER_START, asked = COUNTER_START, begun = COUNTER_START;
  const int half = STEP == 32 ? lane >> 5 : 0, col = STEP == 32 ? lane & 31 : lane;
#pragma unroll 1
  while (c[0].act != ACT_DONE || c[1].act != ACT_DONE) {
    ++begun;
    if (lane == 0) ring_store(&ctl->begun, begun);
    const bool a0 = c[0].act != ACT_DONE, a1 = TWO && c[1].act != ACT_DONE;
    double h0 = 0.0, h1 = 0.0;
    int n0 = ACT_DONE, n1 = ACT_DONE;
    if (a0) split_prepare<NB>(P.t[0], D0, c[0], h0, n0, lane);
    if (a1) split_prepare<NB>(P.t[K], D1, c[1], h1, n1, lane);
    if (D0.mode == MODE_CARTESIAN && a0) split_write_state<NB>(P.t[0], D0, B, c[0].is, lane);
    if (TWO && D1.mode == MODE_CARTESIAN && a1) split_write_state<NB>(P.t[K], D1, B, c[1].is, lane);
    const bool keep = ((n0 | n1) & (SPLIT_J | SPLIT_Q)) != 0;
    if (keep) {
      // PRE; its buffers are free once the message three before it is copied
      if (!wait_for(&ctl->seen, sent - 2, ctl, bound, err, lane)) return;
      for (int q = lane; q < N3; q += WAVE) {
        if (n0 & SPLIT_Q) P.j[0].mv[q] = P.t[0].v[q];
        if (n1 & SPLIT_Q) P.j[K].mv[q] = P.t[K].v[q];
      }
      if (lane == 0) {
        ctl->act[0] = n0; ctl->h[0] = h0; ctl->body[0] = c[0].jb; ctl->index[0] = n0 & SPLIT_SAVE ? P.t[0].count[c[0].jb] - 1 : c[0].is;
        ctl->act[1] = n1; ctl->h[1] = h1; ctl->body[1] = c[1].jb; ctl->index[1] = n1 & SPLIT_SAVE ? P.t[K].count[c[1].jb] - 1 : c[1].is;
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
static __device__ __attribute__((noinline)) void split_pair_jacobian(uint32_t ring, uint32_t slot, double m_i, double m_j, double h, int factored) {
  const bool fact = __builtin_amdgcn_readfirstlane(factored) != 0;
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
  double* mc = fact ? o->c + 36 : o->c + 72;
  for (int rk = 0; rk < 6; ++rk) {
    mc[rk] = jm[rk] * m_j;
    mc[6 + rk] = (((-mj) * dl[rk]) * mijinv) - ((NBG_GNEWT * mi) * kep[rk + 36]);
    mc[12 + rk] = ((mi * dl[rk]) * mijinv) + ((NBG_GNEWT * mj) * kep[rk + 36]);
    mc[18 + rk] = (-jm[rk]) * m_i;
  }
  if (fact) {
    for (int q = 0; q < 36; ++q) o->c[q] = kep[q];
  } else {
    for (int q = 0; q < 36; ++q) {
      o->c[q] = mj * kep[q];
      o->c[36 + q] = mi * kep[q];
    }
  }
  for (int q = 0; q < 6; ++q) o->kh[q] = kep[42 + q];
  o->mi = mi; o->mj = mj;
  o->i = a->i; o->j = a->j;
}

// jij_coef from a JacSlot, without its sign for k of the Kepler block.
template <bool FACT> __device__ __forceinline__ double split_coef(const JacSlot& sl, bool rowi, int rk, int k) {
  constexpr int MC = FACT ? 36 : 72;
  if (k == 6) return sl.c[MC + (rowi ? 0 : 6) + rk];
  if (k == 13) return sl.c[MC + (rowi ? 12 : 18) + rk];
  const int at = rk + 6 * (k < 7 ? k : k - 7);
  const double v = FACT ? (rowi ? sl.mj : sl.mi) * sl.c[at] : sl.c[(rowi ? 0 : 36) + at];
  return rowi == (k < 7) ? v : -v;
}

// The row updates of levels [lev0, lev1) of sweep dir (jij_cols' operations),
// their pair Jacobians in `slots` level by level; STEP lanes a system, every one
// of them taking part: those past the last column compute it again and store
// nothing.  The pairs are taken body by body -- i up and j up, or both down in
// the second sweep, which keeps every body's order -- so that body i's twelve
// rows of J and its error stay in registers over its pairs of these levels and
// body j's next rows are loaded before the arithmetic of the pair at hand.
// Level by level, each pair loaded and stored both bodies' 24 rows: systems
// whose J is not in LDS waited for the L2 cache and what lies behind it (302 GB
// written and 104 read by 250 steps of 4096 systems, 3 TB/s).  Rounds of 200
// steps over 2048 systems in the reference's order 90.7 -> 70.8 ms; factored,
// 250 of 4096, 143.7 -> 137.4.
template <int NB, bool G, int STEP, bool FACT, class R>
__device__ __attribute__((always_inline)) inline void split_rows(R& S, const JacSlot* slots, int dir, int lev0, int lev1, int col) {
  constexpr int N7 = 7 * NB, NC = FACT ? 4 : 6, NL = level_count(NB);
  const int lo = dir == 0 ? lev0 + 1 : NL - lev1 + 1, hi = dir == 0 ? lev1 : NL - lev0;  // i + j in lo .. hi
  const int base = level_start(NB, lev0), turn = dir == 0 ? 1 : -1;
  const int ifirst = level_first(NB, lo), ilast = (hi - 1) / 2;
#pragma unroll 1
  for (int c0 = 0; c0 < N7; c0 += STEP) {
    const bool on = c0 + col < N7;
    const int c = on ? c0 + col : N7 - 1;
#pragma unroll 1
    for (int i = dir == 0 ? ifirst : ilast; i >= ifirst && i <= ilast; i += turn) {
      const int jlo = lo - i > i + 1 ? lo - i : i + 1, jhi = hi - i < NB - 1 ? hi - i : NB - 1;
      if (jlo > jhi) continue;
      int j = dir == 0 ? jlo : jhi;
      const double a6 = (c == 7 * i + 6) ? 1.0 : 0.0;
      const Column<NB, R> Ci(S, 6 * i, c);
      double ai[6], ei[6], aj[6], ej[6];
      auto load = [&](const Column<NB, R>& C, double (&a)[6], double (&e)[6]) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 6; ++k) a[k] = C.j(k);
#pragma unroll
        for (int k = 0; k < 6; ++k) e[k] = C.e(k);
      };
      load(Ci, ai, ei);
      if constexpr (G) load(Column<NB, R>(S, 6 * j, c), aj, ej);
#pragma unroll 1
      while (true) {
        const int sum = i + j, at = level_start(NB, dir == 0 ? sum - 1 : NL - sum) - base + i - level_first(NB, sum);
        const JacSlot& sl = slots[at];
        double cf[NC];
#pragma unroll
        for (int r = 0; r < NC; ++r) cf[r] = sl.c[16 * r + (col & 15)];
        const double mi = sl.mi, mj = sl.mj;
        // G: the next partner's rows are in flight during the arithmetic (the
        // last pair loads its own again); LDS answers too soon for the copies
        // that costs
        const int jn = j + turn < jlo || j + turn > jhi ? j : j + turn;
        const Column<NB, R> Cj(S, 6 * j, c);
        double an[6], en[6];
        if constexpr (G) load(Column<NB, R>(S, 6 * jn, c), an, en);
        else load(Cj, aj, ej);
        __builtin_amdgcn_sched_barrier(0);
        const double a13 = (c == 7 * j + 6) ? 1.0 : 0.0;
        double oi[6], oj[6];
        if constexpr (FACT) {
          double d[6], sk[6];
#pragma unroll
          for (int k = 0; k < 6; ++k) {
            d[k] = ai[k] - aj[k];
            sk[k] = 0.0;
          }
          fmac6<0>(sk, cf, d[0]);
          fmac6<6>(sk, cf, d[1]);
          fmac6<12>(sk, cf, d[2]);
          fmac6<18>(sk, cf, d[3]);
          fmac6<24>(sk, cf, d[4]);
          fmac6<30>(sk, cf, d[5]);
#pragma unroll
          for (int rk = 0; rk < 6; ++rk) {
            oi[rk] = mj * sk[rk];
            oj[rk] = (-mi) * sk[rk];
          }
          fmac6<36>(oi, cf, a6);
          fmac6<42>(oj, cf, a6);
          fmac6<48>(oi, cf, a13);
          fmac6<54>(oj, cf, a13);
        } else {
#pragma unroll
          for (int q = 0; q < 6; ++q) oi[q] = oj[q] = 0.0;
          // k = 0..5: rows of i get +mj*kep * a_i[k], rows of j -mi*kep * a_i[k]
          fmac6<0>(oi, cf, ai[0]);
          fmac6<36, true>(oj, cf, ai[0]);
          fmac6<6>(oi, cf, ai[1]);
          fmac6<42, true>(oj, cf, ai[1]);
          fmac6<12>(oi, cf, ai[2]);
          fmac6<48, true>(oj, cf, ai[2]);
          fmac6<18>(oi, cf, ai[3]);
          fmac6<54, true>(oj, cf, ai[3]);
          fmac6<24>(oi, cf, ai[4]);
          fmac6<60, true>(oj, cf, ai[4]);
          fmac6<30>(oi, cf, ai[5]);
          fmac6<66, true>(oj, cf, ai[5]);
          fmac6<72>(oi, cf, a6);
          fmac6<78>(oj, cf, a6);
          // k = 7..12: rows of i get -mj*kep * a_j[k], rows of j +mi*kep * a_j[k]
          fmac6<0, true>(oi, cf, aj[0]);
          fmac6<36>(oj, cf, aj[0]);
          fmac6<6, true>(oi, cf, aj[1]);
          fmac6<42>(oj, cf, aj[1]);
          fmac6<12, true>(oi, cf, aj[2]);
          fmac6<48>(oj, cf, aj[2]);
          fmac6<18, true>(oi, cf, aj[3]);
          fmac6<54>(oj, cf, aj[3]);
          fmac6<24, true>(oi, cf, aj[4]);
          fmac6<60>(oj, cf, aj[4]);
          fmac6<30, true>(oi, cf, aj[5]);
          fmac6<66>(oj, cf, aj[5]);
          fmac6<84>(oi, cf, a13);
          fmac6<90>(oj, cf, a13);
        }
#pragma unroll
        for (int q = 0; q < 6; ++q) {
          kahan(ai[q], ei[q], oi[q]);
          kahan(aj[q], ej[q], oj[q]);
        }
        if (on) {
#pragma unroll
          for (int k = 0; k < 6; ++k) {
            Cj.j(k) = aj[k];
            Cj.e(k) = ej[k];
          }
        }
        if (jn == j) break;
        j = jn;
        if constexpr (G) {
#pragma unroll
          for (int k = 0; k < 6; ++k) {
            aj[k] = an[k];
            ej[k] = en[k];
          }
        }
      }
      if (on) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          Ci.j(k) = ai[k];
          Ci.e(k) = ei[k];
        }
      }
    }
  }
}

// dqdt_ij (ahl21.jl:743-748) and dq/dt's rows, of cnt pairs level by level.
template <int NB, bool FACT, class R>
__device__ __attribute__((always_inline)) inline void split_rates(R& S, const JacSlot* slots, int cnt, int col) {
#pragma unroll 1
  for (int q = 0; q < cnt; ++q) {
    const JacSlot& sl = slots[q];
    const int i = sl.i, j = sl.j;
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
        dq = (rowi ? sl.mj : -sl.mi) * sl.kh[rk];
        for (int k = 0; k < 14; ++k) s2 = fmad(split_coef<FACT>(sl, rowi, rk, k), q1[k], s2);
      } else {
        for (int k = 0; k < 14; ++k) s2 = fmad(0.0, q1[k], s2);
      }
      const double nd = (dq * 0.5) + (mine + s2);
      S.dqij[col] = nd;
      S.dqdt[rowi ? 7 * i + rk : 7 * j + rk] = nd;
    }
    wsync();
  }
}

template <int NB, bool G, bool TWO, int LIMIT> struct SplitFollow {
  uint32_t head;
  int pos;
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
  constexpr int K = TWO ? 1 : 0, NL = level_count(NB);
  const bool p0 = (n0 & (SPLIT_J | SPLIT_Q)) != 0, p1 = TWO && (n1 & (SPLIT_J | SPLIT_Q)) != 0;
  JacSlot* s0 = P.w[0].slot;
  JacSlot* s1 = L::PHI2 ? P.w[L::NW - 1].slot : P.w[0].slot + L::CH;
  int lev = 0;
  while (lev < NL) {
    const int lev0 = lev;
    int cnt = 0;
    while (lev < NL && cnt + level_width(NB, lev) <= L::CH) cnt += level_width(NB, lev++);
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
        if (dir == 0) split_pair_jacobian<true>(lds_off(a), lds_off(o), m[a->i], m[a->j], hh, FACT);
        else split_pair_jacobian<false>(lds_off(a), lds_off(o), m[a->i], m[a->j], hh, FACT);
      }
    }
    wsync();
    F.head += cnt;
    F.pos += cnt;
    if (F.pos >= L::RR) F.pos -= L::RR;
    publish(&P.ctl.head, F.head, lane);
    const bool j0 = (n0 & SPLIT_J) != 0, q0 = (n0 & SPLIT_Q) != 0, j1 = (n1 & SPLIT_J) != 0, q1 = (n1 & SPLIT_Q) != 0;
    if constexpr (L::HALF) {
      const bool sys = lane >= 32;
      if (sys ? j1 : j0) split_rows<NB, G, 32, FACT>(sys ? P.j[K] : P.j[0], sys ? s1 : s0, dir, lev0, lev, lane & 31);
      if (sys ? q1 : q0) split_rates<NB, FACT>(sys ? P.j[K] : P.j[0], sys ? s1 : s0, cnt, lane & 31);
      wsync();
    } else {
      if (j0) split_rows<NB, G, WAVE, FACT>(P.j[0], s0, dir, lev0, lev, lane);
      if (q0) split_rates<NB, FACT>(P.j[0], s0, cnt, lane);
      if (TWO && j1) split_rows<NB, G, WAVE, FACT>(P.j[K], s1, dir, lev0, lev, lane);
      if (TWO && q1) split_rates<NB, FACT>(P.j[K], s1, cnt, lane);
      wsync();
    }
  }
  return true;
}

// phisalpha! with Jacobian (phisalpha_cols' operations and order) for Kepler
// pairs only, STEP lanes a system, a lane a column of dadq and jac_phi (column
// (d, p): coordinate p of body d, p = 3 its mass).  The terms that depend on a
// column's role in a pair enter as products with 0, 1 or -1 -- exact, and a
// zero added instead of left out changes at most a zero's sign -- where selects
// of 64-bit values took three quarters of the loop's 315 instructions.
template <int NB, int STEP, bool FACT, class R, class WK>
__device__ __attribute__((always_inline)) inline void split_phi(R& S, WK& W, double h, bool needQ, int col) {
  constexpr int N3 = 3 * NB, N4 = 4 * NB, NP = WK::NP, PQ = WK::PQ, PP = (NP + STEP - 1) / STEP;
  double* PHI = W.f.phi;
  double* D = W.f.dadq;
  double* pq = W.f.pq;
  const double coeff = (((2.0 * (h * h * h)) / 96.0) * 2.0) * NBG_GNEWT;
  // loop 1 factors (ahl21.jl:569-575)
#pragma unroll
  for (int u = 0; u < PP; ++u) {
    const int p = col + u * STEP;
    if (p < NP) {
      int i, j;
      pair_at<NB>(p, i, j);
      double rij[3];
      for (int k = 0; k < 3; ++k) rij[k] = S.x[3 * i + k] - S.x[3 * j + k];
      const double r2 = dot3(rij);
      const double fac2 = NBG_GNEWT / (r2 * __builtin_sqrt(r2));
      const double q = 3.0 / r2;
      double* o = pq + p * PQ;
      o[0] = fac2;
      for (int k = 0; k < 3; ++k) {
        o[1 + k] = fac2 * rij[k];
        o[4 + k] = (fac2 * rij[k]) * q;
      }
    }
  }
  wsync();
  // the lane's column; columns past the last work on it again for nothing
  const bool own = col < N4;
  const int cc = own ? col : N4 - 1;
  const int myd = cc < N3 ? cc / 3 : cc - N3, myp = cc < N3 ? cc - 3 * (cc / 3) : 3;
  const double pos = myp < 3 ? 1.0 : 0.0, mass = 1.0 - pos;
  const int ry = myp < 3 ? myp : 0;
  double pk[3];
  for (int k = 0; k < 3; ++k) pk[k] = myp == k ? 1.0 : 0.0;
  // loop 1 (ahl21.jl:567-602), the lane's column: row block b != myd from the
  // pair (b, myd), row block myd over the partners in increasing order
  {
    const double md = S.m[myd], xd = S.x[3 * myd + ry];
    double db[3] = {0.0, 0.0, 0.0}, ab = 0.0;
#pragma unroll 2
    for (int q = 0; q < NB - 1; ++q) {
      const bool after = q >= myd;  // the other body comes after myd
      const int b = after ? q + 1 : q;
      const double* o = pq + (after ? pair_index<NB>(myd, b) : pair_index<NB>(b, myd)) * PQ;
      const double sg = after ? 1.0 : -1.0;  // +1: myd is i
      const double rmy = (sg * pos) * (xd - S.x[3 * b + ry]);
      const double mb = S.m[b], f2 = o[0], mm = sg * mass;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const double fac = o[1 + k], f3 = o[4 + k];
        // row block b: myd is its partner
        const double t1 = fmad(mm, fac, -((f3 * md) * rmy));
        const double t = (0.0 + t1) + pk[k] * (f2 * md);
        if (own) D[(3 * b + k) * N4 + cc] = t;
        // row block myd
        db[k] = (db[k] + (f3 * mb) * rmy) - pk[k] * (f2 * mb);
      }
      const double mf = mb * o[1 + ry];
      ab -= sg * mf;
    }
    if (own)
      for (int k = 0; k < 3; ++k) D[(3 * myd + k) * N4 + cc] = db[k];
    if (own && myp < 3) S.a[3 * myd + myp] = ab;
  }
  wsync();
  // loop 2 factors (ahl21.jl:609-640)
#pragma unroll
  for (int u = 0; u < PP; ++u) {
    const int p = col + u * STEP;
    if (p < NP) {
      int i, j;
      pair_at<NB>(p, i, j);
      double rij[3], aij[3];
      for (int k = 0; k < 3; ++k) {
        aij[k] = S.a[3 * i + k] - S.a[3 * j + k];
        rij[k] = S.x[3 * i + k] - S.x[3 * j + k];
      }
      const double r2 = dot3(rij);
      const double r1 = __builtin_sqrt(r2);
      const double ardot = dot3(aij, rij);
      const double fac1 = coeff / ((r2 * r2) * r1);
      const double mi = S.m[i], mj = S.m[j];
      const double fac2 = ((2.0 * NBG_GNEWT) * (mi + mj)) / r1 + 3.0 * ardot;
      double* o = pq + p * PQ;
      for (int k = 0; k < 3; ++k) {
        o[k] = fac1 * (rij[k] * fac2 - r2 * aij[k]);                                             // fac
        o[4 + k] = (((2.0 * NBG_GNEWT) * fac1) * rij[k]) / r1;                                   // fm
        o[7 + k] = ((-2.0) * fac1) * ((((rij[k] * NBG_GNEWT) * (mi + mj)) / (r2 * r1)) + aij[k]);  // fr
      }
      o[3] = 5.0 / r2;
      o[10] = fac1 * 3.0;
      o[11] = fac1 * fac2;   // fd
      o[12] = (-fac1) * r2;  // fa
    }
  }
  wsync();
  if (needQ) {
    // dqdt_phi, a lane an entry: the pairs of a body in increasing order of
    // its partner, as in the reference's loop
    const double q3h = 3.0 / h;
    for (int e = col; e < N3; e += STEP) {
      const int b = e / 3, k = e - 3 * b;
      double qb = S.dqdt_phi[7 * b + 3 + k];
      for (int q = 0; q < NB - 1; ++q) {
        const bool bi = q >= b;
        const int c = bi ? q + 1 : q;
        const double qm = (q3h * S.m[c]) * pq[(bi ? pair_index<NB>(b, c) : pair_index<NB>(c, b)) * PQ + k];
        qb += bi ? qm : -qm;
      }
      S.dqdt_phi[7 * b + 3 + k] = qb;
    }
  }
  // loop 2 (ahl21.jl:607-698)
  if constexpr (FACT) {
    // pair by pair: the rows of body i receive mj * X, those of body j
    // -mi * X of the same column term X (phisalpha_cols' factored form)
    if (own)
      for (int r = 0; r < N3; ++r) PHI[r * N4 + cc] = 0.0;
    int p = 0;
#pragma unroll 1
    for (int i = 0; i < NB - 1; ++i) {
      double pi[3], xi[3], Di[3];
      for (int k = 0; k < 3; ++k) {
        pi[k] = PHI[(3 * i + k) * N4 + cc];
        xi[k] = S.x[3 * i + k];
        Di[k] = D[(3 * i + k) * N4 + cc];
      }
      const double mi = S.m[i], ai = S.a[3 * i + ry], xr = S.x[3 * i + ry];
      const double si = myd == i ? 1.0 : 0.0;
#pragma unroll 1
      for (int j = i + 1; j < NB; ++j, ++p) {
        const double* o = pq + p * PQ;
        const double mj = S.m[j], sj = myd == j ? 1.0 : 0.0;
        const double sg = pos * (si - sj), mm = mass * (si + sj), ci = mass * si, cj = mass * sj;
        double r[3], dD[3], pj[3];
        for (int k = 0; k < 3; ++k) {
          r[k] = xi[k] - S.x[3 * j + k];
          dD[k] = Di[k] - D[(3 * j + k) * N4 + cc];
          pj[k] = PHI[(3 * j + k) * N4 + cc];
        }
        const double rmy = xr - S.x[3 * j + ry], amy = ai - S.a[3 * j + ry];
        double dot = 0.0;
        for (int k = 0; k < 3; ++k) dot += r[k] * dD[k];
        const double fd = o[11], fa = o[12];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const double fac = o[k], ff = o[10] * r[k];
          const double base = (pk[k] * fd - (fac * o[3]) * rmy) + (o[7 + k] * rmy + ff * amy);
          const double role = fmad(mm, o[4 + k], sg * base);
          const double X = (role + fa * dD[k]) + ff * dot;
          pi[k] += fmad(cj, fac, mj * X);
          pj[k] += fmad(-ci, fac, (-mi) * X);
        }
        if (own)
          for (int k = 0; k < 3; ++k) PHI[(3 * j + k) * N4 + cc] = pj[k];
      }
      if (own)
        for (int k = 0; k < 3; ++k) PHI[(3 * i + k) * N4 + cc] = pi[k];
    }
  } else {
    // one row block at a time over its partners c in increasing order; with
    // r, dD and the like taken from b to c, the signs of the pair's order
    // cancel except in the terms that carry sb
#pragma unroll 1
    for (int b = 0; b < NB; ++b) {
      double pb[3], xb[3], Db[3];
      for (int k = 0; k < 3; ++k) {
        pb[k] = 0.0;
        xb[k] = S.x[3 * b + k];
        Db[k] = D[(3 * b + k) * N4 + cc];
      }
      const double ar = S.a[3 * b + ry], xr = S.x[3 * b + ry], self = myd == b ? 1.0 : 0.0;
#pragma unroll 1
      for (int q = 0; q < NB - 1; ++q) {
        const bool bi = q >= b;
        const int c = bi ? q + 1 : q;
        const double* o = pq + (bi ? pair_index<NB>(b, c) : pair_index<NB>(c, b)) * PQ;
        const double sb = bi ? 1.0 : -1.0, m = S.m[c], other = myd == c ? 1.0 : 0.0;
        const double sg = pos * (self - other);
        const double rs = (sg * sb) * (xr - S.x[3 * c + ry]), as = (sg * sb) * (ar - S.a[3 * c + ry]);
        const double ms = (mass * self) * sb, mo = (mass * other) * sb;
        double r[3], dD[3];
        for (int k = 0; k < 3; ++k) {
          r[k] = xb[k] - S.x[3 * c + k];
          dD[k] = Db[k] - D[(3 * c + k) * N4 + cc];
        }
        double dot = 0.0;
        for (int k = 0; k < 3; ++k) dot += r[k] * dD[k];
        const double fdm = o[11] * m, fam = o[12] * m;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          const double fac = o[k], ff = o[10] * (sb * r[k]), y = o[4 + k] * m;
          const double t1 = fmad(ms, y, fmad(mo, fac, -(((fac * o[3]) * m) * rs)));
          const double t2 = fmad(mo, y, fdm * (sg * pk[k]));
          const double t3 = m * (o[7 + k] * rs + ff * as);
          pb[k] = (((((pb[k] + t1) + t2) + t3) + fam * dD[k]) + (ff * m) * (sb * dot));
        }
      }
      if (own)
        for (int k = 0; k < 3; ++k) PHI[(3 * b + k) * N4 + cc] = pb[k];
    }
  }
}

// The drift of J's position rows (drift_grad!) and, in the reference's order,
// the zero-addend compensated pass over every row that follows it; a body's
// rows at a time, all in flight together.
template <int NB, bool G, int STEP, bool FACT, class R>
__device__ __attribute__((always_inline)) inline void split_drift(R& S, double hh, int col) {
  constexpr int N7 = 7 * NB;
  for (int c = col; c < N7; c += STEP) {
#pragma unroll 1
    for (int b = 0; b < NB; ++b) {
      const Column<NB, R> C(S, 6 * b, c);
      double a[6], e[6];
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        a[k] = C.j(k);
        if (!FACT || k < 3) e[k] = C.e(k);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 3; ++k) kahan(a[k], e[k], hh * a[3 + k]);
      if constexpr (!FACT) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          e[k] += 0.0;
          const double t = a[k] + e[k];
          e[k] += a[k] - t;
          a[k] = t;
        }
      }
#pragma unroll
      for (int k = 0; k < (FACT ? 3 : 6); ++k) {
        C.j(k) = a[k];
        C.e(k) = e[k];
      }
    }
  }
}

// J_vel += Phi * J_pos (step_mid_rest): Phi's rows broadcast along the lanes,
// the columns' position rows in registers.
template <int NB, bool G, int STEP, bool FACT, class R>
__device__ __attribute__((always_inline)) inline void split_vel_product(R& S, const double* B, int col) {
  constexpr int N3 = 3 * NB, N4 = 4 * NB, N7 = 7 * NB, NC = (N4 + 15) / 16;
#pragma unroll 1
  for (int c0 = 0; c0 < N7; c0 += STEP) {
    const bool on = c0 + col < N7;
    const int c = on ? c0 + col : N7 - 1;
    const Column<NB, R> C(S, 0, c);
    double P[N3], u[NB];
#pragma unroll
    for (int d = 0; d < NB; ++d) {
#pragma unroll
      for (int p = 0; p < 3; ++p) P[3 * d + p] = C.j(6 * d + p);
      u[d] = (c == 7 * d + 6) ? 1.0 : 0.0;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
    for (int b = 0; b < NB; ++b) {
      const Column<NB, R> V(S, 6 * b + 3, c);
      double s[3], a[3], e[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        a[k] = V.j(k);
        e[k] = V.e(k);
      }
      double cf[3][NC];
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int r = 0; r < NC; ++r) {
          const int at = 16 * r + (col & 15);
          cf[k][r] = B[(3 * b + k) * N4 + (at < N4 ? at : N4 - 1)];
        }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        s[k] = split_row_product<NB, 0>(0.0, cf[k], P, u);
        kahan(a[k], e[k], s[k]);
      }
      if (on) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          V.j(k) = a[k];
          V.e(k) = e[k];
        }
      }
    }
    if constexpr (!FACT) {
      if (on) zero_add_rows<NB>(S, c, true, false);
    }
  }
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

// The dt/dq rows of a transit (cursor_record) from the final state of its
// gradient step: its dg/dt, the sky separation and velocity, and the
// velocity's rate of change.
template <int NB, class R>
__device__ void split_gradient_rows(R& S, const SysDesc& D, const SysBufs& B, int jb, int64_t cc, double gd, double dx, double dy,
                                    double dvx, double dvy, double ax, double ay, int lane) {
  constexpr int N7 = 7 * NB;
  const int n = NB, ti = D.ti, nb = D.ntbv;
  const auto J_ = jj<NB>(S);
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
      const double dvdt = (dvx * ax + dvy * ay) / vsky;
      dq[1 + nb * base] = (jvx * dvx + jvy * dvy) / vsky + dvdt * d0;
      dq[2 + nb * base] = 2.0 * (jx * dx + jy * dy);
    }
  }
}
template <int NB, class R>
__device__ void split_gradient(R& S, const SysDesc& D, const SysBufs& B, int jb, int64_t cc, int lane) {
  const int ti = D.ti;
  split_gradient_rows<NB>(S, D, B, jb, cc, gdot<NB>(S, ti, jb), S.x[3 * jb] - S.x[3 * ti], S.x[3 * jb + 1] - S.x[3 * ti + 1],
                          S.v[3 * jb] - S.v[3 * ti], S.v[3 * jb + 1] - S.v[3 * ti + 1], S.dqdt[7 * jb + 3] - S.dqdt[7 * ti + 3],
                          S.dqdt[7 * jb + 4] - S.dqdt[7 * ti + 4], lane);
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
                               const Visit& v0, const Visit& v1, int lane, int64_t bound,
                               unsigned long long* err) {
  using L = SplitLds<NB, G, TWO, LIMIT>;
  constexpr int N3 = 3 * NB, N7 = 7 * NB, K = TWO ? 1 : 0;
  constexpr int STEP = L::HALF ? 32 : WAVE;
  SplitCtl* ctl = &P.ctl;
  SplitFollow<NB, G, TWO, LIMIT> F{COUNTER_START, 0, bound, err};
  JacRec<NB, G>& J0 = P.j[0];
  JacRec<NB, G>& J1 = P.j[K];
  typename L::Work& W0 = P.w[0];
  typename L::Work& W1 = P.w[L::NW - 1];
  const bool sys = L::HALF && lane >= 32;
  const int col = L::HALF ? lane & 31 : lane;
  uint32_t seen = COUNTER_START, answered = COUNTER_START;
#pragma unroll 1
  while (true) {
    if (!wait_next(&ctl->sent, seen + 1, ctl, bound, err, lane)) return;
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
    if (D0.mode == MODE_CARTESIAN && j0) split_write_jac<NB>(J0, D0, B, i0, lane);
    if (TWO && D1.mode == MODE_CARTESIAN && j1) split_write_jac<NB>(J1, D1, B, i1, lane);
    if (n0 & SPLIT_SAVE) split_keep_jac<NB>(J0, B.ws + D0.off_ws, false, lane);
    if (n1 & SPLIT_SAVE) split_keep_jac<NB>(J1, B.ws + D1.off_ws, false, lane);
    if constexpr (L::HALF) {
      step_pre<NB, G, 32, FACT, false>(sys ? J1 : J0, W0, sys ? h1 : h0, false, sys ? q1 : q0, false, col);
      if (sys ? j1 : j0) split_drift<NB, G, 32, FACT>(sys ? J1 : J0, 0.5 * (sys ? h1 : h0), col);
    } else {
      step_pre<NB, G, STEP, FACT, false>(J0, W0, h0, false, q0, false, lane);
      if (j0) split_drift<NB, G, WAVE, FACT>(J0, 0.5 * h0, lane);
      if constexpr (TWO) {
        step_pre<NB, G, STEP, FACT, false>(J1, W0, h1, false, q1, false, lane);
        if (j1) split_drift<NB, G, WAVE, FACT>(J1, 0.5 * h1, lane);
      }
    }
    wsync();
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
          split_phi<NB, 32, FACT>(hi ? J1 : J0, hi ? W1 : W0, hi ? h1 : h0, hi ? q1 : q0, lane & 31);
      }
      wsync();
      if constexpr (L::HALF) {
        if (sys ? j1 : j0) split_vel_product<NB, G, 32, FACT>(sys ? J1 : J0, (sys ? W1 : W0).f.phi, col);
        step_mid_rest<NB, G, 32, FACT>(sys ? J1 : J0, sys ? W1 : W0, false, sys ? q1 : q0, col);
      } else {
        if (j0) split_vel_product<NB, G, WAVE, FACT>(J0, W0.f.phi, lane);
        step_mid_rest<NB, G, WAVE, FACT>(J0, W0, false, q0, lane);
        if (j1) split_vel_product<NB, G, WAVE, FACT>(J1, W1.f.phi, lane);
        step_mid_rest<NB, G, WAVE, FACT>(J1, W1, false, q1, lane);
      }
    } else {
      if (j0 || q0) {
        split_phi<NB, WAVE, FACT>(J0, W0, h0, q0, lane);
        wsync();
        if (j0) split_vel_product<NB, G, WAVE, FACT>(J0, W0.f.phi, lane);
        step_mid_rest<NB, G, WAVE, FACT>(J0, W0, false, q0, lane);
      }
      if (TWO && (j1 || q1)) {
        split_phi<NB, WAVE, FACT>(J1, W0, h1, q1, lane);
        wsync();
        if (j1) split_vel_product<NB, G, WAVE, FACT>(J1, W0.f.phi, lane);
        step_mid_rest<NB, G, WAVE, FACT>(J1, W0, false, q1, lane);
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
      step_post<NB, G, 32, FACT, false>(sys ? J1 : J0, W0, sys ? h1 : h0, false, sys ? q1 : q0, false, col);
      if (sys ? j1 : j0) split_drift<NB, G, 32, FACT>(sys ? J1 : J0, 0.5 * (sys ? h1 : h0), col);
    } else {
      step_post<NB, G, STEP, FACT, false>(J0, W0, h0, false, q0, false, lane);
      if (j0) split_drift<NB, G, WAVE, FACT>(J0, 0.5 * h0, lane);
      if constexpr (TWO) {
        step_post<NB, G, STEP, FACT, false>(J1, W0, h1, false, q1, false, lane);
        if (j1) split_drift<NB, G, WAVE, FACT>(J1, 0.5 * h1, lane);
      }
    }
    wsync();
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

// ---------------------------------------------------------------------------
// Three waves (few systems, SplitLds3): the Jacobian wave's work divided in
// two again.  The pair wave turns the ring's slots into pair Jacobians, builds
// Phi and carries dq/dt; the row wave follows with everything that touches J.
// Newton's iterations need the first two only.  Between them: a chunk's pair
// Jacobians in two buffers, Phi in one, a step's header and a transit's
// scalars in two of each.  Cycles a step of the two Jacobian parts as one
// wave: 299k at nine bodies (reference row update; 225k factored) and 64k at
// three, with 210k and 42k for the state's wave beside it; divided, the
// longest of the three is the state's or close to it.  80 gradient steps of
// nine bodies 10.4 -> 8.0 ms, 150 of six with three observables 19.4 -> 11.8.
// ---------------------------------------------------------------------------
struct RowHeader {
  int need, body;
  int64_t index;
  double h;
  double gd, dx, dy, dvx, dvy, ax, ay;  // a gradient step's end (split_gradient)
};
struct RowCtl {
  // counters (counter_reached), from COUNTER_START on
  uint32_t chunks, chunks_done;  // published / released, of all sweeps so far
  uint32_t phis, phis_done;
  uint32_t heads, heads_seen;    // steps announced / read
  uint32_t ends;                 // gradient steps whose scalars are written
  RowHeader hdr[2];
};

template <int NB, int LIMIT> struct SplitLds3 {
  static constexpr int NP = NB * (NB - 1) / 2, N3 = 3 * NB, N4 = 4 * NB, PQ = 13, NS = 1;
  static constexpr int RR = NP;  // a whole sweep's ring
  struct Phi {
    double phi[N3 * N4];
    double dadq[N3 * N4];
    double pq[NP * PQ];
  };
  struct Work {
    static constexpr int NP = SplitLds3::NP, PQ = SplitLds3::PQ;
    Phi f;
  };
  static constexpr size_t FIXED = sizeof(StateRec<NB>) + sizeof(JacRec<NB, false>) + sizeof(Work) + RR * sizeof(RingSlot) +
                                  sizeof(SplitCtl) + sizeof(RowCtl) + 64;
  static constexpr int FIT = (int)(((size_t)LIMIT - FIXED) / (2 * sizeof(JacSlot)));
  // pairs per chunk: half a sweep or less, so that the waves overlap
  static constexpr int CH0 = NP < 4 ? NP : (NP + 1) / 2 < 3 ? 3 : (NP + 1) / 2 > 18 ? 18 : (NP + 1) / 2;
  static constexpr int CH = CH0 < FIT ? CH0 : FIT;
  static_assert(FIXED < (size_t)LIMIT && CH >= (NB / 2 < 1 ? 1 : NB / 2), "a level of pairs must fit");
  StateRec<NB> t[1];
  JacRec<NB, false> j[1];
  Work w;
  JacSlot slot[2][CH];
  RingSlot ring[1][RR];
  SplitCtl ctl;
  RowCtl row;
};

template <int NB, int LIMIT, bool FACT>
__device__ __attribute__((always_inline)) inline bool pair_wave_sweep(SplitLds3<NB, LIMIT>& P, uint32_t& head, int& pos, uint32_t& chunk, int dir,
                                                                      double hh, int need, int lane, int64_t bound,
                                                                      unsigned long long* err) {
  using L = SplitLds3<NB, LIMIT>;
  constexpr int NL = level_count(NB);
  const bool needJ = (need & SPLIT_J) != 0, needQ = (need & SPLIT_Q) != 0;
  JacRec<NB, false>& S = P.j[0];
  int lev = 0;
  while (lev < NL) {
    const int lev0 = lev;
    int cnt = 0;
    while (lev < NL && cnt + level_width(NB, lev) <= L::CH) cnt += level_width(NB, lev++);
    if (!wait_for(&P.ctl.tail, head + cnt, &P.ctl, bound, err, lane)) return false;
    // the buffer the row wave used two chunks ago
    if (!wait_for(&P.row.chunks_done, chunk - 1, &P.ctl, bound, err, lane)) return false;
    JacSlot* slots = P.slot[chunk & 1];
    if (lane < cnt) {
      int at = pos + lane;
      if (at >= L::RR) at -= L::RR;
      const RingSlot* a = &P.ring[0][at];
      if (dir == 0) split_pair_jacobian<true>(lds_off(a), lds_off(slots + lane), S.m[a->i], S.m[a->j], hh, FACT);
      else split_pair_jacobian<false>(lds_off(a), lds_off(slots + lane), S.m[a->i], S.m[a->j], hh, FACT);
    }
    wsync();
    head += cnt;
    pos += cnt;
    if (pos >= L::RR) pos -= L::RR;
    publish(&P.ctl.head, head, lane);
    if (needJ) publish(&P.row.chunks, ++chunk, lane);
    if (needQ) split_rates<NB, FACT>(S, slots, cnt, lane);
  }
  return true;
}

template <int NB, int LIMIT, bool FACT>
__device__ void pair_wave(SplitLds3<NB, LIMIT>& P, const SysDesc& D, const SysBufs& B, const Visit& v, int lane, int64_t bound, unsigned long long* err) {
  constexpr int N3 = 3 * NB, N7 = 7 * NB;
  SplitCtl* ctl = &P.ctl;
  RowCtl* row = &P.row;
  JacRec<NB, false>& S = P.j[0];
  uint32_t seen = COUNTER_START, answered = COUNTER_START, head = COUNTER_START, chunk = COUNTER_START;
  uint32_t steps = COUNTER_START, ends = COUNTER_START;  // announced to the row wave; gradient steps' ends
  int pos = 0;
#pragma unroll 1
  while (true) {
    if (!wait_next(&ctl->sent, seen + 1, ctl, bound, err, lane)) return;
    const int need = __builtin_amdgcn_readfirstlane(ctl->act[0]);
    const bool needJ = need >= 0 && (need & SPLIT_J) != 0, needQ = need >= 0 && (need & SPLIT_Q) != 0;
    const double h = ctl->h[0];
    const int body = ctl->body[0];
    const int64_t index = ctl->index[0];
    if (needJ || need < 0) {
      if (!wait_for(&row->heads_seen, steps - 1, ctl, bound, err, lane)) return;
      RowHeader& H = row->hdr[steps & 1];
      if (lane == 0) {
        H.need = need;
        H.body = body;
        H.index = index;
        H.h = h;
      }
      wsync();
      publish(&row->heads, ++steps, lane);
    }
    if (need < 0) break;
    if (needQ)
      for (int q = lane; q < N3; q += WAVE) S.v[q] = S.mv[q];
    wsync();
    publish(&ctl->seen, ++seen, lane);
    step_pre<NB, false, WAVE, FACT, false>(S, P.w, h, false, needQ, false, lane);
    if (!pair_wave_sweep<NB, LIMIT, FACT>(P, head, pos, chunk, 0, 0.5 * h, need, lane, bound, err)) return;
    if (!wait_for(&ctl->sent, seen + 1, ctl, bound, err, lane)) return;
    for (int q = lane; q < N3; q += WAVE) S.x[q] = S.mx[q];
    wsync();
    publish(&ctl->seen, ++seen, lane);
    // Phi of the last step that had one for the row wave is used up
    if (!wait_for(&row->phis_done, needJ ? steps - 1 : steps, ctl, bound, err, lane)) return;
    split_phi<NB, WAVE, FACT>(S, P.w, h, needQ, lane);
    wsync();
    if (needJ) publish(&row->phis, steps, lane);
    step_mid_rest<NB, false, WAVE, FACT>(S, P.w, false, needQ, lane);
    if (!pair_wave_sweep<NB, LIMIT, FACT>(P, head, pos, chunk, 1, 0.5 * h, need, lane, bound, err)) return;
    if (!wait_for(&ctl->sent, seen + 1, ctl, bound, err, lane)) return;
    if (needQ)
      for (int q = lane; q < N3; q += WAVE) {
        S.x[q] = S.qx[q];
        S.v[q] = S.qv[q];
      }
    wsync();
    publish(&ctl->seen, ++seen, lane);
    step_post<NB, false, WAVE, FACT, false>(S, P.w, h, false, needQ, false, lane);
    publish(&ctl->answered, ++answered, lane);
    if (need & SPLIT_SAVE) {
      const int ti = D.ti, jb = body;
      RowHeader& H = row->hdr[(steps - 1) & 1];
      if (lane == 0) {
        H.gd = gdot<NB>(S, ti, jb);
        H.dx = S.x[3 * jb] - S.x[3 * ti];
        H.dy = S.x[3 * jb + 1] - S.x[3 * ti + 1];
        H.dvx = S.v[3 * jb] - S.v[3 * ti];
        H.dvy = S.v[3 * jb + 1] - S.v[3 * ti + 1];
        H.ax = S.dqdt[7 * jb + 3] - S.dqdt[7 * ti + 3];
        H.ay = S.dqdt[7 * jb + 4] - S.dqdt[7 * ti + 4];
      }
      wsync();
      publish(&row->ends, ++ends, lane);
    } else if ((need & 3) == ACT_MAIN && needQ) {
      for (int q = lane; q < N7; q += WAVE) S.run_dqdt[q] = S.dqdt[q];
      wsync();
    }
  }
}

template <int NB, int LIMIT, bool FACT>
__device__ void row_wave(SplitLds3<NB, LIMIT>& P, const SysDesc& D, const SysBufs& B, const Visit& v, int lane, int64_t bound, unsigned long long* err) {
  using L = SplitLds3<NB, LIMIT>;
  constexpr int NL = level_count(NB);
  SplitCtl* ctl = &P.ctl;
  RowCtl* row = &P.row;
  JacRec<NB, false>& S = P.j[0];
  uint32_t steps = COUNTER_START, ends = COUNTER_START, chunk = COUNTER_START;
#pragma unroll 1
  while (true) {
    if (!wait_next(&row->heads, steps + 1, ctl, bound, err, lane)) return;
    const RowHeader& H = row->hdr[steps & 1];
    const int need = __builtin_amdgcn_readfirstlane(H.need);
    if (need < 0) break;
    const double h = H.h;
    const int body = H.body;
    const int64_t index = H.index;
    ++steps;
    // the header stays until the step's gradient scalars are read from it
    if (!(need & SPLIT_SAVE)) publish(&row->heads_seen, steps, lane);
    if (D.mode == MODE_CARTESIAN) split_write_jac<NB>(S, D, B, index, lane);
    if (need & SPLIT_SAVE) split_keep_jac<NB>(S, B.ws + D.off_ws, false, lane);
    split_drift<NB, false, WAVE, FACT>(S, 0.5 * h, lane);
    wsync();
#pragma unroll 1
    for (int dir = 0; dir < 2; ++dir) {
      int lev = 0;
      while (lev < NL) {
        const int lev0 = lev;
        int cnt = 0;
        while (lev < NL && cnt + level_width(NB, lev) <= L::CH) cnt += level_width(NB, lev++);
        if (!wait_for(&row->chunks, chunk + 1, ctl, bound, err, lane)) return;
        split_rows<NB, false, WAVE, FACT>(S, P.slot[chunk & 1], dir, lev0, lev, lane);
        wsync();
        publish(&row->chunks_done, ++chunk, lane);
      }
      if (dir == 0) {
        if (!wait_for(&row->phis, steps, ctl, bound, err, lane)) return;
        split_vel_product<NB, false, WAVE, FACT>(S, P.w.f.phi, lane);
        wsync();
        publish(&row->phis_done, steps, lane);
      }
    }
    split_drift<NB, false, WAVE, FACT>(S, 0.5 * h, lane);
    wsync();
    if (need & SPLIT_SAVE) {
      if (!wait_for(&row->ends, ++ends, ctl, bound, err, lane)) return;
      const RowHeader G = H;
      split_gradient_rows<NB>(S, D, B, body, index, G.gd, G.dx, G.dy, G.dvx, G.dvy, G.ax, G.ay, lane);
      split_keep_jac<NB>(S, B.ws + D.off_ws, true, lane);
      wsync();
      publish(&row->heads_seen, steps, lane);
    }
  }
  if (v.begin <= D.nsteps) split_store_jac<NB, false>(S, D, B, lane);
}

// calc_dtdelements! (dtdelements) of a finished system, all NWV waves at work:
// wave w takes the transits w, w + NWV, ...; jac_init staged transposed in the
// Jacobian's store (the Jacobian is already stored).
template <int NB, int NWV, class L> __device__ void split_elements(L& P, int k, const SysDesc& D, const SysBufs& B, int wave, int lane) {
  constexpr int N7 = 7 * NB;
  const int n = NB, nb = D.ntbv;
  const auto jt = jj<NB>(P.j[k]);
  const double* jinit = B.jac + D.off_jac + 2 * (int64_t)N7 * N7;
  for (int col = lane; col < N7; col += WAVE)
    for (int cp = wave; cp < N7; cp += NWV) jt[(unsigned)(col + N7 * cp)] = jinit[cp + (int64_t)N7 * col];
  __syncthreads();
  const double* dq = B.dq + D.off_dq;
  double* del = B.del + D.off_del;
  const int64_t ntt = D.ntt;
  int turn = 0;
  for (int b = 0; b < nb; ++b)
    for (int i = 0; i < n; ++i) {
      const int64_t cnt = P.t[k].count[i] < ntt ? P.t[k].count[i] : ntt;
      for (int64_t t = 0; t < cnt; ++t) {
        const bool mine = turn == wave;
        turn = turn + 1 < NWV ? turn + 1 : 0;
        if (!mine) continue;
        for (int col = lane; col < N7; col += WAVE) {
          double acc = 0.0;
          for (int cp = 0; cp < N7; ++cp)
            acc = acc + dq[b + nb * ((int64_t)i + n * (t + ntt * cp))] * jt[(unsigned)(col + N7 * cp)];
          del[b + nb * ((int64_t)i + n * (t + ntt * col))] = acc;
        }
      }
    }
}

// Whether a run ever needs the Jacobian wave.
__device__ inline bool split_follows(const SysDesc& D) { return D.grad || D.mode == MODE_TRANSITS; }

// One visit of a system by a workgroup of three waves.
template <int NB, int LIMIT>
__device__ void split_run3(unsigned char* raw, int wave, const SysDesc& D, const SysBufs& B, int64_t chunk, int64_t bound, unsigned long long* err, int lane) {
  using L = SplitLds3<NB, LIMIT>;
  L& P = *reinterpret_cast<L*>(raw);
  static_assert(sizeof(L) <= (size_t)LIMIT, "LDS");
  const Visit v = visit_of(D, B, chunk), none{1, 1, 0};
  if (wave == 0) {
    split_load_state<NB>(P.t[0], D, B, lane);
    start_counters(P.ctl, lane);
    if (lane == 0) {
      RowCtl& r = P.row;
      r.chunks = r.chunks_done = r.phis = r.phis_done = r.heads = r.heads_seen = r.ends = COUNTER_START;
    }
  } else if (wave == 2) {
    split_load_jac<NB, false>(P.j[0], D, B, lane);
  }
  __syncthreads();
  if (wave == 0) {
    split_state<NB, false>(P, D, D, B, v, none, lane, bound, err);
  } else if (split_follows(D)) {
    if (wave == 1) {
      if (D.rowupd) pair_wave<NB, LIMIT, true>(P, D, B, v, lane, bound, err);
      else pair_wave<NB, LIMIT, false>(P, D, B, v, lane, bound, err);
    } else {
      if (D.rowupd) row_wave<NB, LIMIT, true>(P, D, B, v, lane, bound, err);
      else row_wave<NB, LIMIT, false>(P, D, B, v, lane, bound, err);
    }
  }
  __syncthreads();  // every row is written
  if (D.mode == MODE_TRANSITS && D.grad && v.begin <= D.nsteps && v.end == v.total) split_elements<NB, 3>(P, 0, D, B, wave, lane);
  __syncthreads();
}
template <int N, int HI, int LIMIT>
__device__ __forceinline__ void split_dispatch3(unsigned char* raw, int wave, const SysDesc& D, const SysBufs& B, int64_t chunk,
                                                int64_t bound, unsigned long long* err, int lane) {
  if constexpr (N <= HI) {
    if (D.n == N) {
      split_run3<N, LIMIT>(raw, wave, D, B, chunk, bound, err, lane);
      return;
    }
    split_dispatch3<N + 1, HI, LIMIT>(raw, wave, D, B, chunk, bound, err, lane);
  }
}

// One visit of a system, or of two of equal body count, by a workgroup of two
// waves.
template <int NB, bool G, bool TWO, int LIMIT>
__device__ void split_run(unsigned char* raw, int wave, const SysDesc& D0, const SysDesc& D1, const SysBufs& B, int64_t chunk0,
                          int64_t chunk1, bool pair, int64_t bound, unsigned long long* err, int lane) {
  using L = SplitLds<NB, G, TWO, LIMIT>;
  L& P = *reinterpret_cast<L*>(raw);
  const Visit v0 = visit_of(D0, B, chunk0);
  Visit v1 = visit_of(D1, B, chunk1);
  if (!pair) v1.begin = v1.end = v1.total + 1;  // no second system: as one that finished earlier
  if (wave == 0) {
    split_load_state<NB>(P.t[0], D0, B, lane);
    if (TWO) split_load_state<NB>(P.t[L::NS - 1], D1, B, lane);
    start_counters(P.ctl, lane);
  } else {
    split_load_jac<NB, G>(P.j[0], D0, B, lane);
    if (TWO) split_load_jac<NB, G>(P.j[L::NS - 1], D1, B, lane);
  }
  __syncthreads();
  if (wave == 0) {
    split_state<NB, TWO>(P, D0, D1, B, v0, v1, lane, bound, err);
  } else if (split_follows(D0) || (pair && split_follows(D1))) {
    if (D0.rowupd) split_jacobian<NB, G, TWO, LIMIT, true>(P, D0, D1, B, v0, v1, lane, bound, err);
    else split_jacobian<NB, G, TWO, LIMIT, false>(P, D0, D1, B, v0, v1, lane, bound, err);
  }
  __syncthreads();  // every row is written
  if (D0.mode == MODE_TRANSITS && D0.grad && v0.begin <= D0.nsteps && v0.end == v0.total)
    split_elements<NB, 2>(P, 0, D0, B, wave, lane);
  if (TWO && D1.mode == MODE_TRANSITS && D1.grad && v1.begin <= D1.nsteps && v1.end == v1.total)
    split_elements<NB, 2>(P, L::NS - 1, D1, B, wave, lane);
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
                                               const SysBufs& B, int64_t c0, int64_t c1, bool pair, int64_t bound,
                                               unsigned long long* err, int lane) {
  if constexpr (N <= HI) {
    if (D0.n == N) {
      split_run<N, split_global<N, TWO, LIMIT>(), TWO, LIMIT>(raw, wave, D0, D1, B, c0, c1, pair, bound, err, lane);
      return;
    }
    split_dispatch<N + 1, HI, TWO, LIMIT>(raw, wave, D0, D1, B, c0, c1, pair, bound, err, lane);
  }
}

// Persistent two-wave launch of bodies up to HI: like nbg_run (TWO: like
// nbg_run_duo, one unit of one or two systems at a time).  LIMIT: the
// workgroup's LDS.  units[13] collects wait failures.
template <int HI, bool TWO, int LIMIT, bool THREE = false>
__device__ __forceinline__ void split_body(unsigned char* raw, int* share, const GroupList& gl, const SysBufs& B, int64_t chunk,
                                           int64_t bound, unsigned long long* units,
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
    if constexpr (THREE) split_dispatch3<2, HI, LIMIT>(raw, wave, D0, B, c0, bound, err, lane);
    else split_dispatch<2, HI, TWO, LIMIT>(raw, wave, D0, D1, B, c0, c1, two, bound, err, lane);
    if (threadIdx.x == 0) {
      visit_done(D0, ints0, before0, tr00, it00, B, units);
      if (two) visit_done(D1, ints1, before1, tr01, it01, B, units);
    }
  }
}

}  // namespace nbg
