// Device parts of the barrier-free slot kernels (stream.hip: one wavenumber, sweep.hip: many):
// e^{ikr}, rule selection, the LDS of a workgroup, the hand-over of node sums between waves,
// mid-edge pairs and the tile loop.  The first two serve the derivative kernels (adjoint.hip)
// as well.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "bie_common.hpp"
#include "device_common.hpp"
#include "kernels_math.hpp"
#include "schedule.hpp"

namespace bie {
namespace {

typedef double d8 __attribute__((ext_vector_type(8), aligned(8)));

// The instance is read through the scalar cache where it is needed: fresh(p) keeps the
// compiler from holding its fields in scalar registers across the element loop (it spilled
// some eighty of them).
typedef const __attribute__((address_space(4))) StreamInst* InstPtr;
__device__ __forceinline__ InstPtr fresh(InstPtr p) {
  asm volatile("" : "+s"(p));
  return p;
}
__device__ __forceinline__ d8 sload8(const double* p) {
  return *reinterpret_cast<const __attribute__((address_space(4))) d8*>(
      reinterpret_cast<uintptr_t>(p));
}

__device__ __forceinline__ void lds_wait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

__device__ __forceinline__ unsigned lds_peek(const unsigned* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ unsigned lds_count(unsigned* p, unsigned v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_poke(unsigned* p, unsigned v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Whether this lane's bit of a wave-uniform mask is set (no lane number, no shift).
__device__ __forceinline__ bool lane_of_mask(unsigned long long m) {
  return __builtin_amdgcn_inverse_ballot_w64(m);
}
// The lane number, formed anew: what is computed from it is not kept in registers across the
// element loop (they are short, and a spilled one is a load that waits for column stores).
__device__ __forceinline__ int fresh_lane(int lane) {
  asm volatile("" : "+v"(lane));
  return lane;
}

// ---- one quadrature point ----------------------------------------------------------------

// a * k + c with the constant k in scalar and c in vector registers, and a * b + c, as one
// instruction whose destination is a register of its own (the compiler would copy c there
// first, one more instruction for each polynomial constant).
__device__ __forceinline__ double fma_k(double a, double k, double c) {
  double r;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(k), "v"(c));
  return r;
}
__device__ __forceinline__ double fma_v(double a, double b, double c) {
  double r;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// LDS tables of e^{ikr} and the polynomial constants that stay in vector registers.
struct Trig {
  const double2* cs;   // (cos, sin)(j pi / 64)
  const double* e2;    // 2^(j / 64)
  double s5, s3, c4;   // 1/120, -1/6, 1/24
};
__device__ __forceinline__ Trig make_trig(const double* t) {
  Trig tr{reinterpret_cast<const double2*>(t), t + kTrigDoubles, 1.0 / 120.0, -1.0 / 6.0,
          1.0 / 24.0};
  asm volatile("" : "+v"(tr.s5), "+v"(tr.s3), "+v"(tr.c4));
  return tr;
}

// e^{ikr} in two stages, so that the table entries are under way while the caller reads what
// it needs next: the argument reductions and table reads, then the polynomials.  FAST, for
// |x| < kTabFastMaxArg: sincos_tab without its branch; n = rint(64 x / pi) is formed by adding
// 1.5 * 2^52 to x * 64 / pi inside one fused multiply-add (the sum's unit in the last place is
// 1, so it is rounded to an integer there), the reduction uses n = sum - 1.5 * 2^52 (exact), and
// the table index n mod 128 is the low bits of the sum's mantissa (two's complement for negative
// n).  NaN and infinite x give NaN (the index is masked into the table whatever the bits are).  The damping e^{x}, x = -Im k r: x = (64 i + j) ln 2 / 64 + d with |d| <=
// ln 2 / 128, 2^(j/64) from the table, e^d by its Taylor polynomial to d^5 (truncation below
// 4e-17), the exponent by ldexp; arguments beyond the range of a double are clamped there.
template <bool CPLX, bool FAST>
struct Phase {
  double d, t0, t1, ed, et;
  int ei;
  __device__ __forceinline__ void begin(double krr, double kir, const Trig& tr) {
    constexpr double kShift = 6755399441055744.0;  // 1.5 * 2^52
    if (FAST) {
      constexpr double kInvStep = 20.371832715762602978;       // 64 / pi
      constexpr double kStepHi = 1.5707963267948965580 / 32;   // pi/2 rounded, / 32 (exact)
      constexpr double kStepLo = 6.1232339957367658e-17 / 32;  // its remainder, / 32 (exact)
      const double sh = fma(krr, kInvStep, kShift);
      const double n = sh - kShift;
      d = fma(-n, kStepHi, krr);
      d = fma(-n, kStepLo, d);
      const double2 t = tr.cs[__double2loint(sh) & (kTrigN - 1)];
      t0 = t.x;
      t1 = t.y;
    } else {
      sincos_tab(krr, tr.cs, &t1, &t0);
    }
    if (CPLX) {
      constexpr double kInv = 92.332482616893656977;   // 64 / ln 2
      constexpr double kHi = 0.010830424696249145255;  // ln 2 / 64 rounded
      constexpr double kLo = 3.6235102264711177e-19;   // its remainder
      const double x = fmin(fmax(-kir, -800.0), 800.0);
      const double sh = fma(x, kInv, kShift);
      const double n = sh - kShift;
      ei = __double2loint(sh);
      ed = fma(-n, kHi, x);
      ed = fma(-n, kLo, ed);
      et = tr.e2[ei & (kExpN - 1)];
    }
  }
  __device__ __forceinline__ void end(const Trig& tr, double& sn, double& cs, double& damp) {
    if (FAST) {
      const double d2 = d * d;
      const double sp = fma_v(d2, fma_k(d2, -1.0 / 5040.0, tr.s5), tr.s3);
      const double sd = fma(d * d2, sp, d);
      const double cp = fma(d2, fma_k(d2, -1.0 / 720.0, tr.c4), -0.5);
      const double cd = fma(d2, cp, 1.0);
      sn = fma(t1, cd, t0 * sd);
      cs = fma(t0, cd, -(t1 * sd));
    } else {
      sn = t1;
      cs = t0;
    }
    if (CPLX) {
      double p = fma_k(ed, 1.0 / 120.0, tr.c4);
      p = fma(ed, p, 1.0 / 6.0);
      p = fma(ed, p, 0.5);
      p = fma(ed * ed, p, ed);
      damp = ldexp(fma(et, p, et), ei >> 6);
    }
  }
};

// G = g e^{ikr}, F = t (ikr - 1) G with g = J w / (4 pi r) and t = n.d / r^2
// (greens3d!, freens3d!, kernels.jl:13-37).
template <bool CPLX, bool FAST>
__device__ __forceinline__ void kernels_end(const Phase<CPLX, FAST>& ph, double g, double t,
                                            double krr, double kir, const Trig& tr, double& Fr,
                                            double& Fi, double& Gr, double& Gi) {
  double sn, cs, damp;
  Phase<CPLX, FAST>(ph).end(tr, sn, cs, damp);
  if (CPLX) g *= damp;
  Gr = g * cs;
  Gi = g * sn;
  if (CPLX) {
    const double ar = -1.0 - kir;
    Fr = t * fma(ar, Gr, -krr * Gi);
    Fi = t * fma(ar, Gi, krr * Gr);
  } else {
    Fr = -t * fma(krr, Gi, Gr);
    Fi = t * fma(krr, Gr, -Gi);
  }
}

template <int NP, bool GON>
struct Sums {  // an element's node sums of one row
  double fr[NP], fi[NP], gr[GON ? NP : 1], gi[GON ? NP : 1];
  // adds basis value ph of a point, or (FIRST) begins the sums with it: no zeroing
  template <bool FIRST>
  __device__ __forceinline__ void add(int s, double ph, double Fr, double Fi, double Gr,
                                      double Gi) {
    fr[s] = FIRST ? Fr * ph : fma(Fr, ph, fr[s]);
    fi[s] = FIRST ? Fi * ph : fma(Fi, ph, fi[s]);
    if constexpr (GON) {
      gr[s] = FIRST ? Gr * ph : fma(Gr, ph, gr[s]);
      gi[s] = FIRST ? Gi * ph : fma(Gi, ph, gi[s]);
    }
  }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int s = 0; s < NP; ++s) {
      fr[s] = fi[s] = 0.0;
      if constexpr (GON) gr[s] = gi[s] = 0.0;
    }
  }
  __device__ __forceinline__ void keep(bool on) {  // zero where off
#pragma unroll
    for (int s = 0; s < NP; ++s) {
      fr[s] = on ? fr[s] : 0.0;
      fi[s] = on ? fi[s] : 0.0;
      if constexpr (GON) {
        gr[s] = on ? gr[s] : 0.0;
        gi[s] = on ? gi[s] : 0.0;
      }
    }
  }
};

// Rule of a pair as select_rule, from the element's NP selection nodes P; node(s, d) gives a
// coordinate for the exact comparison of near ties, hyp_of() its kind.
template <int NP, class Node, class HypOf>
__device__ __forceinline__ int select_rule_p(double x0, double x1, double x2,
                                             const double (&P)[NP][3], Node node, int R,
                                             HypOf hyp_of) {
  double d2v_[NP];
#pragma unroll
  for (int s = 0; s < NP; ++s) {
    const double dx = P[s][0] - x0, dy = P[s][1] - x1, dz = P[s][2] - x2;
    d2v_[s] = fma(dx, dx, fma(dy, dy, dz * dz));
  }
  double b = d2v_[0];
#pragma unroll
  for (int s = 1; s < NP; ++s) b = fmin(b, d2v_[s]);
  // Lanes with exactly one distance within 1e-12 of the smallest have their rule; the others
  // (near ties, zero spread, NaN: unordered distances count as near) compare exactly.  The
  // counting runs on lane masks in scalar registers.
  const double lim = b * (1.0 + 1e-12);
  unsigned long long one = 0, two = 0;
  int c = 1;
#pragma unroll
  for (int s = 0; s < NP; ++s) {
    const bool near = !(d2v_[s] > lim);
    const unsigned long long m = __ballot(near);
    two |= one & m;
    one |= m;
    if (s > 0) c = near ? s + 1 : c;
  }
  if (lane_of_mask(two)) {
    double best = INFINITY;
    c = 0;
    const int hyp = hyp_of();
#pragma unroll 1
    for (int s = 0; s < NP; ++s) {
      const double dx = node(s, 0) - x0, dy = node(s, 1) - x1, dz = node(s, 2) - x2;
      const double d = hyp ? scaled_hypot3_inline(dx, dy, dz) : julia_hypot3_inline(dx, dy, dz);
      if (d < best) {
        best = d;
        c = s + 1;
      }
    }
  }
  if (c < 1 || c > R) c = R;
  return c;
}

// The same with the nodes in scalar registers and at Pm in memory.
template <int NP>
__device__ __forceinline__ int select_rule_s(double x0, double x1, double x2,
                                             const double (&P)[NP][3], const double* Pm, int R,
                                             InstPtr in) {
  return select_rule_p<NP>(
      x0, x1, x2, P, [&](int s, int d) { return sload(Pm + 3 * s + d); }, R,
      [&] { return fresh(in)->a.hyp; });
}

// ---- LDS of a workgroup ------------------------------------------------------------------

// Offsets in doubles: slots, tables (basis or flat table, trig, 2^(j/64)), the waves' staged
// rows, 64 row sums of C, then 32-bit words: claims and turns of the slots, counters, and
// two queues of mid-edge pairs.
struct Layout {
  int tab, rows, csum, words, queue, total;
};
__host__ __device__ inline int stage_rows_doubles(int Qc, int rules) {
  return rules * (8 * Qc + 2);  // +2: the rules' rows start in different LDS banks
}
__host__ __device__ inline Layout layout_of(int S, int slot_doubles, int tab_doubles, int waves,
                                            int row_doubles, bool mids) {
  Layout l;
  l.tab = S * slot_doubles;
  l.rows = l.tab + tab_doubles + kTrigDoubles + kExpN;
  l.csum = l.rows + waves * row_doubles;
  l.words = l.csum + 64;
  l.queue = l.words + S + 4;  // 2 S slot words and 8 counters
  l.total = l.queue + (mids ? kStreamMid : 0);
  return l;
}

// How a pair finds its points: flat elements, rows staged in LDS, rows read from memory.
enum { kFlat = 0, kStaged = 1, kRead = 2 };
// after the slot words (kMidN: two; kFailed: a wait of the tile gave up; kPolls: when it does)
enum { kTicket = 0, kTile = 1, kMidN = 2, kFailed = 4, kPolls = 5 };

// Adds v to an LDS counter from one lane; the value before, in every lane.  (Written out: the
// compiler makes a wave-aggregated atomic of it, with a count over the lanes.)
__device__ __forceinline__ unsigned lds_draw(unsigned* p, unsigned v, int lane) {
  const unsigned at =
      (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned*)(p);
  unsigned t = 0;
  if (lane == 0)
    asm volatile("ds_add_rtn_u32 %0, %1, %2\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(t)
                 : "v"(at), "v"(v)
                 : "memory");
  return __builtin_amdgcn_readfirstlane(t);
}

// ---- hand-over of an element's node sums -------------------------------------------------

// 64 rows of a column from `col` (the same in every lane) on, lane's at byte offset `at`.
__device__ __forceinline__ void column_store(double* col, unsigned at, bool shared, double re,
                                             double im) {
  double* x = reinterpret_cast<double*>(reinterpret_cast<char*>(col) + at);
  if (shared) {
    unsafeAtomicAdd(x, re);
    unsafeAtomicAdd(x + 1, im);
  } else {
    __builtin_nontemporal_store(d2v{re, im}, reinterpret_cast<d2v*>(x));
  }
}

// Waits until ready() holds in every lane, at most so many polls (from ctr): then, or once another
// wave of the tile has given up, false.  A wave that gave up neither claims, nor adds, nor frees a
// slot any more for what it waited for: its nodes are then never complete, and whoever was to
// write their columns, or this wave, writes NaN.
template <class P>
__device__ __forceinline__ bool spin(unsigned* ctr, P ready) {
  bool done = !__any(!ready());
  if (!done) {
    const unsigned polls = lds_peek(ctr + kPolls);
#pragma unroll 1
    for (unsigned n = 0; n < polls && !done; ++n) {
      if (lds_peek(ctr + kFailed) != 0) break;
      __builtin_amdgcn_s_sleep(1);
      done = !__any(!ready());
    }
    if (!done) lds_poke(ctr + kFailed, 1u);
  }
  asm volatile("" ::: "memory");  // what follows is read after what was waited for
  return done;
}

struct Roles {
  unsigned long long first, more, last, direct;
};

// Lane s < NP speaks for node s: claims its place among the node's contributions.
// claims[slot] counts claims (low half) and finished contributions (high half).  The slots
// must be free for these nodes before any place is claimed: then a wave that holds a place
// never waits for one that waits for a slot.
template <int NP>
__device__ __forceinline__ Roles claim(const int4& en, int lane, unsigned* claims,
                                       const unsigned* turns, unsigned* ctr, bool& ok) {
  const bool slotted = lane < NP && en.x >= 0;
  // A SIMD issues for its oldest wave first; left alone, some waves run far ahead and then
  // wait here for the others.  A wave that has to wait gives way, one that need not is behind.
  if (__any(slotted && lds_peek(turns + en.x) != (unsigned)en.z))
    __builtin_amdgcn_s_setprio(0);
  else
    __builtin_amdgcn_s_setprio(2);
  ok = spin(ctr, [&] { return !slotted || lds_peek(turns + en.x) == (unsigned)en.z; });
  const bool mine = slotted && ok;
  unsigned old = 0;
  if (mine) old = lds_count(claims + en.x, 1u) & 0xffffu;
  Roles r;
  r.first = __ballot(mine && old == 0);
  r.last = __ballot(mine && old == (unsigned)en.y - 1u);
  r.more = __ballot(mine && old != 0 && old != (unsigned)en.y - 1u);
  r.direct = __ballot(lane < NP && !mine);  // (not ok: NaN to all of them)
  return r;
}

// ---- mid-edge pairs ----------------------------------------------------------------------
// Pairs with a mid-edge split rule (quadrature.jl:117-144), about 1 % of the pairs of
// quadratic meshes: the tiles list them (in LDS, then in memory), a kernel after the dense
// one integrates them and adds them to F, G and C.  They lie where rows and elements are
// close to each other, in few tiles: integrated by their own tile at its end they took as
// long as a quarter of the whole kernel, spread over the chip they are a few per cent.  Four
// lanes share a pair (points q, q + 4, ...), so that the re and im parts of an entry leave in
// one request; the surface is evaluated from the element's six nodes (one round trip of
// loads; tabulated rows would cost one for every point).

__device__ __forceinline__ double quad_swap1(double x) {  // the value of lane ^ 1
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(x), 0xB1, 0xf, 0xf, true),
                          __builtin_amdgcn_mov_dpp(__double2loint(x), 0xB1, 0xf, 0xf, true));
}
__device__ __forceinline__ double quad_swap2(double x) {  // the value of lane ^ 2
  return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(x), 0x4E, 0xf, 0xf, true),
                          __builtin_amdgcn_mov_dpp(__double2loint(x), 0x4E, 0xf, 0xf, true));
}

// What a mid-edge pair is integrated for: one wavenumber's matrices, or (TAY) the k-derivative
// of an order (sweep.hip).
struct MidOut {
  double kr, ki;
  double *F, *G;
  bool sum_c;
  int order;
};

template <bool CPLX, bool GON, bool FAST, bool TAY>
__device__ __forceinline__ void mid_pair_add(InstPtr in, const MidOut& o, int64_t i, int e, int c,
                                             int lane, const double* mid_tab, const Trig& tr) {
  const int sub = lane & 3;
  const int Qm = in->a.len[3];
  const double kr = o.kr, ki = o.ki;
  const double* x = in->a.targets + 3 * i;
  const double x0 = x[0], x1 = x[1], x2 = x[2];
  double X[6][3];
#pragma unroll
  for (int g = 0; g < 6; ++g) {
    const double* p = in->coords + 3 * (size_t)in->topo[(size_t)e * 6 + g];
#pragma unroll
    for (int d = 0; d < 3; ++d) X[g][d] = p[d];
  }
  Sums<6, GON> v;
  v.clear();
  double csum = 0.0;
  const double* pt = mid_tab + (size_t)(c - 3) * Qm * 3;
#pragma unroll 1
  for (int q = sub; q < Qm; q += 4) {
    const double u = pt[3 * q], w = pt[3 * q + 2], vv = pt[3 * q + 1];
    const double l = 1.0 - u - vv;
    const double l2 = 2.0 * l - 1.0, u2 = 2.0 * u - 1.0, v2 = 2.0 * vv - 1.0;
    double N[6] = {l * l2, u * u2, vv * v2, 4.0 * u * l, 4.0 * u * vv, 4.0 * vv * l};
    const double e0 = 1.0 - 4.0 * l, eu = 4.0 * u - 1.0, ev = 4.0 * vv - 1.0;
    double d[3], tu[3], tv[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      d[k] = fma(N[5], X[5][k], fma(N[4], X[4][k], fma(N[3], X[3][k],
             fma(N[2], X[2][k], fma(N[1], X[1][k], N[0] * X[0][k])))));
      const double t0 = e0 * X[0][k];
      tu[k] = fma(eu, X[1][k], fma(4.0 * (l - u), X[3][k], fma(4.0 * vv, X[4][k] - X[5][k], t0)));
      tv[k] = fma(ev, X[2][k], fma(4.0 * (l - vv), X[5][k], fma(4.0 * u, X[4][k] - X[3][k], t0)));
    }
    const double dx = d[0] - x0, dy = d[1] - x1, dz = d[2] - x2;
    const double c0 = tu[2] * tv[1] - tu[1] * tv[2], c1 = tu[0] * tv[2] - tu[2] * tv[0],
                 c2 = tu[1] * tv[0] - tu[0] * tv[1];  // n J
    const double J2 = fma(c0, c0, fma(c1, c1, c2 * c2));
    // n = -c / J is not a number where J is 0 or infinite: F and C are NaN there
    const bool normal = J2 > 0.0 && J2 < INFINITY;
    const double J = normal ? J2 * rsqrt_nr(J2) : J2;
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    const double rinv = rsqrt_nr(r2);
    const double r = r2 * rinv;
    const double krr = kr * r, kir = CPLX ? ki * r : 0.0;
    Phase<CPLX, FAST> ph;
    ph.begin(krr, kir, tr);
    const double nd = normal ? fma(c0, dx, fma(c1, dy, c2 * dz)) : NAN;
    const double g = w * rinv, t = (nd * rinv) * rinv;
    csum = fma(-t, g, csum);
    double Fr, Fi, Gr, Gi;
    if constexpr (TAY) {  // G = r^m g e^{ikr}, F = t (ikr - 1 + m) G, both times i^m below
      double sn, cs, damp, gm = g, rb = r;
      ph.end(tr, sn, cs, damp);
      if (CPLX) gm *= damp;
      for (int m = o.order; m != 0; m >>= 1) {
        if (m & 1) gm *= rb;
        rb *= rb;
      }
      Gr = gm * cs;
      Gi = gm * sn;
      const double am = (double)(o.order - 1) - kir;
      Fr = t * fma(am, Gr, -krr * Gi);
      Fi = t * fma(am, Gi, krr * Gr);
    } else {
      kernels_end<CPLX, FAST>(ph, g, t, krr, kir, tr, Fr, Fi, Gr, Gi);
    }
    Gr *= J;
    Gi *= J;
    if (!in->own_basis) {
      const double* b = in->a.phi + ((size_t)c * in->a.Qmax + q) * 6;
#pragma unroll
      for (int s = 0; s < 6; ++s) N[s] = b[s];
    }
#pragma unroll
    for (int s = 0; s < 6; ++s) v.template add<false>(s, N[s], Fr, Fi, Gr, Gi);
  }
  // sums over the four lanes, each left with one component: F or G (sub / 2), re or im
  const bool hi = (sub & 2) != 0, odd = (sub & 1) != 0;
  const bool out = GON ? (hi || (in->a.flags & BIE_F)) : (!hi && (in->a.flags & BIE_F));
  const int64_t M = in->a.M;
  double* X0 = (hi ? o.G : o.F) + 2 * i + (odd ? 1 : 0);
#pragma unroll
  for (int s = 0; s < 6; ++s) {
    double re = v.fr[s], im = v.fi[s];
    if constexpr (GON) {
      const double gr = v.gr[s], gi = v.gi[s];
      const double tr_ = quad_swap2(hi ? re : gr), ti_ = quad_swap2(hi ? im : gi);
      re = (hi ? gr : re) + tr_;
      im = (hi ? gi : im) + ti_;
    } else {
      re += quad_swap2(re);
      im += quad_swap2(im);
    }
    if constexpr (TAY) {  // times i^m
      if (o.order & 1) {
        const double x1_ = -im;
        im = re;
        re = x1_;
      }
      if (o.order & 2) {
        re = -re;
        im = -im;
      }
    }
    const double other = quad_swap1(odd ? re : im);
    const double mine = (odd ? im : re) + other;
    if (out) unsafeAtomicAdd(X0 + 2 * (size_t)in->a.ptopo[(size_t)e * 6 + s] * (size_t)M, mine);
  }
  csum += quad_swap2(csum);
  csum += quad_swap1(csum);
  if (sub == 0 && o.sum_c) unsafeAtomicAdd(in->a.C + 2 * i, csum);
}

// Listed pairs (queue[0 .. count)), then the tiles whose pairs found no room in the lists:
// those select their pairs again and take them as they come, each tile's elements divided among
// as many waves as there are for it.  (1280 elements with dimpled edges, 2600 targets at their
// centre, every pair a mid-edge one: 887 us, 5380 with all waves on one tile after the other.)
template <bool CPLX, bool GON, bool FAST, bool TAY>
__device__ __forceinline__ void mid_pairs(InstPtr in, const MidOut& o, const double* mid_tab, const Trig& tr,
                                          int first_wave, int waves, int lane) {
  // entries up to the first tile that found no room: mid_count[2] holds where, if any
  const int n = (int)min(sload(in->mid_count), sload(in->mid_count + 2));
  for (int t = first_wave; t * 16 < n; t += waves) {
    const int at = t * 16 + (lane >> 2);
    if (at < n) {
      const int2 q = in->mid_queue[at];
      mid_pair_add<CPLX, GON, FAST, TAY>(in, o, q.x, q.y & 0x0fffffff, 3 + (int)((unsigned)q.y >> 28),
                                    lane, mid_tab, tr);
    }
  }
  const int n_tiles = (int)sload(in->mid_count + 1);
  if (n_tiles == 0) return;
  const int share = max(1, waves / n_tiles);  // waves to a tile, or a wave to several
  for (int k = first_wave / share; k < n_tiles; k += max(1, waves / share)) {
    const int2 tile = in->mid_tiles[k];
    const int64_t i0 = (int64_t)tile.x * 64;
    const int t1 = in->seg_begin[tile.y + 1];
    for (int t = in->seg_begin[tile.y] + first_wave % share; t < t1; t += share) {
      const double* x = in->a.targets + 3 * min(i0 + lane, in->a.M - 1);
      const int e = in->order[t];
      const int cl = select_rule<6>(x[0], x[1], x[2], in->a.selnodes + (size_t)e * 24, in->a.R,
                                    in->a.hyp) - 1;
      unsigned long long left = __ballot(i0 + lane < in->a.M && cl >= 3);
      while (left) {
        unsigned long long m = left;
        for (int j = 0; j < (lane >> 2); ++j) m &= m - 1;
        const int from = m ? __ffsll((long long)m) - 1 : 0;
        const int c = __shfl(cl, from);
        if (m) mid_pair_add<CPLX, GON, FAST, TAY>(in, o, i0 + from, e, c, lane, mid_tab, tr);
        for (int j = 0; j < 16; ++j) left &= left - 1;
      }
    }
  }
}

// One wave moves a finished tile's pairs from its LDS queue to the list in memory.
__device__ __forceinline__ void list_mid_pairs(InstPtr in, int rb, int seg, unsigned n,
                                               const unsigned* queue, int lane) {
  if (n == 0) return;
  unsigned at = 0xffffffffu;
  if (lane == 0) {
    const unsigned cap = in->mid_cap;
    if (n <= (unsigned)kStreamMid &&
        __hip_atomic_load(in->mid_count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < cap) {
      at = atomicAdd(in->mid_count, n);
      if (at + n > cap) {  // the list ends here: what follows belongs to no tile
        atomicMin(in->mid_count + 2, at);
        at = 0xffffffffu;
      }
    }
    if (at == 0xffffffffu)
      in->mid_tiles[atomicAdd(in->mid_count + 1, 1u)] = make_int2(rb, seg);
  }
  at = __builtin_amdgcn_readfirstlane(at);
  if (at == 0xffffffffu) return;
  const int p0 = sload(in->seg_begin + seg);
  for (unsigned t = lane; t < n; t += 64) {
    const unsigned q = queue[t];
    in->mid_queue[at + t] = make_int2(rb * 64 + (int)(q & 63u),
                                      in->order[p0 + (int)(q >> 8)] |
                                          (int)(((q >> 6) & 3u) << 28));
  }
}

// ---- the tile loop -----------------------------------------------------------------------

// Tiles in turn: a workgroup begins with the tile of its own number and draws the next one
// from a counter while it works (the answer is there when it is needed).  Two LDS-only
// barriers lie between tiles; nothing waits for the column stores.  inst_of(tile, rb, seg)
// names the instance, row block and segment of a tile, kmax_of(in, tile) its largest |k|,
// first_of(in, tile) whether it forms C and lists mid-edge pairs, body(in, rb, seg, tile,
// parity) does its work.  SD: doubles of a slot.
template <int SD, int W, bool MIDS, bool FAST, class InstOf, class KmaxOf, class FirstOf,
          class Body>
__device__ __forceinline__ void stream_run(InstOf inst_of, KmaxOf kmax_of, FirstOf first_of,
                                           Body body, int n_tiles, const StreamRun& run) {
  extern __shared__ double lds[];
  const int S = run.S;
  const Layout L = layout_of(S, SD, run.tab_doubles, W, run.row_doubles, run.mids != 0);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  unsigned* words = reinterpret_cast<unsigned*>(lds + L.words);
  unsigned* ctr = words + 2 * S;
  const unsigned* queue = reinterpret_cast<const unsigned*>(lds + L.queue);
  const int total = FAST ? n_tiles : (int)sload(run.counters + kSlowCount);
  int next = blockIdx.x;
  if (next >= total) return;
  const int ntab = run.tab_doubles + kTrigDoubles + kExpN;
  for (int t = threadIdx.x; t < ntab; t += 64 * W) lds[L.tab + t] = run.tab[t];
  if (threadIdx.x < 64) lds[L.csum + threadIdx.x] = 0.0;
  if (threadIdx.x == 0) ctr[kPolls] = (unsigned)run.polls;
  int parity = 0, prev = -1;
  for (;;) {
    // between the barriers nobody works on a tile
    for (int t = threadIdx.x; t < 2 * S; t += 64 * W) words[t] = 0u;  // claims and turns
    if (threadIdx.x == 0) {
      ctr[kTicket] = 0u;
      ctr[kFailed] = 0u;
      ctr[kMidN + parity] = 0u;
    }
    int rb, seg;
    if (prev >= 0 && wave == W - 1) {
      const InstPtr in = inst_of(prev, rb, seg);
      if ((in->a.flags & BIE_C) && first_of(in, prev)) {  // the row sums of C
        const int64_t i = (int64_t)rb * 64 + lane;
        if (i < in->a.M) unsafeAtomicAdd(in->a.C + 2 * i, lds[L.csum + lane]);
        lds[L.csum + lane] = 0.0;
      }
    }
    lds_barrier();
    if constexpr (MIDS)
      if (run.mids && prev >= 0 && wave == W - 1) {
        const InstPtr in = inst_of(prev, rb, seg);
        list_mid_pairs(in, rb, seg, ctr[kMidN + (parity ^ 1)],
                       queue + (parity ^ 1) * kStreamMid, lane);
      }
    if (next >= total) break;
    const int tile = FAST ? next : sload(run.slow + next);
    unsigned drawn = 0;
    if (threadIdx.x == 0 && total > (int)gridDim.x)
      drawn = atomicAdd(run.counters + (FAST ? 0 : kSlowNext), 1u);
    const InstPtr in = inst_of(tile, rb, seg);
    bool skip = false;
    if constexpr (FAST) {
      const double* x = in->a.targets + 3 * min((int64_t)rb * 64 + lane, in->a.M - 1);
      const double cx = x[0] - in->center[0], cy = x[1] - in->center[1], cz = x[2] - in->center[2];
      const double dist = sqrt(fma(cx, cx, fma(cy, cy, cz * cz))) + in->reach;
      // (both bounds at once, as a sum)
      constexpr double kPerDist = 0.5 * kTabFastMaxArg / kFastMaxDist;
      const double far = fma(kmax_of(in, tile), dist, kPerDist * dist);
      skip = run.slow && __any(!(far < 0.5 * kTabFastMaxArg));
      if (skip && threadIdx.x == 0) run.slow[atomicAdd(run.counters + kSlowCount, 1u)] = tile;
    }
    if (!skip) body(in, rb, seg, tile, parity);
    if (threadIdx.x == 0) ctr[kTile] = gridDim.x + drawn;
    lds_barrier();
    next = total > (int)gridDim.x ? (int)__builtin_amdgcn_readfirstlane(ctr[kTile]) : total;
    prev = skip ? -1 : tile;
    parity ^= 1;
  }
}

}  // namespace
}  // namespace bie
