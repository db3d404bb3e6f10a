// Batched frequency sweep: dense F_k, G_k for a list of real wavenumbers k_0..k_{nk-1}
// on one mesh, and the k-derivatives of F and G at one wavenumber (taylor_assemble!,
// src/3d/rosebem.jl:56-157), in one launch per kernel (graph-capturable: no host
// synchronisation, no memset nodes).  The reference has no batched path: it calls
// assemble_parallel! once per k.
//
// The kernel is the stream kernel (stream.hip) with KB matrices at once: tiles are (block of
// KB wavenumbers or orders, segment, 64 rows), an LDS slot holds KB node sums of 64 rows.
// What does not depend on the matrix is formed once per pair or point: rule selection, y - x,
// 1/r, the C integrand (first block only).  Four matrices of F and G (eight of F alone, two
// and four with six-node physics) are 96 registers of sums; eight waves per CU (two per SIMD,
// 256 VGPRs) hold them (eight of F alone on flat elements spill 20 registers; with twelve waves,
// 168 VGPRs, all spilled: 11.9 ms and 10.9 ms where eight take 11.8 and 5.7 for 16 wavenumbers
// and 26 orders on 4002 nodes).  A slot of 8 KB leaves 17 of them, which the surface's segments
// have to fit (44 for 8000 elements).
//   * Uniformly spaced k: e^{i k_b r} = e^{i k_0 r} (e^{i dk r})^b, two sincos per point and
//     one complex product per further k; other blocks form each e^{i k_b r}.  The kernel
//     finds out for every block, so any list of k is exact.
//   * k-derivatives: G_m = (i r)^m G, F_m = (i k r - 1 + m) (n.d / r^2) G_m.  On a flat
//     element n.d is a constant of the pair, and with A_j = sum N (i r)^j e^{ikr} J w / 4 pi r
//     F_m = -(n.d) [k A_{m-1} + (m - 1) A_{m-2}], G_m = A_m:
//     one sequence of sums (two products and six multiply-adds per point and order) gives
//     both.
// 16 wavenumbers on 4002 nodes, 16 points: 17.0 -> 11.5 ms (VALU busy 83 % of the time, 134
// instructions per point and four wavenumbers); 26 orders of F, four points: 8.7 -> 4.9 ms (75 %).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "bie_common.hpp"
#include "stream_device.hpp"

namespace bie {
namespace {

// Shape of a kernel: matrices of a block, waves of a workgroup, doubles of a slot.  F alone of
// the k-derivatives on flat elements (`lean`) keeps sums for one order more than its block and no
// others: twelve waves of 168 registers take six orders (14 registers spill, 25 with complex k),
// and its short rules need the waves (few points a pair: half of the time is the hand-over).  26
// orders on 4002 nodes, four points: 4.99 ms; eight orders and eight waves 5.69, four and sixteen
// 5.43.
struct SweepShape {
  int kb, waves, slot;
};
__host__ __device__ constexpr SweepShape sweep_shape(int NP, bool gon, bool lean,
                                                     bool fast = true) {
  return lean ? SweepShape{6, fast ? 12 : kSlowWaves, 6 * 128}
              : SweepShape{(NP == 6 ? 2 : 4) * (gon ? 1 : 2), 8, (NP == 6 ? 2 : 4) * 256};
}

typedef const __attribute__((address_space(4))) SweepArgs* SweepPtr;

template <int NP, int KB, bool GON>
struct Multi {  // an element's node sums of one row, KB matrices
  double fr[KB][NP], fi[KB][NP], gr[GON ? KB : 1][GON ? NP : 1], gi[GON ? KB : 1][GON ? NP : 1];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int s = 0; s < NP; ++s) {
        fr[b][s] = fi[b][s] = 0.0;
        if constexpr (GON) gr[b][s] = gi[b][s] = 0.0;
      }
  }
  template <class Fn>
  __device__ __forceinline__ void each(Fn fn) {
#pragma unroll
    for (int b = 0; b < KB; ++b)
#pragma unroll
      for (int s = 0; s < NP; ++s) {
        fn(b, fr[b][s], fi[b][s]);
        if constexpr (GON) fn(b, gr[b][s], gi[b][s]);
      }
  }
};

template <bool FIRST>
__device__ __forceinline__ void plus(double& x, double v, double w) {
  x = FIRST ? v * w : fma(v, w, x);
}

// x + iy times i^m.
__device__ __forceinline__ void rotate(int m, double& x, double& y) {
  if (m & 1) {
    const double t = -y;
    y = x;
    x = t;
  }
  if (m & 2) {
    x = -x;
    y = -y;
  }
}

// A block's wavenumbers.
template <int KB>
struct Block {
  double k[KB], dk;
};

// One point of a flat element: K <= KB wavenumbers; the sums leave out J (of G) and n.d J (of
// F).  H = G / r^2 runs through the wavenumbers; not FAST: H = G, and F takes n.d J / r^2 here
// (as point_flat in stream.hip).
template <int KB, int K, bool GON, bool FAST, bool REC, bool FIRST>
__device__ __forceinline__ void sweep_point_flat(const double (&d0)[3], const double (&a)[3],
                                                 const double (&b)[3], double (&n)[4],
                                                 const double* next, const Block<KB>& kv,
                                                 double nd, const Trig& tr, Multi<3, KB, GON>& v,
                                                 double& c3) {
  const double m[4] = {n[0], n[1], n[2], n[3]};
#pragma unroll
  for (int s = 0; s < 4; ++s) n[s] = next[s];
  __builtin_amdgcn_sched_barrier(0);
  const double dx = fma(m[2], b[0], fma(m[1], a[0], d0[0]));
  const double dy = fma(m[2], b[1], fma(m[1], a[1], d0[1]));
  const double dz = fma(m[2], b[2], fma(m[1], a[2], d0[2]));
  const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
  const double rinv = rsqrt_nr(r2);
  const double r = r2 * rinv;
  Phase<false, FAST> e0, e1;
  e0.begin(kv.k[0] * r, 0.0, tr);
  if (REC) e1.begin(kv.dk * r, 0.0, tr);
  const double h = FAST ? (m[3] * rinv) * (rinv * rinv) : m[3] * rinv;
  const double t = FAST ? 1.0 : (nd * rinv) * rinv;
  if constexpr (FAST)
    c3 = FIRST ? h : c3 + h;
  else
    c3 = FIRST ? t * h : fma(t, h, c3);
  double w[3];
  if constexpr (GON) {
#pragma unroll
    for (int s = 0; s < 3; ++s) w[s] = FAST ? m[s] * r2 : m[s];
  }
  double sn, cs, zs = 0.0, zc = 0.0, damp;
  e0.end(tr, sn, cs, damp);
  if (REC) e1.end(tr, zs, zc, damp);
  double Hr = h * cs, Hi = h * sn;
#pragma unroll
  for (int q = 0; q < K; ++q) {
    if (q > 0) {
      if (REC) {
        const double c2 = fma(Hr, zc, -(Hi * zs));
        Hi = fma(Hr, zs, Hi * zc);
        Hr = c2;
      } else {
        Phase<false, FAST> e;
        e.begin(kv.k[q] * r, 0.0, tr);
        e.end(tr, sn, cs, damp);
        Hr = h * cs;
        Hi = h * sn;
      }
    }
    const double krr = kv.k[q] * r;
    double Fr = fma(-krr, Hi, -Hr), Fi = fma(krr, Hr, -Hi);
    if constexpr (!FAST) {
      Fr *= t;
      Fi *= t;
    }
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      plus<FIRST>(v.fr[q][s], Fr, m[s]);
      plus<FIRST>(v.fi[q][s], Fi, m[s]);
      if constexpr (GON) {
        plus<FIRST>(v.gr[q][s], Hr, w[s]);
        plus<FIRST>(v.gi[q][s], Hi, w[s]);
      }
    }
  }
}

template <int KB, int K, bool GON, bool FAST, bool REC>
__device__ __forceinline__ void sweep_pair_flat(const double (&d0)[3], const double (&a)[3],
                                                const double (&b)[3], const double* tab, int Q,
                                                const Block<KB>& kv, double nd, const Trig& tr,
                                                Multi<3, KB, GON>& v, double& c3) {
  double n[4] = {tab[0], tab[1], tab[2], tab[3]};
  sweep_point_flat<KB, K, GON, FAST, REC, true>(d0, a, b, n, tab += 4, kv, nd, tr, v, c3);
#pragma unroll 1
  for (int q = 1; q < Q; ++q)
    sweep_point_flat<KB, K, GON, FAST, REC, false>(d0, a, b, n, tab += 4, kv, nd, tr, v, c3);
}

// A pair on a flat element (d0 = X1 - x, edges a and b, n.d J, J) whose lengths may be anywhere
// in the range, in units of a power of two s near the largest of them (exactly), so that the
// derivatives' 1 / r^3 is formed near 1: k r is k s r then, n.d J w / r^3 and J w / r are what
// they were, and r^m is in units of s^m.  The exponent of s.
__device__ __forceinline__ int pair_unit(double (&d0)[3], double (&a)[3], double (&b)[3],
                                         double& nd, double& J, double& s) {
  double m = 0.0;
#pragma unroll
  for (int d = 0; d < 3; ++d) m = fmax(m, fmax(fabs(d0[d]), fmax(fabs(a[d]), fabs(b[d]))));
  int e = 0;
  if (m > 0.0 && m < INFINITY) (void)frexp(m, &e);
  e = max(-1000, min(1000, e));
  s = ldexp(1.0, e);
  const double u = ldexp(1.0, -e);
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    d0[d] *= u;
    a[d] *= u;
    b[d] *= u;
  }
  nd = ((nd * u) * u) * u;
  J *= u;
  return e;
}

// One point of a flat element for the derivative orders m0 .. m0 + K - 1 (m0 even): sums of N r^j e^{ikr} w / (4 pi r), j = m0 - 2 .., without the factors i^j.
template <int NA, bool CPLX, bool FAST>
__device__ __forceinline__ void taylor_point_flat(const double (&d0)[3], const double (&a)[3],
                                                  const double (&b)[3], double (&n)[4],
                                                  const double* next, double kr, double ki, double unit,
                                                  int m0, const Trig& tr, double (&ac)[NA][3],
                                                  double (&as)[NA][3], double& c3) {
  const double m[4] = {n[0], n[1], n[2], n[3]};
#pragma unroll
  for (int s = 0; s < 4; ++s) n[s] = next[s];
  __builtin_amdgcn_sched_barrier(0);
  const double dx = fma(m[2], b[0], fma(m[1], a[0], d0[0]));
  const double dy = fma(m[2], b[1], fma(m[1], a[1], d0[1]));
  const double dz = fma(m[2], b[2], fma(m[1], a[2], d0[2]));
  const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
  const double rinv = rsqrt_nr(r2);
  const double r = r2 * rinv;
  const double ru = FAST ? r : r * unit;  // (see pair_unit)
  Phase<CPLX, FAST> e;
  e.begin(kr * ru, CPLX ? ki * ru : 0.0, tr);
  double q = m[3] * rinv;
  if (m0 == 0) {
    q *= rinv * rinv;
    c3 += q;
  } else {  // r^(m0 - 2): even, by binary powering
    double p = r2;
    for (int x = (m0 - 2) >> 1; x != 0; x >>= 1) {
      if (x & 1) q *= p;
      p *= p;
    }
  }
  double sn, cs, damp;
  e.end(tr, sn, cs, damp);
  if (CPLX) q *= damp;
  double C = q * cs, S = q * sn;
#pragma unroll
  for (int j = 0; j < NA; ++j) {
    if (j > 0) {
      C *= r;
      S *= r;
    }
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      ac[j][s] = fma(C, m[s], ac[j][s]);
      as[j][s] = fma(S, m[s], as[j][s]);
    }
  }
}

template <int KB, bool CPLX, bool GON, bool FAST>
__device__ __forceinline__ void taylor_pair_flat(const double (&d0)[3], const double (&a)[3],
                                                 const double (&b)[3], const double* tab, int Q,
                                                 double kr, double ki, int m0, double nd,
                                                 double J, double unit, int unit_exp,
                                                 const Trig& tr,
                                                 Multi<3, KB, GON>& v, double& c3) {
  constexpr int NA = KB + (GON ? 2 : 1);
  double ac[NA][3], as[NA][3];
  double n[4] = {tab[0], tab[1], tab[2], tab[3]};
#pragma unroll
  for (int j = 0; j < NA; ++j)
#pragma unroll
    for (int s = 0; s < 3; ++s) ac[j][s] = as[j][s] = 0.0;
  c3 = 0.0;
#pragma unroll 1
  for (int q = 0; q < Q; ++q)
    taylor_point_flat<NA, CPLX, FAST>(d0, a, b, n, tab += 4, kr, ki, unit, m0, tr, ac, as, c3);
  // F_m = (n.d) i^m [(m - 1) A'_{m-2} + i k A'_{m-1}], G_m = J i^m A'_m (A' without i^j)
  if (m0 & 2) {
    nd = -nd;
    J = -J;
  }
  const double kn = nd * (FAST ? kr : kr * unit), kin = CPLX ? nd * (FAST ? ki : ki * unit) : 0.0;
#pragma unroll
  for (int q = 0; q < KB; ++q) {
    const double mn = nd * (double)(m0 + q - 1);
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      double re = fma(mn, ac[q][s], -(kn * as[q + 1][s]));
      double im = fma(mn, as[q][s], kn * ac[q + 1][s]);
      if constexpr (CPLX) {
        re = fma(-kin, ac[q + 1][s], re);
        im = fma(-kin, as[q + 1][s], im);
      }
      rotate(q, re, im);
      if constexpr (!FAST) {  // r^m in units of s^m
        re = ldexp(re, unit_exp * (m0 + q));
        im = ldexp(im, unit_exp * (m0 + q));
      }
      v.fr[q][s] = re;
      v.fi[q][s] = im;
      if constexpr (GON) {
        double gr = J * ac[q + 2][s], gi = J * as[q + 2][s];
        rotate(q, gr, gi);
        if constexpr (!FAST) {
          gr = ldexp(gr, unit_exp * (m0 + q));
          gi = ldexp(gi, unit_exp * (m0 + q));
        }
        v.gr[q][s] = gr;
        v.gi[q][s] = gi;
      }
    }
  }
}

// Pair on an element with tabulated points (rows y, n, J w / (4 pi) in memory, the next one
// always under way; basis values ph in LDS).  REC: spaced wavenumbers.  What a point reads is
// issued before its arithmetic: left to the compiler, some kernels issue it late (16 wavenumbers
// on 2562 quadratic nodes 3.68 ms, 3.29 this way).
template <int NP, int KB, bool TAY, bool CPLX, bool GON, bool FAST, bool REC>
__device__ __forceinline__ void multi_pair_rows(double x0, double x1, double x2,
                                                const double* rows, const double* ph, int Q,
                                                const Block<KB>& kv, double ki, int m0,
                                                const Trig& tr, Multi<NP, KB, GON>& v,
                                                double& csum) {
  v.clear();
  double y[7];
#pragma unroll
  for (int d = 0; d < 7; ++d) y[d] = rows[d];
#pragma unroll 1
  for (int p = 0; p < Q; ++p, ph += NP) {
    const double dx = y[0] - x0, dy = y[1] - x1, dz = y[2] - x2;
    const double nd = fma(y[3], dx, fma(y[4], dy, y[5] * dz)), jw = y[6];
    rows += p + 1 < Q ? 8 : 0;
#pragma unroll
    for (int d = 0; d < 7; ++d) y[d] = rows[d];
    double b[NP];
#pragma unroll
    for (int s = 0; s < NP; ++s) b[s] = ph[s];
    __builtin_amdgcn_sched_barrier(0);
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    const double rinv = rsqrt_nr(r2);
    const double r = r2 * rinv;
    const double g = jw * rinv;
    const double t = nd * (rinv * rinv);
    csum = fma(-t, g, csum);
    double sn, cs, zs = 0.0, zc = 0.0, damp = 1.0;
    Phase<CPLX, FAST> e;
    e.begin(kv.k[0] * r, CPLX ? ki * r : 0.0, tr);
    e.end(tr, sn, cs, damp);
    double gm = g, am = 0.0;
    if constexpr (TAY) {  // G_m without i^(m - m0), F_m = (m - 1 + i k r) t G_m
      if (CPLX) gm *= damp;
      double p2 = r;
      for (int x = m0; x != 0; x >>= 1) {
        if (x & 1) gm *= p2;
        p2 *= p2;
      }
      if (m0 & 2) gm = -gm;
      am = (double)(m0 - 1) - (CPLX ? ki * r : 0.0);
    } else if (REC) {
      Phase<false, FAST> z;
      z.begin(kv.dk * r, 0.0, tr);
      z.end(tr, zs, zc, damp);
    }
    double Gr = gm * cs, Gi = gm * sn;
#pragma unroll
    for (int q = 0; q < KB; ++q) {
      double Fr, Fi;
      if constexpr (TAY) {
        if (q > 0) {
          Gr *= r;
          Gi *= r;
        }
        const double krr = kv.k[0] * r;
        Fr = t * fma(am + (double)q, Gr, -(krr * Gi));
        Fi = t * fma(am + (double)q, Gi, krr * Gr);
      } else {
        if (q > 0) {
          if (REC) {
            const double c2 = fma(Gr, zc, -(Gi * zs));
            Gi = fma(Gr, zs, Gi * zc);
            Gr = c2;
          } else {
            Phase<false, FAST> z;
            z.begin(kv.k[q] * r, 0.0, tr);
            z.end(tr, sn, cs, damp);
            Gr = g * cs;
            Gi = g * sn;
          }
        }
        const double krr = kv.k[q] * r;
        Fr = -t * fma(krr, Gi, Gr);
        Fi = t * fma(krr, Gr, -Gi);
      }
#pragma unroll
      for (int s = 0; s < NP; ++s) {
        v.fr[q][s] = fma(Fr, b[s], v.fr[q][s]);
        v.fi[q][s] = fma(Fi, b[s], v.fi[q][s]);
        if constexpr (GON) {
          v.gr[q][s] = fma(Gr, b[s], v.gr[q][s]);
          v.gi[q][s] = fma(Gi, b[s], v.gi[q][s]);
        }
      }
    }
  }
  if constexpr (TAY) v.each([](int q, double& re, double& im) { rotate(q, re, im); });
}

// First and middle contributions of nb matrices: into the slot (see stream.hip's give).
template <int NP, int KB, bool GON>
__device__ __forceinline__ void give_multi(const int4& en, const Roles& r, int lane, double* acc,
                                           unsigned* claims, unsigned* ctr,
                                           const Multi<NP, KB, GON>& v, int nb, bool& ok) {
  constexpr int SK = GON ? 256 : 128, SD = KB * SK;
  const bool mine_first = lane_of_mask(r.first), mine_more = lane_of_mask(r.more);
#pragma unroll
  for (int s = 0; s < NP; ++s)
    if ((r.first >> s) & 1) {
      double* p = acc + (size_t)__builtin_amdgcn_readlane(en.x, s) * SD + lane;
#pragma unroll
      for (int b = 0; b < KB; ++b) {
        if (b >= nb) break;
        p[b * SK] = v.fr[b][s];
        p[b * SK + 64] = v.fi[b][s];
        if constexpr (GON) {
          p[b * SK + 128] = v.gr[b][s];
          p[b * SK + 192] = v.gi[b][s];
        }
      }
    }
  if (r.first) {
    lds_wait();
    if (mine_first) lds_count(claims + en.x, 0x10000u);
  }
  if (r.more) {
    if (!spin(ctr, [&] { return !mine_more || (lds_peek(claims + en.x) >> 16) != 0; })) {
      ok = false;
      return;
    }
#pragma unroll
    for (int s = 0; s < NP; ++s)
      if ((r.more >> s) & 1) {
        double* p = acc + (size_t)__builtin_amdgcn_readlane(en.x, s) * SD + lane;
#pragma unroll
        for (int b = 0; b < KB; ++b) {
          if (b >= nb) break;
          atomicAdd(p + b * SK, v.fr[b][s]);
          atomicAdd(p + b * SK + 64, v.fi[b][s]);
          if constexpr (GON) {
            atomicAdd(p + b * SK + 128, v.gr[b][s]);
            atomicAdd(p + b * SK + 192, v.gi[b][s]);
          }
        }
      }
    lds_wait();
    if (mine_more) lds_count(claims + en.x, 0x10000u);
  }
}

// Last contributions: to the columns of the block's matrices (see stream.hip's finish).
template <int NP, int KB, bool GON>
__device__ __forceinline__ void finish_multi(InstPtr in, SweepPtr sw, const int4& en,
                                             const Roles& r, int lane, int64_t i0, bool active,
                                             int k0, int nb, const double* acc, unsigned* claims,
                                             unsigned* turns, unsigned* ctr,
                                             const Multi<NP, KB, GON>& v, bool ok) {
  constexpr int SK = GON ? 256 : 128, SD = KB * SK;
  const bool mine = lane_of_mask(r.last);
  if (r.last)
    ok = spin(ctr, [&] {
           return !mine || (lds_peek(claims + en.x) >> 16) == (unsigned)en.y - 1u;
         }) && ok;
  const double bad = ok ? 0.0 : NAN;
  const InstPtr p = fresh(in);
  const bool doF = (p->a.flags & BIE_F) != 0;
  const int64_t M = p->a.M, stride = sw->stride;
  double* F = p->a.F + 2 * (size_t)k0 * stride;
  double* G = p->a.G + 2 * (size_t)k0 * stride;
#pragma unroll
  for (int s = 0; s < NP; ++s) {
    const bool last = (r.last >> s) & 1;
    if (!last && !((r.direct >> s) & 1)) continue;
    const int nw = __builtin_amdgcn_readlane(en.w, s);
    const bool shared = (nw & kSharedBit) != 0;
    const double* q =
        acc + (size_t)(last ? __builtin_amdgcn_readlane(en.x, s) : 0) * SD + lane;
    size_t at = 2 * ((size_t)i0 + (size_t)(nw & ~kSharedBit) * (size_t)M);
#pragma unroll
    for (int b = 0; b < KB; ++b, at += 2 * (size_t)stride) {
      if (b >= nb) break;
      double f0 = v.fr[b][s] + bad, f1 = v.fi[b][s], g0 = 0.0, g1 = 0.0;
      if constexpr (GON) {
        g0 = v.gr[b][s] + bad;
        g1 = v.gi[b][s];
      }
      if (last) {
        f0 += q[b * SK];
        f1 += q[b * SK + 64];
        if constexpr (GON) {
          g0 += q[b * SK + 128];
          g1 += q[b * SK + 192];
        }
      }
      if (active) {
        if (doF) column_store(F + at, 16u * lane, shared, f0, f1);
        if constexpr (GON) column_store(G + at, 16u * lane, shared, g0, g1);
      }
    }
  }
  if (mine && ok) {
    lds_wait();
    lds_poke(claims + en.x, 0u);
    lds_poke(turns + en.x, (unsigned)en.z + 1u);
  }
}

// Elements of the tile's segment, drawn by this wave, for the matrices k0 .. of a block.
template <int NP, bool FLAT, bool TAY, bool CPLX, bool GON, bool FAST>
__device__ __forceinline__ void sweep_tile(InstPtr in, SweepPtr sw, int rb, int seg, int kb,
                                           int S, int tab_doubles, double* lds,
                                           int parity) {
  constexpr SweepShape kShape = sweep_shape(NP, GON, FLAT && TAY && !GON, FAST);
  constexpr int W = kShape.waves, KB = kShape.kb;
  constexpr bool kMids = NP == 6;
  const int lane = threadIdx.x & 63;
  const int R = in->a.R;
  const int Q = in->a.len[0];
  const Layout L = layout_of(S, kShape.slot, tab_doubles, W, 0, kMids && R == 6);
  double* acc = lds;
  const double* tab = lds + L.tab;
  const Trig tr = make_trig(tab + tab_doubles);
  unsigned* claims = reinterpret_cast<unsigned*>(lds + L.words);
  unsigned* turns = claims + S;
  unsigned* ctr = turns + S;
  const int64_t i = (int64_t)rb * 64 + lane;
  const int64_t M = in->a.M;
  const bool active = i < M;
  const double* xt = in->a.targets + 3 * (active ? i : M - 1);
  const double x0 = xt[0], x1 = xt[1], x2 = xt[2];
  const int k0 = kb * KB, nb = min(KB, sw->nk - k0);
  Block<KB> kv;
  double ki = 0.0;
  bool rec = true;
  if constexpr (TAY) {
    kv.k[0] = sw->k_re;
    ki = sw->k_im;
  } else {
#pragma unroll
    for (int q = 0; q < KB; ++q) kv.k[q] = sload(sw->k + min(k0 + q, sw->nk - 1));
    kv.dk = nb > 1 ? kv.k[KB > 1 ? 1 : 0] - kv.k[0] : 0.0;
    // the recurrence forms e^{i (k0 + q dk) r}: taken where that differs from e^{i k_q r} by
    // at most about 2 ulp of k_q r (a rounded linspace does)
#pragma unroll
    for (int q = 2; q < KB; ++q)
      if (q < nb && !(fabs(kv.k[q] - (kv.k[0] + q * kv.dk)) <= 4.5e-16 * fabs(kv.k[q])))
        rec = false;
    rec = __builtin_amdgcn_readfirstlane(rec);
#pragma unroll
    for (int q = 0; q < KB; ++q) asm volatile("" : "+s"(kv.k[q]));
  }
  const int t0 = sload(in->seg_begin + seg), t1 = sload(in->seg_begin + seg + 1);
  const int tab_rule = FLAT ? 4 * Q + 2 : ((Q * NP + 1) & ~1) + 2;
  auto draw = [&]() -> int { return t0 + (int)lds_draw(ctr + kTicket, 1u, lane); };
  double csum = 0.0;
  int pos = draw();
  while (pos < t1) {
    const int nxt = draw();
    const InstPtr u = fresh(in);
    const int l = fresh_lane(lane);
    const int4 en = u->ent[(size_t)pos * NP + min(l, NP - 1)];
    Multi<NP, KB, GON> v;
    if constexpr (FLAT) {
      const double* rec24 = u->flat + (size_t)pos * kFlatDoubles;
      const d8 r0 = sload8(rec24), r1 = sload8(rec24 + 8), r2 = sload8(rec24 + 16);
      const double P[3][3] = {{r0[0], r0[1], r0[2]}, {r0[3], r0[4], r0[5]},
                              {r0[6], r0[7], r1[0]}};
      double ea[3] = {r1[4], r1[5], r1[6]}, eb[3] = {r1[7], r2[0], r2[1]};
      const int c = select_rule_s<3>(x0, x1, x2, P, rec24, R, in) - 1;
      double d0[3] = {r1[1] - x0, r1[2] - x1, r1[3] - x2};
      double nd = fma(r2[2], d0[0], fma(r2[3], d0[1], r2[4] * d0[2]));  // n.d J
      double J = r2[5];
      const double* tc = tab + c * tab_rule;
      double c3 = 0.0;
      if constexpr (TAY) {
        double unit = 1.0;
        int unit_exp = 0;
        if constexpr (!FAST) unit_exp = pair_unit(d0, ea, eb, nd, J, unit);
        taylor_pair_flat<KB, CPLX, GON, FAST>(d0, ea, eb, tc, Q, kv.k[0], ki, k0, nd, J, unit,
                                              unit_exp, tr, v, c3);
        csum = fma(-nd, c3, csum);
      } else {
        if (!rec)
          sweep_pair_flat<KB, KB, GON, FAST, false>(d0, ea, eb, tc, Q, kv, nd, tr, v, c3);
        else if (KB > 4 && nb <= KB / 2)
          sweep_pair_flat<KB, KB / 2, GON, FAST, true>(d0, ea, eb, tc, Q, kv, nd, tr, v, c3);
        else
          sweep_pair_flat<KB, KB, GON, FAST, true>(d0, ea, eb, tc, Q, kv, nd, tr, v, c3);
        csum = FAST ? fma(-nd, c3, csum) : csum - c3;
#pragma unroll
        for (int q = 0; q < KB; ++q)
#pragma unroll
          for (int s = 0; s < 3; ++s) {
            if constexpr (FAST) {
              v.fr[q][s] *= nd;
              v.fi[q][s] *= nd;
            }
            if constexpr (GON) {
              v.gr[q][s] *= J;
              v.gi[q][s] *= J;
            }
          }
      }
    } else {
      int c = 0;
      if (R > 1) {
        double P[NP][3];
        const double* ps = u->psel + (size_t)pos * NP * 3;
#pragma unroll
        for (int s = 0; s < NP; ++s)
#pragma unroll
          for (int d = 0; d < 3; ++d) P[s][d] = sload(ps + 3 * s + d);
        // (no distance below Inf falls to the last rule, a mid-edge one on quadratic geometry:
        // without six nodes to queue it for, such a row, which is NaN, runs along on the third)
        c = select_rule_s<NP>(x0, x1, x2, P, ps, kMids ? R : min(R, 3), in) - 1;
      }
      const bool mid = kMids && c >= 3;
      const int cr = mid ? 0 : c;
      double cs_pair = 0.0;
      auto pair = [&](auto recur) {
        multi_pair_rows<NP, KB, TAY, CPLX, GON, FAST, decltype(recur)::value>(
            x0, x1, x2,
            u->a.elem + ((size_t)sload(u->order + pos) * u->a.Pe + (size_t)cr * Q) * 8,
            tab + (size_t)cr * tab_rule, Q, kv, ki, k0, tr, v, cs_pair);
      };
      if (!TAY && rec)
        pair(std::true_type{});
      else
        pair(std::false_type{});
      if (kMids && R == 6 && __any(mid)) {  // those pairs leave nothing here
        v.each([&](int, double& re, double& im) {
          re = mid ? 0.0 : re;
          im = mid ? 0.0 : im;
        });
        cs_pair = mid ? 0.0 : cs_pair;
        const unsigned long long mask = __ballot(mid && active);
        if (mask && kb == 0) {  // listed once, for every matrix
          const unsigned base = lds_draw(ctr + kMidN + parity, (unsigned)__popcll(mask), lane);
          const unsigned at =
              base + __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                               __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
          if (mid && active && at < (unsigned)kStreamMid)  // position, rule, row of the pair
            reinterpret_cast<unsigned*>(lds + L.queue)[parity * kStreamMid + at] =
                ((unsigned)(pos - t0) << 8) | ((unsigned)(c - 3) << 6) | (unsigned)lane;
        }
      }
      csum += cs_pair;
    }
    bool ok;
    const Roles r = claim<NP>(en, l, claims, turns, ctr, ok);
    give_multi<NP, KB, GON>(en, r, l, acc, claims, ctr, v, nb, ok);
    finish_multi<NP, KB, GON>(in, sw, en, r, l, (int64_t)rb * 64, active, k0, nb, acc, claims,
                              turns, ctr, v, ok);
    pos = nxt;
  }
  if (kb == 0) atomicAdd(lds + L.csum + lane, csum);
}

template <int NP, bool FLAT, bool TAY, bool CPLX, bool GON, bool FAST>
__global__ void __launch_bounds__(64 * sweep_shape(NP, GON, FLAT && TAY && !GON, FAST).waves)
k_sweep(const StreamInst one, const SweepArgs args, int n_tiles, const StreamRun run) {
  extern __shared__ double lds[];
  const auto* base = (const __attribute__((address_space(4))) char*)
      __builtin_amdgcn_kernarg_segment_ptr();
  const InstPtr in = (InstPtr)base;
  const SweepPtr sw = (SweepPtr)(base + ((sizeof(StreamInst) + alignof(SweepArgs) - 1) &
                                         ~(alignof(SweepArgs) - 1)));
  // matrix block outermost, then segment, then row block
  const int per_kb = one.n_segments * one.n_rowblocks;
  auto inst_of = [&](int tile, int& rb, int& seg) -> InstPtr {
    const int t = tile % per_kb, n = in->n_rowblocks;
    seg = t / n;
    rb = t - seg * n;
    return in;
  };
  auto kmax_of = [&](InstPtr, int tile) -> double {
    if constexpr (TAY) {
      return fabs(sw->k_re);
    } else {  // of the block's wavenumbers and of their spacing
      constexpr int KB = sweep_shape(NP, GON, false).kb;
      const int k0 = tile / per_kb * KB;
      double m = 0.0;
      for (int q = k0; q < min(k0 + KB, sw->nk); ++q) m = fmax(m, fabs(sload(sw->k + q)));
      return 2.0 * m;
    }
  };
  constexpr SweepShape kShape = sweep_shape(NP, GON, FLAT && TAY && !GON, FAST);
  stream_run<kShape.slot, kShape.waves, NP == 6, FAST>(
      inst_of, kmax_of, [&](InstPtr, int tile) { return tile < per_kb; },
      [&](InstPtr p, int rb, int seg, int tile, int parity) {
        sweep_tile<NP, FLAT, TAY, CPLX, GON, FAST>(p, sw, rb, seg, tile / per_kb, run.S,
                                                   run.tab_doubles, lds, parity);
      },
      n_tiles, run);
}

// The listed mid-edge pairs, for every matrix (blockIdx.y and on).
template <bool TAY, bool CPLX, bool GON>
__global__ void __launch_bounds__(256)
k_sweep_mid(const StreamInst one, const SweepArgs sw, const double* tab_src, int tab_doubles) {
  extern __shared__ double lds[];
  const InstPtr in = (InstPtr)__builtin_amdgcn_kernarg_segment_ptr();
  const int mid_off = in->mid_off;
  const int ntab = tab_doubles - mid_off + kTrigDoubles + kExpN;
  for (int t = threadIdx.x; t < ntab; t += 256) lds[t] = tab_src[mid_off + t];
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Trig tr = make_trig(lds + tab_doubles - mid_off);
  for (int q = blockIdx.y; q < sw.nk; q += gridDim.y) {
    const size_t at = 2 * (size_t)q * sw.stride;
    const MidOut o{TAY ? sw.k_re : sload(sw.k + q), TAY ? sw.k_im : 0.0, in->a.F + at,
                   in->a.G + at, q == 0 && (in->a.flags & BIE_C), q};
    mid_pairs<CPLX, GON, false, TAY>(in, o, lds, tr, blockIdx.x * 4 + wave, gridDim.x * 4,
                                     threadIdx.x & 63);
  }
}

// Calls fn(kernel, mid-edge kernel) of (NP, flat elements, k-derivatives, complex, G, fast).
template <class Fn>
void with_sweep_kernel(int NP, bool flat, bool tay, bool cplx, bool gon, bool fast, Fn&& fn) {
  using T = std::true_type;
  using F = std::false_type;
  auto by_fast = [&](auto np, auto fl, auto ta, auto cx, auto g) {
    constexpr int N = decltype(np)::value;
    constexpr bool FL = decltype(fl)::value, TA = decltype(ta)::value, CX = decltype(cx)::value,
                   G = decltype(g)::value;
    if (fast)
      fn(k_sweep<N, FL, TA, CX, G, true>, k_sweep_mid<TA, CX, G>);
    else
      fn(k_sweep<N, FL, TA, CX, G, false>, k_sweep_mid<TA, CX, G>);
  };
  auto by_g = [&](auto np, auto fl, auto ta, auto cx) {
    gon ? by_fast(np, fl, ta, cx, T{}) : by_fast(np, fl, ta, cx, F{});
  };
  auto by_kind = [&](auto np, auto fl) {
    if (!tay)
      by_g(np, fl, F{}, F{});
    else
      cplx ? by_g(np, fl, T{}, T{}) : by_g(np, fl, T{}, F{});
  };
  if (NP == 1)
    by_kind(std::integral_constant<int, 1>{}, F{});
  else if (NP == 6)
    by_kind(std::integral_constant<int, 6>{}, F{});
  else if (flat)
    by_kind(std::integral_constant<int, 3>{}, T{});
  else
    by_kind(std::integral_constant<int, 3>{}, F{});
}

}  // namespace

int sweep_block_size(int NP, bool gon, bool lean) { return sweep_shape(NP, gon, lean).kb; }

StreamPlan sweep_plan(const RuleSet& rs, bool flat, bool lean, int slots) {
  const SweepShape sh = sweep_shape(rs.pk, true, lean);
  StreamPlan pl;
  pl.flat = flat;
  pl.waves = sh.waves;
  pl.tab_doubles = stream_tab_doubles(rs, flat);
  pl.mids = uses_mid_rules(rs.R, rs.pk);
  auto bytes = [&](int S) {
    return layout_of(S, sh.slot, pl.tab_doubles, pl.waves, 0, pl.mids).total * 8L;
  };
  while (pl.S < 120 && bytes(pl.S + 1) <= kLdsBytes) ++pl.S;
  if (slots > 0) pl.S = std::min(pl.S, slots);
  pl.shmem = (size_t)bytes(pl.S);
  return pl;
}

void launch_sweep(const StreamInst& in, const SweepArgs& sw, const StreamPlan& pl,
                  const double* d_tab, unsigned* d_counters, int* d_slow, int cus, bool fast,
                  bool prepare_only, hipStream_t s) {
  const bool gon = (in.a.flags & BIE_G) != 0, tay = sw.taylor != 0, cplx = sw.k_im != 0.0;
  const bool lean = pl.flat && tay && !gon;
  const int KB = sweep_shape(in.a.NP, gon, lean).kb;
  const int64_t tiles =
      (int64_t)((sw.nk + KB - 1) / KB) * in.n_segments * (int64_t)in.n_rowblocks;
  BIE_REQUIRE(tiles > 0 && tiles < 2147483647LL, BIE_EINVAL, "too many sweep tiles");
  BIE_REQUIRE(pl.S > 0 && pl.shmem <= (size_t)kLdsBytes, BIE_EINVAL,
              "internal: sweep kernel without LDS slots");
  const StreamRun run{d_tab, d_counters, fast ? nullptr : d_slow, pl.tab_doubles, pl.S, 0,
                      pl.mids ? 1 : 0};
  for (int pass = 0; pass < (fast ? 1 : 2); ++pass)
    with_sweep_kernel(in.a.NP, pl.flat, tay, cplx, gon, pass == 0, [&](auto kern, auto mid) {
      BIE_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                        hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)pl.shmem));
      if (prepare_only) return;
      hipLaunchKernelGGL(kern, dim3((unsigned)std::min<int64_t>(tiles, cus)),
                         dim3(64 * sweep_shape(in.a.NP, gon, lean, pass == 0).waves), pl.shmem, s,
                         in, sw, (int)tiles, run);
      if (pl.mids && pass == (fast ? 0 : 1))
        hipLaunchKernelGGL(mid, dim3(512, (unsigned)std::min(sw.nk, 1024)), dim3(256),
                           sizeof(double) *
                               (size_t)(pl.tab_doubles - in.mid_off + kTrigDoubles + kExpN),
                           s, in, sw, d_tab, pl.tab_doubles);
    });
  BIE_HIP_CHECK(hipGetLastError());
}

}  // namespace bie
