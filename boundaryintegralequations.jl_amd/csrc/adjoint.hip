// Vector-Jacobian product of the dense collocation assembly (gfx950, FP64):
//
//   grad_X, grad_k of  Phi = Re[ sum_i alpha_i sum_j F_ij(X, k) p_j + sum_i beta_i C_i(X) ]
//
// for complex weights alpha (per target), beta (per target) and p (per collocation node),
// with the rule selection held fixed (it is piecewise constant in X).  X are the mesh
// coordinates (3 x Nc); targets that are mesh nodes (tvert[i] >= 0) move with them, field
// targets stay fixed.  This is the building block of the adjoint gradient of objectives
// that go through F, C and a solve; the reference has no counterpart (its shape
// optimisation example differentiates by finite differences,
// examples/2d_optimization.jl:184-216).
//
// Quadrature is recomputed per pair instead of stored: at each rule point
// y = X N, t_u = X dN/du, t_v = X dN/dv, c = t_u x t_v.  Since the reference's normal is
// n = -c/|c| and J = |c|, the integrands times J are
//   f J w = -(c.d) w h(r),   h = e^{ikr}(ikr - 1)/(4 pi r^3)      (kernels.jl:29-37)
//   k0 J w = (c.d) w / (4 pi r^3)                                 (kernels.jl:48-55)
// with d = y - x, so Phi's integrand is (c.d) H with H = -A1 h + A2/(4 pi r^3),
// A1 = alpha p_h w (p_h = physics-basis interpolant of p), A2 = beta w, and
//   dPsi/dd = H c + (c.d) H_r d / r,  dPsi/dc = H d,  dPsi/dk = (c.d) A1 k e^{ikr}/(4 pi r),
//   H_r = -A1 h' + A2 (-3/(4 pi r^4)),  h' = -k^2 e^{ikr}/(4 pi r^2) - 3 h / r.
// The same formulas hold for complex k (the lossy systems' wavenumbers) in complex
// arithmetic; then Phi's derivatives in Re k and Im k are Re(D) and -Im(D) of
// D = sum (c.d) A1 k e^{ikr} / (4 pi r) (F is holomorphic in k).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "bie_common.hpp"
#include "device_common.hpp"
#include "kernels_math.hpp"
#include "stream_device.hpp"

namespace bie {
namespace {

constexpr double kInv4Pi = 0.079577471545947667884;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Calls point({N1, N2, N3, w / (4 pi)}) for the Q points of a flat element's rule in LDS, two
// at a time, the next one always under way (the table has room behind its last point).
template <class Point>
__device__ __forceinline__ void points_flat(const double* tab, int Q, Point point) {
  double m[4], n[4];
  auto load = [&](double (&x)[4]) {
#pragma unroll
    for (int s = 0; s < 4; ++s) x[s] = tab[s];
    tab += 4;
    __builtin_amdgcn_sched_barrier(0);
  };
  load(m);
  if (Q & 1) {
    load(n);
    point(m);
#pragma unroll
    for (int s = 0; s < 4; ++s) m[s] = n[s];
    if (Q == 1) return;
  }
  Q >>= 1;
#pragma unroll 1
  for (int q = 0; q < Q; ++q) {
    load(n);
    point(m);
    load(m);
    point(n);
  }
}

// Curved elements: one target per thread, the element the same for the whole wave (its nodes
// and p in scalar registers, so that two waves fit a SIMD).  Bound by FP64 issue, some 220
// instructions per point.  3242 quadratic nodes, 16 points: 2.72 -> 2.00 ms with the table
// sincos and the second wave.
template <int NG, int NP, bool CPLX, bool FAST>
__global__ void __launch_bounds__(256, 2)
k_adjoint(const AdjointArgs a, int ech, const double* trig) {
  __shared__ double s_trig[kTrigDoubles + kExpN];
  for (int t = threadIdx.x; t < kTrigDoubles + kExpN; t += blockDim.x) s_trig[t] = trig[t];
  __syncthreads();
  const Trig tr = make_trig(s_trig);
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const bool active = i < a.M;
  const int64_t ic = active ? i : (a.M - 1);
  const double x0 = a.targets[3 * ic], x1 = a.targets[3 * ic + 1], x2 = a.targets[3 * ic + 2];
  double2 al = active ? a.alpha[ic] : make_double2(0.0, 0.0);
  double2 be = (active && a.beta) ? a.beta[ic] : make_double2(0.0, 0.0);
  const double k = a.k, ki = CPLX ? a.ki : 0.0;
  double gx0 = 0, gx1 = 0, gx2 = 0, gk = 0, gki = 0;
  const int e0 = blockIdx.y * ech;
  const int e1 = min(a.E, e0 + ech);
  for (int e = e0; e < e1; ++e) {
    const int c =
        select_rule<NP>(x0, x1, x2, a.selnodes + (size_t)e * NP * 4, a.R, a.hyp) - 1;
    double X[NG][3];
#pragma unroll
    for (int q = 0; q < NG; ++q) {
      const int node = sload(a.topo + (size_t)e * NG + q);
#pragma unroll
      for (int d = 0; d < 3; ++d) X[q][d] = sload(a.coords + 3 * (size_t)node + d);
    }
    double pr[NP], pim[NP];
#pragma unroll
    for (int s = 0; s < NP; ++s) {
      const double* v =
          reinterpret_cast<const double*>(a.p + sload(a.ptopo + (size_t)e * NP + s));
      pr[s] = sload(v);
      pim[s] = sload(v + 1);
    }
    double gX[NG][3];
#pragma unroll
    for (int q = 0; q < NG; ++q) gX[q][0] = gX[q][1] = gX[q][2] = 0.0;
    const int Q = a.len[c];
    const double* P0 = a.pts + (size_t)a.off[c] * kPtStride;
    const double* ph0 = a.phi + (size_t)c * a.Qmax * NP;
    for (int q = 0; q < Q; ++q) {
      const double* P = P0 + (size_t)q * kPtStride;
      const double w = P[2];
      double y[3] = {0, 0, 0}, tu[3] = {0, 0, 0}, tv[3] = {0, 0, 0};
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const double N = P[kPtN + g], du = P[kPtDu + g], dv = P[kPtDv + g];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          y[d] = fma(X[g][d], N, y[d]);
          tu[d] = fma(X[g][d], du, tu[d]);
          tv[d] = fma(X[g][d], dv, tv[d]);
        }
      }
      const double cv[3] = {tu[1] * tv[2] - tu[2] * tv[1], tu[2] * tv[0] - tu[0] * tv[2],
                            tu[0] * tv[1] - tu[1] * tv[0]};
      const double d[3] = {y[0] - x0, y[1] - x1, y[2] - x2};
      const double r2 = fma(d[0], d[0], fma(d[1], d[1], d[2] * d[2]));
      const double rinv = rsqrt_nr(r2);
      const double r = r2 * rinv;
      const double cd = fma(cv[0], d[0], fma(cv[1], d[1], cv[2] * d[2]));
      // p interpolated at the point, times alpha and w
      double phr = 0, phi_ = 0;
#pragma unroll
      for (int s = 0; s < NP; ++s) {
        const double b = ph0[q * NP + s];
        phr = fma(b, pr[s], phr);
        phi_ = fma(b, pim[s], phi_);
      }
      const double A1r = w * (al.x * phr - al.y * phi_), A1i = w * (al.x * phi_ + al.y * phr);
      const double A2r = w * be.x;
      double sn, cs, damp;
      Phase<CPLX, FAST> ph;
      ph.begin(k * r, CPLX ? ki * r : 0.0, tr);
      ph.end(tr, sn, cs, damp);
      if (CPLX) {  // e^{ikr} = e^{-Im k r} e^{i Re k r}
        cs *= damp;
        sn *= damp;
      }
      const double i4r = kInv4Pi * rinv;            // 1/(4 pi r)
      const double i4r3 = i4r * rinv * rinv;        // 1/(4 pi r^3)
      const double kr = k * r;
      double hr, hi, hpr, hpi;
      if (CPLX) {
        // h = e^{ikr} (ikr - 1)/(4 pi r^3), ikr - 1 = (-Im k r - 1) + i Re k r
        const double ar = fma(-ki, r, -1.0), ai = kr;
        hr = (cs * ar - sn * ai) * i4r3;
        hi = (cs * ai + sn * ar) * i4r3;
        // h' = -k^2 e^{ikr}/(4 pi r^2) - 3 h / r, k^2 = (Re k^2 - Im k^2) + 2 i Re k Im k
        const double k2r = k * k - ki * ki, k2i = 2.0 * k * ki, s2 = i4r * rinv;
        hpr = -(k2r * cs - k2i * sn) * s2 - 3.0 * hr * rinv;
        hpi = -(k2r * sn + k2i * cs) * s2 - 3.0 * hi * rinv;
      } else {
        hr = (-cs - kr * sn) * i4r3;
        hi = (kr * cs - sn) * i4r3;
        const double k2i4r2 = k * k * i4r * rinv;   // k^2/(4 pi r^2)
        hpr = -k2i4r2 * cs - 3.0 * hr * rinv;
        hpi = -k2i4r2 * sn - 3.0 * hi * rinv;
      }
      // Re(H) = -Re(A1 h) + A2r/(4 pi r^3);  Re(H_r) = -Re(A1 h') - 3 A2r/(4 pi r^4)
      const double ReH = -(A1r * hr - A1i * hi) + A2r * i4r3;
      const double ReHr = -(A1r * hpr - A1i * hpi) - 3.0 * A2r * i4r3 * rinv;
      if (CPLX) {
        // D += cd A1 k e^{ikr} / (4 pi r): d/dRe k = Re D, d/dIm k = -Im D
        const double er = k * cs - ki * sn, ei = k * sn + ki * cs;   // k e^{ikr}
        gk += cd * i4r * (A1r * er - A1i * ei);
        gki -= cd * i4r * (A1r * ei + A1i * er);
      } else {
        // dPsi/dk = cd * Re(A1 k e^{ikr}) / (4 pi r)
        gk += cd * k * i4r * (A1r * cs - A1i * sn);
      }
      const double t = ReHr * cd * rinv;
      const double gd[3] = {fma(t, d[0], ReH * cv[0]), fma(t, d[1], ReH * cv[1]),
                            fma(t, d[2], ReH * cv[2])};
      const double gc[3] = {ReH * d[0], ReH * d[1], ReH * d[2]};
      gx0 -= gd[0];
      gx1 -= gd[1];
      gx2 -= gd[2];
      // d(g.(t_u x t_v))/dt_u = t_v x g,  /dt_v = g x t_u
      const double gtu[3] = {tv[1] * gc[2] - tv[2] * gc[1], tv[2] * gc[0] - tv[0] * gc[2],
                             tv[0] * gc[1] - tv[1] * gc[0]};
      const double gtv[3] = {gc[1] * tu[2] - gc[2] * tu[1], gc[2] * tu[0] - gc[0] * tu[2],
                             gc[0] * tu[1] - gc[1] * tu[0]};
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const double N = P[kPtN + g], du = P[kPtDu + g], dv = P[kPtDv + g];
#pragma unroll
        for (int dd = 0; dd < 3; ++dd)
          gX[g][dd] = fma(N, gd[dd], fma(du, gtu[dd], fma(dv, gtv[dd], gX[g][dd])));
      }
    }
    // the wave shares element e: sum its node gradients over the lanes, one atomic each
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const int node = a.topo[(size_t)e * NG + g];
#pragma unroll
      for (int dd = 0; dd < 3; ++dd) {
        const double v = wave_sum(gX[g][dd]);
        if ((threadIdx.x & 63) == 0) unsafeAtomicAdd(a.gradX + 3 * (size_t)node + dd, v);
      }
    }
  }
  if (active && a.tvert) {
    const int v = a.tvert[i];
    if (v >= 0) {
      unsafeAtomicAdd(a.gradX + 3 * (size_t)v, gx0);
      unsafeAtomicAdd(a.gradX + 3 * (size_t)v + 1, gx1);
      unsafeAtomicAdd(a.gradX + 3 * (size_t)v + 2, gx2);
    }
  }
  const double gks = wave_sum(gk);
  if ((threadIdx.x & 63) == 0 && a.gradk) unsafeAtomicAdd(a.gradk, gks);
  if (CPLX) {
    const double gkis = wave_sum(gki);
    if ((threadIdx.x & 63) == 0 && a.gradk) unsafeAtomicAdd(a.gradk + 1, gkis);
  }
}

// Derivative in k of the assembly, contracted: w = alpha^T (dF/dk) p for every instance of an
// uneven batch.  d/dk of the double-layer integrand e^{ikr}(ikr - 1)(n.d) J w / (4 pi r^3)
// (kernels.jl:29-37; its k-derivative is taylor_freens3d! at order 1, kernels.jl:104-118) is
// -k e^{ikr} (n.d) J w / (4 pi r), holomorphic in k, so complex wavenumbers (the lossy callers)
// are covered.  Every (target, element) pair is included, mid-edge rules too, with the
// assembly's rule selection.
//
// Bound by FP64 issue.  Nothing is written but one number per instance, so a wave works alone:
// a tile is (instance, 64 rows, ech elements), lane = row, and the wave's sum goes to
// w[instance] with one atomic.  Flat elements: the record of the stream kernels by scalar
// loads, n.d J a constant of the pair, sums of N_s e^{ikr} w / (4 pi r) over the rule, and p
// only at the pair's end; 47 instructions per point.  Other elements read the tabulated rows
// (y, n, J w / (4 pi)), the next one always under way.  FAST as in the stream kernels; the
// instances whose arguments may be larger are left to a launch without it.  24 meshes of 500
// to 6000 nodes, 16 points: 26.1 -> 10.3 ms (VALU busy 87 % of the time).
template <int NP, bool FLAT, bool CPLX, bool FAST>
__global__ void __launch_bounds__(256, 4)
k_dfdk_batch(const DfdkInst* insts, int n_inst, int n_tiles, int ech, const double* basis,
             int n_basis, const double* trig) {
  extern __shared__ double lds[];
  for (int t = threadIdx.x; t < n_basis; t += 256) lds[t] = basis[t];
  for (int t = threadIdx.x; t < kTrigDoubles + kExpN; t += 256) lds[n_basis + t] = trig[t];
  __syncthreads();
  const Trig tr = make_trig(lds + n_basis);
  typedef const __attribute__((address_space(4))) DfdkInst* DfdkPtr;
  const DfdkPtr all = (DfdkPtr) reinterpret_cast<uintptr_t>(insts);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int tile = blockIdx.x * 4 + wave; tile < n_tiles; tile += gridDim.x * 4) {
    int lo = 0, hi = n_inst;  // the last instance that begins at or before the tile
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (all[mid].first_tile <= tile)
        lo = mid;
      else
        hi = mid;
    }
    const DfdkPtr a = all + lo;
    if ((a->fast != 0) != FAST) continue;
    const int64_t M = a->M;
    const int rbs = (int)((M + 63) / 64), local = tile - a->first_tile;
    const int ch = local / rbs, rb = local - ch * rbs;
    const int64_t i = (int64_t)rb * 64 + lane;
    const bool active = i < M;
    const double* x = a->targets + 3 * (active ? i : M - 1);
    const double x0 = x[0], x1 = x[1], x2 = x[2];
    double kr = a->kr, ki = CPLX ? a->ki : 0.0;
    asm volatile("" : "+s"(kr), "+s"(ki));
    const int R = a->R, hyp = a->hyp;
    const double2* p = a->p;
    const int* ptopo = a->ptopo;
    double sr = 0.0, si = 0.0;  // sum over pairs and points of (n.d) Jw/(4 pi r) e^{ikr} p_h
    const int e0 = ch * ech, e1 = min(a->E, e0 + ech);
    for (int e = e0; e < e1; ++e) {
      double pr[NP], pi[NP];
#pragma unroll
      for (int s = 0; s < NP; ++s) {
        const double* v = reinterpret_cast<const double*>(p + sload(ptopo + (size_t)e * NP + s));
        pr[s] = sload(v);
        pi[s] = sload(v + 1);
      }
      if constexpr (FLAT) {
        const double* rec = a->flat + (size_t)e * kFlatDoubles;
        const d8 r0 = sload8(rec), r1 = sload8(rec + 8), r2 = sload8(rec + 16);
        const double P[3][3] = {{r0[0], r0[1], r0[2]}, {r0[3], r0[4], r0[5]},
                                {r0[6], r0[7], r1[0]}};
        const double ea[3] = {r1[4], r1[5], r1[6]}, eb[3] = {r1[7], r2[0], r2[1]};
        const int c = select_rule_p<3>(
                          x0, x1, x2, P, [&](int s, int d) { return sload(rec + 3 * s + d); }, R,
                          [&] { return hyp; }) - 1;
        const double d0[3] = {r1[1] - x0, r1[2] - x1, r1[3] - x2};
        const double nd = fma(r2[2], d0[0], fma(r2[3], d0[1], r2[4] * d0[2]));  // n.d J
        const int Q = a->len[0];
        const double* tab = lds + c * (4 * Q + 2);
        double ar[3] = {0, 0, 0}, ai[3] = {0, 0, 0};
        points_flat(tab, Q, [&](const double (&b)[4]) {
          const double dx = fma(b[2], eb[0], fma(b[1], ea[0], d0[0]));
          const double dy = fma(b[2], eb[1], fma(b[1], ea[1], d0[1]));
          const double dz = fma(b[2], eb[2], fma(b[1], ea[2], d0[2]));
          const double r2_ = fma(dx, dx, fma(dy, dy, dz * dz));
          const double rinv = rsqrt_nr(r2_);
          const double r = r2_ * rinv;
          Phase<CPLX, FAST> ph;
          ph.begin(kr * r, CPLX ? ki * r : 0.0, tr);
          double g = b[3] * rinv, sn, cs, damp;
          ph.end(tr, sn, cs, damp);
          if (CPLX) g *= damp;
          const double gr = g * cs, gi = g * sn;
#pragma unroll
          for (int s = 0; s < 3; ++s) {
            ar[s] = fma(gr, b[s], ar[s]);
            ai[s] = fma(gi, b[s], ai[s]);
          }
        });
        double tr_ = 0.0, ti_ = 0.0;
#pragma unroll
        for (int s = 0; s < 3; ++s) {
          tr_ = fma(ar[s], pr[s], fma(-ai[s], pi[s], tr_));
          ti_ = fma(ar[s], pi[s], fma(ai[s], pr[s], ti_));
        }
        sr = fma(nd, tr_, sr);
        si = fma(nd, ti_, si);
      } else {
        const int c =
            select_rule<NP>(x0, x1, x2, a->selnodes + (size_t)e * NP * 4, R, hyp) - 1;
        const double* row = a->elem + ((size_t)e * a->Pe + a->off[c]) * 8;
        const double* ph_ = lds + (size_t)c * a->Qmax * NP;
        const int Q = a->len[c];
        double y[7];
#pragma unroll
        for (int d = 0; d < 7; ++d) y[d] = row[d];
#pragma unroll 1
        for (int q = 0; q < Q; ++q, ph_ += NP) {
          const double dx = y[0] - x0, dy = y[1] - x1, dz = y[2] - x2;
          const double nd = fma(y[3], dx, fma(y[4], dy, y[5] * dz)), jw = y[6];
          row += q + 1 < Q ? 8 : 0;
#pragma unroll
          for (int d = 0; d < 7; ++d) y[d] = row[d];
          const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
          const double rinv = rsqrt_nr(r2);
          const double r = r2 * rinv;
          Phase<CPLX, FAST> ph;
          ph.begin(kr * r, CPLX ? ki * r : 0.0, tr);
          double phr = 0.0, phi_ = 0.0;
#pragma unroll
          for (int s = 0; s < NP; ++s) {
            phr = fma(ph_[s], pr[s], phr);
            phi_ = fma(ph_[s], pi[s], phi_);
          }
          double amp = nd * jw * rinv, sn, cs, damp;  // (n.d) J w / (4 pi r)
          ph.end(tr, sn, cs, damp);
          if (CPLX) amp *= damp;
          sr = fma(amp, fma(cs, phr, -(sn * phi_)), sr);
          si = fma(amp, fma(cs, phi_, sn * phr), si);
        }
      }
    }
    // w += alpha (-k) S
    const double2 al = active ? a->alpha[i] : make_double2(0.0, 0.0);
    const double ur = -(kr * sr - ki * si), ui = -(kr * si + ki * sr);
    const double wr = wave_sum(al.x * ur - al.y * ui), wi = wave_sum(al.x * ui + al.y * ur);
    if (lane == 0) {
      unsafeAtomicAdd(a->w, wr);
      unsafeAtomicAdd(a->w + 1, wi);
    }
  }
}

// ---- adjoint on flat elements ------------------------------------------------------------
// With d = d0 + N2 a + N3 b (a, b the edges from node 1), t_u = a, t_v = b, c = a x b and
// kappa = c.d = c.d0 constants of the pair, the gradient needs sums over the rule of
// H = Re(H) against 1, N2, N3 and of T = Re(H_r) / r against 1, N2, N3, N2^2, N2 N3, N3^2:
//   sum dPsi/dd = c H_1 + kappa (d0 T_1 + a T_2 + b T_3),  sum dPsi/dc = d0 H_1 + a H_2 + b H_3
// and so for the node-weighted ones.  With z = A1 e^{ikr} (A1 = alpha p_h) and w' = w / (4 pi):
//   H = w' (beta - Re[(ikr - 1) z]) / r^3,  T = w' Re(k^2 z) / r^3 - 3 H / r^2.
// Lane = element, the wave runs over rows: an element's sums stay in the lane's registers over
// all of them, and only the row's own gradient (three numbers) is summed over the wave, where
// one target per lane took nine sums over the wave for every element.  Bound by FP64 issue:
// about 66 instructions per point (190 when y, t_u, t_v were formed at every point).  2562
// nodes, 16 points: 1.97 -> 0.71 ms.

// Sum over the wave, the same in every lane: within rows of 16 by DPP, then over the four.
__device__ __forceinline__ double wave_total(double v) {
  auto dpp = [](double x, auto ctrl) {
    constexpr int c = decltype(ctrl)::value;
    return __hiloint2double(
        __builtin_amdgcn_update_dpp(0, __double2hiint(x), c, 0xf, 0xf, true),
        __builtin_amdgcn_update_dpp(0, __double2loint(x), c, 0xf, 0xf, true));
  };
  v += dpp(v, std::integral_constant<int, 0xB1>{});   // lane ^ 1
  v += dpp(v, std::integral_constant<int, 0x4E>{});   // lane ^ 2
  v += dpp(v, std::integral_constant<int, 0x141>{});  // mirrored in 8
  v += dpp(v, std::integral_constant<int, 0x140>{});  // mirrored in 16
  auto at = [&](int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
  };
  return (at(0) + at(16)) + (at(32) + at(48));
}

// LONG: the rules' points stay in memory.  ew: waves that share 64 elements, each taking every
// ew-th row (see launch_adjoint_flat).
template <bool CPLX, bool FAST, bool LONG>
__global__ void __launch_bounds__(256, 2)
k_adjoint_flat(const AdjointArgs a, int rows, int ew, const double* tab_src, int tab_doubles,
               int check) {
  extern __shared__ double lds[];
  const int skip = LONG ? tab_doubles : 0, n_lds = tab_doubles - skip + kTrigDoubles + kExpN;
  double* gx = lds + n_lds;       // rows x 3
  double* ge = gx + 3 * rows;     // (ew > 1) 9 x 64 node gradients of the elements
  for (int t = threadIdx.x; t < n_lds; t += 256) lds[t] = tab_src[skip + t];
  for (int t = threadIdx.x; t < 3 * rows + (ew > 1 ? 576 : 0); t += 256) gx[t] = 0.0;
  __syncthreads();
  const Trig tr = make_trig(lds + tab_doubles - skip);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int e = ew > 1 ? blockIdx.x * 64 + lane : blockIdx.x * 256 + threadIdx.x;
  const bool active = e < a.E;
  const int ec = active ? e : a.E - 1;
  double P[3][3], X1[3], ea[3], eb[3], pr[3], pi[3];
  int node[3];
#pragma unroll
  for (int s = 0; s < 3; ++s) {
    node[s] = a.topo[(size_t)ec * 3 + s];
    const double2 v = a.p[a.ptopo[(size_t)ec * 3 + s]];
    pr[s] = v.x;
    pi[s] = v.y;
#pragma unroll
    for (int d = 0; d < 3; ++d) P[s][d] = a.selnodes[(size_t)ec * 12 + 4 * s + d];
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    X1[d] = a.coords[3 * (size_t)node[0] + d];
    ea[d] = a.coords[3 * (size_t)node[1] + d] - X1[d];
    eb[d] = a.coords[3 * (size_t)node[2] + d] - X1[d];
  }
  const double on = active ? 1.0 : 0.0;  // idle lanes: c = 0, then nothing they add counts
  const double cv[3] = {on * (ea[1] * eb[2] - ea[2] * eb[1]), on * (ea[2] * eb[0] - ea[0] * eb[2]),
                        on * (ea[0] * eb[1] - ea[1] * eb[0])};
  const double k = a.k, ki = CPLX ? a.ki : 0.0;
  const double k2r = k * k - ki * ki, k2i = 2.0 * k * ki;
  const int Q = a.len[0];
  double D[3] = {0, 0, 0}, V[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}, hn[3] = {0, 0, 0};
  double M1 = 0, M2 = 0, M11 = 0, M12 = 0, M22 = 0, gk = 0, gki = 0;
  const int64_t i0 = (int64_t)blockIdx.y * rows, i1 = min(a.M, i0 + rows);
  for (int64_t i = i0 + (ew > 1 ? wave : 0); i < i1; i += ew) {
    const double x0 = sload(a.targets + 3 * i), x1 = sload(a.targets + 3 * i + 1),
                 x2 = sload(a.targets + 3 * i + 2);
    if (check) {  // rows whose |k| r may be large are the other launch's
      const double cx = x0 - a.center[0], cy = x1 - a.center[1], cz = x2 - a.center[2];
      const double dist = sqrt(fma(cx, cx, fma(cy, cy, cz * cz))) + a.reach;
      const bool near = fabs(k) * dist < 0.5 * kTabFastMaxArg && dist < kFastMaxDist;
      if (__builtin_amdgcn_readfirstlane((int)near) != (FAST ? 1 : 0)) continue;
    }
    const double* al = reinterpret_cast<const double*>(a.alpha + i);
    const double alr = sload(al), ali = sload(al + 1);
    const double be = a.beta ? sload(reinterpret_cast<const double*>(a.beta + i)) : 0.0;
    const int c = select_rule_p<3>(
                      x0, x1, x2, P, [&](int s, int d) { return P[s][d]; }, a.R,
                      [&] { return a.hyp; }) - 1;
    double Ar[3], Ai[3];  // alpha p
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      Ar[s] = alr * pr[s] - ali * pi[s];
      Ai[s] = alr * pi[s] + ali * pr[s];
    }
    const double d0[3] = {X1[0] - x0, X1[1] - x1, X1[2] - x2};
    const double kap = fma(cv[0], d0[0], fma(cv[1], d0[1], cv[2] * d0[2]));
    const double* tab = (LONG ? tab_src : lds) + c * (4 * Q + 2);
    double H0 = 0, H1 = 0, H2 = 0, T0 = 0, T1 = 0, T2 = 0, T11 = 0, T12 = 0, T22 = 0, Zr = 0,
           Zi = 0;
    points_flat(tab, Q, [&](const double (&b)[4]) {
      const double dx = fma(b[2], eb[0], fma(b[1], ea[0], d0[0]));
      const double dy = fma(b[2], eb[1], fma(b[1], ea[1], d0[1]));
      const double dz = fma(b[2], eb[2], fma(b[1], ea[2], d0[2]));
      const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
      const double rinv = rsqrt_nr(r2);
      const double r = r2 * rinv;
      const double krr = k * r, kir = CPLX ? ki * r : 0.0;
      Phase<CPLX, FAST> ph;
      ph.begin(krr, kir, tr);
      const double A1r = fma(b[2], Ar[2], fma(b[1], Ar[1], b[0] * Ar[0]));
      const double A1i = fma(b[2], Ai[2], fma(b[1], Ai[1], b[0] * Ai[0]));
      const double rinv2 = rinv * rinv, q1 = b[3] * rinv, q3 = q1 * rinv2;
      double sn, cs, damp;
      ph.end(tr, sn, cs, damp);
      if (CPLX) {
        cs *= damp;
        sn *= damp;
      }
      const double zr = fma(A1r, cs, -(A1i * sn)), zi = fma(A1r, sn, A1i * cs);
      // -Re[(ikr - 1) z]
      const double u = CPLX ? fma(krr, zi, fma(kir, zr, zr)) : fma(krr, zi, zr);
      const double H = q3 * (be + u);
      const double kz = CPLX ? fma(k2r, zr, -(k2i * zi)) : k2r * zr;
      // (FAST: without kappa, which is multiplied in below)
      const double kr2 = FAST ? rinv2 : kap * rinv2;
      const double T = FAST ? fma(q3, kz, -3.0 * rinv2 * H) : fma(kr2 * q1, kz, -3.0 * kr2 * H);
      Zr = fma(q1, zr, Zr);
      if (CPLX) Zi = fma(q1, zi, Zi);
      H0 += H;
      H1 = fma(H, b[1], H1);
      H2 = fma(H, b[2], H2);
      const double t1 = T * b[1], t2 = T * b[2];
      T0 += T;
      T1 += t1;
      T2 += t2;
      T11 = fma(t1, b[1], T11);
      T12 = fma(t1, b[2], T12);
      T22 = fma(t2, b[2], T22);
    });
    const double kapt = FAST ? kap : 1.0;
    T0 *= kapt;
    T1 *= kapt;
    T2 *= kapt;
    hn[0] += H0;
    hn[1] += H1;
    hn[2] += H2;
    M1 += T1;
    M2 += T2;
    M11 = fma(kapt, T11, M11);
    M12 = fma(kapt, T12, M12);
    M22 = fma(kapt, T22, M22);
    double gd[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      D[d] = fma(eb[d], H2, fma(ea[d], H1, fma(d0[d], H0, D[d])));
      V[0][d] = fma(d0[d], T0, V[0][d]);
      V[1][d] = fma(d0[d], T1, V[1][d]);
      V[2][d] = fma(d0[d], T2, V[2][d]);
      gd[d] = fma(eb[d], T2, fma(ea[d], T1, fma(d0[d], T0, cv[d] * H0)));
    }
    if (CPLX) {  // d/dRe k = Re(D), d/dIm k = -Im(D) of D = kappa k Z
      gk = fma(kap, k * Zr - ki * Zi, gk);
      gki = fma(-kap, k * Zi + ki * Zr, gki);
    } else {
      gk = fma(kap * k, Zr, gk);
    }
    if (a.tvert) {
      const double s0 = wave_total(gd[0]), s1 = wave_total(gd[1]), s2 = wave_total(gd[2]);
      if (lane < 3)
        atomicAdd(gx + 3 * (i - i0) + lane, -(lane == 0 ? s0 : lane == 1 ? s1 : s2));
    }
  }
  if (active) {
    const double gtu[3] = {eb[1] * D[2] - eb[2] * D[1], eb[2] * D[0] - eb[0] * D[2],
                           eb[0] * D[1] - eb[1] * D[0]};
    const double gtv[3] = {D[1] * ea[2] - D[2] * ea[1], D[2] * ea[0] - D[0] * ea[2],
                           D[0] * ea[1] - D[1] * ea[0]};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double w0 = fma(cv[d], hn[0], fma(ea[d], M1, fma(eb[d], M2, V[0][d])));
      const double w1 = fma(cv[d], hn[1], fma(ea[d], M11, fma(eb[d], M12, V[1][d])));
      const double w2 = fma(cv[d], hn[2], fma(ea[d], M12, fma(eb[d], M22, V[2][d])));
      const double g[3] = {(w0 - w1 - w2) - (gtu[d] + gtv[d]), w1 + gtu[d], w2 + gtv[d]};
#pragma unroll
      for (int s = 0; s < 3; ++s)
        if (ew > 1)
          atomicAdd(ge + (3 * s + d) * 64 + lane, g[s]);
        else
          unsafeAtomicAdd(a.gradX + 3 * (size_t)node[s] + d, g[s]);
    }
  }
  if (a.gradk) {
    const double s = wave_total(gk);
    if (lane == 0) unsafeAtomicAdd(a.gradk, s);
    if (CPLX) {
      const double t = wave_total(gki);
      if (lane == 0) unsafeAtomicAdd(a.gradk + 1, t);
    }
  }
  if (a.tvert || ew > 1) __syncthreads();
  if (ew > 1 && active) {
#pragma unroll
    for (int q = 0; q < 9; ++q)
      if (q % 4 == wave) unsafeAtomicAdd(a.gradX + 3 * (size_t)node[q / 3] + q % 3, ge[q * 64 + lane]);
  }
  if (a.tvert) {
    for (int t = threadIdx.x; t < 3 * (int)(i1 - i0); t += 256) {
      const int v = a.tvert[i0 + t / 3];
      if (v >= 0) unsafeAtomicAdd(a.gradX + 3 * (size_t)v + t % 3, gx[t]);
    }
  }
}

}  // namespace

void launch_dfdk_batch(const DfdkInst* d_inst, int n_inst, int n_tiles, int ech, int NP,
                       bool flat, bool cplx, bool some_fast, bool some_slow,
                       const double* d_basis, int n_basis, const double* d_trig, int cus,
                       hipStream_t s) {
  if (n_tiles <= 0) return;
  const size_t shmem = sizeof(double) * (size_t)(n_basis + kTrigDoubles + kExpN);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3((unsigned)std::min((n_tiles + 3) / 4, 4 * cus)), dim3(256),
                       shmem, s, d_inst, n_inst, n_tiles, ech, d_basis, n_basis, d_trig);
  };
  auto by = [&](auto np, auto fl) {
    constexpr int N = decltype(np)::value;
    constexpr bool FL = decltype(fl)::value;
    if (some_fast) cplx ? go(k_dfdk_batch<N, FL, true, true>) : go(k_dfdk_batch<N, FL, false, true>);
    if (some_slow)
      cplx ? go(k_dfdk_batch<N, FL, true, false>) : go(k_dfdk_batch<N, FL, false, false>);
  };
  if (NP == 1)
    by(std::integral_constant<int, 1>{}, std::false_type{});
  else if (NP == 6)
    by(std::integral_constant<int, 6>{}, std::false_type{});
  else if (flat)
    by(std::integral_constant<int, 3>{}, std::true_type{});
  else
    by(std::integral_constant<int, 3>{}, std::false_type{});
  BIE_HIP_CHECK(hipGetLastError());
}

// Rows per workgroup (256 elements): whole rounds of about two workgroups a CU, of some 64
// rows each (the lanes' atomics and element data are then a per cent of the work).  Meshes of
// up to 2048 elements leave most of the chip idle that way, and a row's points are a serial
// chain: there the four waves of a workgroup share 64 elements and divide the rows, as long as
// the workgroups fit the chip at once.  Their rows grow as sqrt(M): every further workgroup
// shortens the chain and adds atomics to the same nodes.  (16 points, one wave per element,
// then four: 42 nodes 39 and 18 us, 162 nodes 47 and 28, 642 nodes 95 and 55; 200 field rows
// on 720 elements 71 and 41; one row, or 5120 elements and 30 rows, are 5-10 % slower.)
static void launch_adjoint_flat(const AdjointArgs& a, bool cplx, bool fast, const double* d_tab,
                                int tab_doubles, int cus, hipStream_t s) {
  int64_t eb = (a.E + 255) / 256;
  const int64_t at_once = 2 * (int64_t)cus, eb64 = (a.E + 63) / 64;
  const int64_t rounds = std::max<int64_t>(1, (eb * a.M / 64 + at_once / 2) / at_once);
  const int64_t chunks = std::max<int64_t>(1, rounds * at_once / eb);
  int rows = (int)std::min<int64_t>(512, std::max<int64_t>(8, (a.M + chunks - 1) / chunks));
  const int shared_rows = 4 * (int)std::min(8.0, std::ceil(0.3 * std::sqrt((double)a.M)));
  const int ew = a.M > 4 && eb64 <= 32 &&
                         eb64 * ((a.M + shared_rows - 1) / shared_rows) <= at_once
                     ? 4
                     : 1;
  if (ew > 1) {
    eb = eb64;
    rows = shared_rows;
  }
  const int64_t ny = (a.M + rows - 1) / rows;
  // Rules of up to 48 KB (510 points) come from LDS: with the rows' sums that is below the
  // 64 KB of a plain launch, and two workgroups fit a CU.  Longer ones come from memory.
  const bool in_lds = sizeof(double) * (size_t)tab_doubles <= 48 * 1024;
  const size_t shmem = sizeof(double) * (size_t)((in_lds ? tab_doubles : 0) + kTrigDoubles +
                                                 kExpN + 3 * rows + (ew > 1 ? 576 : 0));
  for (int64_t y0 = 0; y0 < ny; y0 += 65535) {  // (the grid's second dimension ends there)
    AdjointArgs b = a;
    b.targets += 3 * y0 * rows;
    b.alpha += y0 * rows;
    if (b.beta) b.beta += y0 * rows;
    if (b.tvert) b.tvert += y0 * rows;
    b.M -= y0 * rows;
    const dim3 grid((unsigned)eb, (unsigned)std::min<int64_t>(65535, ny - y0));
    b.M = std::min<int64_t>(b.M, (int64_t)grid.y * rows);
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, grid, dim3(256), shmem, s, b, rows, ew, d_tab, tab_doubles,
                         fast ? 0 : 1);
    };
    auto by = [&](auto cx, auto fs) {
      constexpr bool C = decltype(cx)::value, S = decltype(fs)::value;
      in_lds ? go(k_adjoint_flat<C, S, false>) : go(k_adjoint_flat<C, S, true>);
    };
    auto by_fast = [&](auto fs) {
      cplx ? by(std::true_type{}, fs) : by(std::false_type{}, fs);
    };
    by_fast(std::true_type{});
    if (!fast) by_fast(std::false_type{});
  }
  BIE_HIP_CHECK(hipGetLastError());
}

void launch_adjoint(const AdjointArgs& a, int gk, int pk, bool flat, bool cplx, bool fast,
                    const double* d_tab, int tab_doubles, int cus, hipStream_t s) {
  if (a.M == 0 || a.E == 0) return;
  if (flat) return launch_adjoint_flat(a, cplx, fast, d_tab, tab_doubles, cus, s);
  // small problems: workgroups of one wave, so that no waves run for rows there are not (42
  // nodes 24 -> 21 us, 20 field rows on 720 elements 79 -> 37)
  const int bs = a.M * a.E <= 32768 ? 64 : 256;
  const int64_t rowblocks = (a.M + bs - 1) / bs;
  BIE_REQUIRE(rowblocks < 2147483647LL, BIE_EINVAL, "too many targets");
  int64_t chunks = (4096 + rowblocks - 1) / rowblocks;
  if (chunks > a.E) chunks = a.E;
  if (chunks > 65535) chunks = 65535;
  if (chunks < 1) chunks = 1;
  const int ech = (int)((a.E + chunks - 1) / chunks);
  chunks = (a.E + ech - 1) / ech;
  const dim3 grid((unsigned)rowblocks, (unsigned)chunks);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(bs), 0, s, a, ech, d_tab + tab_doubles);
  };
  auto by_fast = [&](auto np, auto cx) {
    constexpr int N = decltype(np)::value;
    constexpr bool C = decltype(cx)::value;
    fast ? go(k_adjoint<6, N, C, true>) : go(k_adjoint<6, N, C, false>);
  };
  auto by_np = [&](auto np) {
    cplx ? by_fast(np, std::true_type{}) : by_fast(np, std::false_type{});
  };
  if (pk == 6)
    by_np(std::integral_constant<int, 6>{});
  else
    by_np(std::integral_constant<int, 3>{});
  BIE_HIP_CHECK(hipGetLastError());
}

}  // namespace bie
