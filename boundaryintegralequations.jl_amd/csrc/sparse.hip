// Sparse near-field assembly (gfx950, FP64): the reference's
//   sparse_assemble_parallel!(mesh, k, sources, physics_function; fOn, gOn, depth, offset)
// (src/3d/assembly_collocation_losses.jl:200-405), the near-field correction behind its
// fast (FMM / H-matrix) operators and the lossy thermal and viscous systems.
//
// * Pattern and rules: built on the host (near_field.cpp): connected_sources' rows and
//   columns, and the six subdivision rules of singular_triangle_integration in the
//   reference triangle (continuous physics) or the polar rules of create_polar_elements
//   around the physics nodes (discontinuous physics, :233-257 there).
// * Pairs: every (row i, connected element e) is integrated with the rule of the element's
//   geometry node closest to source i (find_closest_corner on the element coordinates,
//   :308-309 there), the kernels of sparse_computing_integrals! (:158-186: freens3d!,
//   greens3d!, kernels.jl:13-37) and the physics basis at the rule points; the results add
//   into the row's entries of the element's physics nodes.
//
// One wave per (row, element) pair or per batch of pairs that share an element: lanes take the
// rule's points (a few thousand), the partial sums are reduced across the wave and added into
// the entries with FP64 atomics (a row's entries receive several elements' contributions).
// Bound by instruction issue (VALU busy 94 % of the time, 10242 quadratic nodes, depth 1): curved
// elements cost 290 per point and pair, of which the surface with its exactly rounded normal is
// 200; flat ones 80.  Before and after the cheaper exact divisions, the normal of flat elements
// taken out of the loop and the branch-free sincos (us): 10242 nodes, depth 1: 2350 -> 1686;
// depth 2, quadratic 2562 nodes 3400 -> 1822, linear 1962 nodes 642 -> 515.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <type_traits>
#include <vector>

#include "bie_common.hpp"
#include "device_common.hpp"
#include "kernels_math.hpp"
#include "stream_device.hpp"

namespace bie {
namespace {

constexpr double kInv4PiS = 0.079577471545947667884;

// ---- device ----------------------------------------------------------------------------

struct SparseArgs {
  const double* src;      // 3 x n_rows source points
  const int2* pairs;      // (row, element)
  const int* pos;         // pairs x NP entry index
  int64_t n_pairs;
  const double* coords;   // 3 x Nc
  const int* topo;        // E x NG
  const double* gsel;     // E x NG x 4 geometry node coordinates (selection)
  const double* rules;    // point records (kSparseRec doubles)
  const double* trig;     // (cos, sin)(j pi / 64), j < kTrigN, then 2^(j / 64), j < kExpN
  int off[6], len[6];
  const int* batches;     // 8 ints per batch: element, count, up to 4 pair indices
  int64_t n_batches;
  bool check;             // (batches) waves of near and far rows are a launch each
  double center[3], reach; // every element point is within reach of the centre
  int hyp;
  bool disc;              // discontinuous physics, nodes at beta
  double beta;
  double kr, ki;
  unsigned flags;
  double* F;              // nnz complex
  double* G;
};

// point record: u, v, w, pad (the bases are evaluated per point from u, v: a 26-double
// record with them precomputed made the kernel wait on L2 for 208 bytes per point)
constexpr int kSparseRec = 4;

// The geometry basis and its derivatives at (u, v), operation for operation as the host
// tables (eval_basis, rules.cpp, compiled without fused multiply-adds) and the CPU
// restatement compute them: the geometry below must round as theirs does.
template <int NG>
__device__ __forceinline__ void sparse_geom_basis(double u, double v, double (&N)[NG],
                                                  double (&du)[NG], double (&dv)[NG]) {
#pragma clang fp contract(off)
  if constexpr (NG == 3) {
    N[0] = (1.0 - u) - v;
    N[1] = u;
    N[2] = v;
    du[0] = -1.0;
    du[1] = 1.0;
    du[2] = 0.0;
    dv[0] = -1.0;
    dv[1] = 0.0;
    dv[2] = 1.0;
  } else {
    const double l = (1.0 - v) - u;
    N[0] = l * ((1.0 - 2.0 * v) - 2.0 * u);
    N[1] = u * (2.0 * u - 1.0);
    N[2] = v * (2.0 * v - 1.0);
    N[3] = 4.0 * u * l;
    N[4] = 4.0 * u * v;
    N[5] = 4.0 * v * l;
    const double d0 = -(2.0 * l - 1.0) - 2.0 * l;
    du[0] = d0;
    du[1] = 4.0 * u - 1.0;
    du[2] = 0.0;
    du[3] = 4.0 * l - 4.0 * u;
    du[4] = 4.0 * v;
    du[5] = -4.0 * v;
    dv[0] = d0;
    dv[1] = 0.0;
    dv[2] = 4.0 * v - 1.0;
    dv[3] = -4.0 * u;
    dv[4] = 4.0 * u;
    dv[5] = 4.0 * l - 4.0 * v;
  }
}

// The physics basis at (u, v): continuous three- or six-node triangles (the geometry
// bases), or the discontinuous ones (surface_functions.jl:234-318) with psi(s) =
// (s - beta) / (1 - 3 beta) of the barycentric coordinates 1 - u - v, u, v.
template <int NP>
__device__ __forceinline__ void sparse_phys_basis(bool disc, double beta, double u, double v,
                                                  double (&N)[NP]) {
  if constexpr (NP == 1) {
    N[0] = 1.0;
  } else {
    if (!disc) {
      double du[NP], dv[NP];
      sparse_geom_basis<NP>(u, v, N, du, dv);
      return;
    }
    const double den = 1.0 - 3.0 * beta;
    const double l1 = (((1.0 - u) - v) - beta) / den;
    const double l2 = (u - beta) / den;
    const double l3 = (v - beta) / den;
    if constexpr (NP == 3) {
      N[0] = l1;
      N[1] = l2;
      N[2] = l3;
    } else {
      N[0] = l1 * (2.0 * l1 - 1.0);
      N[1] = l2 * (2.0 * l2 - 1.0);
      N[2] = l3 * (2.0 * l3 - 1.0);
      N[3] = (4.0 * l2) * l1;
      N[4] = (4.0 * l2) * l3;
      N[5] = (4.0 * l3) * l1;
    }
  }
}

// A divisor's reciprocal (estimate refined by two Newton steps) and the quotient from it: the
// residual a - b q is exact, so the correction leaves the correctly rounded a / b (Markstein's
// theorem), the same as the division the oracle performs, at three instructions for each
// further quotient of one divisor.  For divisors and quotients well inside the range.
__device__ __forceinline__ double recip_for_quot(double b) {
  double y = __builtin_amdgcn_rcp(b);
  y = fma(fma(-b, y, 1.0), y, y);
  return fma(fma(-b, y, 1.0), y, y);
}
__device__ __forceinline__ double quot(double a, double b, double y) {
  const double q = a * y;
  return fma(fma(-b, q, a), y, q);
}
// sqrt(s), correctly rounded, for s in [1, 3]: Goldschmidt's coupled iteration for sqrt(s) and
// 1 / (2 sqrt(s)), then two corrections by the exact residual s - g^2.
__device__ __forceinline__ double sqrt_1_3(double s) {
  const double y = __builtin_amdgcn_rsq(s);
  double g = s * y, h = 0.5 * y;
  const double e = fma(-h, g, 0.5);
  g = fma(g, e, g);
  h = fma(h, e, h);
  g = fma(fma(-g, g, s), h, g);
  return fma(fma(-g, g, s), h, g);
}

// J = hypot(c) and the reference's normal n = -c / J: every operation of julia_hypot3 and of
// the three divisions, rounded as they round (six divisions and a square root written out were
// 80 instructions of the 370 of a point; these are 40).  Out of the middle of the range (and
// for infinities, NaN and zero) the operations themselves.
__device__ __forceinline__ void sparse_normal(double c0, double c1, double c2, double (&n)[3],
                                              double& J) {
#pragma clang fp contract(off)
  const double ax = fabs(c0), ay = fabs(c1), az = fabs(c2);
  double mx = ax > ay ? ax : ay;
  mx = mx > az ? mx : az;
  if (mx > 0x1p-300 && mx < 0x1p300) {
    const double y = recip_for_quot(mx);
    const double a = quot(ax, mx, y), b = quot(ay, mx, y), c = quot(az, mx, y);
    double s = a * a;
    s = s + b * b;
    s = s + c * c;
    J = mx * sqrt_1_3(s);
    const double z = recip_for_quot(J);
    n[0] = quot(-c0, J, z);
    n[1] = quot(-c1, J, z);
    n[2] = quot(-c2, J, z);
  } else {
    J = julia_hypot3(c0, c1, c2);
    n[0] = -c0 / J;
    n[1] = -c1 / J;
    n[2] = -c2 / J;
  }
}

// The surface of an element in the oracle's operation order without fused multiply-adds.  On
// the elements around the source node n.d is rounding noise (a flat element contains its own
// node) divided by r^3 at cells ~1e-6 of the element: only geometry that rounds as the CPU
// restatement's does reproduces that noise.  Left out are additions of zero only (the leading
// 0 + and the nodes whose derivative is zero).  On flat elements t_u, t_v, n and J do not
// depend on the point: they are formed once.
template <int NG>
struct Surface {
  double X[NG][3], n[3], J;
  __device__ __forceinline__ void begin() {
#pragma clang fp contract(off)
    if constexpr (NG == 3) {  // -X1 + X2, -X1 + X3
      const double u0 = X[1][0] - X[0][0], u1 = X[1][1] - X[0][1], u2 = X[1][2] - X[0][2];
      const double v0 = X[2][0] - X[0][0], v1 = X[2][1] - X[0][1], v2 = X[2][2] - X[0][2];
      sparse_normal(u1 * v2 - u2 * v1, u2 * v0 - u0 * v2, u0 * v1 - u1 * v0, n, J);
    }
  }
  // y (and on curved elements n, J) at a point from the bases there
  __device__ __forceinline__ void at(const double (&N)[NG], const double (&Du)[NG],
                                     const double (&Dv)[NG], double (&y)[3]) {
#pragma clang fp contract(off)
    double tu[3], tv[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      double a = X[0][d] * N[0];
#pragma unroll
      for (int g = 1; g < NG; ++g) a = a + X[g][d] * N[g];
      y[d] = a;
      if constexpr (NG == 6) {  // Du[2] = Dv[1] = 0
        double b = X[0][d] * Du[0], c = X[0][d] * Dv[0];
        b = b + X[1][d] * Du[1];
        c = c + X[2][d] * Dv[2];
#pragma unroll
        for (int g = 3; g < 6; ++g) {
          b = b + X[g][d] * Du[g];
          c = c + X[g][d] * Dv[g];
        }
        tu[d] = b;
        tv[d] = c;
      }
    }
    if constexpr (NG == 6)
      sparse_normal(tu[1] * tv[2] - tu[2] * tv[1], tu[2] * tv[0] - tu[0] * tv[2],
                    tu[0] * tv[1] - tu[1] * tv[0], n, J);
  }
};

// The kernels at one rule point for a source x: G = e^{ikr} J w / (4 pi r) and
// F = e^{ikr} (ikr - 1) (n.d) J w / (4 pi r^3) (freens3d!, greens3d!, kernels.jl:13-37), d = y - x
// and n.d in the oracle's order.
template <bool CPLX, bool FAST>
__device__ __forceinline__ void sparse_point_kernels(const double (&y)[3], const double (&n)[3],
                                                     double J, const double (&x)[3], double wq,
                                                     double kr, double ki, const Trig& tr,
                                                     double& Fr, double& Fi, double& Gr,
                                                     double& Gi) {
  double dx, dy, dz, nd;
  {
#pragma clang fp contract(off)
    dx = y[0] - x[0];
    dy = y[1] - x[1];
    dz = y[2] - x[2];
    nd = n[0] * dx + n[1] * dy + n[2] * dz;
  }
  const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
  const double rinv = rsqrt_nr(r2);
  const double r = r2 * rinv;
  const double krr = kr * r, kir = CPLX ? ki * r : 0.0;
  Phase<CPLX, FAST> e;
  e.begin(krr, kir, tr);
  const double g = J * wq * kInv4PiS * rinv;  // J w / (4 pi r)
  kernels_end<CPLX, FAST>(e, g, nd * (rinv * rinv), krr, kir, tr, Fr, Fi, Gr, Gi);
}

// Lane = point (q, q + step, ...) of the rule at R0: the sums of B rows, where bit j of m says
// that row j takes part.  The next point's record is always under way.
template <int NG, int NP, int B, bool CPLX, bool FAST>
__device__ __forceinline__ void sparse_rule(const SparseArgs& a, Surface<NG>& sf,
                                            const double (&x)[B][3], unsigned m,
                                            const double* R0, int q, int Q, int step,
                                            const Trig& tr, double (&acc)[B][NP][4]) {
  static_assert(kSparseRec == 4, "a record is two 16-byte loads");
  const double2* rec = reinterpret_cast<const double2*>(R0) + 2 * (size_t)min(q, Q - 1);
  double2 uv = rec[0], wp = rec[1];
  for (; q < Q; q += step) {
    const double u = uv.x, v = uv.y, wq = wp.x;
    rec += q + step < Q ? 2 * (size_t)step : 0;
    uv = rec[0];
    wp = rec[1];
    double Ng[NG], Du[NG], Dv[NG], Np[NP], y[3];
    sparse_geom_basis<NG>(u, v, Ng, Du, Dv);
    sf.at(Ng, Du, Dv, y);
    if constexpr (NP == NG) {
      if (a.disc) {
        sparse_phys_basis<NP>(true, a.beta, u, v, Np);
      } else {
#pragma unroll
        for (int s = 0; s < NP; ++s) Np[s] = Ng[s];
      }
    } else {
      sparse_phys_basis<NP>(a.disc, a.beta, u, v, Np);
    }
    // (tested anew for every point: a loop for each of the sets would interleave its rows and
    // take all registers)
    unsigned now = __builtin_amdgcn_readfirstlane(m);
    if (B > 1) asm volatile("" : "+s"(now));
#pragma unroll
    for (int j = 0; j < B; ++j) {
      if (B > 1 && !((now >> j) & 1u)) continue;
      double Fr, Fi, Gr, Gi;
      sparse_point_kernels<CPLX, FAST>(y, sf.n, sf.J, x[j], wq, a.kr, a.ki, tr, Fr, Fi, Gr, Gi);
#pragma unroll
      for (int s = 0; s < NP; ++s) {
        acc[j][s][0] = fma(Fr, Np[s], acc[j][s][0]);
        acc[j][s][1] = fma(Fi, Np[s], acc[j][s][1]);
        acc[j][s][2] = fma(Gr, Np[s], acc[j][s][2]);
        acc[j][s][3] = fma(Gi, Np[s], acc[j][s][3]);
      }
    }
  }
}

// The block's copy of the trig table (every thread of the block takes part, before any
// leaves).
__device__ __forceinline__ Trig load_trig(const SparseArgs& a, double* s_trig) {
  for (int j = threadIdx.x; j < kTrigDoubles + kExpN; j += blockDim.x) s_trig[j] = a.trig[j];
  __syncthreads();
  return make_trig(s_trig);
}

__device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

template <int NG>
__device__ __forceinline__ void sparse_element(const SparseArgs& a, int e, Surface<NG>& sf) {
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int node = a.topo[(size_t)e * NG + g];
#pragma unroll
    for (int d = 0; d < 3; ++d) sf.X[g][d] = a.coords[3 * (size_t)node + d];
  }
  sf.begin();
}

template <int NP, bool SUM>
__device__ __forceinline__ void sparse_add(const SparseArgs& a, int64_t p, bool writes,
                                           const double (&acc)[NP][4]) {
  const bool doF = (a.flags & BIE_F) != 0, doG = (a.flags & BIE_G) != 0;
#pragma unroll
  for (int s = 0; s < NP; ++s) {
    double v[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) v[t] = SUM ? wave_sum_d(acc[s][t]) : acc[s][t];
    if (writes) {
      const size_t e = 2 * (size_t)a.pos[p * NP + s];
      if (doF) {
        unsafeAtomicAdd(a.F + e, v[0]);
        unsafeAtomicAdd(a.F + e + 1, v[1]);
      }
      if (doG) {
        unsafeAtomicAdd(a.G + e, v[2]);
        unsafeAtomicAdd(a.G + e + 1, v[3]);
      }
    }
  }
}

// One wave per pair.
template <int NG, int NP, bool CPLX, bool FAST>
__global__ void __launch_bounds__(256) k_sparse_pairs(const SparseArgs a) {
  const int64_t p =
      (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  __shared__ double s_trig[kTrigDoubles + kExpN];
  const Trig tr = load_trig(a, s_trig);
  if (p >= a.n_pairs) return;  // the whole wave leaves together
  const int lane = threadIdx.x & 63;
  const int2 pr = a.pairs[p];
  double x[1][3];
#pragma unroll
  for (int d = 0; d < 3; ++d) x[0][d] = a.src[3 * (size_t)pr.x + d];
  // no distance below Inf (non-finite coordinates) falls to the sixth rule, the
  // reference's final else branch (assembly_collocation_losses.jl:390-395)
  const int c = __builtin_amdgcn_readfirstlane(
      select_rule<NG>(x[0][0], x[0][1], x[0][2], a.gsel + (size_t)pr.y * NG * 4, 6, a.hyp) - 1);
  Surface<NG> sf;
  sparse_element<NG>(a, pr.y, sf);
  double acc[1][NP][4] = {};
  const double* R0 = a.rules + (size_t)a.off[c] * kSparseRec;
  if (a.len[c] > 0)
    sparse_rule<NG, NP, 1, CPLX, FAST>(a, sf, x, 1u, R0, lane, a.len[c], 64, tr, acc);
  sparse_add<NP, true>(a, p, lane == 0, acc[0]);
}

// Short rules (the partial near field's gauss_points_triangle(n), n <= 13): one thread per
// pair instead of one wave, the same per-point evaluation; the thread adds its sums into
// the entries with FP64 atomics.
template <int NG, int NP, bool CPLX, bool FAST>
__global__ void __launch_bounds__(256) k_sparse_pairs_short(const SparseArgs a) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  __shared__ double s_trig[kTrigDoubles + kExpN];
  const Trig tr = load_trig(a, s_trig);
  if (p >= a.n_pairs) return;
  const int2 pr = a.pairs[p];
  double x[1][3];
#pragma unroll
  for (int d = 0; d < 3; ++d) x[0][d] = a.src[3 * (size_t)pr.x + d];
  const int c =
      select_rule<NG>(x[0][0], x[0][1], x[0][2], a.gsel + (size_t)pr.y * NG * 4, 6, a.hyp) - 1;
  Surface<NG> sf;
  sparse_element<NG>(a, pr.y, sf);
  double acc[1][NP][4] = {};
  const double* R0 = a.rules + (size_t)a.off[c] * kSparseRec;
  if (a.len[c] > 0)
    sparse_rule<NG, NP, 1, CPLX, FAST>(a, sf, x, 1u, R0, 0, a.len[c], 1, tr, acc);
  sparse_add<NP, false>(a, p, true, acc[0]);
}

// Rows per batch, at two waves a SIMD (256 registers): the most that paid.  One- and three-node
// physics on flat elements fit; with curved elements or six nodes some registers spill (the
// branch-free kernels: 10-14 with three rows of three nodes on curved elements, with two of six
// nodes 35-41 on flat and 121-125 on curved ones).  (Depth 2, two to four
// thousand nodes, us: three six-node rows 3078 against 2992 with two, and in 512 registers 3666;
// four three-node rows 2495 and 3181 on flat and curved elements against 2386 and 1979 with
// three.)
constexpr int batch_rows(int NP) { return NP == 1 ? 4 : NP == 3 ? 3 : 2; }

// Batches of up to B pairs that share an element (built on the host, grouped by the rule
// the mesh sources select): one wave per batch evaluates the surface at each point of a rule
// once and the kernels for every row of the batch that selected that rule - the surface
// (~2/3 of the per-point work) is shared.  Each row's rule is selected here exactly as in
// k_sparse_pairs, so explicit sources stay correct (they only share less).
// CHECK: compiled apart (in the loop's registers its few instructions cost 3 %).
template <int NG, int NP, int B, bool CPLX, bool FAST, bool CHECK>
__global__ void __launch_bounds__(256, 2) k_sparse_batch(const SparseArgs a) {
  const int64_t b =
      (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  __shared__ double s_trig[kTrigDoubles + kExpN];
  const Trig tr = load_trig(a, s_trig);
  if (b >= a.n_batches) return;  // the whole wave leaves together
  const int lane = threadIdx.x & 63;
  const int* rec = a.batches + (size_t)b * 8;
  const int e = rec[0], cnt = rec[1];
  if (CHECK && a.check) {  // whether the batch is this launch's (the whole wave leaves together)
    bool near = true;
    for (int j = 0; j < cnt; ++j) {
      const double* x = a.src + 3 * (size_t)a.pairs[rec[2 + j]].x;
      const double cx = x[0] - a.center[0], cy = x[1] - a.center[1], cz = x[2] - a.center[2];
      const double dist = sqrt(fma(cx, cx, fma(cy, cy, cz * cz))) + a.reach;
      near = near && fabs(a.kr) * dist < 0.5 * kTabFastMaxArg && dist < kFastMaxDist;
    }
    if (__builtin_amdgcn_readfirstlane((int)near) != (FAST ? 1 : 0)) return;
  }
  Surface<NG> sf;
  sparse_element<NG>(a, e, sf);
  double xs[B][3];
  int cr[B], pj[B];
#pragma unroll
  for (int j = 0; j < B; ++j) {
    pj[j] = j < cnt ? rec[2 + j] : -1;
    cr[j] = -1;
    xs[j][0] = xs[j][1] = xs[j][2] = 0.0;
    if (pj[j] >= 0) {
      const int row = a.pairs[pj[j]].x;
      xs[j][0] = a.src[3 * (size_t)row];
      xs[j][1] = a.src[3 * (size_t)row + 1];
      xs[j][2] = a.src[3 * (size_t)row + 2];
      cr[j] = select_rule<NG>(xs[j][0], xs[j][1], xs[j][2], a.gsel + (size_t)e * NG * 4, 6,
                              a.hyp) - 1;
    }
    cr[j] = __builtin_amdgcn_readfirstlane(cr[j]);
  }
  double acc[B][NP][4] = {};
  unsigned done = 0u;
  for (int j0 = 0; j0 < B; ++j0) {
    if (cr[j0] < 0 || ((done >> j0) & 1u)) continue;
    const int c = cr[j0];
    unsigned m = 0u;  // the rows whose rule has these records (filler slots share them)
#pragma unroll
    for (int j = 0; j < B; ++j)
      if (cr[j] >= 0 && a.off[cr[j]] == a.off[c] && a.len[cr[j]] == a.len[c]) m |= 1u << j;
    done |= m;
    const double* R0 = a.rules + (size_t)a.off[c] * kSparseRec;
    if (a.len[c] > 0)
      sparse_rule<NG, NP, B, CPLX, FAST>(a, sf, xs, m, R0, lane, a.len[c], 64, tr, acc);
  }
#pragma unroll
  for (int j = 0; j < B; ++j)
    if (pj[j] >= 0) sparse_add<NP, true>(a, pj[j], lane == 0, acc[j]);
}

}  // namespace

void launch_sparse_pairs(const SparseLaunch& L, hipStream_t s) {
  if (L.n_pairs == 0) return;
  SparseArgs a{};
  a.src = L.src;
  a.pairs = L.pairs;
  a.pos = L.pos;
  a.n_pairs = L.n_pairs;
  a.coords = L.coords;
  a.topo = L.topo;
  a.gsel = L.gsel;
  a.rules = L.rules;
  a.trig = L.trig;
  for (int c = 0; c < 6; ++c) {
    a.off[c] = L.off[c];
    a.len[c] = L.len[c];
  }
  for (int d = 0; d < 3; ++d) a.center[d] = L.center[d];
  a.reach = L.reach;
  a.hyp = L.hyp;
  a.batches = L.batches;
  a.n_batches = L.n_batches;
  a.disc = L.disc;
  a.beta = L.beta;
  a.kr = L.kr;
  a.ki = L.ki;
  a.flags = L.flags;
  a.F = L.F;
  a.G = L.G;
  // every slot's rule short (the partial near field): one thread per pair
  int qmax = 0;
  for (int c = 0; c < 6; ++c) qmax = std::max(qmax, L.len[c]);
  const bool shortr = qmax <= 16;
  const bool batched = !shortr && L.batches != nullptr && L.n_batches > 0;
  const int64_t blocks = shortr    ? (L.n_pairs + 255) / 256
                         : batched ? (L.n_batches + 3) / 4
                                   : (L.n_pairs + 3) / 4;
  BIE_REQUIRE(blocks < 2147483647LL, BIE_EINVAL, "too many sparse pairs");
  const dim3 grid((unsigned)blocks);
  const bool cplx = L.ki != 0.0;
  auto run = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(256), 0, s, a); };
  // geometry nodes 3 or 6; physics nodes 1 (discontinuous constant), 3 or 6
  auto pick = [&](auto ng, auto np, auto cx) {
    constexpr int NG = decltype(ng)::value, NP = decltype(np)::value;
    constexpr bool C = decltype(cx)::value;
    constexpr int B = batch_rows(NP);
    if (shortr)
      L.fast ? run(k_sparse_pairs_short<NG, NP, C, true>)
             : run(k_sparse_pairs_short<NG, NP, C, false>);
    else if (batched) {
      // Explicit sources: the waves whose rows are near and the others are a launch each, the
      // second as a rule empty (4 us).  The full reduction beside the sums of several rows
      // takes more registers than there are: all waves with it, two launches, and sources known
      // to be near (us, depth 2): 1962 linear nodes 606, 557, 515; complex k 931, 663, 638;
      // 2562 quadratic nodes 2095, 1833, 1822; disctrilinear on 720 quadratic elements 935,
      // 704, 690.
      a.check = L.explicit_src && !L.fast;
      if (L.fast) run(k_sparse_batch<NG, NP, B, C, true, false>);
      if (a.check) run(k_sparse_batch<NG, NP, B, C, true, true>);
      if (!L.fast) run(k_sparse_batch<NG, NP, B, C, false, true>);
    } else {
      L.fast ? run(k_sparse_pairs<NG, NP, C, true>) : run(k_sparse_pairs<NG, NP, C, false>);
    }
  };
  auto by_cx = [&](auto ng, auto np) {
    cplx ? pick(ng, np, std::true_type()) : pick(ng, np, std::false_type());
  };
  auto by_np = [&](auto ng) {
    if (L.NP == 1)
      by_cx(ng, std::integral_constant<int, 1>());
    else if (L.NP == 3)
      by_cx(ng, std::integral_constant<int, 3>());
    else
      by_cx(ng, std::integral_constant<int, 6>());
  };
  BIE_REQUIRE((L.NG == 3 || L.NG == 6) && (L.NP == 1 || L.NP == 3 || L.NP == 6), BIE_EINVAL,
              "internal: sparse kernel node counts");
  if (L.NG == 3)
    by_np(std::integral_constant<int, 3>());
  else
    by_np(std::integral_constant<int, 6>());
  BIE_HIP_CHECK(hipGetLastError());
}

int sparse_record_doubles() { return kSparseRec; }

int sparse_batch_rows(int NP) { return batch_rows(NP); }

}  // namespace bie
