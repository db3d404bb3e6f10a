// Dense assembly kernel of the collocation operators (gfx950, FP64): the row loop of
// assemble_parallel! (src/3d/assembly_collocation.jl:314-349, 424-475) for one mesh, or for
// an uneven batch of meshes, in one persistent launch without barriers between elements.
//
// A workgroup takes tiles of 64 target rows (lane = row) x one segment of elements.  Its
// waves draw the segment's elements one at a time from a counter, choose the rule of every
// (row, element) pair (find_closest_corner, :102-115), integrate the pair
// (computing_integrals!, :213-252) and bring the element's node sums to LDS slots:
//   * the first wave to reach a node writes its sums into the slot, the following ones add
//     to it with LDS atomics, the last one reads the slot, adds its own sums and writes the
//     64 rows of the column (1 KB, streaming) - so a slot needs no zero fill and no flush
//     pass, and a node with two elements (a mid-edge node) costs one LDS write and one read;
//   * a node with one element in the segment goes straight from registers to its column;
//   * columns that other segments add to as well take FP64 atomics into zeroed columns.
// What bounds it: FP64 issue and, on curved elements, LDS reads (the table row, the basis
// values and the trig entry of a point are 120 bytes per lane).  A wave waits for nothing
// but its own loads, so sixteen waves per CU (four per SIMD, 128 VGPRs) keep the FP64 pipe
// supplied; with eight waves that met at a barrier after every element the pipe was 40 %
// busy.
//
// Flat elements (three-node geometry): y - x = (X1 - x) + N2 (X2 - X1) + N3 (X3 - X1), n and
// J are constants of the element, so n.d J is one number per pair and a point needs only
// {N1, N2, N3, w} (which are the basis values too).  The element's 24 numbers are read by
// scalar loads.  Curved elements and other physics read y, n, J w / (4 pi) per point from
// rows that the wave staged in LDS.
//
// Before (eight waves, a barrier after every eight elements) and now, F, G and C (us):
// 4002 linear nodes, 16 points 1333 -> 1100 (57 of 71 instructions per point are the formula's);
// 642 nodes, 4 points 144 -> 36; 10242 quadratic nodes, 6 points 2302 -> 1750, of which the
// mid-edge kernel takes 254 and the preparation 48; 3242 quadratic nodes, complex k, 16 points
// 625 -> 420; 24 linear meshes of 500-6000 nodes 16910 -> 12770.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "bie_common.hpp"
#include "stream_device.hpp"

namespace bie {
namespace {

// ---- one pair ----------------------------------------------------------------------------

// Pair on a curved element (or any with tabulated points): rows of 8 doubles y, n,
// J w / (4 pi), 0 and basis values ph (NP per point).  Staged rows (LDS): the next point's y
// and this point's n and J w are read before the point is begun, its basis values behind the
// trig entry, so that every LDS latency is behind arithmetic of the same wave.
template <int NP, bool CPLX, bool GON, bool FAST, bool FIRST, bool AHEAD>
__device__ __forceinline__ void point_row(double x0, double x1, double x2, double (&y)[3],
                                          const double* row, const double* ph, double kr,
                                          double ki, const Trig& tr, Sums<NP, GON>& v,
                                          double& csum) {
  const double dx = y[0] - x0, dy = y[1] - x1, dz = y[2] - x2;
  const double n0 = row[3], n1 = row[4], n2 = row[5], jw = row[6];
  if constexpr (AHEAD) {
#pragma unroll
    for (int d = 0; d < 3; ++d) y[d] = row[8 + d];
    __builtin_amdgcn_sched_barrier(0);
  }
  const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
  const double rinv = rsqrt_nr(r2);
  const double r = r2 * rinv;
  const double krr = kr * r, kir = CPLX ? ki * r : 0.0;
  Phase<CPLX, FAST> e;
  e.begin(krr, kir, tr);
  double b[NP];
#pragma unroll
  for (int s = 0; s < NP; ++s) b[s] = ph[s];
  if constexpr (AHEAD) __builtin_amdgcn_sched_barrier(0);
  const double nd = fma(n0, dx, fma(n1, dy, n2 * dz));
  const double g = jw * rinv;
  const double t = nd * (rinv * rinv);
  csum = fma(-t, g, csum);
  double Fr, Fi, Gr, Gi;
  kernels_end<CPLX, FAST>(e, g, t, krr, kir, tr, Fr, Fi, Gr, Gi);
#pragma unroll
  for (int s = 0; s < NP; ++s) v.template add<FIRST>(s, b[s], Fr, Fi, Gr, Gi);
}

// AHEAD: rows lie in LDS with at least one more row's memory behind them.
template <int NP, bool CPLX, bool GON, bool FAST, bool AHEAD>
__device__ __forceinline__ void pair_rows(double x0, double x1, double x2,
                                          const double* rows, const double* ph, int Q,
                                          double kr, double ki, const Trig& tr,
                                          Sums<NP, GON>& v, double& csum) {
  double y[3] = {rows[0], rows[1], rows[2]};
  point_row<NP, CPLX, GON, FAST, true, AHEAD>(x0, x1, x2, y, rows, ph, kr, ki, tr, v, csum);
  int q = 1;
  if constexpr (AHEAD) {  // two points at a time
    if (!(Q & 1)) {
      point_row<NP, CPLX, GON, FAST, false, true>(x0, x1, x2, y, rows += 8, ph += NP, kr, ki, tr,
                                                  v, csum);
      q = 2;
    }
#pragma unroll 1
    for (; q < Q; q += 2, rows += 16, ph += 2 * NP) {
      point_row<NP, CPLX, GON, FAST, false, true>(x0, x1, x2, y, rows + 8, ph + NP, kr, ki, tr, v,
                                                  csum);
      point_row<NP, CPLX, GON, FAST, false, true>(x0, x1, x2, y, rows + 16, ph + 2 * NP, kr, ki,
                                                  tr, v, csum);
    }
  } else {
#pragma unroll 1
    for (; q < Q; ++q) {
      rows += 8;
      ph += NP;
#pragma unroll
      for (int d = 0; d < 3; ++d) y[d] = rows[d];
      point_row<NP, CPLX, GON, FAST, false, false>(x0, x1, x2, y, rows, ph, kr, ki, tr, v, csum);
    }
  }
}

// Pair on a flat three-node element with its own linear physics: tab holds {N1, N2, N3,
// w / (4 pi)} per point; a, b are the edges from node 1, d0 = X1 - x.  The sums leave out
// the constant factors J (of G) and n.d J (of F and C), which the caller multiplies in; where
// lengths may be anywhere in the range (not FAST) 1 / r^3 is not formed by itself, and F and C
// take n.d J here.
template <bool CPLX, bool GON, bool FAST, bool FIRST>
__device__ __forceinline__ void point_flat(const double (&d0)[3], const double (&a)[3],
                                           const double (&b)[3], double (&n)[4],
                                           const double* next, double kr, double ki, double nd,
                                           const Trig& tr, Sums<3, GON>& v, double& c3) {
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
  const double krr = kr * r, kir = CPLX ? ki * r : 0.0;
  Phase<CPLX, FAST> e;
  e.begin(krr, kir, tr);
  const double g = m[3] * rinv;
  const double t = FAST ? rinv * rinv : (nd * rinv) * rinv;
  c3 = FIRST ? t * g : fma(t, g, c3);
  double Fr, Fi, Gr, Gi;
  kernels_end<CPLX, FAST>(e, g, t, krr, kir, tr, Fr, Fi, Gr, Gi);
#pragma unroll
  for (int s = 0; s < 3; ++s) v.template add<FIRST>(s, m[s], Fr, Fi, Gr, Gi);
}

// (the table has room for one more point behind its last)
template <bool CPLX, bool GON, bool FAST>
__device__ __forceinline__ void pair_flat(const double (&d0)[3], const double (&a)[3],
                                          const double (&b)[3], const double* tab, int Q,
                                          double kr, double ki, double nd, const Trig& tr,
                                          Sums<3, GON>& v, double& c3) {
  double n[4] = {tab[0], tab[1], tab[2], tab[3]};
  point_flat<CPLX, GON, FAST, true>(d0, a, b, n, tab += 4, kr, ki, nd, tr, v, c3);
  int q = 1;
  if (!(Q & 1)) {
    point_flat<CPLX, GON, FAST, false>(d0, a, b, n, tab += 4, kr, ki, nd, tr, v, c3);
    q = 2;
  }
#pragma unroll 1
  for (; q < Q; q += 2, tab += 8) {  // two points at a time
    point_flat<CPLX, GON, FAST, false>(d0, a, b, n, tab + 4, kr, ki, nd, tr, v, c3);
    point_flat<CPLX, GON, FAST, false>(d0, a, b, n, tab + 8, kr, ki, nd, tr, v, c3);
  }
}

// ---- hand-over of an element's node sums -------------------------------------------------

// First and middle contributions: into the slot.
template <int NP, bool GON>
__device__ __forceinline__ void give(const int4& en, const Roles& r, int lane, double* acc,
                                     unsigned* claims, unsigned* ctr, const Sums<NP, GON>& v,
                                     bool& ok) {
  constexpr int SD = GON ? 256 : 128;
  const bool mine_first = lane_of_mask(r.first), mine_more = lane_of_mask(r.more);
#pragma unroll
  for (int s = 0; s < NP; ++s)
    if ((r.first >> s) & 1) {
      double* p = acc + (size_t)__builtin_amdgcn_readlane(en.x, s) * SD + lane;
      p[0] = v.fr[s];
      p[64] = v.fi[s];
      if constexpr (GON) {
        p[128] = v.gr[s];
        p[192] = v.gi[s];
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
        atomicAdd(p, v.fr[s]);
        atomicAdd(p + 64, v.fi[s]);
        if constexpr (GON) {
          atomicAdd(p + 128, v.gr[s]);
          atomicAdd(p + 192, v.gi[s]);
        }
      }
    lds_wait();
    if (mine_more) lds_count(claims + en.x, 0x10000u);
  }
}

// Last contributions: the slot's sums plus this wave's go to the column; the slot is free.
template <int NP, bool GON>
__device__ __forceinline__ void finish(InstPtr in, const int4& en, const Roles& r,
                                       int lane, int64_t i0, bool active, const double* acc,
                                       unsigned* claims, unsigned* turns, unsigned* ctr,
                                       const Sums<NP, GON>& v, bool ok) {
  constexpr int SD = GON ? 256 : 128;
  const bool mine = lane_of_mask(r.last);
  if (r.last)
    ok = spin(ctr, [&] {
           return !mine || (lds_peek(claims + en.x) >> 16) == (unsigned)en.y - 1u;
         }) && ok;
  const double bad = ok ? 0.0 : NAN;
  const InstPtr p = fresh(in);
  const bool doF = (p->a.flags & BIE_F) != 0;
  const int64_t M = p->a.M;
  double *F = p->a.F, *G = p->a.G;
#pragma unroll
  for (int s = 0; s < NP; ++s) {
    const bool last = (r.last >> s) & 1;
    if (!last && !((r.direct >> s) & 1)) continue;
    double f0 = v.fr[s] + bad, f1 = v.fi[s], g0 = 0.0, g1 = 0.0;
    if constexpr (GON) {
      g0 = v.gr[s] + bad;
      g1 = v.gi[s];
    }
    if (last) {
      const double* q = acc + (size_t)__builtin_amdgcn_readlane(en.x, s) * SD + lane;
      f0 += q[0];
      f1 += q[64];
      if constexpr (GON) {
        g0 += q[128];
        g1 += q[192];
      }
    }
    const int nw = __builtin_amdgcn_readlane(en.w, s);
    const bool shared = (nw & kSharedBit) != 0;
    const size_t at = 2 * ((size_t)i0 + (size_t)(nw & ~kSharedBit) * (size_t)M);
    if (active) {
      if (doF) column_store(F + at, 16u * lane, shared, f0, f1);
      if constexpr (GON) column_store(G + at, 16u * lane, shared, g0, g1);
    }
  }
  if (mine && ok) {  // after the slot's reads above (LDS operations of a wave are in order)
    lds_wait();
    lds_poke(claims + en.x, 0u);
    lds_poke(turns + en.x, (unsigned)en.z + 1u);
  }
}

template <bool CPLX, bool GON, bool FAST>
__global__ void __launch_bounds__(256)
k_stream_mid(const StreamInst one, const double* tab_src, int tab_doubles) {
  extern __shared__ double lds[];
  const InstPtr in = (InstPtr)__builtin_amdgcn_kernarg_segment_ptr();
  const int mid_off = in->mid_off;
  const int ntab = tab_doubles - mid_off + kTrigDoubles + kExpN;
  for (int t = threadIdx.x; t < ntab; t += 256) lds[t] = tab_src[mid_off + t];
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const MidOut o{in->a.kr, in->a.ki, in->a.F, in->a.G, (in->a.flags & BIE_C) != 0, 0};
  mid_pairs<CPLX, GON, FAST, false>(in, o, lds, make_trig(lds + tab_doubles - mid_off),
                             blockIdx.x * 4 + wave, gridDim.x * 4, threadIdx.x & 63);
}

// ---- the tile loop -----------------------------------------------------------------------

// Elements of the tile's segment, drawn by this wave.  FAST: every |k| r of the tile is below
// the bound of the branch-free sincos.
template <int NP, int MODE, bool CPLX, bool GON, int W, bool FAST>
__device__ __forceinline__ void stream_tile(InstPtr in, int rb, int seg, int S,
                                            int tab_doubles, double* lds,
                                            int parity) {
  constexpr int SD = GON ? 256 : 128;
  constexpr bool FLAT = MODE == kFlat, STAGED = MODE == kStaged;
  constexpr bool kMids = NP == 6 && !FLAT;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int R = in->a.R;
  const int rules = R < 3 ? R : 3;
  const int Q = in->a.len[0];
  const int row_doubles = STAGED ? stage_rows_doubles(Q, rules) : 0;
  const Layout L = layout_of(S, SD, tab_doubles, W, row_doubles, kMids && R == 6);
  double* acc = lds;
  const double* tab = lds + L.tab;
  const Trig tr = make_trig(tab + tab_doubles);
  double* my_rows = lds + L.rows + (size_t)wave * row_doubles;
  unsigned* claims = reinterpret_cast<unsigned*>(lds + L.words);
  unsigned* turns = claims + S;
  unsigned* ctr = turns + S;
  const int64_t i = (int64_t)rb * 64 + lane;
  const int64_t M = in->a.M;
  const bool active = i < M;
  const double* xt = in->a.targets + 3 * (active ? i : M - 1);
  const double x0 = xt[0], x1 = xt[1], x2 = xt[2];
  double kr = in->a.kr, ki = CPLX ? in->a.ki : 0.0;
  asm volatile("" : "+s"(kr), "+s"(ki));  // stays in registers (not reloaded per point)
  const int t0 = sload(in->seg_begin + seg), t1 = sload(in->seg_begin + seg + 1);
  const int n16 = 4 * Q * rules;                     // 16-byte chunks of an element's rows
  const int tab_rule = FLAT ? 4 * Q + 2 : ((Q * NP + 1) & ~1) + 2;  // table stride of a rule
  auto draw = [&]() -> int { return t0 + (int)lds_draw(ctr + kTicket, 1u, lane); };
  // staged rows of the element at position p: global -> registers, registers -> LDS
  double2 stg[3];
  auto rows_load = [&](int p) {
    typedef unsigned int u4 __attribute__((ext_vector_type(4)));
    const InstPtr u = fresh(in);
    const int l = fresh_lane(lane);
    const int e = sload(u->order + min(p, t1 - 1));
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<double*>(u->a.elem + (size_t)e * u->a.Pe * 8), (short)0, n16 * 16,
        0x00020000);
#pragma unroll
    for (int t = 0; t < 3; ++t)
      stg[t] = __builtin_bit_cast(
          double2, (u4)__builtin_amdgcn_raw_buffer_load_b128(rs, (l + 64 * t) * 16, 0, 0));
  };
  auto rows_store = [&] {
    const int l = fresh_lane(lane);
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const int j = l + 64 * t;
      if (j < n16)
        reinterpret_cast<double2*>(my_rows)[j + (j >= 4 * Q) + (j >= 8 * Q)] = stg[t];
    }
  };
  double csum = 0.0;  // (flat)
  int pos = draw();
  if constexpr (STAGED)
    if (pos < t1) {
      rows_load(pos);
      rows_store();
    }
  while (pos < t1) {
    const int nxt = draw();
    const InstPtr u = fresh(in);
    Sums<NP, GON> v;
    if constexpr (FLAT) {
      const double* rec = u->flat + (size_t)pos * kFlatDoubles;
      const d8 r0 = sload8(rec), r1 = sload8(rec + 8), r2 = sload8(rec + 16);
      const double P[3][3] = {{r0[0], r0[1], r0[2]}, {r0[3], r0[4], r0[5]},
                              {r0[6], r0[7], r1[0]}};
      const double ea[3] = {r1[4], r1[5], r1[6]}, eb[3] = {r1[7], r2[0], r2[1]};
      const int c = select_rule_s<3>(x0, x1, x2, P, rec, R, in) - 1;
      const double d0[3] = {r1[1] - x0, r1[2] - x1, r1[3] - x2};
      const double nd = fma(r2[2], d0[0], fma(r2[3], d0[1], r2[4] * d0[2]));  // n.d J
      const double J = r2[5];
      double c3 = 0.0;
      pair_flat<CPLX, GON, FAST>(d0, ea, eb, tab + c * tab_rule, Q, kr, ki, nd, tr, v, c3);
      csum = FAST ? fma(-nd, c3, csum) : csum - c3;
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        if constexpr (FAST) {
          v.fr[s] *= nd;
          v.fi[s] *= nd;
        }
        if constexpr (GON) {
          v.gr[s] *= J;
          v.gi[s] *= J;
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
      // lanes with a mid-edge rule run along on rule 1 and leave nothing
      const bool mid = kMids && c >= 3;
      double csum = 0.0;
      const int cr = mid ? 0 : c;
      if constexpr (STAGED)
        pair_rows<NP, CPLX, GON, FAST, true>(x0, x1, x2, my_rows + (size_t)cr * (8 * Q + 2),
                                       tab + (size_t)cr * tab_rule, Q, kr, ki, tr, v, csum);
      else  // (the vertex rules come first in the table, Q points each)
        pair_rows<NP, CPLX, GON, FAST, false>(
            x0, x1, x2,
            u->a.elem + ((size_t)sload(u->order + pos) * u->a.Pe + (size_t)cr * Q) * 8,
            tab + (size_t)cr * tab_rule, Q, kr, ki, tr, v, csum);
      if (kMids && R == 6) {  // queue the mid-edge pairs of this element
        const unsigned long long mask = __ballot(mid && active);
        if (__any(mid)) {
          v.keep(!mid);
          csum = mid ? 0.0 : csum;
        }
        if (mask) {
          const unsigned base = lds_draw(ctr + kMidN + parity, (unsigned)__popcll(mask), lane);
          const unsigned at = base + __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
          if (mid && active && at < (unsigned)kStreamMid)  // position, rule, row of the pair
            reinterpret_cast<unsigned*>(lds + L.queue)[parity * kStreamMid + at] =
                ((unsigned)(pos - t0) << 8) | ((unsigned)(c - 3) << 6) | (unsigned)lane;
        }
      }
      atomicAdd(lds + L.csum + fresh_lane(lane), csum);
      if constexpr (STAGED) rows_load(nxt);
    }
    const int l = fresh_lane(lane);
    const int4 en = fresh(in)->ent[(size_t)pos * NP + min(l, NP - 1)];
    bool ok;
    const Roles r = claim<NP>(en, l, claims, turns, ctr, ok);
    give<NP, GON>(en, r, l, acc, claims, ctr, v, ok);
    // before the column stores: loads and stores retire in order, so waiting for the rows
    // behind them would wait for the stores
    if constexpr (STAGED) rows_store();
    finish<NP, GON>(in, en, r, l, (int64_t)rb * 64, active, acc, claims, turns, ctr, v,
                    ok);
    pos = nxt;
  }
  if constexpr (FLAT) atomicAdd(lds + L.csum + lane, csum);
}

template <int NP, int MODE, bool CPLX, bool GON, int W, bool FAST, class InstOf>
__device__ __forceinline__ void run_tiles(InstOf inst_of, int n_tiles, const StreamRun& run) {
  extern __shared__ double lds[];
  stream_run<GON ? 256 : 128, W, NP == 6 && MODE != kFlat, FAST>(
      inst_of, [](InstPtr in, int) { return fabs(in->a.kr); }, [](InstPtr, int) { return true; },
      [&](InstPtr in, int rb, int seg, int, int parity) {
        stream_tile<NP, MODE, CPLX, GON, W, FAST>(in, rb, seg, run.S, run.tab_doubles, lds,
                                                  parity);
      },
      n_tiles, run);
}

template <int NP, int MODE, bool CPLX, bool GON, int W, bool FAST>
__global__ void __launch_bounds__(64 * W)
k_stream(const StreamInst one, int n_tiles, const StreamRun run) {
  // `one` is the first kernel argument: read in place
  const InstPtr in = (InstPtr)__builtin_amdgcn_kernarg_segment_ptr();
  auto inst_of = [&](int tile, int& rb, int& seg) -> InstPtr {
    const int n = in->n_rowblocks;
    seg = tile / n;
    rb = tile - seg * n;
    return in;
  };
  run_tiles<NP, MODE, CPLX, GON, W, FAST>(inst_of, n_tiles, run);
}

// An uneven batch: the tile list names instance, row block and segment; counters, lists and
// tables are shared.
template <int NP, int MODE, bool CPLX, bool GON, int W, bool FAST>
__global__ void __launch_bounds__(64 * W)
k_stream_batch(const BatchInst* insts, const int4* tiles, int n_tiles, const StreamRun run) {
  auto inst_of = [&](int tile, int& rb, int& seg) -> InstPtr {
    typedef int i4 __attribute__((ext_vector_type(4), aligned(16)));
    const i4 t = *reinterpret_cast<const __attribute__((address_space(4))) i4*>(
        reinterpret_cast<uintptr_t>(tiles + tile));
    rb = t.y;
    seg = t.z;
    return (InstPtr) reinterpret_cast<uintptr_t>(&insts[t.x].s);
  };
  run_tiles<NP, MODE, CPLX, GON, W, FAST>(inst_of, n_tiles, run);
}

// The listed mid-edge pairs of every instance (blockIdx.y).
template <bool CPLX, bool GON, bool FAST>
__global__ void __launch_bounds__(256)
k_stream_mid_batch(const BatchInst* insts, const double* tab_src, int tab_doubles) {
  extern __shared__ double lds[];
  const InstPtr in = (InstPtr) reinterpret_cast<uintptr_t>(&insts[blockIdx.y].s);
  const int mid_off = in->mid_off;
  const int ntab = tab_doubles - mid_off + kTrigDoubles + kExpN;
  for (int t = threadIdx.x; t < ntab; t += 256) lds[t] = tab_src[mid_off + t];
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const MidOut o{in->a.kr, in->a.ki, in->a.F, in->a.G, (in->a.flags & BIE_C) != 0, 0};
  mid_pairs<CPLX, GON, FAST, false>(in, o, lds, make_trig(lds + tab_doubles - mid_off),
                             blockIdx.x * 4 + wave, gridDim.x * 4, threadIdx.x & 63);
}

// ---- preparation -------------------------------------------------------------------------

// Per-call preparation of every instance of a batch (blockIdx.y): C zeroed, the columns that
// several segments add to and disabled non-NULL outputs zeroed, the lists emptied.
__global__ void __launch_bounds__(256)
k_stream_batch_prep(const BatchInst* __restrict__ insts, unsigned* counters) {
  const BatchInst& b = insts[blockIdx.y];
  const AssemblyArgs& a = b.s.a;
  const double2 z = make_double2(0.0, 0.0);
  if (blockIdx.x == 0) {
    if (blockIdx.y == 0 && threadIdx.x < kMidCount) counters[threadIdx.x] = 0u;
    if (threadIdx.x < 3 && b.s.mid_queue)
      b.s.mid_count[threadIdx.x] = threadIdx.x == 2 ? b.s.mid_cap : 0u;
    if (a.C)
      for (int64_t r = threadIdx.x; r < a.M; r += 256) reinterpret_cast<double2*>(a.C)[r] = z;
  }
  double* outs[2] = {a.F, a.G};
  const unsigned bits[2] = {BIE_F, BIE_G};
  for (int o = 0; o < 2; ++o) {
    double2* X = reinterpret_cast<double2*>(outs[o]);
    if (!X) continue;
    const bool whole = !(a.flags & bits[o]);
    const int64_t ncols = whole ? a.N : b.n_zero;
    for (int64_t c = blockIdx.x; c < ncols; c += gridDim.x) {
      double2* col = X + (size_t)(whole ? c : b.zero_cols[c]) * a.M;
      for (int64_t r = threadIdx.x; r < a.M; r += 256) col[r] = z;
    }
  }
}

// y, n, J w / (4 pi) of one vertex-rule point of one element (interpolate_elements, jacobian!).
__device__ __forceinline__ void geometry_point(const StreamPrep& p, int64_t t) {
  const int e = (int)(t / p.Pv), q = (int)(t - (int64_t)e * p.Pv);
  const double* P = p.pts + (size_t)q * kPtStride;
  double y[3] = {0, 0, 0}, tu[3] = {0, 0, 0}, tv[3] = {0, 0, 0};
  for (int k = 0; k < p.gk; ++k) {
    const double* X = p.coords + 3 * (size_t)p.topo[(size_t)e * p.gk + k];
    const double N = P[kPtN + k], du = P[kPtDu + k], dv = P[kPtDv + k];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      y[d] += X[d] * N;
      tu[d] += X[d] * du;
      tv[d] += X[d] * dv;
    }
  }
  const double c0 = tu[1] * tv[2] - tu[2] * tv[1], c1 = tu[2] * tv[0] - tu[0] * tv[2],
               c2 = tu[0] * tv[1] - tu[1] * tv[0];
  const double J = sqrt(c0 * c0 + c1 * c1 + c2 * c2);
  double* o = p.elem + ((size_t)e * p.Pe + q) * 8;
  *reinterpret_cast<double4*>(o) = make_double4(y[0], y[1], y[2], -c0 / J);
  *reinterpret_cast<double4*>(o + 4) =
      make_double4(-c1 / J, -c2 / J, J * P[2] * 0.079577471545947667884, 0.0);
}

// The record of one flat element at its position in the stream (order NULL: its number): selection nodes, X1, the
// edges a, b from it, n J = -(a x b), J.
__device__ __forceinline__ void flat_record(const StreamPrep& p, int t) {
  const int e = p.order ? p.order[t] : t;
  double* o = p.flat + (size_t)t * kFlatDoubles;
  double X[3][3];
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      X[k][d] = p.coords[3 * (size_t)p.topo[(size_t)e * 3 + k] + d];
      o[3 * k + d] = p.sources[3 * (size_t)p.ptopo[(size_t)e * 3 + k] + d];
    }
  double a[3], b[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    a[d] = X[1][d] - X[0][d];
    b[d] = X[2][d] - X[0][d];
    o[9 + d] = X[0][d];
    o[12 + d] = a[d];
    o[15 + d] = b[d];
  }
  const double c0 = a[1] * b[2] - a[2] * b[1], c1 = a[2] * b[0] - a[0] * b[2],
               c2 = a[0] * b[1] - a[1] * b[0];
  const double J = sqrt(c0 * c0 + c1 * c1 + c2 * c2);
  // n = -c / J is not a number, or times J not c, where J leaves the range: F and C are NaN
  const bool normal = J > 0.0 && J < INFINITY;
  o[18] = normal ? -c0 : NAN;
  o[19] = normal ? -c1 : NAN;
  o[20] = normal ? -c2 : NAN;
  o[21] = J;
  o[22] = o[23] = 0.0;
}

// Everything a dense call needs before its kernel, in one launch: the geometry, zeros in C,
// in the columns the kernel adds to and in disabled outputs, and the tile counters.  Blocks
// take the columns' zeros first (blockIdx.x < column blocks), then the rest.
__global__ void __launch_bounds__(256) k_stream_prep(const StreamPrep p) {
  const double2 z = make_double2(0.0, 0.0);
  if ((int)blockIdx.x < p.col_blocks) {
    const int ncols = p.n_zero + p.n_whole;
    for (int64_t t = blockIdx.x; t < (int64_t)p.nk * ncols; t += p.col_blocks) {
      const int64_t q = t / ncols;
      const int c = (int)(t - q * ncols);
      // whole outputs: column c of a disabled one; else a listed column of the enabled ones
      const bool whole = c >= p.n_zero;
      const size_t col = (size_t)q * p.stride +
                         (whole ? (size_t)(c - p.n_zero) : (size_t)p.zero_cols[c]) * p.M;
      double2* x[2] = {reinterpret_cast<double2*>(whole == !(p.flags & BIE_F) ? p.F : nullptr),
                       reinterpret_cast<double2*>(whole == !(p.flags & BIE_G) ? p.G : nullptr)};
      for (int o = 0; o < 2; ++o)
        if (x[o])
          for (int64_t r = threadIdx.x; r < p.M; r += 256) x[o][col + r] = z;
    }
    return;
  }
  const int64_t first = (int64_t)(blockIdx.x - p.col_blocks) * 256 + threadIdx.x;
  const int64_t step = (int64_t)(gridDim.x - p.col_blocks) * 256;
  if (first < kStreamCounters) p.counters[first] = first == kMidEnd ? p.mid_cap : 0u;
  for (int64_t r = first; r < p.M; r += step) reinterpret_cast<double2*>(p.C)[r] = z;
  if (p.flat)
    for (int64_t t = first; t < p.E; t += step) flat_record(p, (int)t);
  if (p.elem)
    for (int64_t t = first; t < (int64_t)p.E * p.Pv; t += step) geometry_point(p, t);
}

__global__ void __launch_bounds__(256) k_stream_flat(const StreamPrep p) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t < p.E) flat_record(p, t);
}

// Calls fn with the kernel of (NP, how rows are read, complex, G, fast sincos).
template <bool BATCH, class Fn>
void with_stream_kernel(int NP, int mode, bool cplx, bool gon, bool fast, Fn&& fn) {
  auto pick = [&](auto np, auto md, auto cx, auto g) {
    constexpr int N = decltype(np)::value;
    constexpr int W = stream_waves(N);
    constexpr int MD = decltype(md)::value;
    constexpr bool CX = decltype(cx)::value, G = decltype(g)::value;
    auto by_fast = [&](auto f) {
      constexpr bool FS = decltype(f)::value;
      constexpr int WV = FS || (N < 6 && !CX) ? W : kSlowWaves;
      if constexpr (BATCH)
        fn(k_stream_batch<N, MD, CX, G, WV, FS>, WV);
      else
        fn(k_stream<N, MD, CX, G, WV, FS>, WV);
    };
    fast ? by_fast(std::true_type{}) : by_fast(std::false_type{});
  };
  auto by_c = [&](auto np, auto md) {
    using T = std::true_type;
    using F = std::false_type;
    if (cplx)
      gon ? pick(np, md, T{}, T{}) : pick(np, md, T{}, F{});
    else
      gon ? pick(np, md, F{}, T{}) : pick(np, md, F{}, F{});
  };
  using Staged = std::integral_constant<int, kStaged>;
  auto by_mode = [&](auto np) {
    mode == kStaged ? by_c(np, Staged{}) : by_c(np, std::integral_constant<int, kRead>{});
  };
  switch (NP) {
    case 1: by_mode(std::integral_constant<int, 1>{}); break;
    case 3:
      if (mode == kFlat)
        by_c(std::integral_constant<int, 3>{}, std::integral_constant<int, kFlat>{});
      else
        by_mode(std::integral_constant<int, 3>{});
      break;
    case 6: by_mode(std::integral_constant<int, 6>{}); break;
    default:
      if constexpr (!BATCH) {  // quadrilaterals
        if (NP == 4) return by_mode(std::integral_constant<int, 4>{});
        if (NP == 8) return by_mode(std::integral_constant<int, 8>{});
        if (NP == 9) return by_mode(std::integral_constant<int, 9>{});
      }
      throw Error{BIE_EINVAL, "internal: no assembly kernel for this node count"};
  }
}

// Calls fn with the mid-edge kernel of (complex, G, fast sincos).
template <bool BATCH, class Fn>
void with_mid_kernel(bool cplx, bool gon, bool fast, Fn&& fn) {
  auto by_fast = [&](auto cx, auto g) {
    constexpr bool CX = decltype(cx)::value, G = decltype(g)::value;
    if constexpr (BATCH)
      fast ? fn(k_stream_mid_batch<CX, G, true>) : fn(k_stream_mid_batch<CX, G, false>);
    else
      fast ? fn(k_stream_mid<CX, G, true>) : fn(k_stream_mid<CX, G, false>);
  };
  using T = std::true_type;
  using F = std::false_type;
  if (cplx)
    gon ? by_fast(T{}, T{}) : by_fast(T{}, F{});
  else
    gon ? by_fast(F{}, T{}) : by_fast(F{}, F{});
}

}  // namespace

// The tables of the kernel: basis values of the vertex rules (or {N1, N2, N3, w / (4 pi)} of
// flat elements), each rule's part padded so that the rules start in different LDS banks,
// then the trig table and 2^(j/64).
std::vector<double> stream_tables(const RuleSet& rs, bool flat) {
  const int Q = rs.len[0], rules = std::min(rs.R, 3);
  const int stride = flat ? 4 * Q + 2 : ((Q * rs.pk + 1) & ~1) + 2;
  std::vector<double> t((size_t)stream_tab_doubles(rs, flat) + kTrigDoubles + kExpN, 0.0);
  for (int c = 0; c < rules; ++c)
    for (int q = 0; q < Q; ++q) {
      const double* p = &rs.pts[(size_t)(rs.off[c] + q) * kPtStride];
      if (flat) {
        for (int s = 0; s < 3; ++s) t[(size_t)c * stride + 4 * q + s] = p[kPtN + s];
        t[(size_t)c * stride + 4 * q + 3] = p[2] * 0.079577471545947667884;
      } else {
        for (int s = 0; s < rs.pk; ++s)
          t[(size_t)c * stride + q * rs.pk + s] = rs.phi[((size_t)c * rs.Qmax + q) * rs.pk + s];
      }
    }
  if (uses_mid_rules(rs.R, rs.pk)) {  // (u, v, w / (4 pi)) of the mid-edge rules
    double* p = t.data() + rules * stride;
    for (int q = rs.off[3]; q < rs.off[5] + rs.len[5]; ++q) {
      const double* x = &rs.pts[(size_t)q * kPtStride];
      *p++ = x[0];
      *p++ = x[1];
      *p++ = x[2] * 0.079577471545947667884;
    }
  }
  double* e = t.data() + stream_tab_doubles(rs, flat);
  for (int j = 0; j < kTrigN; ++j) {  // (cos, sin)(j pi / 64), rounded from long double
    const long double th = (long double)j * (3.14159265358979323846264338327950288L / 64);
    *e++ = (double)cosl(th);
    *e++ = (double)sinl(th);
  }
  for (int j = 0; j < kExpN; ++j) *e++ = (double)exp2l((long double)j / kExpN);
  return t;
}

int stream_polls() {
  const char* v = std::getenv("BIE_AMD_POLLS");
  return v ? std::max(0, std::atoi(v)) : 1 << 22;
}

int stream_tab_doubles(const RuleSet& rs, bool flat) {
  const int mid = uses_mid_rules(rs.R, rs.pk) ? (9 * rs.len[3] + 1) & ~1 : 0;
  return stream_mid_offset(rs, flat) + mid;
}

int stream_mid_offset(const RuleSet& rs, bool flat) {
  const int Q = rs.len[0], rules = std::min(rs.R, 3);
  return rules * (flat ? 4 * Q + 2 : ((Q * rs.pk + 1) & ~1) + 2);
}

// LDS plan: rows are staged up to kStageMaxQ points, and only when that leaves room for the
// slots; slots = 0 when nothing fits (the all-atomic kernel takes such rules).
StreamPlan stream_plan(const RuleSet& rs, bool flat, bool gon, int slots) {
  StreamPlan pl;
  pl.flat = flat;
  pl.waves = stream_waves(rs.pk);
  pl.tab_doubles = stream_tab_doubles(rs, flat);
  const int Q = rs.len[0], rules = std::min(rs.R, 3);
  pl.row_doubles = flat || Q > kStageMaxQ ? 0 : stage_rows_doubles(Q, rules);
  pl.mids = uses_mid_rules(rs.R, rs.pk);
  const int sd = gon ? 256 : 128;
  int S = 0;
  for (int s = 1; s <= 120; ++s)
    if (layout_of(s, sd, pl.tab_doubles, pl.waves, pl.row_doubles, pl.mids).total * 8L <=
        kLdsBytes)
      S = s;
  if (slots > 0) S = std::min(S, slots);
  pl.S = S;
  pl.shmem = (size_t)layout_of(S, sd, pl.tab_doubles, pl.waves, pl.row_doubles, pl.mids).total * 8;
  return pl;
}

void launch_stream_prep(const StreamPrep& p0, hipStream_t s) {
  StreamPrep p = p0;
  p.col_blocks = (int)std::min<int64_t>((int64_t)(p.n_zero + p.n_whole) * p.nk, 4096);
  const int64_t work = std::max({p.M, p.elem ? (int64_t)p.E * p.Pv : 0, (int64_t)p.E, (int64_t)kStreamCounters});
  const int64_t rest = std::min<int64_t>((work + 255) / 256, 4096);
  hipLaunchKernelGGL(k_stream_prep, dim3((unsigned)(p.col_blocks + rest)), dim3(256), 0, s, p);
  BIE_HIP_CHECK(hipGetLastError());
}

static size_t mid_shmem(const StreamPlan& pl, int mid_off) {
  return sizeof(double) * (size_t)(pl.tab_doubles - mid_off + kTrigDoubles + kExpN);
}

void launch_stream(const StreamInst& in, const StreamPlan& pl, const double* d_tab,
                   unsigned* d_counters, int* d_slow, int cus, bool fast, hipStream_t s) {
  const int64_t tiles = (int64_t)in.n_rowblocks * in.n_segments;
  BIE_REQUIRE(tiles > 0 && tiles < 2147483647LL, BIE_EINVAL, "tile count out of range");
  BIE_REQUIRE(pl.S > 0 && pl.shmem <= (size_t)kLdsBytes, BIE_EINVAL,
              "internal: assembly kernel without LDS slots");
  const bool cplx = in.a.ki != 0.0, gon = (in.a.flags & BIE_G) != 0;
  const int grid = (int)std::min<int64_t>(tiles, cus);
  const int mode = pl.flat ? kFlat : (pl.row_doubles ? kStaged : kRead);
  // (fast: no list, no tile is left out)
  const StreamRun run{d_tab, d_counters, fast ? nullptr : d_slow, pl.tab_doubles, pl.S, pl.row_doubles,
                      pl.mids ? 1 : 0};
  // not known to be fast: the tiles that are not are left to a second launch
  for (int pass = 0; pass < (fast ? 1 : 2); ++pass) {
    with_stream_kernel<false>(in.a.NP, mode, cplx, gon, pass == 0, [&](auto kern, int waves) {
      BIE_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                        hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)pl.shmem));
      hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * waves), pl.shmem, s, in,
                         (int)tiles, run);
    });
  }
  BIE_HIP_CHECK(hipGetLastError());
}

void launch_stream_mid(const StreamInst& in, const StreamPlan& pl, const double* d_tab,
                       bool fast, hipStream_t s) {
  if (!pl.mids) return;
  with_mid_kernel<false>(in.a.ki != 0.0, (in.a.flags & BIE_G) != 0, fast, [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(2048), dim3(256), mid_shmem(pl, in.mid_off), s, in, d_tab,
                       pl.tab_doubles);
  });
  BIE_HIP_CHECK(hipGetLastError());
}

void launch_stream_flat(const StreamPrep& p, hipStream_t s) {
  if (p.E <= 0) return;
  hipLaunchKernelGGL(k_stream_flat, dim3((p.E + 255) / 256), dim3(256), 0, s, p);
  BIE_HIP_CHECK(hipGetLastError());
}

void launch_stream_batch(const BatchInst* d_inst, int n_inst, int64_t max_cols,
                         const int4* d_tiles, int n_tiles, const StreamPlan& pl, int NP,
                         bool cplx, bool gon, bool fast, const double* d_tab, int mid_off,
                         unsigned* d_counters, int* d_slow, int cus, hipStream_t s) {
  if (n_inst <= 0) return;
  BIE_REQUIRE(n_inst <= 65535, BIE_EINVAL, "too many batch instances");
  const int64_t blocks = std::max<int64_t>(1, std::min<int64_t>(max_cols, 1024));
  hipLaunchKernelGGL(k_stream_batch_prep, dim3((unsigned)blocks, (unsigned)n_inst), dim3(256), 0,
                     s, d_inst, d_counters);
  BIE_HIP_CHECK(hipGetLastError());
  if (n_tiles <= 0) return;
  BIE_REQUIRE(pl.S > 0 && pl.shmem <= (size_t)kLdsBytes, BIE_EINVAL,
              "internal: batch kernel without LDS slots");
  const int mode = pl.flat ? kFlat : (pl.row_doubles ? kStaged : kRead);
  // (fast: no list, no tile is left out)
  const StreamRun run{d_tab, d_counters, fast ? nullptr : d_slow, pl.tab_doubles, pl.S, pl.row_doubles,
                      pl.mids ? 1 : 0};
  for (int pass = 0; pass < (fast ? 1 : 2); ++pass) {
    with_stream_kernel<true>(NP, mode, cplx, gon, pass == 0, [&](auto kern, int waves) {
      BIE_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                        hipFuncAttributeMaxDynamicSharedMemorySize,
                                        (int)pl.shmem));
      hipLaunchKernelGGL(kern, dim3((unsigned)std::min(n_tiles, cus)), dim3(64 * waves),
                         pl.shmem, s, d_inst, d_tiles, n_tiles, run);
    });
  }
  if (pl.mids)
    with_mid_kernel<true>(cplx, gon, fast, [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(256, (unsigned)n_inst), dim3(256), mid_shmem(pl, mid_off), s,
                         d_inst, d_tab, pl.tab_doubles);
    });
  BIE_HIP_CHECK(hipGetLastError());
}

}  // namespace bie
