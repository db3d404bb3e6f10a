// Shared host-side declarations of the bie_amd library (gfx950).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/bie_amd.h"

namespace bie {

void set_error(const std::string& msg);

struct Error {
  int code;
  std::string msg;
};

#define BIE_HIP_CHECK(expr)                                                       \
  do {                                                                            \
    hipError_t _e = (expr);                                                       \
    if (_e != hipSuccess)                                                         \
      throw ::bie::Error{BIE_EHIP, std::string(#expr) + ": " + hipGetErrorString(_e)}; \
  } while (0)

#define BIE_REQUIRE(cond, code, msg)                         \
  do {                                                       \
    if (!(cond)) throw ::bie::Error{(code), std::string(msg)}; \
  } while (0)

constexpr double kPi = 3.14159265358979323846;

// Bound on |x| for the branch-free table sincos (Phase with FAST, stream_device.hpp): 2^46,
// so that 64 |x| / pi stays below 2^51 and its rounding by an added 1.5 * 2^52 is exact.
// The host chooses that form only when |k| times a bound on every target-to-element-point
// distance is below it.
constexpr double kTabFastMaxArg = 70368744177664.0;
// The kernels of that form divide by up to r^5 at once: it is taken up to these distances; the
// other form stays in range as far as r^2 does.
constexpr double kFastMaxDist = 1e50;

// Point record of the concatenated rule set: u, v, w, then N, dN/du, dN/dv of the
// geometry basis (6 slots each, unused slots zero).
constexpr int kPtStride = 30;
// offsets in a point record of N, dN/du and dN/dv (9 geometry nodes each)
constexpr int kPtN = 3, kPtDu = 12, kPtDv = 21;

// All quadrature rules one assembly uses, for a geometry and a physics kind.  Triangles:
// rules 1..3 cluster at the corners (Q = n*m each); rules 4..6 at the edge mid points of
// quadratic elements (Q = 2*n*m', m' = m rounded up to even).  Quadrilaterals: one tensor
// Gauss-Legendre rule on [-1, 1]^2 (Q = n*m, R = 1).
struct RuleSet {
  int gk = 3, pk = 3, n = 0, m = 0;  // geometry and physics nodes per element
  int gkind = 3;                     // geometry kind (BIE_TRI3 .. BIE_QUAD9)
  int pkind = 3;                     // physics kind (BIE_TRI3 .. BIE_DTRI6)
  double beta = 0.0;                 // node offset of BIE_DTRI3 / BIE_DTRI6
  int R = 3;          // number of rules
  int Qc = 0, Qm = 0; // corner / mid-edge rule sizes
  int Pe = 0;         // points per element over all rules
  int Qmax = 0;
  int off[6] = {0, 0, 0, 0, 0, 0};
  int len[6] = {0, 0, 0, 0, 0, 0};
  std::vector<double> pts;  // Pe x kPtStride
  std::vector<double> phi;  // R x Qmax x pk physics basis at the rule points
};

RuleSet build_ruleset(int gkind, int pkind, double beta, int n, int m);

// Element kinds: the low byte is the node count; BIE_DTRI* / BIE_DQUAD* are discontinuous,
// BIE_QUAD* / BIE_DQUAD* quadrilaterals (one Gauss rule, no selection).
inline int physics_nodes(int pkind) { return pkind & 0xff; }
inline int geometry_nodes(int gkind) { return gkind & 0xff; }
inline bool physics_discontinuous(int pkind) { return (pkind & 0x100) != 0; }
inline bool kind_is_quad(int kind) { return (kind >> 9) != 0; }
// physics kinds whose nodes sit at the offset bie_mesh.physics_beta
inline bool kind_has_beta(int pkind) {
  return pkind == BIE_DTRI3 || pkind == BIE_DTRI6 || pkind == BIE_DQUAD4 || pkind == BIE_DQUAD9;
}
// The mid-edge split rules 4-6 exist on quadratic geometry (R = 6) and are chosen only when
// the nearest of six physics nodes is an edge node.
inline bool uses_mid_rules(int gk, int pk) { return gk == 6 && pk == 6; }
void gauss_legendre01(int n, std::vector<double>& x, std::vector<double>& w);
void gauss_legendre_pm1(int n, std::vector<double>& x, std::vector<double>& w);

// Device-side launch parameters for one assembly.
struct AssemblyArgs {
  const double* targets;   // 3 x M
  int64_t M;
  int64_t N;               // columns of F, G
  int E;
  int NP;                  // physics nodes per element
  const double* elem;      // E x Pe x 8: y(3), n(3), J*w/(4 pi), 0
  int Pe;
  const double* selnodes;  // E x NP x 4 selection node coordinates
  const int* ptopo;        // E x NP physics node indices (0-based, element-major)
  const double* phi;       // R x Qmax x NP
  int Qmax;
  int off[6];
  int len[6];
  int R;
  int hyp;                 // rule-selection distance: 0 julia_hypot3, 1 scaled_hypot3
  double kr, ki;
  unsigned flags;
  double* F;
  double* G;
  double* C;
};

constexpr int kSlotWaves = 8;   // elements per step of the schedule check
constexpr int kSlotCount = 64;  // LDS slots of the schedule check (64 rows x 4 doubles each)
constexpr int kLdsBytes = 160 * 1024;  // LDS per CU (one workgroup of the slot kernels)

// Vertex rules up to this length are staged in LDS per wave: three rules of 16 rows are three
// 16-byte loads per lane, all that the registers hold beside a pair; longer ones are read from
// memory in the point loop.
constexpr int kStageMaxQ = 16;

// Table of (cos, sin)(j pi / 64), j < kTrigN, for the table-driven sincos of the slot
// kernels.
constexpr int kTrigN = 128;
constexpr int kTrigDoubles = 2 * kTrigN;

// Stream kernel (stream.hip): dense assembly of one mesh or of a batch.
constexpr int kExpN = 64;         // entries of its table 2^(j / 64)
constexpr int kStreamMid = 2048;  // mid-edge pairs a tile may queue in LDS (4 bytes each)
// Counters of a call: tiles drawn, slow tiles listed and drawn, then StreamInst::mid_count:
// mid-edge pairs listed, tiles without room for theirs, end of the list.
enum { kSlowCount = 1, kSlowNext = 2, kMidCount = 3, kMidEnd = 5, kStreamCounters = 6 };
constexpr int kFlatDoubles = 24;  // record of a flat element
// Waves of its workgroup (one per CU): four per SIMD with 128 VGPRs each; eight- and nine-node
// physics keep 32 and 36 sums per lane and take two per SIMD.
constexpr int stream_waves(int NP) { return NP >= 8 ? 8 : 16; }
// and of the kernels for large arguments with six-node physics or complex k, whose reduction
// does not fit 128 VGPRs beside a pair (2562 quadratic nodes 1210 us with sixteen waves, 466 with
// eight; 4002 linear nodes, real k, 1163 and 1248)
constexpr int kSlowWaves = 8;

struct StreamInst {
  AssemblyArgs a;
  const int* seg_begin;     // n_segments + 1
  const int* order;         // element at each position
  const int4* ent;          // E x NP schedule entries (StreamEntry), by position
  const double* psel;       // E x NP x 3 selection nodes, by position
  const double* flat;       // E x kFlatDoubles records of flat elements, by position
  const double* coords;     // geometry nodes and topology (mid-edge pairs)
  const int* topo;
  unsigned* mid_count;      // mid-edge pairs listed, tiles without room, end of the list
  int2* mid_queue;          // (row, element | (rule - 4) << 28)
  int2* mid_tiles;          // (row block, segment) of tiles whose pairs are not listed
  unsigned mid_cap;
  int own_basis;            // the physics basis is the geometry basis
  int mid_off;              // of the mid-edge points in the tables
  int n_segments, n_rowblocks;
  double center[3], reach;  // every element point is within reach of the centre
};

// Device lists of a call: tile counters, mid-edge pairs (quadratic physics) and the tiles they
// have no room for, tiles left to the launch for large arguments.
struct StreamLists {
  unsigned* counters = nullptr;  // kStreamCounters
  int2* mid_queue = nullptr;
  int2* mid_tiles = nullptr;
  int64_t mid_cap = 0, mid_tiles_cap = 0;
  int* slow = nullptr;
  int64_t slow_cap = 0;
};

// 2^22, which no wait of a valid schedule comes near; BIE_AMD_POLLS sets another number (tests).
int stream_polls();
struct StreamRun {
  const double* tab;        // stream_tables
  unsigned* counters;       // kStreamCounters
  int* slow;                // tiles left to the second launch, or NULL: there is none
  int tab_doubles, S, row_doubles, mids;
  int polls = stream_polls();  // of a wait for another wave, before it gives up
};

struct StreamPlan {
  bool flat = false, mids = false;
  int waves = 16, S = 0, tab_doubles = 0, row_doubles = 0;
  size_t shmem = 0;
};

struct StreamPrep {
  int64_t M;
  int E, Pe, Pv, gk;        // Pv: points of the vertex rules
  unsigned flags;
  double *F, *G, *C;
  const int* zero_cols;     // columns of enabled outputs to zero
  int n_zero, n_whole;      // n_whole: columns of disabled outputs to zero (N or 0)
  int nk;                   // matrices of F and G, `stride` complex entries apart
  int64_t stride;
  int col_blocks;
  unsigned* counters;       // kStreamCounters
  unsigned mid_cap;
  const double *coords, *sources, *pts;
  const int *topo, *ptopo, *order;
  double* flat;             // records to write, or NULL
  double* elem;             // element tables to write, or NULL
};

std::vector<double> stream_tables(const RuleSet& rs, bool flat);
int stream_tab_doubles(const RuleSet& rs, bool flat);
int stream_mid_offset(const RuleSet& rs, bool flat);
// slots: at most so many LDS slots (0: as many as fit)
StreamPlan stream_plan(const RuleSet& rs, bool flat, bool gon, int slots = 0);
void launch_stream_prep(const StreamPrep& p, hipStream_t s);
void launch_stream(const StreamInst& in, const StreamPlan& pl, const double* d_tab,
                   unsigned* d_counters, int* d_slow, int cus, bool fast, hipStream_t s);
// the mid-edge pairs it listed
void launch_stream_mid(const StreamInst& in, const StreamPlan& pl, const double* d_tab,
                       bool fast, hipStream_t s);

// One instance of an uneven batch: its assembly and schedule, and the columns to zero.
struct BatchInst {
  StreamInst s;
  const int* zero_cols;
  int n_zero;
  int pad;
};
void launch_stream_flat(const StreamPrep& p, hipStream_t s);
// n_tiles tiles (instance, row block, segment); d_counters: kMidCount of them
void launch_stream_batch(const BatchInst* d_inst, int n_inst, int64_t max_cols,
                         const int4* d_tiles, int n_tiles, const StreamPlan& pl, int NP,
                         bool cplx, bool gon, bool fast, const double* d_tab, int mid_off,
                         unsigned* d_counters, int* d_slow, int cus, hipStream_t s);

// Batched frequency sweep and k-derivatives (sweep.hip).
struct SweepArgs {
  const double* k;           // nk real wavenumbers (device)
  int64_t stride;            // complex elements between consecutive F_k (and G_k)
  double k_re, k_im;
  int nk;
  int taylor;                // 1: the nk matrices are d^q/dk^q, q = 0..nk-1, at k_re + i k_im
};
// lean: F alone of the k-derivatives on flat elements
int sweep_block_size(int NP, bool gon, bool lean);  // matrices per block of the kernel
// slots: at most so many LDS slots (0: as many as fit)
StreamPlan sweep_plan(const RuleSet& rs, bool flat, bool lean, int slots);
// prepare_only: sets the kernels' attributes, launches nothing
void launch_sweep(const StreamInst& in, const SweepArgs& sw, const StreamPlan& pl,
                  const double* d_tab, unsigned* d_counters, int* d_slow, int cus, bool fast,
                  bool prepare_only, hipStream_t s);

// Vector-Jacobian product of the assembly (adjoint.hip).
struct AdjointArgs {
  const double* targets;   // 3 x M
  int64_t M;
  const int* tvert;        // M: mesh node a target sits on (moves with X), -1 fixed; or NULL
  const double2* alpha;    // M complex weights of F rows
  const double2* beta;     // M complex weights of C (or NULL)
  const double2* p;        // N complex values at the collocation nodes
  const double* coords;    // 3 x Nc
  const int* topo;         // E x NG
  const int* ptopo;        // E x NP
  const double* selnodes;  // E x NP x 4
  const double* pts;       // rule points (kPtStride)
  const double* phi;       // R x Qmax x NP
  int Qmax;
  int off[6];
  int len[6];
  int R;
  int E;
  int hyp;                 // rule-selection distance (as AssemblyArgs::hyp)
  double k;               // Re k
  double ki;              // Im k (complex-k entry point; 0 for real k)
  double center[3], reach; // every element point is within reach of the centre
  double* gradX;           // 3 x Nc, accumulated
  double* gradk;           // d/dRe k (and d/dIm k after it for complex k), accumulated, or NULL
};

// One instance of the batched k-derivative w = alpha^T (dF/dk) p (adjoint.hip).
struct DfdkInst {
  const double* targets;   // 3 x M (the instance's collocation nodes)
  int64_t M;
  int E;
  int Pe;
  int first_tile;          // of the instance's (row block, element chunk) tiles
  int fast;                // every |k| r is below the fast sincos bound
  const double* flat;      // E x kFlatDoubles records of flat elements, or NULL
  const double* elem;      // element tables of the assembly (E x Pe x 8)
  const double* selnodes;  // E x NP x 4
  const int* ptopo;        // E x NP
  const double* phi;       // R x Qmax x NP
  int Qmax;
  int R;
  int hyp;
  int off[6];
  int len[6];
  double kr, ki;
  const double2* alpha;    // M
  const double2* p;        // N
  double* w;               // complex result (2 doubles), accumulated
};

// Sparse near-field assembly (sparse.hip).
struct SparseLaunch {
  const double* src;      // 3 x rows source points (device)
  const int2* pairs;      // (row, element) per pair (device)
  const int* pos;         // pairs x NP entry indices (device)
  int64_t n_pairs;
  const double* coords;   // 3 x Nc (device)
  const int* topo;        // E x NG (device)
  const double* gsel;     // E x NG x 4 geometry node coordinates (device)
  const double* rules;    // point records (u, v, w, 0), sparse_record_doubles() each (device)
  const double* trig;     // (cos, sin)(j pi / 64), interleaved, then 2^(j / 64) (device)
  bool fast;              // every |k| r is below the fast sincos bound
  bool explicit_src = false;  // the caller's sources: not known here whether they are
  double center[3], reach;    // every element point is within reach of the centre
  int off[6], len[6];     // per geometry node: first record and point count
  int NG, NP, hyp;
  const int* batches = nullptr;  // pair batches sharing an element (device; 8 ints each)
  int64_t n_batches = 0;
  bool disc;              // discontinuous physics (basis at beta)
  double beta;
  double kr, ki;
  unsigned flags;
  double* F;              // nnz complex (device), zeroed
  double* G;
};
void subdivision_rule(const double src[3], std::vector<double>& u, std::vector<double>& v,
                      std::vector<double>& w);
bool gauss_points_triangle(int n, std::vector<double>& u, std::vector<double>& v,
                           std::vector<double>& w);
void sparse_pattern(const int* ptopo, int NP, int64_t E, int64_t N, int depth,
                    std::vector<int64_t>& row_ptr, std::vector<int>& cols,
                    std::vector<int64_t>& pair_ptr, std::vector<int>& pair_elem);
// connected_sources of discontinuous physics (row r belongs to element r / NP; N == E * NP);
// topo: the geometry topology (E x NG), whose first three nodes are the corners.
void sparse_pattern_disc(const int* topo, int NG, const int* ptopo, int NP, int64_t E,
                         int64_t N, int depth, std::vector<int64_t>& row_ptr,
                         std::vector<int>& cols, std::vector<int64_t>& pair_ptr,
                         std::vector<int>& pair_elem);
// The polar rule of a discontinuous element around its physics node (pu, pv): three
// sub-triangles from the node to the reference triangle's sides, polar_gaussian(n) on each.
void polar_rule(double pu, double pv, int n, std::vector<double>& u, std::vector<double>& v,
                std::vector<double>& w);
// Local (u, v) of node c of a discontinuous triangular physics kind.
void discontinuous_node(int pkind, double beta, int c, double* u, double* v);
// Physics basis of any physics kind at (u, v) (rules.cpp); N holds 9 entries.
void physics_basis(int pkind, double beta, double u, double v, double* N);
void launch_sparse_pairs(const SparseLaunch& L, hipStream_t s);
int sparse_record_doubles();
// Rows per batch of the batched sparse kernel (k_sparse_batch) for NP physics nodes.
int sparse_batch_rows(int NP);
// Geometry basis of a geometry kind and its derivatives at (u, v) (rules.cpp); N, du, dv
// hold 9 entries each (slots beyond the kind's node count are zeroed).
void geometry_basis(int kind, double u, double v, double* N, double* du, double* dv);

// Launchers (assemble.hip)
void launch_fill_zero(double* p, int64_t n_doubles, hipStream_t s);
void launch_geometry(const double* coords, const int* topo, int gk, int E,
                     const double* d_pts, int Pe, double* elem, hipStream_t s);
void launch_gather_selnodes(const double* sources, const int* ptopo, int NP, int E,
                            double* selnodes, hipStream_t s);
void launch_assemble(const AssemblyArgs& a, hipStream_t s);
void zgemv_batched_device(int64_t M, int64_t K, const double* dA, int64_t strideA, int64_t lda,
                          const double* dX, int64_t ldx, double* dY, int64_t ldy,
                          const int32_t* d_idx, int32_t n_idx, hipStream_t s);
// Y = sum_t coef_t A_t over n_terms arrays of n complex entries spaced strideA apart
// (apply_taylor_expansion, src/3d/rosebem.jl:164-199); coef on the host.
constexpr int kTaylorMaxOrders = 64;
void taylor_expand_device(int n_terms, int64_t n, const double* dA, int64_t strideA,
                          const double* coef, double* dY, hipStream_t s);
void zgemm_device(int64_t M, int64_t nrhs, int64_t K, const double* dA, int64_t lda,
                  const double* dX, int64_t ldx, double* dY, int64_t ldy, hipStream_t s);
// Capacity of the allocation-free apply's scratch array, in complex128 entries (16 MiB).
constexpr int64_t kApplyScratchComplex = int64_t(1) << 20;
// As zgemm_device with the packed X in the device scratch array instead of an allocated
// workspace: K * ceil(nrhs/32)*32 <= kApplyScratchComplex.
void zgemm_device_noalloc(int64_t M, int64_t nrhs, int64_t K, const double* dA, int64_t lda,
                          const double* dX, int64_t ldx, double* dY, int64_t ldy,
                          hipStream_t s);
// d_tab: stream_tables; fast: every |k| r is below the fast sincos bound
void launch_adjoint(const AdjointArgs& a, int gk, int pk, bool flat, bool cplx, bool fast,
                    const double* d_tab, int tab_doubles, int cus, hipStream_t s);
// tiles: (64-row block, chunk of ech elements) of every instance, rows fastest; d_basis: flat
// table or basis values, d_trig: (cos, sin) and 2^(j/64) tables
void launch_dfdk_batch(const DfdkInst* d_inst, int n_inst, int n_tiles, int ech, int NP,
                       bool flat, bool cplx, bool some_fast, bool some_slow,
                       const double* d_basis, int n_basis, const double* d_trig, int cus,
                       hipStream_t s);
// Solves on the device (solve.hip)
void lu_factor_device(int64_t n, double* dA, int64_t lda, const double* dC, int32_t* d_ipiv,
                      hipStream_t s);
void lu_solve_device(int64_t n, const double* dA, int64_t lda, const int32_t* d_ipiv, int trans,
                     double* dB, int64_t ldb, int64_t nrhs, hipStream_t s);
void zgemv_device(int trans, int64_t m, int64_t n, const double* dA, int64_t lda,
                  const double* dx, double* dy, hipStream_t s);
void gmres_batched_device(int64_t n, int nsys, const double* dF, int64_t strideF, int64_t ldf,
                          const double* dC, const double* dB, int64_t ldb, double* dX,
                          int64_t ldx, double tol, int restart, int maxiter, int32_t* iters,
                          double* resid, hipStream_t s);
void launch_select(const double* targets, int64_t M, const double* selnodes, int NP, int E,
                   int R, int hyp, int8_t* out, hipStream_t s);

}  // namespace bie

// Device-resident mesh and its cached rule-dependent tables.
struct bie_dmesh {
  int device = 0;
  int gk = 3, pk = 3;           // geometry nodes, physics nodes per element
  int gkind = 3;                // geometry kind (BIE_TRI3 .. BIE_QUAD9)
  int pkind = 3;                // physics kind (BIE_TRI3 .. BIE_DTRI6)
  double beta = 0.0;            // node offset of BIE_DTRI3 / BIE_DTRI6
  int hyp = 0;                  // rule-selection distance (BIE_MESH_SCALED_HYPOT)
  int64_t Nc = 0, E = 0, N = 0;
  double* d_coords = nullptr;
  int* d_topo = nullptr;        // E x gk, element-major
  double* d_sources = nullptr;  // 3 x N
  int* d_ptopo = nullptr;       // E x pk, element-major
  double* d_selnodes = nullptr; // E x pk x 4
  // rule-dependent cache
  int cn = -1, cm = -1;
  bie::RuleSet rs;
  double* d_pts = nullptr;
  double* d_phi = nullptr;
  double* d_elem = nullptr;
  bool geom_valid = false;      // d_elem holds the geometry of the cached rule set
  // bounding sphere of the mesh: centre, radius over the coordinates and over the sources
  double center[3] = {0.0, 0.0, 0.0};
  double coord_radius = 0.0, source_radius = 0.0;
  // host copies for scheduling
  std::vector<double> h_coords, h_sources;
  std::vector<int> h_topo, h_ptopo;
  // stream schedule of the dense kernel (stream.hip) and what goes with it
  struct Stream {
    int S = -1;                  // slots it was built for
    int64_t key = -1;            // and what the segments were chosen for
    int64_t rowblocks = -1;      // (single-mesh calls) of the last call, and its rule length
    int Q = -1;
    int segments = 0, zero_cols = 0;
    int* d_seg_begin = nullptr;
    int* d_order = nullptr;
    int4* d_ent = nullptr;
    double* d_psel = nullptr;    // selection nodes by position
    double* d_flat = nullptr;    // records of flat elements by position
    int* d_zero_cols = nullptr;
    std::vector<int> h_seg_begin;  // (batch) host copy, for the tile list
  };
  double* d_eflat = nullptr;     // records of flat elements in element order (k-derivatives)
  Stream stream[2][2];  // of single-mesh calls (own rows or others, without or with G)
  // of batches, and of sweeps and k-derivatives: the last few that were asked for, shared with
  // the batches and graphs that use them
  static constexpr size_t kBatchStreams = 4, kSweepStreams = 8;
  std::vector<std::shared_ptr<Stream>> bstreams, sstreams;
  struct {
    int Q = -1, segments = 0;
    int64_t tiles = -1;
  } sweep_choice[2];             // the last choice of segments, for few and for many matrices
  bie::StreamLists lists[2][2], blists, slists;  // (lists: as stream)
  double* d_stab = nullptr;      // its tables for the cached rule set (stream_tables)
  // tile shape of the frequency sweep (bie_sweep_tune): elements per tile (0: one segment per
  // row block) and LDS slots (0: as many as fit)
  int sweep_elems_per_tile = 0;
  int sweep_slots = 0;
  // calls on the handle share the scratch above: each call's work waits for the previous
  // call's (recorded in `done` on `done_stream`) when it runs on another stream
  hipEvent_t done = nullptr;
  hipStream_t done_stream = nullptr;
  bool done_valid = false;
  std::mutex mu;
};

// An uneven batch: several device meshes (same element kinds) assembled with one rule set
// in one persistent launch (bie_batch_* in include/bie_amd.h).
struct bie_batch {
  int device = 0;
  int gk = 3, pk = 3, n = 0, m = 0;
  int pkind = 3;
  double beta = 0.0;
  std::vector<bie_dmesh*> meshes;
  // schedule configuration (chosen by bie_batch_tune)
  bool fitted = true;        // segments chosen from the batch's work (not configured)
  int elems_per_tile = 64;   // else: target elements per segment
  int slots = 64;            // LDS slots per workgroup (0: as many as fit)
  int slots_used = 64;       // the slot count the tile list was built with
  int order = 0;             // 0: longest tiles first, 1: instances interleaved
  int64_t configured_key = -1;  // configuration the tile list was built for
  // device state
  bie::BatchInst* d_inst = nullptr;
  bie::BatchInst* h_inst = nullptr;  // pinned staging for the per-call table
  hipEvent_t staged = nullptr;       // the last upload of h_inst has completed
  int4* d_tiles = nullptr;
  int n_tiles = 0;
  int* d_slow = nullptr;             // tiles left to the launch for large arguments
  unsigned* d_counter = nullptr;
  std::vector<int64_t> rowblocks;
  std::vector<std::shared_ptr<bie_dmesh::Stream>> streams;  // per instance: what it indexes
  std::mutex mu;
};
