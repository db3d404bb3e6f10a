// Host schedules of the assembly kernels.
//
// The dense assembly writes F[i, j] = sum over elements e incident to node j of that
// element's contribution for target i.  A workgroup owns 64 target rows and one *segment* of
// elements, an ordered list that its waves draw from one element at a time; a node's
// contributions meet in an LDS *slot*, which it occupies from its first element in the segment
// to a few positions past its last (build_stream_schedule; stream.hip has the hand-over).
// Nodes whose elements all lie in one segment ("owned") are written once with a plain store;
// nodes touched by several segments ("shared") are added atomically into columns zeroed
// beforehand.
//
// Segments come from recursive coordinate splitting of the element centroids into the
// requested number of parts; each is swept along its longest axis, which keeps the number
// of occupied slots (the sweep front) near the segment's width.  Segments are split
// further until their front fits the slot budget.
//
// build_slot_schedule is the same for waves that meet at a barrier after every step of W
// elements: a node is flushed during the step after its last element, and its slot is free one
// step later.  No kernel runs by it: bie_schedule_check reports its statistics.
#include <algorithm>
#include <cmath>
#include <deque>
#include <numeric>

#include "schedule.hpp"

namespace bie {
namespace {

struct SegOrder {
  std::vector<int> elems;  // sweep order
};

int longest_axis(const std::vector<int>& idx, const double* cent) {
  double lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  for (int e : idx)
    for (int d = 0; d < 3; ++d) {
      lo[d] = std::min(lo[d], cent[3 * (size_t)e + d]);
      hi[d] = std::max(hi[d], cent[3 * (size_t)e + d]);
    }
  int ax = 0;
  for (int d = 1; d < 3; ++d)
    if (hi[d] - lo[d] > hi[ax] - lo[ax]) ax = d;
  return ax;
}

void sort_along(std::vector<int>& idx, const double* cent, int ax) {
  std::stable_sort(idx.begin(), idx.end(), [&](int a, int b) {
    return cent[3 * (size_t)a + ax] < cent[3 * (size_t)b + ax];
  });
}

// Largest number of slots occupied at any step when idx (already in sweep order) is
// swept in steps of W elements: a node occupies its slot from its first step through
// the step after its last.
int front_width(const std::vector<int>& idx, const int* ptopo, int NP, int W,
                std::vector<int>& first, std::vector<int>& last, std::vector<int>& touched) {
  touched.clear();
  const int nsteps = ((int)idx.size() + W - 1) / W;
  for (size_t t = 0; t < idx.size(); ++t) {
    const int step = (int)t / W;
    for (int s = 0; s < NP; ++s) {
      const int node = ptopo[(size_t)idx[t] * NP + s];
      if (first[node] < 0) {
        first[node] = step;
        touched.push_back(node);
      }
      last[node] = step;
    }
  }
  std::vector<int> delta(nsteps + 2, 0);
  for (int node : touched) {
    delta[first[node]] += 1;
    delta[last[node] + 2] -= 1;
  }
  int live = 0, best = 0;
  for (int t = 0; t < nsteps; ++t) {
    live += delta[t];
    best = std::max(best, live);
  }
  for (int node : touched) first[node] = last[node] = -1;
  return best;
}

// Splits idx into `parts` segments of nearly equal size along longest axes (halves of
// the part count at every level, so any count is reachable), then splits further any
// segment whose front exceeds S slots.
template <class Fits>
void split(std::vector<int> idx, int parts, const double* cent, const Fits& fits,
           std::vector<SegOrder>& out) {
  const int ax = longest_axis(idx, cent);
  sort_along(idx, cent, ax);
  if ((int)idx.size() < parts) parts = std::max(1, (int)idx.size());
  if (parts <= 1) {
    if (idx.size() <= 1 || fits(idx)) {
      out.push_back(SegOrder{std::move(idx)});
      return;
    }
    parts = 2;
  }
  const int pa = parts / 2, pb = parts - pa;
  const size_t h = idx.size() * (size_t)pa / (size_t)parts;
  std::vector<int> a(idx.begin(), idx.begin() + h), b(idx.begin() + h, idx.end());
  split(std::move(a), pa, cent, fits, out);
  split(std::move(b), pb, cent, fits, out);
}

}  // namespace

SlotSchedule build_slot_schedule(const int* ptopo, int NP, int E, int N, const double* cent,
                                 int W, int S, int min_segments) {
  SlotSchedule sc;
  sc.W = W;
  sc.S = S;
  sc.NP = NP;
  std::vector<int> first(N, -1), last(N, -1), touched;
  std::vector<SegOrder> segs;
  if (E > 0) {
    std::vector<int> all(E);
    std::iota(all.begin(), all.end(), 0);
    auto fits = [&](const std::vector<int>& idx) {
      return front_width(idx, ptopo, NP, W, first, last, touched) <= S;
    };
    split(std::move(all), std::max(1, min_segments), cent, fits, segs);
  }
  sc.n_segments = (int)segs.size();
  // how many segments touch each node
  std::vector<int> nseg(N, 0), mark(N, -1);
  for (int g = 0; g < sc.n_segments; ++g)
    for (int e : segs[g].elems)
      for (int s = 0; s < NP; ++s) {
        const int node = ptopo[(size_t)e * NP + s];
        if (mark[node] != g) {
          mark[node] = g;
          nseg[node] += 1;
        }
      }
  for (int j = 0; j < N; ++j)
    if (nseg[j] != 1) sc.zero_cols.push_back(j);  // shared or untouched
  sc.n_shared = 0;
  for (int j = 0; j < N; ++j) sc.n_shared += nseg[j] > 1;

  sc.slot_of.assign((size_t)E * NP, -1);
  std::vector<int> node_slot(N, -1);
  sc.seg_step_begin.push_back(0);
  sc.flush_begin.push_back(0);
  sc.max_live = 0;
  for (int g = 0; g < sc.n_segments; ++g) {
    const std::vector<int>& el = segs[g].elems;
    const int nsteps = ((int)el.size() + W - 1) / W;
    // first / last step per node within this segment
    touched.clear();
    for (size_t t = 0; t < el.size(); ++t) {
      const int step = (int)t / W;
      for (int s = 0; s < NP; ++s) {
        const int node = ptopo[(size_t)el[t] * NP + s];
        if (first[node] < 0) {
          first[node] = step;
          touched.push_back(node);
        }
        last[node] = step;
      }
    }
    std::vector<std::vector<int>> starts(nsteps), ends(nsteps);
    for (int node : touched) {
      starts[first[node]].push_back(node);
      ends[last[node]].push_back(node);
    }
    // free slots, lowest index first; slots of nodes that ended at the previous step are
    // released after this step (they are flushed during it)
    std::vector<int> freelist, pending;
    for (int q = S - 1; q >= 0; --q) freelist.push_back(q);
    int live = 0;
    for (int t = 0; t < nsteps; ++t) {
      std::sort(starts[t].begin(), starts[t].end());
      for (int node : starts[t]) {
        if (freelist.empty()) throw Error{BIE_EINVAL, "slot schedule overflow"};
        node_slot[node] = freelist.back();
        freelist.pop_back();
        ++live;
      }
      sc.max_live = std::max(sc.max_live, live);
      for (int w = 0; w < W; ++w) {
        const size_t p = (size_t)t * W + w;
        const int e = p < el.size() ? el[p] : -1;
        sc.step_elems.push_back(e);
        if (e >= 0)
          for (int s = 0; s < NP; ++s)
            sc.slot_of[(size_t)e * NP + s] = node_slot[ptopo[(size_t)e * NP + s]];
      }
      std::sort(ends[t].begin(), ends[t].end());
      for (int node : ends[t]) {
        sc.flush_node.push_back(node);
        sc.flush_slot.push_back(node_slot[node] | (nseg[node] > 1 ? kSharedBit : 0));
      }
      for (int sl : pending) {
        freelist.push_back(sl);
        --live;
      }
      pending.clear();
      for (int node : ends[t]) pending.push_back(node_slot[node]);
      sc.flush_begin.push_back((int)sc.flush_node.size());
    }
    for (int node : touched) first[node] = last[node] = -1;
    sc.seg_step_begin.push_back(sc.seg_step_begin.back() + nsteps);
  }
  sc.n_steps = sc.seg_step_begin.back();
  return sc;
}

// Replays a schedule and checks every invariant the slot kernel relies on: each element
// is swept exactly once; a slot holds one node from its first to its last step; every
// touched node is flushed exactly once per segment, from the slot it occupies; owned and
// shared flags agree with the segment count; zero_cols = shared + untouched columns.
void validate_slot_schedule(const SlotSchedule& sc, const int* ptopo, int NP, int E, int N) {
  auto fail = [](const std::string& m) { throw Error{BIE_EINVAL, "schedule: " + m}; };
  if ((int)sc.step_elems.size() != sc.n_steps * sc.W) fail("step_elems size");
  if ((int)sc.flush_begin.size() != sc.n_steps + 1) fail("flush_begin size");
  std::vector<int> seen(E, 0), nseg(N, 0), seg_mark(N, -1);
  std::vector<int> slot_node(sc.S, -1), node_slot(N, -1), flushed(N, -1);
  for (int g = 0; g < sc.n_segments; ++g) {
    std::vector<int> pending;  // slots flushed during the current step, free after it
    for (int t = sc.seg_step_begin[g]; t < sc.seg_step_begin[g + 1]; ++t) {
      for (int w = 0; w < sc.W; ++w) {
        const int e = sc.step_elems[(size_t)t * sc.W + w];
        if (e < 0) continue;
        if (e >= E) fail("element id out of range");
        if (seen[e]++) fail("element swept twice");
        for (int s = 0; s < NP; ++s) {
          const int node = ptopo[(size_t)e * NP + s];
          const int sl = sc.slot_of[(size_t)e * NP + s];
          if (sl < 0 || sl >= sc.S) fail("slot out of range");
          if (seg_mark[node] != g) {
            seg_mark[node] = g;
            nseg[node]++;
          }
          if (node_slot[node] < 0) {  // first touch in this segment
            if (flushed[node] == g) fail("node touched after its flush");
            if (slot_node[sl] >= 0) fail("slot reused while occupied");
            slot_node[sl] = node;
            node_slot[node] = sl;
          } else if (node_slot[node] != sl) {
            fail("node moved between slots");
          }
        }
      }
      // the flush of step t - 1 runs during step t: its slots are free from step t + 1
      for (int sl : pending) slot_node[sl] = -1;
      pending.clear();
      for (int f = sc.flush_begin[t]; f < sc.flush_begin[t + 1]; ++f) {
        const int node = sc.flush_node[f];
        const int sl = sc.flush_slot[f] & 0xffff;
        if (node < 0 || node >= N) fail("flush node out of range");
        if (node_slot[node] != sl || slot_node[sl] != node) fail("flush of a slot not held");
        if (flushed[node] == g) fail("node flushed twice in a segment");
        flushed[node] = g;
        node_slot[node] = -1;
        pending.push_back(sl);
      }
    }
    for (int sl : pending) slot_node[sl] = -1;
    for (int q = 0; q < sc.S; ++q)
      if (slot_node[q] >= 0) fail("slot still occupied at segment end");
  }
  for (int e = 0; e < E; ++e)
    if (seen[e] != 1) fail("element not swept");
  std::vector<char> zero(N, 0);
  for (int j : sc.zero_cols) zero[j] = 1;
  for (int j = 0; j < N; ++j)
    if ((nseg[j] != 1) != (zero[j] != 0)) fail("zero_cols disagrees with segment counts");
  for (size_t f = 0; f < sc.flush_node.size(); ++f) {
    const bool shared = (sc.flush_slot[f] & kSharedBit) != 0;
    if (shared != (nseg[sc.flush_node[f]] > 1)) fail("shared flag wrong");
  }
}

namespace {

// Nodes of a segment in stream order: first and last position and number of contributions.
struct StreamNodes {
  std::vector<int> first, last, count, touched;
  explicit StreamNodes(int N) : first(N, -1), last(N, -1), count(N, 0) {}
  void sweep(const std::vector<int>& idx, const int* ptopo, int NP) {
    for (int node : touched) first[node] = -1, count[node] = 0;
    touched.clear();
    for (size_t t = 0; t < idx.size(); ++t)
      for (int s = 0; s < NP; ++s) {
        const int node = ptopo[(size_t)idx[t] * NP + s];
        if (first[node] < 0) {
          first[node] = (int)t;
          touched.push_back(node);
        }
        last[node] = (int)t;
        ++count[node];
      }
  }
  // the most contributions to one node
  int most() const {
    int best = 0;
    for (int node : touched) best = std::max(best, count[node]);
    return best;
  }
  // the largest number of slots held at once: a node holds one from its first position to
  // kStreamLag past its last; a node with a single contribution needs none
  int front(size_t n) const {
    std::vector<int> delta(n + kStreamLag + 2, 0);
    for (int node : touched)
      if (count[node] > 1) {
        ++delta[first[node]];
        --delta[last[node] + kStreamLag];
      }
    int live = 0, best = 0;
    for (size_t t = 0; t < n; ++t) best = std::max(best, live += delta[t]);
    return best;
  }
};

}  // namespace

StreamSchedule build_stream_schedule(const int* ptopo, int NP, int E, int N, const double* cent,
                                     int S, int min_segments) {
  StreamSchedule sc;
  sc.S = S;
  sc.NP = NP;
  StreamNodes nd(N);
  std::vector<SegOrder> segs;
  if (E > 0) {
    std::vector<int> all(E);
    std::iota(all.begin(), all.end(), 0);
    auto fits = [&](const std::vector<int>& idx) {
      nd.sweep(idx, ptopo, NP);
      return nd.front(idx.size()) <= S && nd.most() <= kStreamMost;
    };
    split(std::move(all), std::max(1, min_segments), cent, fits, segs);
  }
  sc.n_segments = (int)segs.size();
  std::vector<int> nseg(N, 0), mark(N, -1);
  for (int g = 0; g < sc.n_segments; ++g)
    for (int e : segs[g].elems)
      for (int s = 0; s < NP; ++s) {
        const int node = ptopo[(size_t)e * NP + s];
        if (mark[node] != g) {
          mark[node] = g;
          ++nseg[node];
        }
      }
  for (int j = 0; j < N; ++j) {
    if (nseg[j] != 1) sc.zero_cols.push_back(j);
    sc.n_shared += nseg[j] > 1;
  }
  sc.order.reserve(E);
  sc.ent.reserve((size_t)E * NP);
  sc.seg_begin.push_back(0);
  std::vector<int> slot(N, -1), turn_of(N, 0), turns(S);
  for (const SegOrder& seg : segs) {
    const std::vector<int>& el = seg.elems;
    nd.sweep(el, ptopo, NP);
    std::fill(turns.begin(), turns.end(), 0);
    std::vector<std::vector<int>> release(el.size() + kStreamLag + 1);  // slots by position
    // slots change hands in the order they were given back: the longest possible distance
    // between a node's last contribution and its slot's next node
    std::deque<int> freelist;
    for (int q = 0; q < S; ++q) freelist.push_back(q);
    for (size_t t = 0; t < el.size(); ++t) {
      for (int q : release[t]) freelist.push_back(q);
      for (int s = 0; s < NP; ++s) {
        const int node = ptopo[(size_t)el[t] * NP + s];
        if (nd.first[node] == (int)t && nd.count[node] > 1 && slot[node] < 0) {
          if (freelist.empty()) throw Error{BIE_EINVAL, "stream schedule overflow"};
          slot[node] = freelist.front();
          freelist.pop_front();
          turn_of[node] = turns[slot[node]]++;
          release[nd.last[node] + kStreamLag].push_back(slot[node]);
        }
        sc.ent.push_back(StreamEntry{slot[node], nd.count[node], turn_of[node],
                                     node | (nseg[node] > 1 ? kSharedBit : 0)});
      }
      sc.max_live = std::max(sc.max_live, S - (int)freelist.size());
      sc.order.push_back(el[t]);
    }
    for (int node : nd.touched) slot[node] = -1, turn_of[node] = 0;
    sc.seg_begin.push_back((int)sc.order.size());
  }
  return sc;
}

// Replays a stream schedule: every element once; a node keeps one slot within a segment,
// its entries agree on count and turn; a slot changes hands only after all contributions of
// the node before, at least kStreamLag positions later, with the turn counted up by one.
void validate_stream_schedule(const StreamSchedule& sc, const int* ptopo, int NP, int E, int N) {
  auto fail = [](const std::string& m) { throw Error{BIE_EINVAL, "stream schedule: " + m}; };
  if ((int)sc.order.size() != E || sc.ent.size() != (size_t)E * NP) fail("sizes");
  if ((int)sc.seg_begin.size() != sc.n_segments + 1 || sc.seg_begin[sc.n_segments] != E)
    fail("segment bounds");
  std::vector<int> seen(E, 0), nseg(N, 0), mark(N, -1);
  struct Hold {
    int node = -1, got = 0, count = 0, turn = -1, freed = 0;
  };
  for (int g = 0; g < sc.n_segments; ++g) {
    std::vector<Hold> hold(sc.S);
    for (int t = sc.seg_begin[g]; t < sc.seg_begin[g + 1]; ++t) {
      const int e = sc.order[t];
      if (e < 0 || e >= E || seen[e]++) fail("element swept twice or out of range");
      for (int s = 0; s < NP; ++s) {
        const StreamEntry& x = sc.ent[(size_t)t * NP + s];
        const int node = ptopo[(size_t)e * NP + s];
        if ((x.node & ~kSharedBit) != node) fail("entry of another node");
        if (mark[node] != g) {
          mark[node] = g;
          ++nseg[node];
        } else if (x.slot < 0) {
          fail("direct node with several contributions");
        }
        if (x.slot < 0) {
          if (x.count != 1) fail("direct node with several contributions");
          continue;
        }
        if (x.slot >= sc.S || x.count < 2 || x.count > kStreamMost) fail("slot out of range");
        Hold& h = hold[x.slot];
        if (h.node != node) {
          if (h.got != h.count) fail("slot handed on before its node is complete");
          if (h.node >= 0 && t < h.freed) fail("slot handed on too early");
          if (x.turn != h.turn + 1) fail("turn");
          h = Hold{node, 0, x.count, x.turn, 0};
        }
        if (x.count != h.count || x.turn != h.turn) fail("entries of a node disagree");
        if (++h.got > h.count) fail("more contributions than counted");
        if (h.got == h.count) h.freed = t + kStreamLag;
      }
    }
    for (const Hold& h : hold)
      if (h.got != h.count) fail("node incomplete at the segment's end");
  }
  std::vector<char> zero(N, 0);
  for (int j : sc.zero_cols) zero[j] = 1;
  for (int j = 0; j < N; ++j)
    if ((nseg[j] != 1) != (zero[j] != 0)) fail("zero_cols disagrees with segment counts");
  for (const StreamEntry& x : sc.ent)
    if (((x.node & kSharedBit) != 0) != (nseg[x.node & ~kSharedBit] > 1)) fail("shared flag");
}

}  // namespace bie
