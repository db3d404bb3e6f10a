// Schedules of the assembly kernels' LDS slots (built by schedule.cpp).
#pragma once

#include <cstdint>
#include <string>
#include <vector>

#include "bie_common.hpp"

namespace bie {

constexpr int kSharedBit = 1 << 30;

// Slot schedule in steps of W elements (bie_schedule_check's statistics; no kernel runs by it).
struct SlotSchedule {
  int W = 0;            // elements per step (waves per workgroup)
  int S = 0;            // LDS slots available
  int NP = 0;
  int n_segments = 0;
  int n_steps = 0;
  int n_shared = 0;     // nodes touched by more than one segment
  int max_live = 0;     // largest number of live slots over all steps
  std::vector<int> seg_step_begin;  // n_segments + 1
  std::vector<int> step_elems;      // n_steps * W (element id or -1)
  std::vector<int> slot_of;         // E * NP slot of each element-local node
  std::vector<int> flush_begin;     // n_steps + 1
  std::vector<int> flush_node;      // node column flushed after the step
  std::vector<int> flush_slot;      // slot | kSharedBit when the node is shared
  std::vector<int> zero_cols;       // columns to zero before the kernel
};

// min_segments: the number of segments to aim for (exactly that many unless a segment's
// front exceeds S slots, which splits it further).
SlotSchedule build_slot_schedule(const int* ptopo, int NP, int E, int N, const double* cent,
                                 int W, int S, int min_segments);

// Stream schedule of the barrier-free slot kernels (stream.hip): every segment is an ordered
// list of elements that the waves of a workgroup take one at a time; a node's contributions
// meet in an LDS slot, which the wave that brings the last one writes out.
struct StreamEntry {  // one per (position, element node): an int4 on the device
  int slot;           // LDS slot, or -1: the node's only element of the segment is this one
  int count;          // contributions the node receives in the segment
  int turn;           // how many nodes held the slot before (it must have been freed so often)
  int node;           // column | kSharedBit when other segments add to it as well
};
struct StreamSchedule {
  int S = 0, NP = 0, n_segments = 0, n_shared = 0, max_live = 0;
  std::vector<int> seg_begin;      // n_segments + 1 positions
  std::vector<int> order;          // element at each position
  std::vector<StreamEntry> ent;    // E * NP, by position
  std::vector<int> zero_cols;      // columns the kernel adds to, or does not touch at all
};
// A slot is handed to a new node kStreamLag positions after its last contribution at the
// earliest (any positive distance is correct; a few positions keep the waves, which run
// that far apart, from waiting for each other).
constexpr int kStreamLag = 6;
// A slot's claims and finished contributions are counted in 16 bits each.
constexpr int kStreamMost = 0xffff;
StreamSchedule build_stream_schedule(const int* ptopo, int NP, int E, int N, const double* cent,
                                     int S, int min_segments);
void validate_stream_schedule(const StreamSchedule& sc, const int* ptopo, int NP, int E, int N);

void validate_slot_schedule(const SlotSchedule& sc, const int* ptopo, int NP, int E, int N);

}  // namespace bie
