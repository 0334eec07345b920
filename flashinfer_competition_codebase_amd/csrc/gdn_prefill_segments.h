// gdn_prefill_segments.h - what each unit of the prefill's two segment scan
// launches starts from and where it ends (included by gdn_prefill.hip; plain
// C++, so that the rules can be checked on the host).

#pragma once

namespace gdn_pf {

// A 128 x 128 block a unit starts from or ends in, per (sequence, v-head).
// kState and kNewState are the caller's state and new_state (the same block
// for an in-place call), the others the workspace's of one segment.
enum class SegBlock {
  kNone,         // nowhere; as a start: zeros
  kIdentity,     // as a start only
  kState,
  kNewState,
  kStart,        // the state at the segment's start
  kZeroEnd,      // the state at its end from a zero start
  kTransition,   // its transition
};

struct SegUnit {
  int seg;             // the segment it scans
  SegBlock from;       // its start, of segment `seg`
  SegBlock to;         // its end, of segment `to_seg`
  int to_seg;
  bool keep_start;     // also copies its start to kStart of segment `seg`
};

// Unit u of a sequence of nseg segments (nseg >= 2 in the first launch).
// First launch (out false), 2 nseg - 3 units: segment 0 from the sequence's
// state, segments 1 .. nseg-2 from a zero start and from the identity.
// Second launch (out true), nseg units: every segment from its start, the
// last one's end being the new state.  In the second launch nothing orders
// the last segment's unit after segment 0's: in place (state and new_state
// the same block), segment 0 then starts from the copy that the first launch
// kept, and only a sequence of one segment, whose one unit reads before it
// writes, from the state itself.
constexpr SegUnit seg_unit(bool out, int nseg, int u, bool in_place) {
  if (!out) {
    const int mid = nseg - 2;
    if (u == 0) return SegUnit{0, SegBlock::kState, SegBlock::kStart, 1, in_place};
    if (u <= mid) return SegUnit{u, SegBlock::kNone, SegBlock::kZeroEnd, u, false};
    return SegUnit{u - mid, SegBlock::kIdentity, SegBlock::kTransition, u - mid, false};
  }
  const SegBlock from =
      u == 0 && (nseg == 1 || !in_place) ? SegBlock::kState : SegBlock::kStart;
  return SegUnit{u, from, u == nseg - 1 ? SegBlock::kNewState : SegBlock::kNone, u, false};
}

}  // namespace gdn_pf
