// Where the work-groups of a launch run, as host and device code both reckon it: work-group
// i on XCD (i + r) % n_xcc, r being the rotation of the stream's hardware queue.
#pragma once

namespace drt {

// The rotation that work-group i sees, running on XCD xcc. One below n_xcc where the count
// is right; a count that is too small leaves XCDs past it, and rotations that differ.
constexpr int xcd_rotation(int xcc, int i, int n_xcc) {
  const int r = xcc - i % n_xcc;
  return r < 0 ? r + n_xcc : r;
}

// What a work-group that finds itself a rotation r away from the forward's reports in the
// error word besides bit 0, the placement's.
constexpr int placement_bit(int r) { return 1 << (8 + r); }

// A drained stream's error word without its placement reports, if every one of them names the
// rotation that the stream has now and every arrival counter is back at zero (at_rest); other
// kernels' bits stay. Else the word as it is.
// The counters tell a rotation that moved between launches from one that moved inside one:
// there a block's slices counted in two XCDs' L2s, neither reached the block's count, and
// what either wrote back is neither zero nor the count. Every later launch then ends its
// block early by as much and leaves the same remainder.
constexpr int settled_word(int word, int rotation, bool at_rest) {
  constexpr int any = ((1 << 16) - 1) << 8;
  if (rotation < 0 || !at_rest || (word & any) != placement_bit(rotation)) return word;
  return word & ~(1 | placement_bit(rotation));
}

}  // namespace drt
