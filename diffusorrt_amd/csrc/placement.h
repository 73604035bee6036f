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
// rotation that the stream has now; other kernels' bits stay. Else the word as it is.
constexpr int settled_word(int word, int rotation) {
  constexpr int any = ((1 << 16) - 1) << 8;
  if (rotation < 0 || (word & any) != placement_bit(rotation)) return word;
  return word & ~(1 | placement_bit(rotation));
}

}  // namespace drt
