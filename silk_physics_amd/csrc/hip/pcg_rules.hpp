// Rules of the persistent PCG that have no device code in them, so that host
// code can check them.
#pragma once

namespace silk::amd {

/// Place of entry e of a row (lane `lane` of its slice) in the slot-ELL, whose
/// slice starts at `off` and holds `width` entries per row.  An entry the row
/// does not have is read at place 0, which every table has: a slice of width 0
/// (only padding and vertices of no face) owns no storage, and past its start
/// the table may end.
constexpr int sell_place(int off, int width, int e, int slice, int lane) {
  return e < width ? off + e * slice + lane : 0;
}

/// Epoch the one-exchange kernel leaves in its counter after a solve that found
/// `before` there and whose last exchange was `last`; the next solve starts
/// one above it.  Epoch last + 1 is left out: M0 r went out under it when the
/// last step was taken.  The parity is such that the first exchanges of
/// consecutive solves use different buffers, so that solves that end at their
/// first exchange (a scene at rest) leave no word older than two solves in
/// either: the level-1 sums carry 16 bits of their epoch only, and one left
/// alone for 65,536 epochs would be taken for a new one.
constexpr unsigned one_last_epoch(unsigned before, unsigned last) {
  const unsigned next = last + 1;
  return ((next - before) & 1u) != 0 ? next : next + 1;
}

}  // namespace silk::amd
