// Index rules of the persistent PCG that have no device code in them, so that
// host code can check them.
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

}  // namespace silk::amd
