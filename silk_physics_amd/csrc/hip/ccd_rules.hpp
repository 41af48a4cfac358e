// Rules of the CCD's root search that have no device code in them, so that host
// code can check them.
#pragma once

namespace silk::amd {

/// When a search re-reads the running minimum: 32 passes after the last time.
/// A pass can count for two (a half without a root is done with in its
/// parent's), so the count may step over any given number.
struct CutRefresh {
  int next = 32;
  constexpr bool due(int iter) {
    if (iter < next) return false;
    next = iter + 32;
    return true;
  }
};

}  // namespace silk::amd
