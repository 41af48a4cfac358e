// Memory the workgroups of a persistent PCG exchange data through.  No device
// code, so that host code can check it.
#pragma once

namespace silk::amd {

/// Buf<T>: a device buffer with zero(stream).
template <template <class> class Buf>
struct PcgWords {
  // Epoch-tagged words (hip/pcg_exchange.hpp): the two-exchange kernel's z0 of
  // the slots, sums of the level-1 nodes, corrections of the coarse nodes and
  // r.z_coarse of the coarse banks; the one-exchange kernel's two buffers;
  // both kernels' partial sums and dx.
  Buf<unsigned long long> tz, tn, tc, tcp, tw, tp, tdx;
  Buf<unsigned> bar;  // per system: the epoch of the last solve's last exchange
  Buf<int> abort;     // a wait gave up

  template <class Fn>
  void each(Fn&& fn) {
    fn(tz);
    fn(tn);
    fn(tc);
    fn(tcp);
    fn(tw);
    fn(tp);
    fn(tdx);
    fn(bar);
    fn(abort);
  }

  /// Before the first solve, and after one in which a wait gave up.  The epochs
  /// start again at 1, so no word may keep a tag: one left by an abandoned
  /// exchange would be taken for the same epoch's of the next solve.
  template <class Stream>
  void clear(Stream s) {
    each([&](auto& b) { b.zero(s); });
  }
};

}  // namespace silk::amd
