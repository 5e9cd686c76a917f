// ha_mark.h -- a slab's full mark: a word beside its counter that says the
// count is at or above the busy threshold, so that a probe need not load the
// counter itself.  Shared by the device code and the host test that runs the
// interleavings.
//
// The mark is not part of the counter's atomic, so stores to it can pass each
// other.  A mark of 1 that is out of date costs one visit to the head search,
// which clears it.  A mark of 0 that is out of date would last: groups would
// probe a full slab to the end of their tries.  So once every group is done,
// a count at the threshold has its mark set:
//   * the add that takes the count to the threshold sets it;
//   * whoever clears it looks at the slab again once the 0 is in place, and
//     sets it if an add came in between; an add that comes later finds a count
//     below the threshold and sets it itself.  The slab may by then hold
//     another class, so the second look takes the threshold of its class now;
//   * an add that is taken back (the slab had passed to another class) does
//     not mark, so an add on top of it may have found the count at the
//     threshold already: what is left after the give-back decides.
//
// M: set(v) stores the mark, get() loads it, settle() waits until the store is
// in place, full() loads the slab's class and count and compares.
#pragma once

#include "ha_bits.h"

namespace ha {

template <class M>
HA_HD inline void mark_clear(M m) {
  m.set(0);
  m.settle();
  if (m.full()) m.set(1);
}
// a group's add took the count from oc to nc
template <class M>
HA_HD inline void mark_added(M m, u32 oc, u32 nc, u32 thr) {
  if (oc < thr && nc >= thr) m.set(1);
}
// a free took it from oc to nc
template <class M>
HA_HD inline void mark_freed(M m, u32 oc, u32 nc, u32 thr) {
  if (oc >= thr && nc < thr) mark_clear(m);
}
// a group took its add back
template <class M>
HA_HD inline void mark_taken_back(M m, u32 oc, u32 nc, u32 thr) {
  if (nc >= thr) m.set(1);
  else mark_freed(m, oc, nc, thr);
}
// a head search read the count c
template <class M>
HA_HD inline void mark_checked(M m, u32 c, u32 thr) {
  if (c >= thr) m.set(1);
  else if (m.get()) mark_clear(m);
}

}  // namespace ha
