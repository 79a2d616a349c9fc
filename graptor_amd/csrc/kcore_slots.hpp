// kcore_slots.hpp -- which list and which count the phases of the k-core
// peeling use.
//
// List r has its lengths in slot kc_slot(r) of three and its entries in buffer
// r & 1.  A pass appends to its list; round r reads list r and appends to list
// r + 1.  Between two barriers blocks are unordered: each reads a list's
// lengths after the first and goes on into the phase that they ask for, while
// others may not have read them yet.  So no phase appends to, or clears, the
// slot that was read before it: a round appends one slot on and clears the one
// after that, and a pass, which follows a list read as empty, skips that list
// (kc_after_empty).
#pragma once

#ifdef __HIPCC__
#define KC_FN __host__ __device__ constexpr
#else
#define KC_FN constexpr
#endif

namespace gpr {

KC_FN unsigned kc_slot(unsigned r) { return r % 3; }
// the list that a pass fills after list r was read as empty
KC_FN unsigned kc_after_empty(unsigned r) { return r + 1; }
// cleared during round r, and during the pass that fills list r
KC_FN unsigned kc_cleared_by_round(unsigned r) { return kc_slot(r + 2); }
KC_FN unsigned kc_cleared_by_pass(unsigned r) { return kc_slot(r + 1); }

} // namespace gpr
