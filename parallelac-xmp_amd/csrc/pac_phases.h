/*
 * pac_phases.h -- how the triangle / edge emptiness runs over a number of
 * simplices (plain C++: the rule is tested on the host).
 */
#ifndef PAC_PHASES_H
#define PAC_PHASES_H
#include <cstdint>

namespace pac {

/* Simplices from this many on are packed by the blocks that scan them: the
 * dead and closed ones leave most lanes of a wave idle otherwise; fewer do
 * not fill the chip as they are. */
constexpr int64_t kPackItems = 1 << 17;
/* A packing block marks those it leaves to phase B untested with this bit of
 * their id; ids that need the bit for themselves are not packed, and phase B
 * then takes every entry as an id. */
constexpr uint32_t kRestWhole = 0x80000000u;

struct LowPhases {
  bool pack;
  uint32_t whole; /* phase B: the mark, 0 if there is none */
};
/* marks: covered edges are marked (most simplices are decided at once);
 * budget: phase A's pairs a simplex (0: one phase) */
inline LowPhases low_phases(bool marks, int64_t items, int budget) {
  const bool p = marks && budget > 0 && items >= kPackItems &&
                 items <= (int64_t)kRestWhole;
  return LowPhases{p, p ? kRestWhole : 0u};
}
/* an entry of phase B's list: the simplex, and the pairs tested before */
constexpr uint32_t left_id(uint32_t x, uint32_t whole) { return x & ~whole; }
constexpr int left_tested(uint32_t x, uint32_t whole, int budget) {
  return (x & whole) ? 0 : budget;
}

}  // namespace pac
#endif
