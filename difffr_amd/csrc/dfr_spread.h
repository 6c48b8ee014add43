// How a scene's gather passes are spread over the chip.  Plain C++, no HIP.
#pragma once
#include <cstdint>

namespace dfr {

// A pass of a few bricks costs the chain of one wavefront: staging, then some 40
// pairs one after the other per lane, and up to 20 boundary samples a group at a
// time.  There, 2^parts workgroups share a brick's particles (each stages the whole
// halo) and four lanes share a particle's pairs.  The step's own passes still add in
// list order (Terms in dfr_tile.h): a solve's masks flip on an ulp, and a trajectory
// would hang on the scene's size.  The reverse passes, linear in what they carry, add
// each lane's partial sum.
//
// The two kinds turn at different sizes.  Velocity + recompute and the reverse delta +
// update + factor, us with one lane and one workgroup -> parts 1, 2 (full tanks at rest
// density, 12, 20 and 30 particles deep; the boundary's share differs between them):
//   particles   forward          forward          forward          reverse
//    28,000     29 -> 26, 21     32 -> 31, 26     31 -> 31, 24     53 -> 37, 32
//    36,000     31 -> 33, 28     31 -> 27, 25     32 -> 35, 28     58 -> 45, 43
//    42,000     31 -> 35, 29     31 -> 28, 27     32 -> 34, 29     55 -> 48, 47
//    45,000     31 -> 37, 31     31 -> 28, 27     32 -> 34, 29     56 -> 50, 49
//    50,000     30 -> 36, 31     32 -> 38, 34     31 -> 35, 29     54 -> 50, 52
//    55,000     32 -> 37, 34     32 -> 39, 35     35 -> 40, 31     61 -> 53, 60
//    78,000                      37 -> 44, 43                      75 -> 67, 74
// (2,000 particles: forward 22 -> 20, 13.)  Parts 1 never pay forward.  Parts 2 do up to some 45,000 particles as long as these
// fill few bricks (the rows above up to 45,000: 64 to 108, but the first column's last,
// 128).  Shallow tanks of ten layers at spacing 2 r, which have fewer pairs, a whole step
// of two divergence and four pressure iterations: 22,000 particles in 72 bricks 267 -> 252
// us, 26,000 in 98 265 -> 263, 30,000 in 98 260 -> 271, 36,000 in 128 251 -> 280, 42,000
// in 162 263 -> 303.  The reverse passes gain with parts 1 up to 80,000 particles.
// Beyond (98,000: velocity 15.7 -> 19.0, delta 24.5 -> 24.6) the chip is full with one
// workgroup a brick and the halo is staged again for nothing.
//
// The grid covers the domain, and a workgroup of an empty brick still costs about
// half a nanosecond: few particles in a large domain pay 2^parts times the empty
// workgroups.  Velocity + recompute and the reverse delta + update, us with one
// lane -> parts 2 (parts 1):
//   bricks  1,000 particles                            16,000 particles
//      729  23 -> 19 (22)   28 -> 16 (19)   30 -> 28 (31)   36 -> 27 (29)
//    1,331  23 -> 21 (23)   28 -> 18 (20)   31 -> 31 (31)   37 -> 31 (29)
//    2,744  24 -> 25 (25)   28 -> 21 (22)   31 -> 36 (33)   38 -> 35 (31)
//    4,913  26 -> 44 (29)   30 -> 36 (24)   35 -> 54 (44)   42 -> 51 (40)
// So the spread grid stays within 5,120 workgroups: 1,280 bricks with parts 2, 2,560
// with parts 1.  (A step of 30,000 particles in 117,649 bricks with two divergence
// and four pressure iterations: 1.84 ms with one workgroup a brick, 7.75 with four.)
constexpr uint32_t SPREAD_GRID = 5120;
inline bool spread_fits(uint32_t nbricks, int parts) { return ((uint64_t)nbricks << parts) <= SPREAD_GRID; }
// log2 of the workgroups a brick (0: one, and one lane per particle).  filled: the
// bricks that hold particles when the scene starts; not looked at from
// FORWARD_PARTICLES on.
constexpr int FORWARD_PARTICLES = 44000;
inline int forward_parts_log2(int nf, uint32_t nbricks, uint32_t filled) {
  return nf < FORWARD_PARTICLES && filled <= 112 && spread_fits(nbricks, 2) ? 2 : 0;
}
inline int reverse_parts_log2(int nf, uint32_t nbricks) {
  if (nf < 44000 && spread_fits(nbricks, 2)) return 2;
  return nf < 80000 && spread_fits(nbricks, 1) ? 1 : 0;
}
// The list build goes by cells where the reverse passes are spread: 28,000 particles
// 31 us (60 by particles), 56,000 55 (61), 78,000 69 (78); 16,000 in 2,744 bricks 46
// (58), in 4,913 61 (63), in 9,261 81 (66).
inline bool build_by_cells(int nf, uint32_t nbricks) { return reverse_parts_log2(nf, nbricks) > 0; }

}  // namespace dfr
