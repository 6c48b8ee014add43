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
// Measured, us a launch with one lane and one workgroup -> parts 2 (parts 1):
//   particles   velocity            recompute           adjoint delta        adjoint div. update
//     2,000     11.6 ->  7.2 (10.6) 10.5 ->  6.2 ( 9.2) 15.7 ->  6.7 (10.1)  20.7 ->  9.0 (12.4)
//     8,500     14.9 ->  9.2 (10.8) 10.5 ->  7.9 ( 9.4) 16.4 ->  9.1 (10.9)  22.6 -> 11.1 (13.8)
//    35,000     14.3 -> 10.8 (12.0) 11.9 ->  9.5 (10.5) 17.4 -> 11.6 (12.5)  20.6 -> 12.6 (13.6)
//    56,000     15.2 -> 13.9 (17.0) 13.7 -> 15.3 (13.6) 21.4 -> 17.1 (17.3)  28.1 -> 19.1 (18.6)
//    98,000     15.7 -> 19.7 (19.0) 15.7 -> 22.3 (18.4) 24.5 -> 27.3 (24.6)  25.5 -> 30.0 (25.6)
// At 98,000 the chip is full with one workgroup a brick and the halo is staged
// again for nothing.
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
inline int gather_parts_log2(int nf, uint32_t nbricks) {
  int parts = nf < 40000 ? 2 : nf < 80000 ? 1 : 0;
  while (parts > 0 && ((uint64_t)nbricks << parts) > SPREAD_GRID) --parts;
  return parts;
}

}  // namespace dfr
