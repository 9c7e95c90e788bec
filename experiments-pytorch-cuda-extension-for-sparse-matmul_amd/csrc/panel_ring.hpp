// The ring of panel buffers of weight_panels.hip: how many buffers and fetching waves there are, and when a buffer may be filled
// again.  Free of HIP, so that a test builds the same rule with g++ and walks through every order in which the waves can run
// (tests/test_panel_ring.py).
#pragma once

#if defined(__HIPCC__)
#define BSA_RING __host__ __device__ __forceinline__
#else
#define BSA_RING inline
#endif

namespace bsa {

// panels in LDS at a time: as many as a compute unit's 160 KB hold beside the lists of the widest contraction
BSA_RING constexpr int panel_stages(int rt) { return rt <= 3 ? 4 : 3; }
constexpr int PANEL_FETCHERS = 3;               // waves that do nothing but fetch them: panel s is wave s % PANEL_FETCHERS'

// Flags: ready[buffer] is one more than the last panel that has arrived in it, done[wave] the first panel a multiplying wave may
// still read.
constexpr int PANEL_READY = 0, PANEL_DONE = 4;

// Panel s may be fetched where the flag that each lane watches has reached panel_refill_from: the panel before in this buffer,
// s - stages, has been read by all, and it has ARRIVED.  Neither follows from the other: a wave is done with a panel in which it
// has no block without having waited for it, and where there are more buffers than fetching waves another wave has requested it.
// Filled before that, the late panel lands over panel s, and its flag goes back behind the wave that waits for panel s.
BSA_RING constexpr int panel_refill_flag(int lane, int walkers, int s, int stages)
{
    return lane < walkers ? PANEL_DONE + lane : PANEL_READY + s % stages;
}
BSA_RING constexpr int panel_refill_from(int s, int stages) { return s - stages + 1; }

}  // namespace bsa
