// pbb_slot.h -- the occupancy word of a pool slot: its state bits and the number
// of explorers inside.  No HIP header is included, so the rules also build on
// their own.
#pragma once

#ifdef __HIPCC__
#define PBB_HD __host__ __device__ __forceinline__
#else
#define PBB_HD inline
#endif

namespace pbb {

// RUNNING: admitted, explorers may join.  DONE: the search ended, its result is
// recorded.  CLOSING: a workgroup has left or is about to.
enum { POOL_RUNNING = 1 << 30, POOL_DONE = 1 << 29, POOL_CLOSING = 1 << 28, POOL_MEMBERS = (1 << 28) - 1 };

// A workgroup of W explorers that joins takes the member indices from the count
// on, so the count may only grow while workgroups can still join: they leave
// after DONE, or earlier on the launch's deadline or stop word, which each of them
// reads for itself, and the first one to leave closes the slot before it lowers
// the count.  Otherwise one that joined later would get indices still in use, and
// two explorers a mask bit: donors that claim it one after the other may address
// one mailbox.
PBB_HD bool slot_open(int occ, int W, int epi)
{
    return (occ & POOL_RUNNING) && !(occ & (POOL_DONE | POOL_CLOSING)) && (occ & POOL_MEMBERS) + W <= epi;
}

}  // namespace pbb
