// Bookkeeping of a wave's slot table in the wave-per-source search: plain integer arithmetic, for the
// kernel and for a host program alike.
//
// Slots are numbered in the order in which nodes are expanded.  The newest lie in an LDS ring, slot s at
// s % kRing; those below `out` have left it for the wave's part of the global table.
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define RL_BOTH __host__ __device__ __forceinline__
#else
#define RL_BOTH inline
#endif

namespace rl {

constexpr uint32_t kRing = 512;
constexpr uint32_t kRingMask = kRing - 1U;
constexpr uint32_t kLeave = 64;            // slots that leave the ring together; a step adds at most as many
// Slots of a source: one less than the table's 2,048 records, so that every slot number up to and including
// the number of slots, which a node without expanded children records, fits the 11 bits of an fx entry.
constexpr uint32_t kMostSlots = 2047;

// What a slot records of its children: the slot of the first expanded one and how many there are.
RL_BOTH uint32_t fx_pack(uint32_t slot, uint32_t count) { return slot | count << 11U; }
RL_BOTH uint32_t fx_slot(uint32_t fx) { return fx & 0x7FFU; }
RL_BOTH uint32_t fx_count(uint32_t fx) { return fx >> 11U; }

// The number of slots up to which a step needs no room made: the end of the ring, and of the table.
RL_BOTH uint32_t slot_limit(uint32_t out) { return out + kRing < kMostSlots ? out + kRing : kMostSlots; }

// A step that processed the slots before `end` and brings their number to `tail`, above slot_limit(out):
// whether kLeave slots can leave the ring for it.  Otherwise the source goes to the per-lane search.
RL_BOTH bool slots_can_leave(uint32_t tail, uint32_t out, uint32_t end) {
    return tail <= kMostSlots && out + kLeave <= end;
}

// The masses of expanded children are pulled into their parents from the last slot on, up to 64 slots at
// a time: of the slots [first, first + 64) below hi, the ones above the last that has a child below hi
// (`open`, a bit per slot).  Children follow their parents, so slot hi - 1 is never open, and the result is
// below hi.
RL_BOTH uint32_t pull_from(uint32_t first, uint64_t open) {
    return open == 0 ? first : first + 64U - static_cast<uint32_t>(__builtin_clzll(open));
}

}  // namespace rl
