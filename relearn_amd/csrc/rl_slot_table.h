// Bookkeeping of a wave's slot table in the wave-per-source search: plain integer arithmetic, for the
// kernel and for a host program alike.
//
// Slots are numbered in the order in which nodes are expanded.  [out, out + kRing) lie in an LDS ring, slot s
// at s % kRing; those below have left it for the wave's part of the global table, and those that were
// expanded while the ring was full of waiting ones wait there for their place.
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
// Slots of a source: every slot number up to and including the number of slots, which a node without expanded
// children records, fits the 11 bits of an fx entry.  The table's last record takes the slots beyond of the step
// that needs more.
constexpr uint32_t kMostSlots = 2047;
constexpr uint32_t kSlotRecords = kMostSlots + 1;

// What a slot records of its children: the slot of the first expanded one and how many there are.
RL_BOTH uint32_t fx_pack(uint32_t slot, uint32_t count) { return slot | count << 11U; }
RL_BOTH uint32_t fx_slot(uint32_t fx) { return fx & 0x7FFU; }
RL_BOTH uint32_t fx_count(uint32_t fx) { return fx >> 11U; }

// The number of slots up to which a step appends to the ring as it is: the end of the ring, and of the table.
RL_BOTH uint32_t slot_limit(uint32_t out) { return out + kRing < kMostSlots ? out + kRing : kMostSlots; }

// The record in which a slot waits outside the ring.
RL_BOTH uint32_t waiting_record(uint32_t slot) { return slot < kMostSlots ? slot : kMostSlots; }

// Whether the first kLeave slots leave the ring after a step that processed the slots before `end` and went
// beyond slot_limit(out).  While slots wait outside, that is asked after every step, and a step processes 8:
// they enter the ring long before their turn.
RL_BOTH bool slots_leave(uint32_t out, uint32_t end) { return out + kLeave <= end; }

// The masses of expanded children are pulled into their parents from the last slot on, up to 64 slots at
// a time: of the slots [first, first + 64) below hi, the ones above the last that has a child below hi
// (`open`, a bit per slot).  Children follow their parents, so slot hi - 1 is never open, and the result is
// below hi.
RL_BOTH uint32_t pull_from(uint32_t first, uint64_t open) {
    return open == 0 ? first : first + 64U - static_cast<uint32_t>(__builtin_clzll(open));
}

}  // namespace rl
