// A wave's slot table on the CPU: the traversal's steps, the ring's eviction and the pull of the masses as
// the wave-per-source search does them, over the same functions (rl_slot_table.h), for trees given by the
// number of expanded children of every slot.  Usage: slot_table_check SLOTS WAITING SEED [--end-full]
//   SLOTS      slots that the source needs
//   WAITING    slots that wait at most (the width of the tree)
//   --end-full the last slots get all their children in one step
// Prints "done" or "overflow"; exit status 1 if a record is wrong or the pull makes no progress.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "rl_slot_table.h"

using namespace rl;

namespace {

int fail(const char* what, uint32_t at) {
    std::printf("wrong: %s at %u\n", what, at);
    return 1;
}

// Expanded children per slot, in queue order: `slots` in all, about `waiting` of them waiting at a time.
std::vector<uint32_t> tree(uint32_t slots, uint32_t waiting, bool end_full, std::mt19937& gen) {
    std::vector<uint32_t> kids;
    uint32_t tail = 1;
    for (uint32_t k = 0; k < tail; k++) {
        const uint32_t left = slots - tail;
        const uint32_t queued = tail - k - 1;
        uint32_t c = queued < waiting ? std::min<uint32_t>(8, waiting - queued) : 0;
        c = c == 0 ? 0 : gen() % (c + 1);
        c = std::max(c, queued == 0 ? 1U : 0U);
        if (end_full && left <= 64 && queued >= 8 && queued < 16) {
            c = 8;
        } else if (end_full && left <= 64 && queued > 0) {
            c = 0;
        }
        c = std::min(c, left);
        kids.push_back(c);
        tail += c;
    }
    return kids;
}

}  // namespace

int main(int argc, char** argv) {
    if (argc < 4) {
        return 2;
    }
    const uint32_t slots = static_cast<uint32_t>(std::atoi(argv[1]));
    const uint32_t waiting = static_cast<uint32_t>(std::atoi(argv[2]));
    std::mt19937 gen(static_cast<uint32_t>(std::atoi(argv[3])));
    const std::vector<uint32_t> kids = tree(slots, waiting, argc > 4, gen);

    std::vector<double> ms(kRing, -1.0), t_ms(kSlotRecords, -1.0);
    std::vector<uint32_t> my(kRing, ~0U), t_my(kSlotRecords, ~0U), t_fx(kSlotRecords, ~0U);
    std::vector<uint16_t> fx(kRing, 0xFFFF);
    // an entry of the queue stands for its own slot number, its mass is 1
    uint32_t tail = 1, out = 0, limit = slot_limit(0), most_waiting = 0;
    my[0] = 0;
    // a step covers up to 8 queue entries, read before the step ahead of it appends its own
    uint32_t kb = 0, end = 1;
    std::vector<uint32_t> entry{ my[0] };
    while (true) {
        const uint32_t next_end = std::min(end + 8, tail);
        std::vector<uint32_t> next;
        for (uint32_t k = end; k < next_end; k++) {
            next.push_back(my[k & kRingMask]);
        }
        const uint32_t before = tail;
        uint32_t to = tail;
        for (uint32_t k = kb; k < end; k++) {
            if (entry[k - kb] != k) {
                return fail("queue entry", k);
            }
            fx[k & kRingMask] = static_cast<uint16_t>(fx_pack(to, kids[k]));
            ms[k & kRingMask] = 1.0;
            to += kids[k];
        }
        for (uint32_t s = before; s < to; s++) {
            if (waiting_record(s) >= kSlotRecords || (to <= limit && s >= out + kRing)) {
                return fail("slot out of range", s);
            }
            (to <= limit || s < out + kRing ? my[s & kRingMask] : t_my[waiting_record(s)]) = s;
        }
        tail = to;
        most_waiting = std::max(most_waiting, tail - end);
        if (tail > limit) {
            if (tail > kMostSlots) {
                std::printf("overflow %u %u\n", tail, most_waiting);
                return 0;
            }
            if (slots_leave(out, end)) {
                for (uint32_t s = out; s < out + kLeave; s++) {
                    t_my[s] = my[s & kRingMask];
                    t_fx[s] = fx[s & kRingMask];
                    t_ms[s] = ms[s & kRingMask];
                    if (s + kRing < tail) {
                        my[s & kRingMask] = t_my[s + kRing];
                    }
                }
                out += kLeave;
                limit = slot_limit(out);
            }
        }
        if (end >= tail) {
            break;
        }
        kb = end;
        end = next_end;
        entry = next;
    }
    if (tail != slots) {
        return fail("number of slots", tail);
    }
    // records as the draws read them
    uint32_t first_child = 1;
    for (uint32_t s = 0; s < tail; s++) {
        const uint32_t f = s >= out ? fx[s & kRingMask] : t_fx[s];
        const uint32_t m = s >= out ? my[s & kRingMask] : t_my[s];
        if (m != s || fx_count(f) != kids[s] || (kids[s] != 0 && fx_slot(f) != first_child)) {
            return fail("record", s);
        }
        first_child += kids[s];
    }
    // the pull
    uint32_t hi = tail;
    while (hi > 0) {
        const uint32_t first = hi > 64 ? hi - 64 : 0;
        uint64_t open = 0;
        for (uint32_t s = first; s < hi; s++) {
            const uint32_t f = s >= out ? fx[s & kRingMask] : t_fx[s];
            open |= fx_count(f) != 0 && fx_slot(f) < hi ? 1ULL << (s - first) : 0;
        }
        const uint32_t lo = pull_from(first, open);
        if (lo >= hi) {
            return fail("no progress of the pull", hi);
        }
        for (uint32_t s = lo; s < hi; s++) {
            const uint32_t f = s >= out ? fx[s & kRingMask] : t_fx[s];
            for (uint32_t c = 0; c < fx_count(f); c++) {
                const uint32_t k = fx_slot(f) + c;
                (s >= out ? ms[s & kRingMask] : t_ms[s]) += k >= out ? ms[k & kRingMask] : t_ms[k];
            }
        }
        hi = lo;
    }
    if ((out == 0 ? ms[0] : t_ms[0]) != static_cast<double>(slots)) {
        return fail("mass of the root", slots);
    }
    std::printf("done %u %u\n", slots, most_waiting);
    return 0;
}
