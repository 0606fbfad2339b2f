// Wavefront-cooperative Barnes-Hut target search.
//
// One wavefront handles one source neuron at a time.  The lanes form 8 groups of 8; in the
// traversal a group takes one expanded node and each of its lanes tests one child, so a wavefront
// tests the children of 8 nodes per step.  The traversal is breadth-first over exactly the nodes
// that BarnesHutBase::get_nodes_to_consider (source/algorithm/BarnesHutInternal/BarnesHutBase.h:
// 129-206) tests -- the children of every expanded node, each with test_acceptance_criterion
// (:72-114) -- so the acceptance-test count equals the CPU path's.
//
// Expanded nodes get a slot in a per-wave table: node, first expanded-child slot and count, and
// the node's mass = total probability of the accepted candidates below it.  A group sums the
// probabilities of its accepted children with a DPP butterfly; after the traversal the masses of
// expanded children are pulled into their parents, last slots first.  The mass of a node is the
// span its subtree occupies in the reference's candidate list (descending Morton order = children
// visited in descending octant order), so a draw r is resolved top-down
// (ProbabilityPicker::pick_target, source/util/ProbabilityPicker.h:46-112): at each expanded node
// the children are scanned in descending octant order with the running sum of their masses and the
// first child whose running sum reaches r is entered, or returned when it is an accepted candidate.
// Up to 8 draws (one per group) are resolved at once.  The descents below a picked node
// (BarnesHutBase::find_target_neuron, :223-255) usually accept all children of the node; a group
// then does the whole level -- test, sum, draw, pick -- on its own, in parallel for all axons of the
// neuron.  Levels that need expansion (rare) run through the general traversal afterwards.
//
// Sums are formed in a fixed order, so results are deterministic and independent of launch
// geometry; they differ from the CPU's left-to-right sums only by rounding, so only draws within
// ~1e-15 of a cumulative boundary can resolve differently.
//
// Work distribution: persistent waves; active sources in Morton order are split into one
// contiguous segment per XCD so that an XCD's L2 caches one region of the tree; waves take sources
// from their XCD's segment, then from the others.  A source whose slot table would overflow is handed
// to the per-lane kernel.
#include <algorithm>

#include "rl_search_eval.h"
#include "rl_slot_table.h"

namespace rl {
namespace {

constexpr int kWave = 64;
constexpr int kXcds = kCursorSlots;

struct CoopArgs {
    SearchArgs s;
    const uint32_t* work;
    const uint64_t* nwork;        // device count of work; XCD segment x is [nwork x / 8, nwork (x + 1) / 8)
    unsigned long long* cursor;   // kXcds counters
    uint32_t chunk;               // sources taken from a segment per cursor increment
    uint32_t* t_my;               // per wave: cap slots, of which those outside the LDS ring are used
    uint32_t* t_fexp;
    double* t_mass;
    uint32_t cap;                 // records per wave: kSlotRecords
    uint32_t* overflow;
    unsigned long long* n_overflow;
    uint4* slow;                  // (slot, source, node, level) of descents for the per-lane kernel
    unsigned long long* n_slow;
    uint64_t run_below;           // the kernel returns at once when *nwork >= run_below
};

// The slot table of the source a wave works on: per expanded node its packed child range (which also makes
// the table the traversal's queue), the slot of its first expanded child with their number, and its
// mass.  LDS holds a ring of kRing slots, the wave's part of the global table the others: a source expands
// about 110 nodes at 1,000 neurons, 340 at 52,000, 550 at 1M and 640 at 4M (theta 0.3), so few slots or
// none leave the ring, and those are the top of the tree.
//
// A level has up to about 4/3 pi / theta^3 expanded nodes: 155 at theta 0.3, 393 at 0.22, 523 at 0.2, so at
// small theta more slots wait than the ring holds.  They wait in the global table.  While such sources were
// handed to the per-lane search, the 1M-neuron update took 87.8 ms at theta 0.22 (a quarter of the sources),
// now 19.2, and 106.2 ms in FP64, now 24.8.  Sources that need more than the table are handed over still.
//
// What bounds the search are its vector instructions (units 0.99 busy at 1M neurons, both precisions) and the data
// path of its loads (0.97), so every instruction of a step counts; the scalar unit is 0.58 busy, L2 hits
// 0.97.  With the whole table in global memory behind LDS staging rings, the level boundaries
// tracked in every step and the reference's formulas inlined, a step took about 150 instructions and
// the FP32-mixed kernel 96 VGPRs (5 waves per SIMD); now 105 and 80 (6 waves, 22 per CU by LDS).  1M
// neurons: FP32-mixed 12.1 -> 8.7 ms, FP64 16.0 -> 11.3 ms.
template <bool kMixed>
struct CoopShared {
    double ms[kRing];
    double2 exp_table[kMixed ? 1 : 32]; // 2^(i/32), first and second part (FP64 search only)
    uint32_t my[kRing];
    uint16_t fx[kRing];                 // fx_pack(first expanded child's slot, expanded children)
};

__device__ __forceinline__ uint32_t lane() {
    return __lane_id();
}

// Set bits of `mask` below the calling lane (v_mbcnt_lo/hi: two instructions instead of a masked
// 64-bit population count).
__device__ __forceinline__ uint32_t rank_below(uint64_t mask) {
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32U),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0U));
}

__device__ __forceinline__ double uniform_f64(double v) {
    const int lo = __builtin_amdgcn_readfirstlane(__double2loint(v));
    const int hi = __builtin_amdgcn_readfirstlane(__double2hiint(v));
    return __hiloint2double(hi, lo);
}

// Lanes whose DPP source lies outside their row read 0 (bound_ctrl).
template <int kCtrl>
__device__ __forceinline__ double dpp_f64(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), kCtrl, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), kCtrl, 0xF, 0xF, true);
    return __hiloint2double(hi, lo);
}

// Sum over the 8 lanes of a group, valid in the group's first lane: ((p0+p1)+(p2+p3))+((p4+p5)+(p6+p7)).
__device__ __forceinline__ double group_sum8(double v) {
    v = v + dpp_f64<0xB1>(v);   // quad_perm [1,0,3,2]
    v = v + dpp_f64<0x4E>(v);   // quad_perm [2,3,0,1]
    v = v + dpp_f64<0x104>(v);  // row_shl:4
    return v;
}

// Running sum in descending child order within a group: lane j gets sum of lanes j..7 of its group.
__device__ __forceinline__ double group_suffix8(double v) {
    const uint32_t j = lane() & 7U;
#pragma unroll
    for (int d = 1; d < 8; d <<= 1) {
        const double t = __shfl_down(v, d, kWave);
        if (j + d < 8) {
            v += t;
        }
    }
    return v;
}

// Element i of a wave-uniform array whose byte offsets fit 32 bits (slot tables; node arrays of
// fewer than 2^28 nodes): the address is a scalar base plus a 32-bit lane offset.
template <typename T>
__device__ __forceinline__ T& at(T* base, uint32_t i) {
    const uint32_t off = i * static_cast<uint32_t>(sizeof(T));
    return *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + off);
}

template <typename T>
__device__ __forceinline__ const T& at(const T* base, uint32_t i) {
    const uint32_t off = i * static_cast<uint32_t>(sizeof(T));
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off);
}

struct NodeData {
    uint2 m;
    uint4 r32;
    double4 r64;
};

// Loads the count/link word and the position record of `node` (both issued together).  The loads
// are issued in every lane (node 0 stands in for inactive lanes) so that no branch hides them from
// the compiler's memory-counter bookkeeping: a load in a skippable branch makes the next wait drain
// every outstanding load, prefetches included.
template <bool kMixed, bool kMu0>
__device__ __forceinline__ NodeData load_node(const Lane& L, uint32_t node, bool active) {
    const uint32_t x = active ? node : 0U;
    NodeData d;
    d.m = at(L.meta, x);
    if (kMixed) {
        d.r32 = at(L.rec32, x);
        d.r64 = make_double4(0.0, 0.0, 0.0, 0.0);
    } else {
        d.r32 = make_uint4(0U, 0U, 0U, 0U);
        d.r64 = L.rec64[x];
    }
    return d;
}

struct ExactEval {
    int st;
    double p;
};

// The reference's own test and probability of a node, for the few that the test on squares leaves open.
// Out of line: inlined into the traversal its divisions, square root and exponential cost the FP32-mixed
// kernel a wave per SIMD (96 VGPRs instead of 80).
__device__ __noinline__ ExactEval eval_reference(double theta, double mu, double scale64, double dx, double dy,
                                                 double dz, double side, uint32_t count, bool leaf) {
#pragma clang fp contract(off)
    ExactEval e;
    const double d = hypot3_exact(dx, dy, dz);
    e.st = d == 0.0 ? kDiscard : (leaf || side < theta * d ? kAccept : kExpand);
    const double exponent = ((d - mu) * (d - mu)) * scale64;
    e.p = e.st == kAccept ? (exp(exponent) * 1.0) * static_cast<double>(count) : 0.0;
    return e;
}

// Lanes that accept, and lanes that expand, their node.
struct Verdict {
    uint64_t accept, expand;
};

// Below this a squared distance is left to the formulas of the CPU path: squares of distances under about
// 1e-125 lose bits to underflow.
constexpr double kTiny = 1.0e-250;

// Acceptance test and probability of a loaded node (test_acceptance_criterion, BarnesHutBase.h:72-114;
// Kernel::calculate_attractiveness_to_connect, Kernel.h:61-75) for the lanes in `act`; p = 0 in lanes
// that do not accept.  The verdicts are lane masks combined in scalar registers, which the scalar unit
// does beside the vector arithmetic that bounds the kernel.
//
// Both precisions decide on squares, side^2 against theta^2 d^2, and leave what is too close (and
// distances of 0) to the reference's own comparison under one wave-uniform branch.  FP32: exact
// fixed-point differences, a leaf's squared side is -infinity, hence accepted.  FP64: a relative margin
// of 1e-13, a thousand times the rounding of both sides, so a decision outside it is the
// reference's; the Gaussian takes d^2 itself, which is rounded less than the square of the reference's
// scaled hypot.  That hypot (three divisions and a square root, about 75 of the 210 vector
// instructions of an FP64 step) and the library's exp made the FP64 search of 1M neurons 24.4 ms; with
// squares and exp_gauss it takes 16.0 ms (and 11.3 with the ring table above).
template <bool kMixed, bool kMu0>
__device__ __forceinline__ Verdict eval_node(const SearchArgs& a, const Lane& L, const NodeData& d, uint32_t node,
                                             uint64_t act, const double2* table, double* p_out) {
#pragma clang fp contract(off)
    // The source's own leaf lies at distance 0 and is discarded by the test, so the kernel's
    // self-exclusion (Kernel.h:61-75) never applies here.
    const uint64_t valid = act & __builtin_amdgcn_ballot_w64(d.m.x != 0);
    Verdict v;
    uint64_t unsure;
    double p;
    if (kMixed) {
        const float dx = static_cast<float>(static_cast<int32_t>(d.r32.x) - L.qx);
        const float dy = static_cast<float>(static_cast<int32_t>(d.r32.y) - L.qy);
        const float dz = static_cast<float>(static_cast<int32_t>(d.r32.z) - L.qz);
        const float d2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
        const float s2 = __uint_as_float(d.r32.w);
        const float g = __builtin_fmaf(a.theta2f, d2, -s2);
        // the squared distance of integer differences is 0 exactly at a coincidence
        const uint64_t coinc = __builtin_amdgcn_ballot_w64(d2 == 0.0f);
        const uint64_t near = __builtin_amdgcn_ballot_w64(fabsf(g) <= __builtin_fmaf(a.guard, s2, a.guard_abs));
        const uint64_t pos = __builtin_amdgcn_ballot_w64(g > 0.0f);
        float x;
        if (kMu0) {
            x = d2 * L.k2q;
        } else {
            const float dd = sqrtf(d2) * L.inv_q - a.muf;
            x = dd * dd * a.k2f;
        }
        const float w = __builtin_amdgcn_exp2f(x) * static_cast<float>(d.m.x);
        unsure = valid & (coinc | near);
        v.accept = valid & ~unsure & pos;
        v.expand = valid & ~unsure & ~pos;
        float wa = __builtin_amdgcn_inverse_ballot_w64(v.accept) ? w : 0.0f;
        __asm__ volatile("" : "+v"(wa));   // select in FP32, then one conversion
        p = static_cast<double>(wa);
    } else {
        const double dx = d.r64.x - L.px;
        const double dy = d.r64.y - L.py;
        const double dz = d.r64.z - L.pz;
        const double d2 = __builtin_fma(dx, dx, __builtin_fma(dy, dy, dz * dz));
        const double t = a.theta2 * d2;
        const double s2 = d.r64.w * d.r64.w;
        const uint64_t leaf = __builtin_amdgcn_ballot_w64((d.m.y >> kLinkBits) == 0);
        const uint64_t above = leaf | __builtin_amdgcn_ballot_w64(s2 < t * (1.0 - 1.0e-13));
        const uint64_t below = __builtin_amdgcn_ballot_w64(s2 > t * (1.0 + 1.0e-13));
        unsure = valid & (__builtin_amdgcn_ballot_w64(!(d2 > kTiny)) | ~(above | below));
        v.accept = valid & ~unsure & above;
        v.expand = valid & ~unsure & ~above;
        double x;
        if (kMu0) {
            x = d2 * a.scale64;
        } else {
            const double dd = sqrt(d2) - a.mu;
            x = (dd * dd) * a.scale64;
        }
        // exp is 0 below -745.2; the clamp keeps the exponent arithmetic in range
        const double w = exp_gauss(fmax(x, -800.0), table) * static_cast<double>(d.m.x);
        p = __builtin_amdgcn_inverse_ballot_w64(v.accept) ? w : 0.0;
    }
    if (unsure != 0) {
        int st = kDiscard;
        if (__builtin_amdgcn_inverse_ballot_w64(unsure)) {
            const bool leaf = (d.m.y >> kLinkBits) == 0;
            const double4 r = kMixed ? L.rec64[node] : d.r64;
            const ExactEval e = eval_reference(a.theta, a.mu, a.scale64, r.x - L.px, r.y - L.py, r.z - L.pz, r.w, d.m.x, leaf);
            st = e.st;
            p = e.p;
        }
        v.accept |= __builtin_amdgcn_ballot_w64(st == kAccept);
        v.expand |= __builtin_amdgcn_ballot_w64(st == kExpand);
    }
    *p_out = p;
    return v;
}

struct Bfs {
    double total;
    uint64_t accepted;   // not 0: the list has candidates
    uint32_t tests;
    bool overflow;
};


// One BFS step's input: up to 8 queue entries [kb, end) (one per group) and this lane's child of
// its group's node (loaded).
struct StepIn {
    uint32_t kb;     // first queue entry (= slot) of the step
    uint32_t end;    // one past the last entry the step covers
    uint32_t k;      // this group's entry
    uint32_t child;
    uint64_t groups; // lanes of the groups with an entry
    uint64_t act;    // lanes with a child
    NodeData nd;
};

// Lanes of the first `n` groups of 8.
__device__ __forceinline__ uint64_t group_lanes(uint32_t n) {
    return n >= 8U ? ~0ULL : ((1ULL << (8U * n)) - 1ULL);
}

struct SlotTable {   // the global part, indexed by slot
    uint32_t* my;
    uint32_t* fx;
    double* ms;
};

// Reads the entries [kb, min(kb + 8, tail)) of the queue and issues the loads of their children.
template <bool kMixed, bool kMu0>
__device__ __forceinline__ StepIn fetch_step(const Lane& L, const CoopShared<kMixed>& sh, uint32_t kb, uint32_t tail) {
    const uint32_t ln = lane();
    const uint32_t q = ln >> 3U, j = ln & 7U;
    StepIn x;
    // kb and end are wave-uniform; keeping them in scalar registers keeps the step's control flow scalar
    x.kb = __builtin_amdgcn_readfirstlane(kb);
    x.end = __builtin_amdgcn_readfirstlane(min(kb + 8U, tail));
    x.k = kb + q;
    x.groups = group_lanes(x.end - x.kb);
    const uint32_t packed = sh.my[x.k & kRingMask];   // groups without an entry read a stale one
    x.child = (packed & kLinkMask) + j;
    x.act = x.groups & __builtin_amdgcn_ballot_w64(j < (packed >> kLinkBits));
    x.nd = load_node<kMixed, kMu0>(L, x.child, __builtin_amdgcn_inverse_ballot_w64(x.act));
    return x;
}

struct BfsState {
    uint32_t nslots;   // queue tail = slots allocated; 0 after a step that went beyond the limit, and then
    uint32_t tail;     // the slots allocated
    uint32_t out;      // slots below left the ring for the global table
    uint32_t limit;    // slot_limit(out)
};

// Tests the children of one step's entries, sums the accepted probabilities per group, appends the
// expanded children to the ring and records the entries' masses.  In a step that goes beyond b.limit, those for
// which the ring has no room wait in the global table, and bfs() has to make room or give up.
template <bool kMixed, bool kMu0>
__device__ __forceinline__ void bfs_step(const CoopArgs& a, const Lane& L, CoopShared<kMixed>& sh, const SlotTable& t,
                                         const StepIn& x, BfsState& b, Bfs& r) {
    const uint32_t ln = lane();
    const uint32_t q = ln >> 3U;
    double p;
    const Verdict v = eval_node<kMixed, kMu0>(a.s, L, x.nd, x.child, x.act, sh.exp_table, &p);
    r.tests += static_cast<uint32_t>(__popcll(x.act));
    r.accepted |= v.accept;
    const double gsum = group_sum8(p);
    const uint64_t em = v.expand;
    const uint32_t ns = __builtin_amdgcn_readfirstlane(b.nslots);
    const uint32_t tail = ns + static_cast<uint32_t>(__popcll(em));
    // lane 8q (the one that writes group q's record) has rank_below(em) = the group's first slot
    const uint32_t slot = ns + rank_below(em);
    if (__builtin_amdgcn_inverse_ballot_w64(x.groups & 0x0101010101010101ULL)) {
        const uint32_t gem = static_cast<uint32_t>(em >> (8U * q)) & 0xFFU;
        const uint32_t gi = x.k & kRingMask;
        sh.ms[gi] = gsum;
        sh.fx[gi] = static_cast<uint16_t>(fx_pack(slot, static_cast<uint32_t>(__popc(gem))));
    }
    if (tail > b.limit) {
        if (__builtin_amdgcn_inverse_ballot_w64(em)) {
            if (slot < b.out + kRing) {
                sh.my[slot & kRingMask] = x.nd.m.y;
            } else {
                at(t.my, waiting_record(slot)) = x.nd.m.y;
            }
        }
        b.tail = tail;
        b.nslots = 0;
        return;
    }
    if (__builtin_amdgcn_inverse_ballot_w64(em)) {
        sh.my[slot & kRingMask] = x.nd.m.y;
    }
    b.nslots = tail;
}

// Breadth-first traversal below `root` (inner, with vacant dendrites) filling the slot table.  The queue
// is consumed 8 entries per step across level boundaries; the next step's child records are
// loaded before the current step is evaluated (two alternating step buffers, so no registers are
// copied).  *out gets the number of slots in the global table.
template <bool kMixed, bool kMu0>
__device__ Bfs bfs(const CoopArgs& a, const Lane& L, uint32_t root_meta_y, CoopShared<kMixed>& sh, uint64_t base,
                   uint32_t* out) {
    const uint32_t ln = lane();
    Bfs r{ 0.0, 0, 0, false };
    SlotTable t;
    t.my = a.t_my + base;
    t.fx = a.t_fexp + base;
    t.ms = a.t_mass + base;
    if (ln == 0) {
        sh.my[0] = root_meta_y;
    }
    __syncthreads();
    BfsState b{ 1U, 1U, 0U, slot_limit(0U) };
    StepIn xa = fetch_step<kMixed, kMu0>(L, sh, 0U, 1U);
    // Wait for the first step's data here, so that the loop header carries no pending load.
    if (kMixed) {
        __asm__ volatile("" ::"v"(xa.nd.m.x), "v"(xa.nd.m.y), "v"(xa.nd.r32.x), "v"(xa.nd.r32.y), "v"(xa.nd.r32.z),
                         "v"(xa.nd.r32.w));
    } else {
        __asm__ volatile("" ::"v"(xa.nd.m.x), "v"(xa.nd.m.y), "v"(xa.nd.r64.x), "v"(xa.nd.r64.y), "v"(xa.nd.r64.z),
                         "v"(xa.nd.r64.w));
    }
    // After a step whose successor starts at slot `next`, when that is no slot: the traversal ends, or the step
    // went beyond the limit.  Both share the exit test, and the room is made out of the step, whose registers it
    // would take: 18 more spilled in the FP32-mixed kernel.  1M neurons at theta 0.3: 8.67 ms FP32-mixed and
    // 11.40 FP64, against 8.80 and 11.43 with the room made in the step and no slots outside the ring.
    auto ends = [&](uint32_t next) -> bool {
        if (b.nslots != 0) {
            return true;
        }
        if (b.tail > kMostSlots) {
            r.overflow = true;
            return true;
        }
        if (slots_leave(b.out, next)) {
            const uint32_t sl = b.out + ln;
            at(t.my, sl) = sh.my[sl & kRingMask];
            at(t.fx, sl) = sh.fx[sl & kRingMask];
            at(t.ms, sl) = sh.ms[sl & kRingMask];
            if (sl + kRing < b.tail) {   // a slot that waits outside takes the place
                __threadfence_block();
                sh.my[sl & kRingMask] = at(t.my, sl + kRing);
            }
            b.out += kLeave;
            b.limit = slot_limit(b.out);
        }
        b.nslots = b.tail;
        return next >= b.nslots;
    };
    while (true) {
        const StepIn xb = fetch_step<kMixed, kMu0>(L, sh, xa.end, b.nslots);
        __builtin_amdgcn_sched_barrier(0);   // keep the prefetch ahead of this step's work
        bfs_step<kMixed, kMu0>(a, L, sh, t, xa, b, r);
        if (xb.kb >= b.nslots && ends(xb.kb)) {
            break;
        }
        xa = fetch_step<kMixed, kMu0>(L, sh, xb.end, b.nslots);
        __builtin_amdgcn_sched_barrier(0);
        bfs_step<kMixed, kMu0>(a, L, sh, t, xb, b, r);
        if (xa.kb >= b.nslots && ends(xa.kb)) {
            break;
        }
    }
    if (r.overflow) {
        return r;
    }
    __syncthreads();
    // Pull the masses of expanded children into their parents, last slots first, up to 64 at a time: all
    // children of the slots [lo, hi) lie at or beyond hi and have their final masses.
    *out = b.out;
    uint32_t hi = __builtin_amdgcn_readfirstlane(b.nslots);
    while (hi > 0) {
        const uint32_t first = hi > kWave ? hi - kWave : 0U;
        const uint32_t sl = first + ln;
        const bool in_lds = first >= b.out;   // then the children are too
        uint32_t fx = 0;
        if (sl < hi) {
            fx = in_lds || sl >= b.out ? sh.fx[sl & kRingMask] : at(t.fx, sl);
        }
        const uint32_t f = fx_slot(fx);
        const uint32_t ne = fx_count(fx);
        const uint32_t lo = pull_from(first, __builtin_amdgcn_ballot_w64(ne != 0 && f < hi));
        if (sl >= lo && ne != 0) {
            double m8[8];
            if (in_lds) {
#pragma unroll
                for (uint32_t c = 0; c < 8; c++) {
                    m8[c] = sh.ms[(f + c) & kRingMask];
                }
            } else {
#pragma unroll
                for (uint32_t c = 0; c < 8; c++) {
                    const uint32_t k = f + (c < ne ? c : 0U);
                    m8[c] = k >= b.out ? sh.ms[k & kRingMask] : at(t.ms, k);
                }
            }
            double sum = 0.0;
#pragma unroll
            for (uint32_t c = 0; c < 8; c++) {
                if (c < ne) {
                    sum += m8[c];
                }
            }
            if (in_lds || sl >= b.out) {
                sh.ms[sl & kRingMask] += sum;
            } else {
                at(t.ms, sl) += sum;
            }
        }
        __syncthreads();
        hi = lo;
    }
    r.total = b.out == 0 ? sh.ms[0] : t.ms[0];
    return r;
}

// Resolves the draws of the active groups top-down through the slot table (one draw per group).
// Returns the picked node in every lane of the group, kNone when the list had no positive mass.
template <bool kMixed, bool kMu0>
__device__ uint32_t navigate(const CoopArgs& a, const Lane& L, const CoopShared<kMixed>& sh, uint32_t out, double rr,
                             bool gact, uint64_t base, uint32_t* tests) {
    const SearchArgs& s = a.s;
    const uint32_t ln = lane();
    const uint32_t q = ln >> 3U, j = ln & 7U;
    const uint32_t g0 = 8U * q;
    const uint32_t* const tmy = a.t_my + base;
    const uint32_t* const tfx = a.t_fexp + base;
    const double* const tms = a.t_mass + base;
    uint32_t slot = 0;
    bool done = !gact;
    uint32_t res = kNone;
    for (uint32_t guard = 0; guard < kMaxLevels + 2; guard++) {
        if (__ballot(!done) == 0) {
            break;
        }
        // slot < kMostSlots always holds: it only advances to a checked child slot
        uint32_t fx, my;
        if (__builtin_amdgcn_ballot_w64(slot < out) == 0) {
            fx = sh.fx[slot & kRingMask];
            my = sh.my[slot & kRingMask];
        } else {
            fx = slot >= out ? sh.fx[slot & kRingMask] : at(tfx, slot);
            my = slot >= out ? sh.my[slot & kRingMask] : at(tmy, slot);
        }
        if (done) {
            fx = 0;
            my = 0;
        }
        const uint32_t fc = my & kLinkMask;
        const uint32_t nc = my >> kLinkBits;
        const uint32_t f = fx_slot(fx);
        const uint32_t nexp = fx_count(fx);
        const bool act = !done && j < nc;
        // the children and the masses of the expanded ones, loaded together
        const NodeData nd = load_node<kMixed, kMu0>(L, fc + j, act);
        const uint32_t mk = j < nexp ? f + j : slot;
        double mj;
        if (__builtin_amdgcn_ballot_w64(mk < out) == 0) {
            mj = sh.ms[mk & kRingMask];
        } else {
            mj = mk >= out ? sh.ms[mk & kRingMask] : at(tms, mk);
        }
        double p;
        const uint64_t actm = __builtin_amdgcn_ballot_w64(act);
        const Verdict v = eval_node<kMixed, kMu0>(s, L, nd, fc + j, actm, sh.exp_table, &p);
        *tests += static_cast<uint32_t>(__popcll(actm));
        const uint64_t em = v.expand;
        const uint32_t gem = static_cast<uint32_t>((em >> g0) & 0xFFULL);
        const uint32_t rk = static_cast<uint32_t>(__popc(gem & ((1U << j) - 1U)));
        const double mexp = __shfl(mj, static_cast<int>(g0 + (rk & 7U)), kWave);
        const double mass = __builtin_amdgcn_inverse_ballot_w64(em) ? mexp : p;   // p is 0 unless accepted
        const double cum = group_suffix8(mass);
        const double cum_next_raw = __shfl_down(cum, 1, kWave);
        const double cum_next = (j + 1 < 8) ? cum_next_raw : 0.0;
        const uint32_t gcm = static_cast<uint32_t>((__ballot(act && mass > 0.0 && cum >= rr) >> g0) & 0xFFULL);
        const uint32_t gpm = static_cast<uint32_t>((__ballot(act && mass > 0.0) >> g0) & 0xFFULL);
        int jstar = -1;
        if (gcm != 0) {
            jstar = 31 - __clz(static_cast<int>(gcm));
        } else if (gpm != 0) {
            jstar = __ffs(static_cast<int>(gpm)) - 1;
        }
        const uint32_t src_lane = g0 + static_cast<uint32_t>(jstar < 0 ? 0 : jstar);
        const bool accj = ((v.accept >> src_lane) & 1ULL) != 0;
        const double before = __shfl(cum_next, static_cast<int>(src_lane), kWave);
        if (!done) {
            if (jstar < 0) {
                done = true;
                res = kNone;
            } else if (accj) {
                done = true;
                res = fc + static_cast<uint32_t>(jstar);
            } else {
                rr = rr - before;
                const uint32_t next = f + static_cast<uint32_t>(__popc(gem & ((1U << jstar) - 1U)));
                if (nexp == 0 || next >= kMostSlots) {
                    done = true;
                    res = kNone;
                } else {
                    slot = next;
                }
            }
        }
    }
    return res;
}

struct ListResult {
    double total;
    bool any;        // the list has candidates
    uint32_t tests;
    uint32_t out;    // slots in the global table
    bool overflow;   // slot table overflow or a Gaussian sum of 0: the per-lane kernel redoes the source
};

// Candidate list of the subtree of `root`; a list whose Gaussian sum underflows to 0 needs the
// reference's fallbacks (Kernel::create_probability_interval, Kernel.h:109-126), which the per-lane
// kernel implements, so the source is handed over.  Sums near the smallest FP64 number stay: probabilities are
// multiples of it there, rounded once more by exp_gauss, and their sums are exact.  A few sources of one lane
// each take longer than this kernel for all: with sums below 1e-250 handed over, 20,000 neurons 100 um apart
// at sigma 5 um took 5.2 ms for 113 such sources.
template <bool kMixed, bool kMu0>
__device__ ListResult list_of(const CoopArgs& a, const Lane& L, uint32_t root, CoopShared<kMixed>& sh, uint64_t base) {
    ListResult lr{ 0.0, false, 0, 0, false };
    const uint2 mr = L.meta[root];
    if (mr.x == 0) {
        return lr;
    }
    const Bfs b = bfs<kMixed, kMu0>(a, L, mr.y, sh, base, &lr.out);
    lr.tests = b.tests;
    lr.total = b.total;
    lr.any = b.accepted != 0;
    lr.overflow = b.overflow || (lr.any && b.total == 0.0);
    return lr;
}


// Per-draw descent state, identical in the 8 lanes of the draw's group.
enum : int { kDrawActive = 0, kDrawDone = 1, kDrawFailed = 2, kDrawSlow = 3, kDrawIdle = 4 };

// Levels >= 2 of the groups' draws (BarnesHutBase::find_target_neuron, :223-255), one draw per group
// of 8 lanes, each lane testing one child of the draw's current node.  Below an accepted node the
// candidate list is normally the node's children, all accepted; the group then sums, draws and picks
// on its own.  A level that needs expansion, or whose Gaussian sum is 0 (the reference's fallbacks),
// ends in kDrawSlow with (node, level) where the general per-lane traversal takes over.
template <bool kMixed, bool kMu0>
__device__ __forceinline__ int descend_fast(const SearchArgs& s, const Lane& L, const double2* table, uint32_t jd, int state, uint32_t& node,
                                            uint32_t& level, uint32_t& tests, unsigned long long& exec) {
    const uint32_t ln = lane();
    const uint32_t j = ln & 7U;
    const uint32_t g0 = ln & ~7U;
    for (uint32_t guard = 0; guard < kMaxLevels + 2; guard++) {
        uint32_t my = 0;
        if (state == kDrawActive) {
            if (node >= s.m) {
                state = kDrawFailed;
            } else {
                const uint2 mn = L.meta[node];
                my = mn.y;
                if ((my >> kLinkBits) == 0) {
                    node = my & kLinkMask;  // leaf: the target neuron
                    state = kDrawDone;
                } else if (mn.x == 0) {
                    state = kDrawFailed;  // no vacant dendrites: empty list
                }
            }
        }
        if (__builtin_amdgcn_ballot_w64(state == kDrawActive) == 0) {
            break;
        }
        const bool act_g = state == kDrawActive;
        const uint32_t fc = my & kLinkMask;
        const uint32_t nc = act_g ? (my >> kLinkBits) : 0U;
        const bool act = act_g && j < nc;
        double p;
        const NodeData cd = load_node<kMixed, kMu0>(L, fc + j, act);
        const uint64_t actm = __builtin_amdgcn_ballot_w64(act);
        const Verdict v = eval_node<kMixed, kMu0>(s, L, cd, fc + j, actm, table, &p);
        exec += static_cast<uint32_t>(__popcll(actm));
        const uint32_t gexp = static_cast<uint32_t>(v.expand >> g0) & 0xFFU;
        const uint32_t gacc = static_cast<uint32_t>(v.accept >> g0) & 0xFFU;
        const double gsum = __shfl(group_sum8(p), static_cast<int>(g0), kWave);
        if (act_g) {
            if (gexp != 0 || (gacc != 0 && gsum == 0.0)) {
                state = kDrawSlow;
            } else {
                tests += nc;
                if (gacc == 0) {
                    state = kDrawFailed;
                }
            }
        }
        const bool pick = state == kDrawActive;
        const double r = pick ? draw_to_uniform(pick_draw(L.seed, L.local, L.step, jd, level), nextafter(gsum, gsum + 0.00001))
                              : 0.0;
        const double cum = group_suffix8(p);
        const uint32_t gcm = static_cast<uint32_t>((__builtin_amdgcn_ballot_w64(p > 0.0 && cum >= r) >> g0) & 0xFFULL);
        const uint32_t gpm = static_cast<uint32_t>((__builtin_amdgcn_ballot_w64(p > 0.0) >> g0) & 0xFFULL);
        if (pick) {
            int jstar = -1;
            if (gcm != 0) {
                jstar = 31 - __clz(static_cast<int>(gcm));
            } else if (gpm != 0) {
                jstar = __ffs(static_cast<int>(gpm)) - 1;
            }
            if (jstar < 0) {
                state = kDrawFailed;
            } else {
                node = fc + static_cast<uint32_t>(jstar);
                level++;
            }
        }
    }
    return state;
}

// One wave per source builds the candidate list of the root once (BarnesHutBase::find_target_neuron
// re-derives it for every axon, BarnesHutBase.h:223-255), resolves the source's level-1 draws against
// it 8 at a time, and continues each draw's descent in its group.  Results go to slot_target; descents
// that need the general traversal are queued for the per-lane kernel.  Registers: FP32-mixed is held to 6
// waves per SIMD (80 VGPRs; 11.0 against 11.3 ms per 1M-neuron update at 5), FP64 to 5 (96).
template <bool kMixed, bool kMu0>
__global__ void __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(kMixed ? 6 : 5, 8))) k_level1(CoopArgs a) {
    __shared__ CoopShared<kMixed> sh;
    const SearchArgs& s = a.s;
    const uint32_t ln = lane();
    const uint32_t q = ln >> 3U, j = ln & 7U;
    const uint64_t base = static_cast<uint64_t>(blockIdx.x) * a.cap;
    int seg = static_cast<int>(blockIdx.x % kXcds);
    unsigned long long acc_exec = 0;
    const uint64_t nw = *a.nwork;
    if (nw >= a.run_below) {
        return;   // the group walk takes this update
    }
    if (!kMixed) {
        if (ln < 32) {
            sh.exp_table[ln] = make_double2(kExpTable[ln][0], kExpTable[ln][1]);
        }
        __syncthreads();
    }
    const uint32_t step = *s.step;
    const uint32_t chunk = grab_size(nw, a.chunk);
    uint64_t w_next = 0, w_lim = 0;   // the wave's current chunk of its segment
    while (true) {
        if (w_next >= w_lim) {
            const uint64_t seg_end = nw * static_cast<uint64_t>(seg + 1) / kXcds;
            uint64_t w0 = 0;
            if (ln == 0) {
                w0 = nw * static_cast<uint64_t>(seg) / kXcds + atomicAdd(&a.cursor[seg * kCursorStride], static_cast<unsigned long long>(chunk));
            }
            w0 = __shfl(w0, 0, kWave);
            if (w0 >= seg_end) {
                seg = next_segment(a.cursor, nw, seg);
                if (seg < 0) {
                    break;
                }
                continue;
            }
            w_next = w0;
            w_lim = std::min<uint64_t>(w0 + chunk, seg_end);
        }
        const uint64_t w = w_next++;
        const uint32_t src = __builtin_amdgcn_readfirstlane(a.work[w]);
        const uint32_t na = __builtin_amdgcn_readfirstlane(s.vac_axon[src]);
        const uint32_t slot0 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(s.slot_off[src]));
        // source data is wave-uniform: keep it in scalar registers
        Lane L;
        L.src = src;
        L.sig = __builtin_amdgcn_readfirstlane(s.signal[src] == 0 ? 0 : 1);
        lane_bind(s, L);
        const uint32_t net = __builtin_amdgcn_readfirstlane(s.net_of[src]);
        L.root = net;
        L.local = src - __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(s.net_off[net]));
        L.step = step;
        L.seed = (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(s.net_seed[net] >> 32U)))) << 32U) |
                 static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(s.net_seed[net] & 0xFFFFFFFFULL)));
        L.k2q = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(s.net_k2q[net])));
        L.inv_q = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(s.net_invq[net])));
        L.px = uniform_f64(s.pos[src]);
        L.py = uniform_f64(s.pos[s.n + src]);
        L.pz = uniform_f64(s.pos[2 * s.n + src]);
        if (kMixed) {
            L.qx = __builtin_amdgcn_readfirstlane(static_cast<int32_t>(s.qpos[src]));
            L.qy = __builtin_amdgcn_readfirstlane(static_cast<int32_t>(s.qpos[s.n + src]));
            L.qz = __builtin_amdgcn_readfirstlane(static_cast<int32_t>(s.qpos[2 * s.n + src]));
        } else {
            L.qx = L.qy = L.qz = 0;
        }
        const ListResult l1 = list_of<kMixed, kMu0>(a, L, L.root, sh, base);
        acc_exec += l1.tests;
        if (l1.overflow) {
            if (ln == 0) {
                const unsigned long long k = atomicAdd(a.n_overflow, 1ULL);
                a.overflow[k] = src;
                s.found[src] = kOverflowMark;
            }
        } else if (!l1.any) {
            if (ln == 0) {
                s.slot_tests[slot0] = l1.tests;   // slot_target[slot0] stays kNone: one failed search
            }
        } else {
            const double next1 = nextafter(l1.total, l1.total + 0.00001);
            uint32_t nav_tests = 0;
            for (uint32_t j0 = 0; j0 < na; j0 += 8) {
                const bool gact = j0 + q < na;
                const double r = gact ? draw_to_uniform(pick_draw(L.seed, L.local, L.step, j0 + q, 1U), next1) : 0.0;
                uint32_t node = navigate<kMixed, kMu0>(a, L, sh, l1.out, r, gact, base, &nav_tests);
                uint32_t level = 2, tests = l1.tests;
                int state = !gact ? kDrawIdle : (node == kNone ? kDrawFailed : kDrawActive);
                state = descend_fast<kMixed, kMu0>(s, L, sh.exp_table, j0 + q, state, node, level, tests, acc_exec);
                const bool lead = gact && j == 0;
                const uint64_t sm = __builtin_amdgcn_ballot_w64(lead && state == kDrawSlow);
                unsigned long long at0 = 0;
                if (ln == 0 && sm != 0) {
                    at0 = atomicAdd(a.n_slow, static_cast<unsigned long long>(__popcll(sm)));
                }
                at0 = __shfl(at0, 0, kWave);
                if (lead) {
                    const uint32_t slot = slot0 + j0 + q;
                    s.slot_tests[slot] = tests;
                    if (state == kDrawSlow) {
                        a.slow[at0 + rank_below(sm)] = make_uint4(slot, src, node, level);
                    } else {
                        s.slot_target[slot] = state == kDrawDone ? node : kNone;
                    }
                }
            }
            acc_exec += nav_tests;
        }
        __syncthreads();
    }
    if (ln == 0 && acc_exec != 0) {
        // beside the wave's XCD's cursor; k_emit_requests adds the eight up
        atomicAdd(&a.cursor[(blockIdx.x % kXcds) * kCursorStride + 1], acc_exec);
    }
}

// Per source, in axon order: a search that fails ends the source's searches (find_target_neurons,
// BarnesHutBase.h:283-289).  Counts the searches, the successful ones and the reference's tests.
// Neurons in index order, grid-stride, so that neighbouring lanes read neighbouring slots (the work
// list is in Morton order, whose slots are scattered).  The totals are summed per block and added
// with one atomic per block and counter: same-address atomics pass one after another.  At 1M neurons the
// kernel took 58 us with 2,048 blocks, 21 us now.
__global__ void __launch_bounds__(kCountThreads) k_finalize(SearchArgs s) {
    unsigned long long ref = 0, searched_n = 0;
    const bool over = s.counters[kCtrOverCap] != 0;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t src = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; src < s.n; src += stride) {
        // the active sources that k_search_reset flags: enabled, with vacant axons, and no over-capacity update
        if (over || s.enabled[src] == 0 || s.vac_axon[src] == 0 || s.found[src] == kOverflowMark) {
            continue;
        }
        const uint32_t na = s.vac_axon[src];
        const uint64_t slot0 = s.slot_off[src];
        uint32_t found = 0, searched = 0;
        uint32_t jj = 0;
        for (; jj < na; jj++) {
            searched++;
            ref += s.slot_tests[slot0 + jj];
            if (s.slot_target[slot0 + jj] == kNone) {
                break;
            }
            found++;
        }
        // draws after the first failure were resolved speculatively: the reference never makes them
        for (jj = jj + 1; jj < na; jj++) {
            s.slot_target[slot0 + jj] = kNone;
            s.slot_tests[slot0 + jj] = 0;
        }
        s.found[src] = found;
        s.searched[src] = searched;
        searched_n += searched;
    }
    unsigned long long sum[2] = { ref, searched_n };
    block_totals(sum);
    if (threadIdx.x == 0 && sum[1] != 0) {
        atomicAdd(&s.counters[kCtrTestsRef], sum[0]);
        atomicAdd(&s.counters[kCtrSearches], sum[1]);
    }
}

}  // namespace

// Cooperative search over the active sources (c->coop_work, count in sa.nwork): the search kernel,
// the per-lane general descents it hands over, then the per-source finalisation.  Sources that
// overflow the slot table (or whose root list sums to 0) go to c->coop_overflow, counted in
// counters[kCtrOverflow], for the per-lane kernel.  All counts stay on the device.
int launch_search_coop(rl_bh_ctx* c, const SearchArgs& sa) {
    const bool timed = !c->capturing;
    if (timed) RL_HIP(c, hipEventRecord(c->ev2, c->stream));
    if (uses_walk(c)) {   // the tuned setting is the walk's
        RL_TRY(launch_level1(c, sa, c->coop_work, sa.nwork, UINT64_MAX, c->cus * kMixedWavesPerCu, kMixedChunk));
    } else {
        RL_TRY(launch_level1(c, sa, c->coop_work, sa.nwork, UINT64_MAX, c->coop_blocks, c->search_chunk));
    }
    if (timed) RL_HIP(c, hipEventRecord(c->ev3, c->stream));
    RL_TRY(launch_descend_lane(c, sa, c->slow_items, c->counters + kCtrSlow));
    return launch_finalize(c, sa);
}

// The wave-per-source kernel over work[0, *nwork) on `blocks` persistent waves taking `chunk` sources
// per cursor increment, skipped on the device when *nwork >= run_below.
int launch_level1(rl_bh_ctx* c, const SearchArgs& sa, const uint32_t* work, const uint64_t* nwork,
                  uint64_t run_below, uint32_t blocks, uint32_t chunk) {
    hipStream_t s = c->stream;
    CoopArgs a{};
    a.s = sa;
    a.work = work;
    a.nwork = nwork;
    a.run_below = run_below;
    a.cursor = c->coop_cursor;
    a.chunk = std::max<uint32_t>(chunk, 1U);
    a.t_my = c->coop_node;
    a.t_fexp = c->coop_fexp;
    a.t_mass = c->coop_mass;
    a.cap = c->coop_cap;
    a.overflow = c->coop_overflow;
    a.n_overflow = c->counters + kCtrOverflow;
    a.slow = c->slow_items;
    a.n_slow = c->counters + kCtrSlow;
    const bool mixed = c->cfg.precision == RL_PREC_FP32_MIXED;
    const bool mu0 = c->cfg.mu == 0.0;
    if (mixed && mu0) {
        k_level1<true, true><<<blocks, kWave, 0, s>>>(a);
    } else if (mixed) {
        k_level1<true, false><<<blocks, kWave, 0, s>>>(a);
    } else if (mu0) {
        k_level1<false, true><<<blocks, kWave, 0, s>>>(a);
    } else {
        k_level1<false, false><<<blocks, kWave, 0, s>>>(a);
    }
    RL_HIP(c, hipGetLastError());
    return RL_OK;
}

int launch_finalize(rl_bh_ctx* c, const SearchArgs& sa) {
    k_finalize<<<count_blocks(c->n), kCountThreads, 0, c->stream>>>(sa);
    RL_HIP(c, hipGetLastError());
    return RL_OK;
}

}  // namespace rl
