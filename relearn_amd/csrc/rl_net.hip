// Network graph of the synaptic input on the device: creation and deletion of synapses.
//
// The synaptic input of a neuron (SynapticEquallyWeightedActivityInputCPU::update_local_input,
// source/neurons/input/SynapticEquallyWeightedActivityInputCPU.cpp:21-50) sums the weights of its
// in-edges (NetworkGraph::get_local_in_edges) whose source fired in the last step.  The device keeps
// those in-edges as a CSR by target with one entry per (source, target) pair whose weight is the sum
// of the pair's synapses, as NetworkGraph::add_synapse merges them; a pair whose weight returns to 0
// is dropped at the next append.
//
// Creation: every commit appends the synapses it created (Neurons::update_connectivity adds them to
// the graph, source/neurons/Neurons.cpp:458-476), weight +1 for an excitatory source and -1 for an
// inhibitory one (ForwardConnector::process_requests, source/algorithm/Connector.cpp:33-121).  The
// new synapses are counted per target, prefix-summed and staged; one lane per target then merges
// them into the target's pairs, writing the merged list into the second buffer, and the compacted
// graph is copied back.  Counts come from device memory and nothing allocates, so the append can be
// captured with the commit; an append that would not fit appends nothing and raises a device flag.
//
// Deletion (SynapseDeletionFinderCPU::delete_synapses, source/neurons/helper/SynapseDeletionFinderCPU.cpp,
// with RandomSynapseDeletionFinder::find_synapses_on_neuron, SynapseDeletionFinder.cpp:53-69): after
// the element commit of one type, a neuron that lost k bound elements of that type deletes k of its
// synapse units of that kind, drawn uniformly without replacement: axons its outgoing synapses,
// dendrites its incoming synapses of the dendrite's sign; a pair of weight w counts |w| units
// (SynapseDeletionFinderBase::register_synapses, SynapseDeletionFinderBase.cpp:33-151).  Every deleted
// unit lowers the pair's weight by one and disconnects one element of the partner
// (commit_deletions, ElementBaseBase::disconnect_elements, ElementBaseBase.h:311-319).  The draw is
// counter-based: the k units with the smallest deletion_key(...) over (partner, copy), so the subset
// does not depend on the order the pairs are stored in.
#include <algorithm>
#include <cstring>
#include <vector>

#include "rl_device.h"
#include "rl_internal.h"

namespace rl {
namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(uint64_t n, int block = kBlock) {
    const uint64_t g = (n + block - 1) / block;
    return static_cast<unsigned>(g == 0 ? 1 : g);
}

__device__ __forceinline__ int32_t unit_sign(int32_t w) {
    return w < 0 ? -1 : 1;
}

// The lists of 64 neighbouring targets, whose entries [lo, lo + m) a wave goes through in order, so that
// its loads are consecutive; a lane finds its entry's list by bisection over the 64 starts.
struct WaveLists {
    uint64_t lo;
    uint32_t start;   // of this lane's list, relative to lo
    uint32_t m;

    // Entry j's list: the last one that starts at or before it.  For all lanes of the wave together.
    __device__ __forceinline__ uint32_t list_of(uint32_t j) const {
        uint32_t k = 0;
#pragma unroll
        for (uint32_t step = 32; step != 0; step >>= 1) {
            const uint32_t at = __shfl(start, static_cast<int>(k + step));
            k += at <= j ? step : 0U;
        }
        return k;
    }
};

__device__ __forceinline__ WaveLists wave_lists(uint64_t t0, uint64_t t1, const uint64_t* __restrict__ off) {
    const uint64_t t = t0 + (threadIdx.x & 63U);
    const uint64_t mine = off[t < t1 ? t : t1];
    WaveLists l;
    l.lo = __shfl(static_cast<unsigned long long>(mine), 0);
    l.start = static_cast<uint32_t>(mine - l.lo);
    l.m = static_cast<uint32_t>(off[t0 + 64 < t1 ? t0 + 64 : t1] - l.lo);
    return l;
}

// ---------------------------------------------------------------- append

__global__ void k_net_count(const uint64_t* __restrict__ n_req, const uint8_t* __restrict__ ok,
                            const uint32_t* __restrict__ tgt, uint32_t* __restrict__ ncnt) {
    const uint64_t m = *n_req;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < m; i += stride) {
        if (ok[i] != 0) {
            atomicAdd(&ncnt[tgt[i]], 1U);
        }
    }
}

// New synapses staged per target at npre[t]: their sources (the weight follows from the source's
// signal type).  ncnt returns to zero.  The merge writes target t's list at off[t] + npre[t] of the second
// buffer, room for its old entries and its new synapses: an append that does not fit the capacity in
// that layout is left out, and the counts stay.
__global__ void k_net_stage(uint64_t n, const uint64_t* __restrict__ off, uint64_t cap,
                            const uint64_t* __restrict__ n_req, const uint8_t* __restrict__ ok,
                            const uint32_t* __restrict__ tgt, const uint32_t* __restrict__ rsrc,
                            const uint64_t* __restrict__ npre, uint32_t* __restrict__ ncnt, uint32_t* __restrict__ stage,
                            unsigned long long* __restrict__ counters) {
    const uint64_t add = npre[n];
    const bool over = off[n] + add > cap;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        counters[kCtrNetOver] = over ? 1ULL : 0ULL;
        counters[kCtrNetNew] = over ? 0ULL : add;
        if (over) {
            counters[kCtrSticky] += 1ULL;
        }
    }
    if (over) {
        return;
    }
    const uint64_t m = *n_req;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < m; i += stride) {
        if (ok[i] == 0) {
            continue;
        }
        const uint32_t t = tgt[i];
        stage[npre[t] + atomicSub(&ncnt[t], 1U) - 1U] = rsrc[i];
    }
}

// Target t's list, its non-zero pairs and then its new synapses (added to the pair of their source or
// appended as a new pair), at off[t] + npre[t] of the second buffer; ncnt[t] gets its length.  A wave copies
// the lists of 64 targets as they are; then the lanes whose target lost a pair or has new synapses, a
// few in a hundred, close the gaps and add them.  One lane per list from end to end, whose loads were 32
// bytes apart and followed one another, took 283 us for 16M pairs of 2M targets;
// 102 us now (2.5 of about 5 TB/s).
__global__ void k_net_merge(uint64_t n, const uint64_t* __restrict__ off, const uint64_t* __restrict__ npre,
                            const uint32_t* __restrict__ src, const int32_t* __restrict__ w,
                            const uint32_t* __restrict__ stage, const uint8_t* __restrict__ signal,
                            uint32_t* src2, int32_t* w2, uint32_t* __restrict__ ncnt,
                            const unsigned long long* __restrict__ counters) {
    if (counters[kCtrNetOver] != 0) {
        return;
    }
    const uint32_t lane = threadIdx.x & 63U;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t t0 = blockIdx.x * static_cast<uint64_t>(blockDim.x) + (threadIdx.x & ~63U); t0 < n; t0 += stride) {
        const WaveLists l = wave_lists(t0, n, off);
        const uint64_t t = t0 + lane < n ? t0 + lane : n;
        const uint64_t before = npre[t];   // new synapses of the targets before
        const uint64_t first = __shfl(static_cast<unsigned long long>(before), 0);
        const uint32_t shift = static_cast<uint32_t>(before - first);
        uint64_t gaps = 0;                 // lists with a pair of weight 0
        for (uint32_t j0 = 0; j0 < l.m; j0 += 64) {
            const uint32_t j = j0 + lane;
            const bool in = j < l.m;
            const uint32_t s = in ? src[l.lo + j] : 0U;
            const int32_t we = in ? w[l.lo + j] : 1;
            const uint32_t k = l.list_of(j);
            const uint64_t to = l.lo + j + first + __shfl(shift, static_cast<int>(k));
            if (in) {
                src2[to] = s;
                w2[to] = we;
            }
            for (uint64_t zero = __ballot(we == 0); zero != 0; zero &= zero - 1) {
                gaps |= 1ULL << __shfl(k, __ffsll(static_cast<unsigned long long>(zero)) - 1);
            }
        }
        __threadfence_block();   // the wave's copies before its lanes' reads
        if (t >= n) {
            continue;
        }
        const uint64_t base = l.lo + l.start + before;
        const uint64_t end = npre[t + 1];
        uint32_t k = static_cast<uint32_t>(off[t + 1] - off[t]);
        if ((gaps >> lane & 1ULL) != 0) {
            const uint32_t had = k;
            k = 0;
            for (uint32_t j = 0; j < had; j++) {
                const int32_t we = w2[base + j];
                if (we != 0) {
                    src2[base + k] = src2[base + j];
                    w2[base + k] = we;
                    k++;
                }
            }
        }
        for (uint64_t q = before; q < end; q++) {
            const uint32_t s = stage[q];
            const int32_t dw = signal[s] != 0 ? -1 : 1;
            uint32_t j = 0;
            while (j < k && src2[base + j] != s) {
                j++;
            }
            if (j < k) {
                w2[base + j] += dw;
            } else {
                src2[base + k] = s;
                w2[base + k] = dw;
                k++;
            }
        }
        ncnt[t] = k;
    }
}

// Compacted lists back into the primary arrays, at the prefix sum noff of the merged counts, which become
// the offsets (a list's old offset is read by its own lane only).  Copied by the wave as in k_net_merge:
// 226 -> 64 us for 16M pairs of 2M targets (4 TB/s).
__global__ void k_net_copyback(uint64_t n, uint64_t* __restrict__ off, const uint64_t* __restrict__ npre,
                               const uint64_t* __restrict__ noff, const uint32_t* __restrict__ src2,
                               const int32_t* __restrict__ w2, uint32_t* __restrict__ src, int32_t* __restrict__ w,
                               const unsigned long long* __restrict__ counters) {
    if (counters[kCtrNetOver] != 0) {
        return;
    }
    const uint32_t lane = threadIdx.x & 63U;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t t0 = blockIdx.x * static_cast<uint64_t>(blockDim.x) + (threadIdx.x & ~63U); t0 < n; t0 += stride) {
        const WaveLists l = wave_lists(t0, n, noff);
        const uint64_t t = t0 + lane;
        // how far this lane's list moves; it moves at least as far as the list before it
        uint64_t moves = 0;
        if (t < n) {
            moves = off[t] + npre[t] - (l.lo + l.start);
            off[t] = l.lo + l.start;
        }
        if (t0 + 64 >= n && lane == 0) {
            off[n] = l.lo + l.m;
        }
        const uint64_t first = __shfl(static_cast<unsigned long long>(moves), 0);
        const uint32_t more = static_cast<uint32_t>(moves - first);
        for (uint32_t j0 = 0; j0 < l.m; j0 += 64) {
            const uint32_t j = j0 + lane;
            const uint64_t from = l.lo + j + first + __shfl(more, static_cast<int>(l.list_of(j)));
            if (j < l.m) {
                src[l.lo + j] = src2[from];
                w[l.lo + j] = w2[from];
            }
        }
    }
}

// ---------------------------------------------------------------- pairs by source

// The pairs grouped by source come from a counting sort in two levels, without global atomics.  Sources
// fall into bins of 2^shift.  k_out_bins<false> counts the pairs of each block of targets per bin; after
// a prefix sum over (bin, block), k_out_bins<true> writes them there as 16-byte records, so that a
// block's records of one bin are consecutive.  k_out_sort then sorts a bin's records by source in LDS
// and writes them in order.  One count and one scatter over all sources, each with one global atomic per
// pair, were bound by the atomics (26 G/s) and by 4-byte writes to lines that had left L2 by the next
// write: 608 + 1,256 us for 16M pairs of 2M sources, against 83 + 258 + 144 us and 10 us of prefix sum
// (1.2 GB moved); axon deletions needed 666 us more for lists of their own.  9 periods of 300,001
// neurons in all: 235 -> 71 us.
//
// More bins cost k_out_bins partly written lines (a block's open line per bin, 32 x bins x 128 B in an
// XCD's L2), fewer cost k_out_sort: k_out_bins<true> + k_out_sort took 199 + 551 us with 512 bins,
// 239 + 333 with 2,048 and 258 + 222 with 4,096 when k_out_sort scattered to memory; with the records
// sorted in LDS 258 + 144 us with 4,096 bins and 286 + 188 with 8,192.  One block per CU: 512 blocks do
// not gain.
constexpr uint64_t kOutBlocks = 256;
constexpr uint32_t kOutThreads = 1024;
constexpr uint32_t kOutBins = 4096;        // below; more once a bin's counters would not fit into 64 KB of LDS
constexpr uint32_t kOutMinShift = 8;
constexpr uint32_t kOutMaxShift = 14;
constexpr uint32_t kOutHeld = 8;           // records per thread that k_out_sort holds
constexpr uint32_t kOutStaged = kOutHeld * kOutThreads;
constexpr uint32_t kOutStageShift = 12;    // staging area and counters share the LDS up to this bin size
// Small graphs are sorted by one block in one launch: the four launches of the larger sort take about
// 5 us each, and the one block 21 us for 8,000 pairs (1,000 neurons) and more in proportion, so that
// by the capacity's bound of 32,768 it is at worst some 50 us behind.
constexpr uint64_t kOutOneSources = 2048;
constexpr uint64_t kOutOnePairs = 32768;

uint32_t out_shift(uint64_t n) {
    uint32_t shift = kOutMinShift;
    while (shift < kOutMaxShift && (n >> shift) >= kOutBins) {
        shift++;
    }
    return shift;
}

uint64_t out_bins(uint64_t n) {
    return (n + (1ULL << out_shift(n)) - 1) >> out_shift(n);
}

uint64_t out_blocks(uint64_t n) {
    return std::min<uint64_t>(kOutBlocks, (n + kOutThreads - 1) / kOutThreads);
}

// f(entry, target, source, weight) for the non-zero pairs of targets [t0, min(t0 + 64, t1)).
template <typename F>
__device__ __forceinline__ void wave_pairs(uint64_t t0, uint64_t t1, const uint64_t* __restrict__ off,
                                           const uint32_t* __restrict__ src, const int32_t* __restrict__ w, F f) {
    const WaveLists l = wave_lists(t0, t1, off);
    for (uint32_t j0 = 0; j0 < l.m; j0 += 64) {
        const uint32_t j = j0 + (threadIdx.x & 63U);
        const bool in = j < l.m;
        const uint32_t s = in ? src[l.lo + j] : 0U;
        const int32_t we = in ? w[l.lo + j] : 0;
        const uint32_t k = l.list_of(j);
        if (we != 0) {
            f(l.lo + j, t0 + k, s, we);
        }
    }
}

// Block b takes targets [b per, (b + 1) per).  kWrite: records to the bin's place, else counts per bin.
template <bool kWrite>
__global__ void __launch_bounds__(kOutThreads) k_out_bins(uint64_t n, uint64_t per, uint32_t shift, uint32_t bins,
                                                          const uint64_t* __restrict__ off,
                                                          const uint32_t* __restrict__ src,
                                                          const int32_t* __restrict__ w, uint32_t* __restrict__ cnt,
                                                          const uint64_t* __restrict__ place, uint4* __restrict__ rec) {
    extern __shared__ uint32_t bin[];   // counts, or the next place
    // places of more than 32 bits are held relative to the bin's first
    const bool wide = kWrite && place[static_cast<uint64_t>(bins) * gridDim.x] >> 32U != 0;
    for (uint32_t b = threadIdx.x; b < bins; b += kOutThreads) {
        const uint64_t at = static_cast<uint64_t>(b) * gridDim.x;
        bin[b] = kWrite ? static_cast<uint32_t>(place[at + blockIdx.x] - (wide ? place[at] : 0)) : 0U;
    }
    __syncthreads();
    const uint64_t first = blockIdx.x * per;
    const uint64_t last = first + per < n ? first + per : n;
    for (uint64_t t0 = first + (threadIdx.x & ~63U); t0 < last; t0 += kOutThreads) {
        wave_pairs(t0, last, off, src, w, [&](uint64_t e, uint64_t t, uint32_t s, int32_t we) {
            const uint32_t b = s >> shift;
            const uint32_t at = atomicAdd(&bin[b], 1U);
            if (kWrite) {
                rec[at + (wide ? place[static_cast<uint64_t>(b) * gridDim.x] : 0)] =
                    make_uint4(s, static_cast<uint32_t>(t), static_cast<uint32_t>(we), static_cast<uint32_t>(e));
            }
        });
    }
    if (!kWrite) {
        __syncthreads();
        for (uint32_t b = threadIdx.x; b < bins; b += kOutThreads) {
            cnt[static_cast<uint64_t>(b) * gridDim.x + blockIdx.x] = bin[b];
        }
    }
}

// The counts of 2^shift sources become their exclusive prefix sums, the list offsets of sources
// [s0, min(s0 + 2^shift, n)) at `base`.
__device__ __forceinline__ void out_offsets(uint32_t* cnt, uint32_t shift, uint64_t s0, uint64_t n, uint64_t base,
                                            uint64_t* __restrict__ out_off) {
    constexpr uint32_t kMost = (1U << kOutMaxShift) / kOutThreads;
    const uint32_t size = 1U << shift;
    const uint32_t each = size > kOutThreads ? size / kOutThreads : 1U;
    const uint32_t first = threadIdx.x * each;
    const uint32_t lane = threadIdx.x & 63U;
    const uint32_t wave = threadIdx.x >> 6U;
    uint32_t v[kMost];
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < kMost; k++) {
        v[k] = k < each && first + k < size ? cnt[first + k] : 0U;
        sum += v[k];
    }
    uint32_t inc = sum;
#pragma unroll
    for (uint32_t o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(inc, o);
        inc += lane >= o ? y : 0U;
    }
    __syncthreads();   // every count is in registers: the array's start holds the waves' sums now
    if (lane == 63) {
        cnt[wave] = inc;
    }
    __syncthreads();
    uint32_t run = inc - sum;
#pragma unroll
    for (uint32_t k = 0; k < kOutThreads / 64; k++) {
        run += k < wave ? cnt[k] : 0U;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < kMost; k++) {
        if (k < each && first + k < size) {
            cnt[first + k] = run;
            if (s0 + first + k < n) {
                out_off[s0 + first + k] = base + run;
            }
            run += v[k];
        }
    }
    __syncthreads();
}

// Block b sorts the records of bin b by source (order inside a source arbitrary).  Up to kOutStaged
// records are read once, held in registers and written in order from LDS; a bin with more is read twice
// and scattered.
__global__ void __launch_bounds__(kOutThreads) k_out_sort(uint64_t n, uint32_t shift, uint32_t blocks,
                                                          const uint64_t* __restrict__ place,
                                                          const uint4* __restrict__ rec, uint64_t* __restrict__ out_off,
                                                          uint2* __restrict__ out_pair, uint32_t* __restrict__ out_entry) {
    extern __shared__ uint32_t cnt[];   // 2^shift counters, then the staging area
    const uint32_t size = 1U << shift;
    const uint64_t base = place[static_cast<uint64_t>(blockIdx.x) * blocks];
    const uint64_t end = place[(static_cast<uint64_t>(blockIdx.x) + 1) * blocks];
    const uint64_t s0 = static_cast<uint64_t>(blockIdx.x) << shift;
    const uint32_t m = static_cast<uint32_t>(end - base);
    for (uint32_t k = threadIdx.x; k < size; k += kOutThreads) {
        cnt[k] = 0;
    }
    if (blockIdx.x + 1 == gridDim.x && threadIdx.x == 0) {
        out_off[n] = end;
    }
    __syncthreads();
    if (m <= kOutStaged && shift <= kOutStageShift) {
        uint2* pair = reinterpret_cast<uint2*>(cnt + size);
        uint32_t* entry = reinterpret_cast<uint32_t*>(pair + kOutStaged);
        uint4 r[kOutHeld];
        uint32_t rank[kOutHeld];
#pragma unroll
        for (uint32_t k = 0; k < kOutHeld; k++) {
            const uint32_t j = k * kOutThreads + threadIdx.x;
            if (j < m) {
                r[k] = rec[base + j];
            }
        }
#pragma unroll
        for (uint32_t k = 0; k < kOutHeld; k++) {
            if (k * kOutThreads + threadIdx.x < m) {
                rank[k] = atomicAdd(&cnt[r[k].x & (size - 1U)], 1U);
            }
        }
        __syncthreads();
        out_offsets(cnt, shift, s0, n, base, out_off);
#pragma unroll
        for (uint32_t k = 0; k < kOutHeld; k++) {
            if (k * kOutThreads + threadIdx.x < m) {
                const uint32_t at = cnt[r[k].x & (size - 1U)] + rank[k];
                pair[at] = make_uint2(r[k].y, r[k].z);
                entry[at] = r[k].w;
            }
        }
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < m; j += kOutThreads) {
            out_pair[base + j] = pair[j];
            out_entry[base + j] = entry[j];
        }
        return;
    }
    for (uint32_t j = threadIdx.x; j < m; j += kOutThreads) {
        atomicAdd(&cnt[rec[base + j].x & (size - 1U)], 1U);
    }
    __syncthreads();
    out_offsets(cnt, shift, s0, n, base, out_off);
    for (uint32_t j = threadIdx.x; j < m; j += kOutThreads) {
        const uint4 r = rec[base + j];
        const uint64_t at = base + atomicAdd(&cnt[r.x & (size - 1U)], 1U);
        out_pair[at] = make_uint2(r.y, r.z);
        out_entry[at] = r.w;
    }
}

// The same in one block for at most kOutOneSources sources, from the graph itself.
__global__ void __launch_bounds__(kOutThreads) k_out_one(uint64_t n, const uint64_t* __restrict__ off,
                                                         const uint32_t* __restrict__ src,
                                                         const int32_t* __restrict__ w, uint64_t* __restrict__ out_off,
                                                         uint2* __restrict__ out_pair, uint32_t* __restrict__ out_entry) {
    __shared__ uint32_t cnt[kOutOneSources];   // 2^11
    __shared__ uint32_t total;
    for (uint32_t k = threadIdx.x; k < kOutOneSources; k += kOutThreads) {
        cnt[k] = 0;
    }
    if (threadIdx.x == 0) {
        total = 0;
    }
    __syncthreads();
    uint32_t mine = 0;
    for (uint64_t t0 = threadIdx.x & ~63U; t0 < n; t0 += kOutThreads) {
        wave_pairs(t0, n, off, src, w, [&](uint64_t, uint64_t, uint32_t s, int32_t) {
            atomicAdd(&cnt[s], 1U);
            mine++;
        });
    }
    atomicAdd(&total, mine);
    __syncthreads();
    out_offsets(cnt, 11U, 0, n, 0, out_off);
    for (uint64_t t0 = threadIdx.x & ~63U; t0 < n; t0 += kOutThreads) {
        wave_pairs(t0, n, off, src, w, [&](uint64_t e, uint64_t t, uint32_t s, int32_t we) {
            const uint32_t at = atomicAdd(&cnt[s], 1U);
            out_pair[at] = make_uint2(static_cast<uint32_t>(t), static_cast<uint32_t>(we));
            out_entry[at] = static_cast<uint32_t>(e);
        });
    }
    if (threadIdx.x == 0) {
        out_off[n] = total;
    }
}

// ---------------------------------------------------------------- synaptic input by push

// acc[t] += the weights of the pairs whose source has fired set (acc starts at zero).
__global__ void k_syn_push_all(uint64_t n, const uint8_t* __restrict__ fired, const uint64_t* __restrict__ out_off,
                               const uint2* __restrict__ out_pair, int32_t* __restrict__ acc) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t s = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; s < n; s += stride) {
        if (fired[s] != 0) {
            for (uint64_t e = out_off[s]; e < out_off[s + 1]; e++) {
                const uint2 tw = out_pair[e];
                atomicAdd(&acc[tw.x], static_cast<int32_t>(tw.y));
            }
        }
    }
}

// ---------------------------------------------------------------- deletion

struct DelArgs {
    uint64_t n;
    const uint32_t* net_of;
    const uint64_t* net_off;
    const uint64_t* net_seed;
    const uint32_t* step;        // device: plasticity update index
    const uint32_t* deleted;     // units to delete per neuron (this type)
    const uint8_t* signal;
    const uint64_t* off;         // graph
    const uint32_t* src;
    int32_t* w;
    uint32_t* conn[3];
    uint32_t* vac[3];
    unsigned long long* counters;
};

// A unit (partner, copy) of a neuron with its key; units compare by (key, partner, copy).
struct Unit {
    uint64_t key;
    uint32_t partner;
    uint32_t copy;
};

__device__ __forceinline__ bool unit_less(const Unit& a, const Unit& b) {
    if (a.key != b.key) return a.key < b.key;
    if (a.partner != b.partner) return a.partner < b.partner;
    return a.copy < b.copy;
}

// f(entry, pair) for the m entries of a neuron, pair = (partner, weight) = load(entry); eight loads in flight, where
// one at a time cost a round trip each.
constexpr uint32_t kEntriesAhead = 8;
template <typename Load, typename F>
__device__ __forceinline__ void each_entry(uint32_t m, Load load, F f) {
    for (uint32_t j0 = 0; j0 < m; j0 += kEntriesAhead) {
        uint2 pw[kEntriesAhead];
#pragma unroll
        for (uint32_t k = 0; k < kEntriesAhead; k++) {
            pw[k] = load(j0 + k < m ? j0 + k : j0);
        }
#pragma unroll
        for (uint32_t k = 0; k < kEntriesAhead; k++) {
            if (j0 + k < m) {
                f(j0 + k, pw[k]);
            }
        }
    }
}

// Deletes up to `want` units of neuron `id` among its m entries: those with the smallest keys.  load(j) gives entry
// j's (partner, weight), units(w) the units that a pair of this weight counts, and drop(j, partner, weight, count)
// takes `count` of entry j.  Returns the number deleted.
//
// One lane per neuron, and few neurons delete, so a neuron's chain of loads and Philox draws is the time: the entries
// are loaded eight at a time, a partner of the neuron's own network costs no look-up, and the usual cases
// (one unit, or all of them) need one pass over the keys or none, where counting, k passes and a last one to
// find the k-th key's entries were made before.  The three kernels of a period: 32 -> 20 us for 1,000 neurons,
// 77 -> 47 us for 300,001, 262 -> 227 us for 2M.
template <typename Load, typename Units, typename Drop>
__device__ __forceinline__ uint32_t delete_units(const DelArgs& a, uint32_t id, uint32_t type, uint32_t m, uint32_t want,
                                                 Load load, Units units, Drop drop) {
    uint32_t all = 0;
    each_entry(m, load, [&](uint32_t, const uint2& pw) { all += units(static_cast<int32_t>(pw.y)); });
    if (all <= want) {
        each_entry(m, load, [&](uint32_t j, const uint2& pw) {
            const uint32_t count = units(static_cast<int32_t>(pw.y));
            if (count != 0) {
                drop(j, pw.x, static_cast<int32_t>(pw.y), count);
            }
        });
        return all;
    }
    const uint32_t step = *a.step;
    const uint32_t g = a.net_of[id];
    const uint64_t seed = a.net_seed[g];
    const uint32_t first = static_cast<uint32_t>(a.net_off[g]);
    const uint32_t size = static_cast<uint32_t>(a.net_off[g + 1]) - first;
    const uint32_t self = id - first;
    // a partner's id in its network, nearly always the neuron's own
    auto local = [&](uint32_t i) {
        return i - first < size ? i - first : i - static_cast<uint32_t>(a.net_off[a.net_of[i]]);
    };
    Unit last{ 0, 0, 0 };
    uint32_t entry = 0;
    uint2 pair = make_uint2(0U, 0U);
    for (uint32_t pass = 0; pass < want; pass++) {
        Unit best{ ~0ULL, ~0U, ~0U };
        bool found = false;
        each_entry(m, load, [&](uint32_t j, const uint2& pw) {
            const uint32_t count = units(static_cast<int32_t>(pw.y));
            for (uint32_t c = 0; c < count; c++) {
                const uint32_t partner = local(pw.x);
                const Unit u{ deletion_key(seed, self, step, partner, type, c), partner, c };
                if ((pass == 0 || unit_less(last, u)) && (!found || unit_less(u, best))) {
                    best = u;
                    found = true;
                    entry = j;
                    pair = pw;
                }
            }
        });
        last = best;
    }
    if (want == 1) {
        drop(entry, pair.x, static_cast<int32_t>(pair.y), 1U);
        return 1;
    }
    each_entry(m, load, [&](uint32_t j, const uint2& pw) {
        const uint32_t count = units(static_cast<int32_t>(pw.y));
        uint32_t selected = 0;
        for (uint32_t c = 0; c < count; c++) {
            const uint32_t partner = local(pw.x);
            const Unit u{ deletion_key(seed, self, step, partner, type, c), partner, c };
            selected += unit_less(last, u) ? 0U : 1U;
        }
        if (selected != 0) {
            drop(j, pw.x, static_cast<int32_t>(pw.y), selected);
        }
    });
    return want;
}

// Axons: source s deletes deleted[s] units among its outgoing pairs; each unit lowers the pair's
// weight and disconnects one dendrite (of s's signal type) of the target.  The lists by source hold the
// weights as they are before this kernel.
__global__ void k_del_axons(DelArgs a, const uint64_t* __restrict__ out_off, const uint2* __restrict__ out_pair,
                            const uint32_t* __restrict__ out_entry) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    unsigned long long done = 0, short_of = 0;
    for (uint64_t s = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; s < a.n; s += stride) {
        const uint32_t want = a.deleted[s];
        if (want == 0) {
            continue;
        }
        const uint64_t o = out_off[s];
        const uint32_t m = static_cast<uint32_t>(out_off[s + 1] - o);
        const int sig = a.signal[s] != 0 ? 1 : 0;
        const uint32_t got = delete_units(
            a, static_cast<uint32_t>(s), 0U, m, want, [&](uint32_t j) { return out_pair[o + j]; },
            [](int32_t w) { return static_cast<uint32_t>(w < 0 ? -w : w); },
            [&](uint32_t j, uint32_t t, int32_t w, uint32_t count) {
                a.w[out_entry[o + j]] = w - unit_sign(w) * static_cast<int32_t>(count);
                atomicSub(&a.conn[1 + sig][t], count);
                atomicAdd(&a.vac[1 + sig][t], count);
            });
        done += got;
        short_of += want - got;
    }
    if (done != 0) atomicAdd(&a.counters[kCtrDeleted], done);
    if (short_of != 0) atomicAdd(&a.counters[kCtrDelShort], short_of);
}

// Dendrites of `type` (1 excitatory: pairs of positive weight, 2 inhibitory: negative): target t
// deletes deleted[t] units among its incoming pairs of that sign; each disconnects one axon of the
// source.
__global__ void k_del_dendrites(DelArgs a, uint32_t type) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    unsigned long long done = 0, short_of = 0;
    for (uint64_t t = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; t < a.n; t += stride) {
        const uint32_t want = a.deleted[t];
        if (want == 0) {
            continue;
        }
        const uint64_t o = a.off[t];
        const uint32_t m = static_cast<uint32_t>(a.off[t + 1] - o);
        const uint32_t got = delete_units(
            a, static_cast<uint32_t>(t), type, m, want,
            [&](uint32_t j) { return make_uint2(a.src[o + j], static_cast<uint32_t>(a.w[o + j])); },
            [&](int32_t w) { return (type == 1 ? w > 0 : w < 0) ? static_cast<uint32_t>(w < 0 ? -w : w) : 0U; },
            [&](uint32_t j, uint32_t s, int32_t w, uint32_t count) {
                a.w[o + j] = w - unit_sign(w) * static_cast<int32_t>(count);
                atomicSub(&a.conn[0][s], count);
                atomicAdd(&a.vac[0][s], count);
            });
        done += got;
        short_of += want - got;
    }
    if (done != 0) atomicAdd(&a.counters[kCtrDeleted], done);
    if (short_of != 0) atomicAdd(&a.counters[kCtrDelShort], short_of);
}

// The arrays of `cap` entries beside the graph's own.
int net_alloc_scratch(rl_bh_ctx* c, uint64_t cap) {
    NetGraph& g = c->net;
    RL_TRY(dalloc(c, &g.scratch, cap));
    g.src2 = reinterpret_cast<uint32_t*>(g.scratch);
    g.w2 = reinterpret_cast<int32_t*>(g.src2 + cap);
    RL_TRY(dalloc(c, &g.out_pair, cap));
    RL_TRY(dalloc(c, &g.out_entry, cap));
    g.cap = cap;
    return RL_OK;
}

int net_alloc_edges(rl_bh_ctx* c, uint64_t cap) {
    NetGraph& g = c->net;
    RL_TRY(dalloc(c, &g.src, cap));
    RL_TRY(dalloc(c, &g.w, cap));
    return net_alloc_scratch(c, cap);
}

// Counts the accepted requests of the last commit per target into ncnt (cleared by the commit) and their
// prefix into npre.
int enqueue_net_count(rl_bh_ctx* c) {
    NetGraph& g = c->net;
    const uint64_t n = c->n;
    k_net_count<<<stream_blocks(c->slots_cap), kBlock, 0, c->stream>>>(c->req_off + n, c->req_ok, c->req_target, g.ncnt);
    RL_HIP(c, hipGetLastError());
    return scan_counts(c, g.ncnt, n, g.npre);
}

// Stage, merge, compact.  The staging area is the commit's grouped-index scratch (slots_cap entries,
// at least the accepted requests), free once the commit has run.
int enqueue_net_merge(rl_bh_ctx* c) {
    NetGraph& g = c->net;
    const uint64_t n = c->n;
    hipStream_t s = c->stream;
    k_net_stage<<<stream_blocks(c->slots_cap), kBlock, 0, s>>>(n, g.off, g.cap, c->req_off + n, c->req_ok, c->req_target,
                                                               c->req_source, g.npre, g.ncnt, c->c_sidx, c->counters);
    RL_HIP(c, hipGetLastError());
    k_net_merge<<<grid_for(n), kBlock, 0, s>>>(n, g.off, g.npre, g.src, g.w, c->c_sidx, c->signal, g.src2, g.w2, g.ncnt,
                                               c->counters);
    RL_HIP(c, hipGetLastError());
    RL_TRY(scan_counts(c, g.ncnt, n, g.off2));
    k_net_copyback<<<grid_for(n), kBlock, 0, s>>>(n, g.off, g.npre, g.off2, g.src2, g.w2, g.src, g.w, c->counters);
    RL_HIP(c, hipGetLastError());
    return RL_OK;
}

DelArgs del_args(rl_bh_ctx* c, int type) {
    DelArgs a{};
    a.n = c->n;
    a.net_of = c->net_of;
    a.net_off = c->net_off;
    a.net_seed = c->net_seed;
    a.step = c->d_steps + 1;
    a.deleted = c->neurons.deleted + static_cast<uint64_t>(type) * c->n;
    a.signal = c->signal;
    a.off = c->net.off;
    a.src = c->net.src;
    a.w = c->net.w;
    for (int t = 0; t < 3; t++) {
        a.conn[t] = c->conn[t];
        a.vac[t] = c->vac[t];
    }
    a.counters = c->counters;
    return a;
}

}  // namespace

void net_free(rl_bh_ctx* c) {
    NetGraph& g = c->net;
    dfree(&g.off);
    dfree(&g.src);
    dfree(&g.w);
    dfree(&g.off2);
    dfree(&g.ncnt);
    dfree(&g.npre);
    dfree(&g.out_off);
    dfree(&g.out_pair);
    dfree(&g.out_entry);
    dfree(&g.bin_cnt);
    dfree(&g.bin_off);
    dfree(&g.scratch);
    g.src2 = nullptr;
    g.w2 = nullptr;
    dfree(&g.acc[0]);
    g.acc[1] = nullptr;
    g.cap = 0;
    g.ready = false;
    g.out_valid = false;
    g.syn_valid = false;
}

int net_init(rl_bh_ctx* c, uint64_t capacity, const uint64_t* in_offsets, const uint32_t* sources,
             const int32_t* weights) {
    const uint64_t n = c->n;
    if (n == 0) {
        return fail(c, RL_ESTATE, "rl_net_init: no neurons (rl_bh_init first)");
    }
    // merge repeated (source, target) pairs and drop zero weights, as NetworkGraph keeps them
    std::vector<uint64_t> off(n + 1, 0);
    std::vector<uint32_t> src;
    std::vector<int32_t> w;
    if (in_offsets != nullptr) {
        if (in_offsets[0] != 0) {
            return fail(c, RL_EINVAL, "rl_net_init: in_offsets[0] must be 0");
        }
        for (uint64_t t = 0; t < n; t++) {
            if (in_offsets[t + 1] < in_offsets[t]) {
                return fail(c, RL_EINVAL, "rl_net_init: in_offsets must be non-decreasing");
            }
        }
        const uint64_t edges = in_offsets[n];
        if (edges > 0 && (sources == nullptr || weights == nullptr)) {
            return fail(c, RL_EINVAL, "rl_net_init: null sources or weights");
        }
        for (uint64_t e = 0; e < edges; e++) {
            if (sources[e] >= n) {
                return fail(c, RL_EINVAL, "rl_net_init: edge source out of range");
            }
        }
        std::vector<std::pair<uint32_t, int64_t>> pairs;
        for (uint64_t t = 0; t < n; t++) {
            pairs.clear();
            for (uint64_t e = in_offsets[t]; e < in_offsets[t + 1]; e++) {
                pairs.emplace_back(sources[e], weights[e]);
            }
            std::sort(pairs.begin(), pairs.end());
            int64_t in_weight = 0;   // the synaptic input sums a neuron's in-weights in 32 bits
            for (size_t i = 0; i < pairs.size();) {
                int64_t sum = 0;
                size_t j = i;
                for (; j < pairs.size() && pairs[j].first == pairs[i].first; j++) {
                    sum += pairs[j].second;
                }
                if (sum != 0) {
                    in_weight += sum < 0 ? -sum : sum;
                    if (sum > INT32_MAX || sum < INT32_MIN || in_weight > INT32_MAX) {
                        return fail(c, RL_EINVAL, "rl_net_init: pair weight or summed in-weight of a neuron out of range");
                    }
                    src.push_back(pairs[i].first);
                    w.push_back(static_cast<int32_t>(sum));
                }
                i = j;
            }
            off[t + 1] = src.size();
        }
    }
    if (src.size() > capacity) {
        return fail(c, RL_EINVAL, "rl_net_init: more edges than the capacity");
    }
    destroy_graph(c);  // a captured period without the graph must be captured again
    net_free(c);
    NetGraph& g = c->net;
    RL_TRY(dalloc(c, &g.off, n + 1));
    RL_TRY(dalloc(c, &g.off2, n + 1));
    RL_TRY(dalloc(c, &g.ncnt, n));
    RL_TRY(dalloc(c, &g.npre, n + 1));
    RL_TRY(dalloc(c, &g.out_off, n + 1));
    RL_TRY(dalloc(c, &g.bin_cnt, out_bins(n) * out_blocks(n)));
    RL_TRY(dalloc(c, &g.bin_off, out_bins(n) * out_blocks(n) + 1));
    RL_TRY(dalloc(c, &g.acc[0], 2 * n));
    g.acc[1] = g.acc[0] + n;
    RL_TRY(net_alloc_edges(c, std::max<uint64_t>(capacity, 1)));
    hipStream_t s = c->stream;
    RL_HIP(c, hipMemcpyAsync(g.off, off.data(), (n + 1) * sizeof(uint64_t), hipMemcpyHostToDevice, s));
    if (!src.empty()) {
        RL_HIP(c, hipMemcpyAsync(g.src, src.data(), src.size() * sizeof(uint32_t), hipMemcpyHostToDevice, s));
        RL_HIP(c, hipMemcpyAsync(g.w, w.data(), w.size() * sizeof(int32_t), hipMemcpyHostToDevice, s));
    }
    RL_HIP(c, hipStreamSynchronize(s));
    g.entries_bound = src.size();
    g.ready = true;
    g.out_valid = false;
    g.syn_valid = false;
    return RL_OK;
}

int net_get(rl_bh_ctx* c, uint64_t capacity, uint64_t* in_offsets, uint32_t* sources, int32_t* weights,
            uint64_t* num_edges) {
    NetGraph& g = c->net;
    if (!g.ready) {
        return fail(c, RL_ESTATE, "rl_net_get_edges: no network graph (rl_net_init)");
    }
    const uint64_t n = c->n;
    hipStream_t s = c->stream;
    std::vector<uint64_t> off(n + 1);
    RL_HIP(c, hipMemcpyAsync(off.data(), g.off, (n + 1) * sizeof(uint64_t), hipMemcpyDeviceToHost, s));
    RL_HIP(c, hipStreamSynchronize(s));
    const uint64_t edges = off[n];
    if (num_edges != nullptr) {
        *num_edges = edges;
    }
    if (in_offsets == nullptr && sources == nullptr && weights == nullptr) {
        return RL_OK;
    }
    if (capacity < edges) {
        return fail(c, RL_EINVAL, "rl_net_get_edges: capacity too small");
    }
    if (in_offsets != nullptr) {
        std::memcpy(in_offsets, off.data(), (n + 1) * sizeof(uint64_t));
    }
    if (edges > 0) {
        if (sources != nullptr) RL_HIP(c, hipMemcpyAsync(sources, g.src, edges * sizeof(uint32_t), hipMemcpyDeviceToHost, s));
        if (weights != nullptr) RL_HIP(c, hipMemcpyAsync(weights, g.w, edges * sizeof(int32_t), hipMemcpyDeviceToHost, s));
    }
    RL_HIP(c, hipStreamSynchronize(s));
    return RL_OK;
}

// Groups the graph's non-zero pairs by source.  Allocates nothing and reads no count on the host, so a
// captured period can end with it.
int enqueue_out_lists(rl_bh_ctx* c) {
    NetGraph& g = c->net;
    const uint64_t n = c->n;
    if (!g.ready || n == 0) {
        return RL_OK;
    }
    hipStream_t s = c->stream;
    if (n <= kOutOneSources && g.cap <= kOutOnePairs) {
        k_out_one<<<1, kOutThreads, 0, s>>>(n, g.off, g.src, g.w, g.out_off, g.out_pair, g.out_entry);
        RL_HIP(c, hipGetLastError());
        return RL_OK;
    }
    const uint32_t shift = out_shift(n);
    const uint32_t bins = static_cast<uint32_t>(out_bins(n));
    const unsigned blocks = static_cast<unsigned>(out_blocks(n));
    const uint64_t per = (n + blocks - 1) / blocks;
    k_out_bins<false><<<blocks, kOutThreads, bins * sizeof(uint32_t), s>>>(n, per, shift, bins, g.off, g.src, g.w,
                                                                           g.bin_cnt, nullptr, nullptr);
    RL_HIP(c, hipGetLastError());
    RL_TRY(scan_counts(c, g.bin_cnt, static_cast<uint64_t>(bins) * blocks, g.bin_off));
    k_out_bins<true><<<blocks, kOutThreads, bins * sizeof(uint32_t), s>>>(n, per, shift, bins, g.off, g.src, g.w, nullptr,
                                                                          g.bin_off, g.scratch);
    RL_HIP(c, hipGetLastError());
    const size_t lds = (sizeof(uint32_t) << shift) +
                       (shift <= kOutStageShift ? kOutStaged * (sizeof(uint2) + sizeof(uint32_t)) : 0);
    k_out_sort<<<bins, kOutThreads, lds, s>>>(n, shift, blocks, g.bin_off, g.scratch, g.out_off, g.out_pair, g.out_entry);
    RL_HIP(c, hipGetLastError());
    return RL_OK;
}

// The accumulators from the fired status of fired_buf[parity] and the lists by source: the state the step
// kernel expects at that parity.  Capturable as well.
int enqueue_syn_push(rl_bh_ctx* c, int parity) {
    NetGraph& g = c->net;
    const uint64_t n = c->n;
    if (!g.ready || n == 0 || !c->neurons.ready) {
        return RL_OK;
    }
    RL_TRY(fill_u32(c, reinterpret_cast<uint32_t*>(g.acc[0]), 0U, 2 * n));   // both
    k_syn_push_all<<<stream_blocks(n), kBlock, 0, c->stream>>>(n, c->neurons.fired_buf[parity], g.out_off, g.out_pair,
                                                            g.acc[parity]);
    RL_HIP(c, hipGetLastError());
    return RL_OK;
}

int syn_prepare(rl_bh_ctx* c) {
    NetGraph& g = c->net;
    if (!g.ready || g.syn_valid || c->n == 0 || !c->neurons.ready) {
        return RL_OK;
    }
    if (!g.out_valid) {
        RL_TRY(enqueue_out_lists(c));
        g.out_valid = true;
    }
    RL_TRY(enqueue_syn_push(c, c->neurons.parity));
    g.syn_valid = true;
    return RL_OK;
}

int enqueue_net_append(rl_bh_ctx* c) {
    if (!c->net.ready || c->n == 0) {
        return RL_OK;
    }
    RL_TRY(enqueue_net_count(c));
    return enqueue_net_merge(c);
}

// Grows the edge arrays to hold `need` entries (at least doubling), keeping the current pairs.  A
// captured period refers to the old arrays and is released.
static int net_grow(rl_bh_ctx* c, uint64_t have, uint64_t need) {
    NetGraph& g = c->net;
    hipStream_t s = c->stream;
    destroy_graph(c);
    const uint64_t cap = std::max<uint64_t>(2 * g.cap, need);
    uint32_t* src = nullptr;
    int32_t* w = nullptr;
    RL_TRY(dalloc(c, &src, cap));
    RL_TRY(dalloc(c, &w, cap));
    if (have > 0) {
        RL_HIP(c, hipMemcpyAsync(src, g.src, have * sizeof(uint32_t), hipMemcpyDeviceToDevice, s));
        RL_HIP(c, hipMemcpyAsync(w, g.w, have * sizeof(int32_t), hipMemcpyDeviceToDevice, s));
    }
    RL_HIP(c, hipStreamSynchronize(s));
    dfree(&g.src);
    dfree(&g.w);
    dfree(&g.scratch);
    dfree(&g.out_pair);
    dfree(&g.out_entry);
    g.src = src;
    g.w = w;
    g.out_valid = false;
    g.syn_valid = false;
    return net_alloc_scratch(c, cap);
}

// Merges the counted synapses (ncnt, npre of the last commit), growing the arrays first when they
// would not fit.
static int net_merge_grow(rl_bh_ctx* c) {
    NetGraph& g = c->net;
    const uint64_t n = c->n;
    hipStream_t s = c->stream;
    uint64_t have = 0, add = 0;
    RL_HIP(c, hipMemcpyAsync(&have, g.off + n, sizeof(uint64_t), hipMemcpyDeviceToHost, s));
    RL_HIP(c, hipMemcpyAsync(&add, g.npre + n, sizeof(uint64_t), hipMemcpyDeviceToHost, s));
    RL_HIP(c, hipStreamSynchronize(s));
    if (have + add > g.cap) {
        RL_TRY(net_grow(c, have, have + add));
    }
    g.entries_bound = have + add;   // the merge keeps at most the old entries and the new synapses
    return enqueue_net_merge(c);
}

int net_append(rl_bh_ctx* c) {
    if (!c->net.ready || c->n == 0) {
        return RL_OK;
    }
    c->net.out_valid = false;
    c->net.syn_valid = false;
    RL_TRY(enqueue_net_count(c));
    return net_merge_grow(c);
}

// A captured append that did not fit left the counts of its synapses (ncnt, npre) and the graph
// untouched: grow and merge them now.
int net_append_retry(rl_bh_ctx* c) {
    if (!c->net.ready || c->n == 0) {
        return RL_OK;
    }
    c->net.out_valid = false;
    c->net.syn_valid = false;
    RL_TRY(net_merge_grow(c));
    unsigned long long over = 0;
    RL_HIP(c, hipMemcpyAsync(&over, c->counters + kCtrNetOver, sizeof(over), hipMemcpyDeviceToHost, c->stream));
    RL_HIP(c, hipStreamSynchronize(c->stream));
    if (over != 0) {
        return fail(c, RL_EHIP, "network graph append: still over capacity after growing");
    }
    return RL_OK;
}

// Deletes the synapses of the elements of `type` that the element commit unbound (neurons.deleted).
int enqueue_net_delete(rl_bh_ctx* c, int type) {
    NetGraph& g = c->net;
    const uint64_t n = c->n;
    if (!g.ready || n == 0) {
        return RL_OK;
    }
    hipStream_t s = c->stream;
    const DelArgs a = del_args(c, type);
    if (type == 0) {
        k_del_axons<<<grid_for(n), kBlock, 0, s>>>(a, g.out_off, g.out_pair, g.out_entry);
    } else {
        k_del_dendrites<<<grid_for(n), kBlock, 0, s>>>(a, static_cast<uint32_t>(type));
    }
    RL_HIP(c, hipGetLastError());
    return RL_OK;
}

}  // namespace rl
