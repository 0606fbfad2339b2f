// Exclusive prefix sums and fills for the update pipeline.  Sizes come from the host (fixed per
// context) or are read from device memory by the kernels, and nothing here issues a memset, an
// allocation or a host synchronisation, so the pipeline that uses them can be captured into a HIP
// graph and replayed.  The sums are deterministic: the tile partition and the reduction order do not
// depend on timing.
#include <algorithm>

#include "rl_caller_memory.h"
#include "rl_internal.h"

namespace rl {
namespace {

constexpr int kScanBlock = 256;
constexpr int kScanItems = 16;                      // counts per thread
constexpr uint64_t kScanTile = kScanBlock * kScanItems;
constexpr int kTopBlock = 1024;                     // the single block that scans the tile sums
constexpr int kTopItems = 8;
// Launches of a scan.  A small kernel costs 5-8 us from launch to launch whatever it does, in a captured
// graph too, so up to kOneBlockCounts counts are scanned by one block (two passes of 16,384), and while
// the tile sums are few (kOwnPrefixTiles) every block of the last kernel adds up those before its own
// instead of waiting for a kernel that does.  With three launches at every size the scans of a
// 1,000-neuron update took 15 of its 48 launches.
constexpr uint64_t kOneBlockCounts = 32768;
constexpr uint64_t kOwnPrefixTiles = 1024;
constexpr int kWave = 64;

// Thread t of tile b owns counts [b * 4096 + 16 t, + 16); counts at or beyond n read as 0.
__device__ __forceinline__ void load_counts(const uint32_t* __restrict__ in, uint64_t first, uint64_t n,
                                            uint32_t (&v)[kScanItems]) {
    if (first + kScanItems <= n) {
        const uint4* p = reinterpret_cast<const uint4*>(in + first);
#pragma unroll
        for (int k = 0; k < kScanItems / 4; k++) {
            const uint4 w = p[k];
            v[4 * k] = w.x;
            v[4 * k + 1] = w.y;
            v[4 * k + 2] = w.z;
            v[4 * k + 3] = w.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; k++) {
            v[k] = first + k < n ? in[first + k] : 0U;
        }
    }
}

// Exclusive scan of one value per thread over the block; *total receives the block's sum.
template <int kThreads>
__device__ __forceinline__ uint64_t block_exclusive(uint64_t x, uint64_t* wave_sums, uint64_t* total) {
    const int ln = static_cast<int>(threadIdx.x) & (kWave - 1);
    const int w = static_cast<int>(threadIdx.x) / kWave;
    unsigned long long inc = x;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const unsigned long long y = __shfl_up(inc, o, kWave);
        if (ln >= o) {
            inc += y;
        }
    }
    if (ln == kWave - 1) {
        wave_sums[w] = inc;
    }
    __syncthreads();
    uint64_t off = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < kThreads / kWave; k++) {
        const uint64_t s = wave_sums[k];
        off += k < w ? s : 0;
        tot += s;
    }
    __syncthreads();  // wave_sums may be reused by the caller
    *total = tot;
    return off + inc - x;
}

// Writes the exclusive prefix sums `run`, run + v[0], ... of a thread's counts.
__device__ __forceinline__ void store_prefix(uint64_t* __restrict__ out, uint64_t first, uint64_t n, uint64_t run,
                                             const uint32_t (&v)[kScanItems]) {
    uint64_t o[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        o[k] = run;
        run += v[k];
    }
    if (first + kScanItems <= n) {
        ulonglong2* p = reinterpret_cast<ulonglong2*>(out + first);
#pragma unroll
        for (int k = 0; k < kScanItems / 2; k++) {
            p[k] = make_ulonglong2(o[2 * k], o[2 * k + 1]);
        }
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; k++) {
            if (first + k < n) {
                out[first + k] = o[k];
            }
        }
    }
}

__device__ __forceinline__ uint64_t sum_counts(const uint32_t (&v)[kScanItems]) {
    uint64_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        s += v[k];
    }
    return s;
}

__global__ void __launch_bounds__(kScanBlock) k_scan_reduce(const uint32_t* __restrict__ in, uint64_t n,
                                                            uint64_t* __restrict__ part) {
    __shared__ uint64_t ws[kScanBlock / kWave];
    uint32_t v[kScanItems];
    load_counts(in, blockIdx.x * kScanTile + threadIdx.x * static_cast<uint64_t>(kScanItems), n, v);
    uint64_t tot = 0;
    (void)block_exclusive<kScanBlock>(sum_counts(v), ws, &tot);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = tot;
    }
}

// One block scans everything.
__global__ void __launch_bounds__(kTopBlock) k_scan_one(const uint32_t* __restrict__ in, uint64_t n,
                                                        uint64_t* __restrict__ out, uint64_t* __restrict__ total) {
    __shared__ uint64_t ws[kTopBlock / kWave];
    uint64_t carry = 0;
    for (uint64_t base = 0; base < n; base += static_cast<uint64_t>(kTopBlock) * kScanItems) {
        const uint64_t first = base + threadIdx.x * static_cast<uint64_t>(kScanItems);
        uint32_t v[kScanItems];
        load_counts(in, first, n, v);
        uint64_t tot = 0;
        const uint64_t run = carry + block_exclusive<kTopBlock>(sum_counts(v), ws, &tot);
        store_prefix(out, first, n, run, v);
        carry += tot;
    }
    if (threadIdx.x == 0) {
        out[n] = carry;
        if (total != nullptr) {
            *total = carry;
        }
    }
}

// One block: exclusive scan of the tile sums in place, and the grand total into out[n].
__global__ void __launch_bounds__(kTopBlock) k_scan_top(uint64_t* __restrict__ part, uint64_t tiles,
                                                        uint64_t* __restrict__ out_total,
                                                        uint64_t* __restrict__ total) {
    __shared__ uint64_t ws[kTopBlock / kWave];
    uint64_t carry = 0;
    for (uint64_t base = 0; base < tiles; base += static_cast<uint64_t>(kTopBlock) * kTopItems) {
        const uint64_t first = base + threadIdx.x * static_cast<uint64_t>(kTopItems);
        uint64_t v[kTopItems];
        uint64_t s = 0;
#pragma unroll
        for (int k = 0; k < kTopItems; k++) {
            v[k] = first + k < tiles ? part[first + k] : 0;
            s += v[k];
        }
        uint64_t tot = 0;
        uint64_t run = carry + block_exclusive<kTopBlock>(s, ws, &tot);
#pragma unroll
        for (int k = 0; k < kTopItems; k++) {
            if (first + k < tiles) {
                part[first + k] = run;
            }
            run += v[k];
        }
        carry += tot;
    }
    if (threadIdx.x == 0) {
        *out_total = carry;
        if (total != nullptr) {
            *total = carry;
        }
    }
}

// kOwnPrefix: part holds the tiles' sums, and the block adds up the ones before its own (at most
// kOwnPrefixTiles); the last block writes the total.  Else part holds their prefix sums.
template <bool kOwnPrefix>
__global__ void __launch_bounds__(kScanBlock) k_scan_down(const uint32_t* __restrict__ in, uint64_t n,
                                                          const uint64_t* __restrict__ part, uint64_t* __restrict__ out,
                                                          uint64_t* __restrict__ total) {
    __shared__ uint64_t ws[kScanBlock / kWave];
    const uint64_t first = blockIdx.x * kScanTile + threadIdx.x * static_cast<uint64_t>(kScanItems);
    uint32_t v[kScanItems];
    load_counts(in, first, n, v);
    uint64_t before = 0;
    if (kOwnPrefix) {
        uint64_t mine = 0;
#pragma unroll
        for (uint64_t k = 0; k < kOwnPrefixTiles / kScanBlock; k++) {
            const uint64_t t = k * kScanBlock + threadIdx.x;
            mine += t < blockIdx.x ? part[t] : 0;
        }
        (void)block_exclusive<kScanBlock>(mine, ws, &before);
    } else {
        before = part[blockIdx.x];
    }
    uint64_t tot = 0;
    const uint64_t run = before + block_exclusive<kScanBlock>(sum_counts(v), ws, &tot);
    store_prefix(out, first, n, run, v);
    if (kOwnPrefix && blockIdx.x + 1 == gridDim.x && threadIdx.x == 0) {
        out[n] = before + tot;
        if (total != nullptr) {
            *total = before + tot;
        }
    }
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t value, uint64_t n) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < n; i += stride) {
        p[i] = value;
    }
}

constexpr int kCopyBlock = 256;
constexpr int kCopyAhead = 4;            // loads in flight per thread
constexpr unsigned kCopyBlocks = 256;    // per array

struct CopyList {
    const char* src[kMaxCopies];
    char* dst[kMaxCopies];
    uint64_t bytes[kMaxCopies];
};

template <typename T>
__device__ __forceinline__ void copy_words(const char* __restrict__ from, char* __restrict__ to, uint64_t bytes) {
    const T* const src = reinterpret_cast<const T*>(from);
    T* const dst = reinterpret_cast<T*>(to);
    const uint64_t words = bytes / sizeof(T);
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kCopyBlock;
    for (uint64_t i = blockIdx.x * static_cast<uint64_t>(kCopyBlock) + threadIdx.x; i < words; i += kCopyAhead * stride) {
        T v[kCopyAhead];
#pragma unroll
        for (int k = 0; k < kCopyAhead; k++) {
            const uint64_t j = i + k * stride;
            v[k] = src[j < words ? j : i];
        }
#pragma unroll
        for (int k = 0; k < kCopyAhead; k++) {
            const uint64_t j = i + k * stride;
            if (j < words) {
                dst[j] = v[k];
            }
        }
    }
    const uint64_t done = words * sizeof(T);
    if (blockIdx.x == 0 && threadIdx.x < bytes - done) {
        to[done + threadIdx.x] = from[done + threadIdx.x];
    }
}

// Array blockIdx.y, in the widest words that source and destination are aligned to.
__global__ void __launch_bounds__(kCopyBlock) k_copy_list(CopyList l) {
    const char* const from = l.src[blockIdx.y];
    char* const to = l.dst[blockIdx.y];
    const uintptr_t low = reinterpret_cast<uintptr_t>(from) | reinterpret_cast<uintptr_t>(to);
    if ((low & 15U) == 0) {
        copy_words<uint4>(from, to, l.bytes[blockIdx.y]);
    } else if ((low & 3U) == 0) {
        copy_words<uint32_t>(from, to, l.bytes[blockIdx.y]);
    } else {
        copy_words<uint8_t>(from, to, l.bytes[blockIdx.y]);
    }
}

__global__ void k_set_u32(uint32_t* __restrict__ p, uint32_t a, uint32_t b) {
    if (threadIdx.x == 0) {
        p[0] = a;
        p[1] = b;
    }
}

}  // namespace

uint64_t scan_scratch_entries(uint64_t n) {
    return (n + kScanTile - 1) / kScanTile + 1;
}

hipError_t scan_counts_on(hipStream_t s, const uint32_t* in, uint64_t n, uint64_t* out, uint64_t* part,
                          uint64_t* total) {
    if (n <= kOneBlockCounts) {
        k_scan_one<<<1, kTopBlock, 0, s>>>(in, n, out, total);
        return hipGetLastError();
    }
    const uint64_t tiles = (n + kScanTile - 1) / kScanTile;
    k_scan_reduce<<<static_cast<unsigned>(tiles), kScanBlock, 0, s>>>(in, n, part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        return e;
    }
    if (tiles <= kOwnPrefixTiles) {
        k_scan_down<true><<<static_cast<unsigned>(tiles), kScanBlock, 0, s>>>(in, n, part, out, total);
        return hipGetLastError();
    }
    k_scan_top<<<1, kTopBlock, 0, s>>>(part, tiles, out + n, total);
    e = hipGetLastError();
    if (e == hipSuccess) {
        k_scan_down<false><<<static_cast<unsigned>(tiles), kScanBlock, 0, s>>>(in, n, part, out, nullptr);
        e = hipGetLastError();
    }
    return e;
}

int scan_counts(rl_bh_ctx* c, const uint32_t* in, uint64_t n, uint64_t* out, uint64_t* total) {
    if ((reinterpret_cast<uintptr_t>(in) & 15U) != 0 || (reinterpret_cast<uintptr_t>(out) & 15U) != 0) {
        return fail(c, RL_EINVAL, "scan_counts: operands must be 16-byte aligned");
    }
    if (scan_scratch_entries(n) > c->scan_part_cap) {
        return fail(c, RL_ESTATE, "scan_counts: scratch smaller than the scan");
    }
    RL_HIP(c, scan_counts_on(c->stream, in, n, out, c->scan_part, total));
    return RL_OK;
}

int fill_u32(rl_bh_ctx* c, uint32_t* p, uint32_t value, uint64_t n) {
    k_fill_u32<<<stream_blocks(n), 256, 0, c->stream>>>(p, value, n);
    RL_HIP(c, hipGetLastError());
    return RL_OK;
}

// One launch for the arrays that the device can address (page-locked host arrays, memory of the own GPU);
// the rest by copies.  Each copy of its own costs 9 to 10 us whatever its size: with one launch per
// call, and the counts written to page-locked memory by the kernels that form them, a 1,000-neuron update
// takes 271 us instead of 341, a 1,000-neuron period 938 instead of 1,039.  Large arrays move at the host
// link's rate, 57 GB/s, either way (16M neurons: 174.8 ms with both).
int copy_arrays(rl_bh_ctx* c, const CopyItem* items, int count, hipMemcpyKind kind) {
    CopyList l{};
    unsigned listed = 0;
    size_t most = 0;
    for (int k = 0; k < count; k++) {
        const CopyItem& it = items[k];
        if (it.bytes == 0) {
            continue;
        }
        const void* src = it.src;
        void* dst = it.dst;
        if (kind == hipMemcpyHostToDevice) {
            src = mapped_host(it.src, it.bytes);
        } else if (kind == hipMemcpyDeviceToHost) {
            dst = mapped_host(it.dst, it.bytes);
        } else if (!own_device(c->cfg.device, it.src, it.bytes)) {
            src = nullptr;
        }
        if (src == nullptr || dst == nullptr || listed == kMaxCopies) {
            RL_HIP(c, hipMemcpyAsync(it.dst, it.src, it.bytes, kind, c->stream));
            continue;
        }
        l.src[listed] = static_cast<const char*>(src);
        l.dst[listed] = static_cast<char*>(dst);
        l.bytes[listed] = it.bytes;
        listed++;
        most = std::max(most, it.bytes);
    }
    if (listed != 0) {
        constexpr size_t kPerBlock = kCopyBlock * sizeof(uint4);
        const size_t blocks = std::min<size_t>(kCopyBlocks, (most + kPerBlock - 1) / kPerBlock);
        k_copy_list<<<dim3(static_cast<unsigned>(blocks), listed), kCopyBlock, 0, c->stream>>>(l);
        RL_HIP(c, hipGetLastError());
    }
    return RL_OK;
}

int set_steps(rl_bh_ctx* c, uint32_t neuron_step, uint32_t update) {
    k_set_u32<<<1, 64, 0, c->stream>>>(c->d_steps, neuron_step, update);
    RL_HIP(c, hipGetLastError());
    return RL_OK;
}

}  // namespace rl
