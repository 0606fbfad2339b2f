// Device helpers shared by the kernels.  All translation units are compiled with
// -ffp-contract=off so that FP64 expressions round exactly like the CPU path's.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace rl {

// Three-argument std::hypot of libstdc++ (<cmath>, __hypot3): scale by the largest magnitude,
// sum the three squared quotients left to right, square root, rescale.  The reference computes
// every distance on the path this way (Vec3::calculate_2_norm, external/cpp-utility/
// data-structure/Vec3.hpp:548-551).  Division and sqrt are IEEE correctly rounded on gfx950.
__device__ __forceinline__ double hypot3_exact(double x, double y, double z) {
#pragma clang fp contract(off)
    x = fabs(x);
    y = fabs(y);
    z = fabs(z);
    const double a = x < y ? (y < z ? z : y) : (x < z ? z : x);
    if (a != 0.0) {
        const double xa = x / a;
        const double ya = y / a;
        const double za = z / a;
        return a * sqrt(xa * xa + ya * ya + za * za);
    }
    return a != a ? a : 0.0;
}

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw: "Parallel random numbers: as easy as 1, 2, 3", SC'11).
// Each round's two 32x32 -> 64-bit products are written as 64-bit multiplies, which compile to one
// v_mad_u64_u32 each instead of a v_mul_lo_u32 + v_mul_hi_u32 pair (all quarter-rate instructions).
__device__ __forceinline__ uint4 philox4x32_10(uint4 c, uint2 k) {
#pragma unroll
    for (int round = 0; round < 10; round++) {
        if (round > 0) {
            k.x += 0x9E3779B9U;
            k.y += 0xBB67AE85U;
        }
        const uint64_t p0 = static_cast<uint64_t>(c.x) * 0xD2511F53ULL;
        const uint64_t p1 = static_cast<uint64_t>(c.z) * 0xCD9E8D57ULL;
        c = make_uint4(static_cast<uint32_t>(p1 >> 32U) ^ c.y ^ k.x, static_cast<uint32_t>(p1),
                       static_cast<uint32_t>(p0 >> 32U) ^ c.w ^ k.y, static_cast<uint32_t>(p0));
    }
    return c;
}

// Draw for the pick at `level` of axon j of neuron `neuron` in plasticity step `step` (tag 1).
__device__ __forceinline__ uint32_t pick_draw(uint64_t seed, uint32_t neuron, uint32_t step, uint32_t j,
                                              uint32_t level) {
    const uint4 o = philox4x32_10(make_uint4(neuron, step, (j << 8U) | (level & 0xFFU), 1U),
                                  make_uint2(static_cast<uint32_t>(seed), static_cast<uint32_t>(seed >> 32U)));
    return o.x;
}

// 64-bit commit priority of request (source, j) (tag 2).
__device__ __forceinline__ uint64_t commit_priority(uint64_t seed, uint32_t source, uint32_t step, uint32_t j) {
    const uint4 o = philox4x32_10(make_uint4(source, step, j, 2U),
                                  make_uint2(static_cast<uint32_t>(seed), static_cast<uint32_t>(seed >> 32U)));
    return (static_cast<uint64_t>(o.x) << 32U) | o.y;
}

// 64-bit key of synapse unit `copy` between `neuron` and `partner` (ids inside their network) when
// `neuron` deletes `type` elements (0 axon, 1 excitatory, 2 inhibitory dendrite) in plasticity update
// `step`: the deleted units are the ones with the smallest keys, a uniform random subset whatever
// the order the synapses are stored in.  The low two bits of the last counter word are 0, so the
// stream never meets the tags 1-3 of the other draws.
__device__ __forceinline__ uint64_t deletion_key(uint64_t seed, uint32_t neuron, uint32_t step, uint32_t partner,
                                                 uint32_t type, uint32_t copy) {
    const uint4 o = philox4x32_10(make_uint4(neuron, step, partner, (copy << 4U) | (type << 2U)),
                                  make_uint2(static_cast<uint32_t>(seed), static_cast<uint32_t>(seed >> 32U)));
    return (static_cast<uint64_t>(o.x) << 32U) | o.y;
}

// uniform_real_distribution(0, next) of a 32-bit engine: (k / 2^32) * (next - 0) + 0
// (boost::random::detail::generate_uniform_real; ProbabilityPicker.h:108-109).
__device__ __forceinline__ double draw_to_uniform(uint32_t k, double next) {
#pragma clang fp contract(off)
    const double numerator = static_cast<double>(k);
    return numerator / 4294967296.0 * (next - 0.0) + 0.0;
}

// 2^(i/32), i = 0..31, each as the nearest FP64 number and the nearest one to the rest.
static __constant__ const double kExpTable[32][2] = {
    { 0x1.0000000000000p+0, 0x0.0p+0 },
    { 0x1.059b0d3158574p+0, 0x1.d73e2a475b465p-55 },
    { 0x1.0b5586cf9890fp+0, 0x1.8a62e4adc610bp-54 },
    { 0x1.11301d0125b51p+0, -0x1.6c51039449b3ap-54 },
    { 0x1.172b83c7d517bp+0, -0x1.19041b9d78a76p-55 },
    { 0x1.1d4873168b9aap+0, 0x1.e016e00a2643cp-54 },
    { 0x1.2387a6e756238p+0, 0x1.9b07eb6c70573p-54 },
    { 0x1.29e9df51fdee1p+0, 0x1.612e8afad1255p-55 },
    { 0x1.306fe0a31b715p+0, 0x1.6f46ad23182e4p-55 },
    { 0x1.371a7373aa9cbp+0, -0x1.63aeabf42eae2p-54 },
    { 0x1.3dea64c123422p+0, 0x1.ada0911f09ebcp-55 },
    { 0x1.44e086061892dp+0, 0x1.89b7a04ef80d0p-59 },
    { 0x1.4bfdad5362a27p+0, 0x1.d4397afec42e2p-56 },
    { 0x1.5342b569d4f82p+0, -0x1.07abe1db13cadp-55 },
    { 0x1.5ab07dd485429p+0, 0x1.6324c054647adp-54 },
    { 0x1.6247eb03a5585p+0, -0x1.383c17e40b497p-54 },
    { 0x1.6a09e667f3bcdp+0, -0x1.bdd3413b26456p-54 },
    { 0x1.71f75e8ec5f74p+0, -0x1.16e4786887a99p-55 },
    { 0x1.7a11473eb0187p+0, -0x1.41577ee04992fp-55 },
    { 0x1.82589994cce13p+0, -0x1.d4c1dd41532d8p-54 },
    { 0x1.8ace5422aa0dbp+0, 0x1.6e9f156864b27p-54 },
    { 0x1.93737b0cdc5e5p+0, -0x1.75fc781b57ebcp-57 },
    { 0x1.9c49182a3f090p+0, 0x1.c7c46b071f2bep-56 },
    { 0x1.a5503b23e255dp+0, -0x1.d2f6edb8d41e1p-54 },
    { 0x1.ae89f995ad3adp+0, 0x1.7a1cd345dcc81p-54 },
    { 0x1.b7f76f2fb5e47p+0, -0x1.5584f7e54ac3bp-56 },
    { 0x1.c199bdd85529cp+0, 0x1.11065895048ddp-55 },
    { 0x1.cb720dcef9069p+0, 0x1.503cbd1e949dbp-56 },
    { 0x1.d5818dcfba487p+0, 0x1.2ed02d75b3707p-55 },
    { 0x1.dfc97337b9b5fp+0, -0x1.1a5cd4f184b5cp-54 },
    { 0x1.ea4afa2a490dap+0, -0x1.e9c23179c2893p-54 },
    { 0x1.f50765b6e4540p+0, 0x1.9d3e12dd8a18bp-54 },
};

// exp(x) of a Gaussian exponent (x <= 0) in FP64.
//   x = (32 e + i) ln2/32 + r,  exp(x) = 2^e 2^(i/32) exp(r),  |r| <= ln2/64
// with ln2/32 in two parts (the fused x - k ln2/32 of the first is exact), 2^(i/32) in two parts from the
// table (a copy of kExpTable in LDS), and the Taylor polynomial of exp(r) - 1 to r^6 (the next term is below 4e-18).  Largest error
// against 64-bit-mantissa values at 2 million points of [-700, 0]: 0.55 units in the last place (the math
// library's exp: 0.86); about 20 vector instructions instead of 34.
__device__ __forceinline__ double exp_gauss(double x, const double2* table) {
#pragma clang fp contract(off)
    const double k = __builtin_rint(x * 46.16624130844683);
    double r = __builtin_fma(k, -0x1.62e42fefa39efp-6, x);
    r = __builtin_fma(k, -0x1.abc9e3b39803fp-61, r);
    const int n = static_cast<int>(k);
    const double2 t = table[n & 31];
    double q = __builtin_fma(r, 1.0 / 720.0, 1.0 / 120.0);
    q = __builtin_fma(r, q, 1.0 / 24.0);
    q = __builtin_fma(r, q, 1.0 / 6.0);
    q = __builtin_fma(r, q, 0.5);
    q = __builtin_fma(r * r, q, r);
    return ldexp(t.x + __builtin_fma(t.x, q, t.y), n >> 5);
}

// Kernels that visit every neuron or group and end by adding to a device counter: blocks of 1,024
// threads, two per CU of a 256-CU GPU, so that few atomics meet at the counter.
constexpr int kCountThreads = 1024;
constexpr unsigned kCountBlocks = 512;

inline unsigned count_blocks(uint64_t n) {
    const uint64_t b = (n + kCountThreads - 1) / kCountThreads;
    return static_cast<unsigned>(b == 0 ? 1 : (b < kCountBlocks ? b : kCountBlocks));
}

// Sums each of the N values over a block of kCountThreads threads; thread 0 gets the totals.
template <int N>
__device__ __forceinline__ void block_totals(unsigned long long (&v)[N]) {
    __shared__ unsigned long long part[N][kCountThreads / 64];
    const uint32_t ln = threadIdx.x & 63U;
#pragma unroll
    for (int k = 0; k < N; k++) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            v[k] += __shfl_xor(v[k], o, 64);
        }
        if (ln == 0) {
            part[k][threadIdx.x / 64U] = v[k];
        }
    }
    __syncthreads();
    if (threadIdx.x < 64U) {
#pragma unroll
        for (int k = 0; k < N; k++) {
            unsigned long long t = ln < kCountThreads / 64U ? part[k][ln] : 0;
#pragma unroll
            for (int o = 8; o > 0; o >>= 1) {
                t += __shfl_xor(t, o, 64);
            }
            v[k] = t;
        }
    }
}

}  // namespace rl
