// Fused per-step neuron update: background input, Izhikevich membrane update, calcium integrator and
// the growth-curve deltas of the three synaptic element types, one lane per neuron, in FP64 (the
// counter-based background draw, normal_input below, is FP32) and in the CPU path's operation order, but for
// the growth curves' exponential, which is exp_gauss (files compiled with -ffp-contract=off):
//   IzhikevichModelCPU::update_activity   (source/neurons/models/izhikevich/IzhikevichModelCPU.cpp:75-125)
//   CalciumCalculatorCPU::update_current_calcium (source/neurons/calcium/CalciumCalculatorCPU.cpp:40-103)
//   update_number_elements_openmp + gaussian_growth_curve
//                                       (source/neurons/synaptic_elements/SynapticElementsCPU.cpp:25-49,
//                                        GrowthCurves.h:30-54)
// and, at plasticity steps, ElementBaseBase::update (ElementBaseBase.h:420-487) per element type.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "rl_caller_memory.h"
#include "rl_device.h"
#include "rl_internal.h"

namespace rl {
namespace {

constexpr int kBlock = 256;

inline unsigned grid_for(uint64_t n, int block = kBlock) {
    const uint64_t g = (n + block - 1) / block;
    return static_cast<unsigned>(g == 0 ? 1 : g);
}

// The growth curve of one element type; branch-free, so that the three types interleave.  table: kExpTable.
__device__ __forceinline__ double growth_curve(double current, double eta, double epsilon, const double2* table) {
#pragma clang fp contract(off)
    constexpr double factor = 1.6651092223153955127063292897904020952611777045288814583336582344;
    constexpr double factor_inv = 1.0 / factor;
    const double xi = (eta + epsilon) * 0.5;
    const double zeta = (eta - epsilon) * factor_inv;
    const double difference = current - xi;
    const double quotient = difference / zeta;
    const double product = quotient * quotient;
    // exp is 0 below -745.2; the clamp keeps the exponent arithmetic in range and lets a NaN through
    const double x = product > 800.0 ? -800.0 : -product;
    const double curve = (2.0 * exp_gauss(x, table)) - 1.0;
    return eta == epsilon ? (current == eta ? 0.0 : -1.0) : curve;
}

// Normal(mean, stddev) from two Philox words (tag 3) by the Box-Muller transform in FP32 on 24-bit
// uniforms: background noise needs no more (|z| <= 5.77, the mass beyond is 8e-9), and the FP32
// transcendentals take a third of what the FP64 ones cost in this kernel.  This input mode has no
// counterpart in the reference's stream (its normal input comes from Boost); the caller-array mode
// is the one to compare with the CPU path.
__device__ __forceinline__ double normal_input(uint64_t seed, uint32_t neuron, uint32_t step, double mean, double sd) {
    const uint4 o = philox4x32_10(make_uint4(neuron, step, 0U, 3U),
                                  make_uint2(static_cast<uint32_t>(seed), static_cast<uint32_t>(seed >> 32U)));
    const float u1 = static_cast<float>((o.x >> 8U) + 1U) * 5.9604644775390625e-8f;  // (0, 1]
    const float u2 = static_cast<float>(o.y >> 8U) * 5.9604644775390625e-8f;         // [0, 1)
    const float z = sqrtf(-2.0f * logf(u1)) * cospif(2.0f * u2);
    return mean + sd * static_cast<double>(z);
}

struct StepArgs {
    uint64_t n;
    rl_step_params p;
    const uint32_t* net_of;      // network of each neuron, or null: one network
    const uint64_t* net_off;     // first neuron of each network
    const uint64_t* net_seed;    // draw seed of each network
    const double* net_nu;        // growth rates per network (3 each) or null: p.nu for all
    const double* min_ca;        // 3n per-neuron minimum calcium (type-major) or null: p.eta
    const uint32_t* step_base;   // device step base of a captured period (step = *step_base + step) or null
    uint32_t step;
    uint32_t count;              // steps of a launch (1 with synaptic input)
    double* x;
    double* u;
    double* ca;
    const double* input;
    const uint8_t* fired_prev;   // fired status of the previous step (disabled carry)
    uint8_t* fired;
    const double* target_ca;     // per-neuron target calcium, or null: target_value for all
    double target_value;
    double* delta;
    const uint8_t* enabled;
    // synaptic input, or null: acc_cur holds the summed weights that the sources which fired in the
    // previous step pushed; a neuron that fires in this step pushes its out-pairs into acc_next
    int32_t* acc_cur;
    int32_t* acc_next;
    const uint64_t* out_off;
    const uint2* out_pair;       // target, weight
    double conductance;
    // 1 / h and -1 / tau_ca, divided once on the host (IEEE division is correctly rounded on both
    // sides, so the values are the ones the reference's loops use)
    double scale;
    double tau_inv;
};

// Element i of an array that the whole launch shares: scalar base, 32-bit byte offset (at most 2^28
// neurons of 8 bytes).
template <typename T>
__device__ __forceinline__ T& at(T* base, uint32_t i) {
    return *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + i * static_cast<uint32_t>(sizeof(T)));
}

template <typename T>
__device__ __forceinline__ const T& at(const T* base, uint32_t i) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + i * static_cast<uint32_t>(sizeof(T)));
}

// A neuron that fired adds the weight of each of its out-pairs [e0, e1) to the target's input of the
// next step (integer atomics: the sums do not depend on their order).  Few neurons fire per step, so
// this replaces a gather over every in-edge of every neuron.
// The step reads the first kPushAhead pairs before the growth curves and the rest, kPushBatch at a time,
// after them: a launch that fits the chip at once ends with the last wave that pushes, whose three
// round trips (offsets, pairs, pairs) are then mostly behind the arithmetic.  Period of 100 steps with 8
// pairs per neuron: 300,001 neurons 2,570 us with no pair ahead, 2,520 with 4, 2,450 with 8, 2,402 with 12 and
// 2,410 with 16; 1,000 neurons 955, 929, 874, 828 and 834 us; 2M neurons 11.78, 11.69, 11.70, 11.74 and 11.96 ms.
// With the loads free of branches, and skipped whole by waves in which no neuron fired, 1,000 neurons went
// from 843 to 829 us and 2M from 11.42 to 11.33 ms.
// 12 holds the whole list of a neuron with up to 12 partners, as the simulated networks of 3 to 10 synapses
// per neuron have them; each further 8 pairs are a round trip more.  With 5, 12, 24 and 60 pairs per neuron the
// period of 1,000 neurons takes 727, 815, 1,046 and 1,795 us, that of 300,001 2.34, 2.58, 3.03 and 4.69 ms.
constexpr uint32_t kPushAhead = 12;
constexpr uint32_t kPushBatch = 8;

// The first kCount of m > 0 pairs at p (weight 0 beyond the last), without branches between the loads.
template <uint32_t kCount>
__device__ __forceinline__ void load_pairs(const uint2* p, uint32_t m, uint2 (&tw)[kCount]) {
#pragma unroll
    for (uint32_t k = 0; k < kCount; k++) {
        tw[k] = p[k < m ? k : 0U];
    }
#pragma unroll
    for (uint32_t k = 0; k < kCount; k++) {
        tw[k].y = k < m ? tw[k].y : 0U;
    }
}

template <uint32_t kCount>
__device__ __forceinline__ void push_pairs(const StepArgs& a, const uint2 (&tw)[kCount]) {
#pragma unroll
    for (uint32_t k = 0; k < kCount; k++) {
        if (tw[k].y != 0) {
            atomicAdd(&a.acc_next[tw[k].x], static_cast<int32_t>(tw[k].y));
        }
    }
}

// All m pairs at p.
__device__ __forceinline__ void push_out_pairs(const StepArgs& a, const uint2* p, uint32_t m) {
    for (uint32_t k = 0; k < m; k += kPushBatch) {
        uint2 tw[kPushBatch];
        load_pairs(p + k, m - k, tw);
        push_pairs(a, tw);
    }
}

// One wave per block: a wave starts when its own registers are free and waits for no other, and a small
// network's waves lie on compute units of their own.  Period of 100 steps with 64, 128, 256 and 512 threads per block:
// 1,000 neurons 770, 784, 820 and 917 us; 300,001 neurons 2,355, 2,418, 2,409 and 2,480 us; 2M neurons
// 11.34, 11.38, 11.49 and 11.66 ms.  Registers held to 8 waves per SIMD (64): 865, 2,515 us and 11.84 ms.
constexpr int kStepBlock = 64;

// One step of one neuron per lane.
//
// At 1M neurons the kernel moves its 106 bytes per neuron at 4.2 TB/s, 0.8 of what a device copy
// reaches; below about 500,000 neurons (one round of waves) the time is a wave's own chain of loads and
// about 545 vector instructions.  They were about 650, with 64-bit addresses, the library's exp in three
// divergent branches, vector keys for Philox and a loop over the substeps.  1M neurons without synaptic
// input: 28.0 -> 25.5 us; 2M with it: 62 -> 57 us.  Fewer resident waves, so that rounds overlap, are
// slower (6 blocks per CU instead of 8: +2%, 4: +6%).
// kSub: substeps of a step (the reference's 10) unrolled, or 0 for p.h of any number.  kSynaptic: with
// synaptic input (its pairs in flight take 28 registers, which the step without it does not pay).  kMany:
// a.count steps with counter-based input, the state in registers; without synaptic input no neuron waits
// for another, so a captured period's steps share launches: period of 100 steps without synaptic input
// 676 -> 393 us for 1,000 neurons, 2,170 -> 1,622 us for 300,001, 10.63 -> 8.55 ms for 2M.
template <uint32_t kSub, bool kSynaptic, bool kMany>
__global__ void __launch_bounds__(kStepBlock) k_step(StepArgs a) {
#pragma clang fp contract(off)
    __shared__ double2 table[32];
    const uint32_t n = static_cast<uint32_t>(a.n);
    const uint32_t lane_i = blockIdx.x * static_cast<uint32_t>(kStepBlock) + threadIdx.x;
    const bool in = lane_i < n;
    const uint32_t i = in ? lane_i : n - 1U;
    const rl_step_params& p = a.p;
    // every per-neuron load first, so that they are in flight together instead of one round trip
    // after another
    const uint8_t en = at(a.enabled, i);
    const uint8_t fprev = at(a.fired_prev, i);
    const uint32_t g = a.net_of != nullptr ? at(a.net_of, i) : 0U;
    double xv = at(a.x, i);
    double uv = at(a.u, i);
    double c = at(a.ca, i);
    const double tgt = a.target_ca != nullptr ? at(a.target_ca, i) : a.target_value;
    double* const delta[3] = { a.delta, a.delta + a.n, a.delta + 2 * a.n };
    double dl[3] = { at(delta[0], i), at(delta[1], i), at(delta[2], i) };
    double input = p.input_mode == 0 ? at(a.input, i) : 0.0;
    const int32_t syn = kSynaptic ? at(a.acc_cur, i) : 0;
    if (threadIdx.x < 32) {
        table[threadIdx.x] = make_double2(kExpTable[threadIdx.x][0], kExpTable[threadIdx.x][1]);
    }
    __syncthreads();
    if (!in) {
        return;
    }
    if (en == 0) {
        at(a.fired, i) = fprev;  // the step leaves a disabled neuron's status as it was
        if (kSynaptic) {
            at(a.acc_cur, i) = 0;
            if (fprev != 0) {
                const uint64_t e0 = a.out_off[i];
                push_out_pairs(a, a.out_pair + e0, static_cast<uint32_t>(a.out_off[i + 1] - e0));
            }
        }
        return;
    }
    const uint32_t step0 = a.step_base != nullptr && p.input_mode != 0 ? *a.step_base + a.step : a.step;
    const double scale = a.scale;
    const double ab = p.a * p.b;
    const double tau_inv = a.tau_inv;
    const uint32_t h = kSub != 0 ? kSub : p.h;
    bool spiked;
    for (uint32_t rep = 0;; rep++) {
        if (p.input_mode != 0) {
            const uint32_t step = step0 + rep;
            // Neurons of one network are neighbours, so nearly always the wave's lanes share one, whose seed and
            // first neuron then lie in scalar registers.  Other waves draw with per-lane keys: 50 steps of 50,000
            // networks of 4 neurons take 428 us, of 10,000 networks of 16 369 us (1,042 and 472 with one pass per
            // network over scalar keys).
            const uint32_t g0 = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(g)));
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(g != g0) == 0, 1)) {
                const uint64_t seed = a.net_seed[g0];
                const uint32_t first = static_cast<uint32_t>(a.net_off[g0]);
                const uint32_t s0 = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(seed)));
                const uint32_t s1 = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(seed >> 32U)));
                input = normal_input(s0 | static_cast<uint64_t>(s1) << 32U, i - first, step, p.input_mean, p.input_stddev);
            } else {
                input = normal_input(a.net_seed[g], i - static_cast<uint32_t>(a.net_off[g]), step, p.input_mean,
                                     p.input_stddev);
            }
        }
        if (kSynaptic) {
            // SynapticEquallyWeightedActivityInputCPU::update_local_input: the weights of the in-edges
            // whose source fired in the previous step, times the conductance.  The sum was pushed by those
            // sources; it is an integer, which the reference's FP64 accumulation of integer weights
            // yields exactly.  CombinedActivityInputCPU adds it to the background input.
            input = input + static_cast<double>(syn) * a.conductance;
            if (syn != 0) {
                at(a.acc_cur, i) = 0;
            }
        }
        spiked = false;
#pragma unroll
        for (uint32_t s = 0; s < h; s++) {
            const double x_increase = (p.k1 * xv * xv) + (p.k2 * xv) + p.k3 - uv + input;
            const double u_increase = (ab * xv) - (p.a * uv);
            xv += x_increase * scale;
            uv += u_increase * scale;
            if (xv >= p.v_spike) {
                xv = p.c;
                uv += p.d;
                spiked = true;
                break;
            }
        }
        if (!kMany) {
            at(a.fired, i) = spiked ? 1 : 0;
            at(a.x, i) = xv;
            at(a.u, i) = uv;
        }
        uint64_t e0 = 0, e1 = 0;   // read here, used at the end
        if (kSynaptic && spiked) {
            e0 = a.out_off[i];
            e1 = a.out_off[i + 1];
        }
        const double local_beta = p.beta_ca * (spiked ? 1.0 : 0.0);
#pragma unroll
        for (uint32_t s = 0; s < h; s++) {
            c += scale * (c * tau_inv + local_beta);
        }
        if (!kMany) {
            at(a.ca, i) = c;
        }
        uint2 tw[kPushAhead];
        const uint32_t pairs = static_cast<uint32_t>(e1 - e0);
        const bool push = kSynaptic && pairs != 0;
        if (push) {
            load_pairs(a.out_pair + e0, pairs, tw);
        }
#pragma unroll
        for (int t = 0; t < 3; t++) {
            const double eta = a.min_ca != nullptr ? at(a.min_ca + t * a.n, i) : p.eta[t];
            const double clamped_target = tgt < eta ? eta : tgt;  // std::max(target, eta)
            const double dz = growth_curve(c, eta, clamped_target, table);
            const double nu = a.net_nu != nullptr ? a.net_nu[3 * static_cast<uint64_t>(g) + t] : p.nu[t];
            dl[t] = dl[t] + dz * nu;
            if (!kMany) {
                at(delta[t], i) = dl[t];
            }
        }
        if (push) {
            push_pairs(a, tw);
            if (pairs > kPushAhead) {
                push_out_pairs(a, a.out_pair + e0 + kPushAhead, pairs - kPushAhead);
            }
        }
        if (!kMany || rep + 1 == a.count) {
            break;
        }
    }
    if (kMany) {
        at(a.fired, i) = spiked ? 1 : 0;
        at(a.x, i) = xv;
        at(a.u, i) = uv;
        at(a.ca, i) = c;
#pragma unroll
        for (int t = 0; t < 3; t++) {
            at(delta[t], i) = dl[t];
        }
    }
}

constexpr uint32_t kStepsPerLaunch = 256;   // 60 ms for 16M neurons

template <bool kSynaptic, bool kMany>
void launch_step_of(const StepArgs& a, hipStream_t s) {
    if (a.p.h == 10) {
        k_step<10, kSynaptic, kMany><<<grid_for(a.n, kStepBlock), kStepBlock, 0, s>>>(a);
    } else {
        k_step<0, kSynaptic, kMany><<<grid_for(a.n, kStepBlock), kStepBlock, 0, s>>>(a);
    }
}

void launch_step(const StepArgs& a, hipStream_t s) {
    if (a.acc_cur != nullptr) {
        launch_step_of<true, false>(a, s);
    } else if (a.count > 1) {
        launch_step_of<false, true>(a, s);
    } else {
        launch_step_of<false, false>(a, s);
    }
}

// Vacant retract ratios of the element commit: per neuron (3n, type-major) or one per type.
struct Retract {
    const double* per_neuron;
    double r[3];
};

// Element types [k0 / n, k1 / n) of every neuron: index k = type * n + neuron.  The first lane clears the
// deletion counters (unless counters is null).
__global__ void k_elements_update(uint64_t n, uint64_t k0, uint64_t k1, double* __restrict__ grown,
                                  double* __restrict__ delta, uint32_t* __restrict__ c0, uint32_t* __restrict__ c1,
                                  uint32_t* __restrict__ c2, uint32_t* __restrict__ v0, uint32_t* __restrict__ v1,
                                  uint32_t* __restrict__ v2, uint32_t* __restrict__ deleted, Retract rr,
                                  unsigned long long* __restrict__ counters) {
#pragma clang fp contract(off)
    const uint64_t k = k0 + blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x;
    if (k >= k1) {
        return;
    }
    if (counters != nullptr && k == k0) {
        counters[kCtrDeleted] = 0;
        counters[kCtrDelShort] = 0;
    }
    const int t = static_cast<int>(k / n);
    const uint64_t i = k - static_cast<uint64_t>(t) * n;
    uint32_t* connected = t == 0 ? c0 : (t == 1 ? c1 : c2);
    uint32_t* vacant = t == 0 ? v0 : (t == 1 ? v1 : v2);
    const double current_count = grown[k];
    const double current_delta = delta[k];
    const uint32_t connected_integral = connected[i];
    const double retract = rr.per_neuron != nullptr ? rr.per_neuron[k] : (t == 0 ? rr.r[0] : (t == 1 ? rr.r[1] : rr.r[2]));
    const double current_connected = static_cast<double>(connected_integral);
    const double current_vacant = current_count - current_connected;
    const double new_vacant = current_vacant + current_delta;
    if (new_vacant >= 0.0) {
        const double new_vacant_after_retract = (1 - retract) * new_vacant;
        grown[k] = new_vacant_after_retract + current_connected;
        delta[k] = 0.0;
        vacant[i] = static_cast<uint32_t>(new_vacant_after_retract);
        deleted[k] = 0;
        return;
    }
    if (current_count + current_delta <= 0.0) {
        grown[k] = 0.0;
        delta[k] = 0.0;
        vacant[i] = 0;
        connected[i] = 0;
        deleted[k] = connected_integral;
        return;
    }
    const double new_count = current_count + current_delta;
    const double new_connected_count = floor(new_count);
    const double num_vacant = new_count - new_connected_count;
    grown[k] = ((1 - retract) * num_vacant) + new_connected_count;
    delta[k] = 0.0;
    vacant[i] = 0;
    connected[i] = static_cast<uint32_t>(new_connected_count);
    deleted[k] = static_cast<uint32_t>(current_connected - new_connected_count);
}

}  // namespace

void neurons_free(rl_bh_ctx* c) {
    destroy_graph(c);
    Neurons& s = c->neurons;
    dfree(&s.x);
    dfree(&s.u);
    dfree(&s.ca);
    dfree(&s.target_ca);
    dfree(&s.input);
    dfree(&s.fired_buf[0]);
    dfree(&s.fired_buf[1]);
    s.fired = nullptr;
    s.parity = 0;
    dfree(&s.grown);
    dfree(&s.delta);
    dfree(&s.deleted);
    dfree(&s.net_nu);
    dfree(&s.min_ca);
    dfree(&s.retract);
    s.ready = false;
}

int neurons_set_element_params(rl_bh_ctx* c, const double* min_calcium, const double* retract_ratio) {
    Neurons& s = c->neurons;
    if (!s.ready) {
        return fail(c, RL_ESTATE, "rl_neurons_set_element_params before rl_neurons_init");
    }
    const size_t cnt = 3 * static_cast<size_t>(c->n);
    for (size_t k = 0; min_calcium != nullptr && k < cnt; k++) {
        if (!std::isfinite(min_calcium[k])) {
            return fail(c, RL_EINVAL, "rl_neurons_set_element_params: minimum calcium must be finite");
        }
    }
    for (size_t k = 0; retract_ratio != nullptr && k < cnt; k++) {
        if (!(retract_ratio[k] >= 0.0 && retract_ratio[k] <= 1.0)) {
            return fail(c, RL_EINVAL, "rl_neurons_set_element_params: retract ratios must lie in [0, 1]");
        }
    }
    destroy_graph(c);  // a captured period holds the old pointers
    dfree(&s.min_ca);
    dfree(&s.retract);
    if (min_calcium != nullptr && cnt > 0) {
        RL_TRY(dalloc(c, &s.min_ca, cnt));
        RL_HIP(c, hipMemcpyAsync(s.min_ca, min_calcium, cnt * sizeof(double), hipMemcpyHostToDevice, c->stream));
    }
    if (retract_ratio != nullptr && cnt > 0) {
        RL_TRY(dalloc(c, &s.retract, cnt));
        RL_HIP(c, hipMemcpyAsync(s.retract, retract_ratio, cnt * sizeof(double), hipMemcpyHostToDevice, c->stream));
    }
    RL_HIP(c, hipStreamSynchronize(c->stream));
    return RL_OK;
}

int neurons_set_network_growth(rl_bh_ctx* c, const double* nu) {
    Neurons& s = c->neurons;
    if (!s.ready) {
        return fail(c, RL_ESTATE, "rl_neurons_set_network_growth before rl_neurons_init");
    }
    destroy_graph(c);  // a captured period holds the old growth-rate pointer
    if (nu == nullptr) {
        dfree(&s.net_nu);
        return RL_OK;
    }
    const size_t cnt = 3 * static_cast<size_t>(c->num_networks);
    for (size_t k = 0; k < cnt; k++) {
        if (!std::isfinite(nu[k])) {
            return fail(c, RL_EINVAL, "rl_neurons_set_network_growth: growth rates must be finite");
        }
    }
    RL_TRY(dalloc(c, &s.net_nu, cnt));
    RL_HIP(c, hipMemcpyAsync(s.net_nu, nu, cnt * sizeof(double), hipMemcpyHostToDevice, c->stream));
    RL_HIP(c, hipStreamSynchronize(c->stream));
    return RL_OK;
}

int neurons_init(rl_bh_ctx* c, const rl_step_params* p, const double* x, const double* u, const double* ca,
                 const double* target_ca, const double* grown, const uint32_t* connected) {
    const uint64_t n = c->n;
    Neurons& s = c->neurons;
    hipStream_t st = c->stream;
    neurons_free(c);
    s.p = *p;
    RL_TRY(dalloc(c, &s.x, n));
    RL_TRY(dalloc(c, &s.u, n));
    RL_TRY(dalloc(c, &s.ca, n));
    RL_TRY(dalloc(c, &s.target_ca, n));
    RL_TRY(dalloc(c, &s.input, n));
    RL_TRY(dalloc(c, &s.fired_buf[0], n));
    RL_TRY(dalloc(c, &s.fired_buf[1], n));
    s.parity = 0;
    s.fired = s.fired_buf[0];
    RL_TRY(dalloc(c, &s.grown, 3 * n));
    RL_TRY(dalloc(c, &s.delta, 3 * n));
    RL_TRY(dalloc(c, &s.deleted, 3 * n));
    auto up = [&](double* d, const double* h, uint64_t cnt) -> int {
        if (h != nullptr) {
            RL_HIP(c, hipMemcpyAsync(d, h, cnt * sizeof(double), hipMemcpyHostToDevice, st));
        } else {
            RL_HIP(c, hipMemsetAsync(d, 0, cnt * sizeof(double), st));
        }
        return RL_OK;
    };
    RL_TRY(up(s.x, x, n));
    RL_TRY(up(s.u, u, n));
    RL_TRY(up(s.ca, ca, n));
    RL_TRY(up(s.target_ca, target_ca, n));
    // the same bits everywhere (not merely equal values: -0 and +0 stay per-neuron)
    s.target_uniform = n > 0 && target_ca != nullptr &&
                       std::all_of(target_ca, target_ca + n,
                                   [&](double v) { return std::memcmp(&v, target_ca, sizeof(double)) == 0; });
    s.target_value = n > 0 && target_ca != nullptr ? target_ca[0] : 0.0;
    RL_TRY(up(s.grown, grown, 3 * n));
    RL_HIP(c, hipMemsetAsync(s.delta, 0, 3 * n * sizeof(double), st));
    RL_HIP(c, hipMemsetAsync(s.fired_buf[0], 0, n, st));
    RL_HIP(c, hipMemsetAsync(s.fired_buf[1], 0, n, st));
    for (int t = 0; t < 3; t++) {
        if (connected != nullptr) {
            RL_HIP(c, hipMemcpyAsync(c->conn[t], connected + t * n, n * sizeof(uint32_t), hipMemcpyHostToDevice, st));
        }
    }
    RL_HIP(c, hipStreamSynchronize(st));
    s.ready = true;
    c->net.syn_valid = false;   // new fired status
    return RL_OK;
}

namespace {

StepArgs step_args(rl_bh_ctx* c) {
    Neurons& s = c->neurons;
    StepArgs a{};
    a.n = c->n;
    a.p = s.p;
    a.net_of = c->num_networks > 1 ? c->net_of : nullptr;   // one network: every neuron is in network 0
    a.net_off = c->net_off;
    a.net_seed = c->net_seed;
    a.net_nu = s.net_nu;
    a.min_ca = s.min_ca;
    a.step_base = nullptr;
    a.step = 0;
    a.count = 1;
    a.x = s.x;
    a.u = s.u;
    a.ca = s.ca;
    a.input = s.input;
    a.fired_prev = s.fired_buf[s.parity];
    a.fired = s.fired_buf[s.parity ^ 1];
    a.target_ca = s.target_uniform ? nullptr : s.target_ca;
    a.target_value = s.target_value;
    a.delta = s.delta;
    a.enabled = c->enabled;
    a.scale = 1.0 / static_cast<double>(s.p.h);
    a.tau_inv = -1.0 / s.p.tau_ca;
    if (s.p.synaptic_input != 0) {
        a.acc_cur = c->net.acc[s.parity];
        a.acc_next = c->net.acc[s.parity ^ 1];
        a.out_off = c->net.out_off;
        a.out_pair = c->net.out_pair;
        a.conductance = s.p.synapse_conductance;
    }
    return a;
}

__global__ void k_copy_u8(uint64_t n, const uint8_t* __restrict__ from, uint8_t* __restrict__ to) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < n; i += stride) {
        to[i] = from[i];
    }
}

Retract retract_of(const Neurons& s) {
    Retract r{};
    r.per_neuron = s.retract;
    for (int t = 0; t < 3; t++) {
        r.r[t] = s.p.retract_ratio[t];
    }
    return r;
}

int check_synaptic(rl_bh_ctx* c) {
    if (c->neurons.p.synaptic_input != 0 && !c->net.ready) {
        return fail(c, RL_ESTATE, "synaptic input needs the network graph (rl_net_init)");
    }
    return RL_OK;
}

}  // namespace

int neurons_step(rl_bh_ctx* c, uint32_t step, const double* input) {
    Neurons& s = c->neurons;
    if (!s.ready) {
        return fail(c, RL_ESTATE, "rl_neurons_step called before rl_neurons_init");
    }
    if (s.p.input_mode == 0 && input == nullptr) {
        return fail(c, RL_EINVAL, "input_mode 0 needs an input array");
    }
    const uint64_t n = c->n;
    if (n == 0) {
        return RL_OK;
    }
    RL_TRY(check_synaptic(c));
    if (s.p.synaptic_input != 0) {
        RL_TRY(syn_prepare(c));
    }
    StepArgs a = step_args(c);
    a.step = step;
    if (s.p.input_mode == 0) {
        // Page-locked input is read by the step kernel itself: 8 bytes per neuron at the host link's rate,
        // under which the step's own loads and arithmetic disappear, where a copy before the kernel added
        // its time and its start.  100,003 neurons, 10 steps and the state read back: 513 -> 349 us.
        const void* mapped = mapped_host(input, n * sizeof(double));
        if (mapped != nullptr) {
            a.input = static_cast<const double*>(mapped);
        } else {
            RL_HIP(c, hipMemcpyAsync(s.input, input, n * sizeof(double), hipMemcpyHostToDevice, c->stream));
        }
    }
    launch_step(a, c->stream);
    RL_HIP(c, hipGetLastError());
    s.parity ^= 1;
    s.fired = s.fired_buf[s.parity];
    return RL_OK;
}

// The last step's fired status into fired_buf[0], where a captured period expects it.
int normalize_fired(rl_bh_ctx* c) {
    Neurons& s = c->neurons;
    if (!s.ready || s.parity == 0) {
        return RL_OK;
    }
    k_copy_u8<<<kStreamBlocks, kBlock, 0, c->stream>>>(c->n, s.fired_buf[1], s.fired_buf[0]);
    RL_HIP(c, hipGetLastError());
    s.parity = 0;
    s.fired = s.fired_buf[0];
    c->net.syn_valid = false;   // the accumulators were those of parity 1
    return RL_OK;
}

// `steps` neuron steps d_steps[0] + k on the context's stream (counter-based input only).
int enqueue_neuron_steps(rl_bh_ctx* c, uint32_t steps) {
    Neurons& s = c->neurons;
    if (!s.ready || s.p.input_mode == 0) {
        return fail(c, RL_ESTATE, "captured neuron steps need rl_neurons_init with counter-based input");
    }
    if (c->n == 0) {
        return RL_OK;
    }
    RL_TRY(check_synaptic(c));
    if (s.parity != 0) {
        return fail(c, RL_ESTATE, "captured neuron steps start from fired_buf[0]");
    }
    // step k reads fired_buf[k & 1] and writes the other; an odd count copies the last status back,
    // so every replay starts and ends with it in fired_buf[0]
    StepArgs a = step_args(c);
    a.step_base = c->d_steps;
    if (a.acc_cur == nullptr) {
        // a lane reads and writes its own neuron's status only: in place
        a.fired_prev = s.fired_buf[0];
        a.fired = s.fired_buf[0];
        for (uint32_t k = 0; k < steps; k += a.count) {
            a.step = k;
            a.count = std::min(steps - k, kStepsPerLaunch);
            launch_step(a, c->stream);
            RL_HIP(c, hipGetLastError());
        }
        return RL_OK;
    }
    for (uint32_t k = 0; k < steps; k++) {
        a.step = k;
        a.fired_prev = s.fired_buf[k & 1U];
        a.fired = s.fired_buf[(k + 1) & 1U];
        a.acc_cur = c->net.acc[k & 1U];
        a.acc_next = c->net.acc[(k + 1) & 1U];
        launch_step(a, c->stream);
        RL_HIP(c, hipGetLastError());
    }
    if ((steps & 1U) != 0) {
        k_copy_u8<<<kStreamBlocks, kBlock, 0, c->stream>>>(c->n, s.fired_buf[1], s.fired_buf[0]);
        RL_HIP(c, hipGetLastError());
    }
    return RL_OK;
}

// ElementBaseBase::update for the three element types.  With a network graph the types are committed
// one after the other, each followed by the deletion of the synapses its shrunken elements held
// (SynapseDeletionFinderCPU::delete_synapses: axons, then excitatory, then inhibitory dendrites, each
// seeing the disconnections of the previous ones); the deletion draws use the update index in
// d_steps[1].  Without a graph the deletions are only counted (neurons.deleted).
int enqueue_elements_commit(rl_bh_ctx* c) {
    Neurons& s = c->neurons;
    if (!s.ready) {
        return fail(c, RL_ESTATE, "rl_neurons_commit_elements called before rl_neurons_init");
    }
    const uint64_t n = c->n;
    if (n == 0) {
        return RL_OK;
    }
    if (!c->net.ready) {
        k_elements_update<<<grid_for(3 * n), kBlock, 0, c->stream>>>(n, 0, 3 * n, s.grown, s.delta, c->conn[0], c->conn[1],
                                                                      c->conn[2], c->vac[0], c->vac[1], c->vac[2], s.deleted,
                                                                      retract_of(s), nullptr);
        RL_HIP(c, hipGetLastError());
        return RL_OK;
    }
    // axons are deleted among the pairs by source; a captured period with synaptic input starts with valid
    // lists (rl_bh_graph_launch) and its steps leave the pairs alone
    if (c->capturing ? s.p.synaptic_input == 0 : !c->net.out_valid) {
        RL_TRY(enqueue_out_lists(c));
    }
    for (int t = 0; t < 3; t++) {
        k_elements_update<<<grid_for(n), kBlock, 0, c->stream>>>(n, t * n, (t + 1) * n, s.grown, s.delta, c->conn[0],
                                                                  c->conn[1], c->conn[2], c->vac[0], c->vac[1], c->vac[2],
                                                                  s.deleted, retract_of(s),
                                                                  t == 0 ? c->counters : nullptr);
        RL_HIP(c, hipGetLastError());
        RL_TRY(enqueue_net_delete(c, t));
    }
    return RL_OK;
}

int neurons_commit(rl_bh_ctx* c, uint32_t update, uint32_t* deleted) {
    if (c->neurons.ready && c->n > 0) {
        RL_TRY(set_steps(c, 0, update));
    }
    const int status = enqueue_elements_commit(c);
    c->net.out_valid = false;   // deletions change the pairs
    c->net.syn_valid = false;
    RL_TRY(status);
    if (deleted != nullptr && c->n > 0) {
        RL_HIP(c, hipMemcpyAsync(deleted, c->neurons.deleted, 3 * c->n * sizeof(uint32_t), hipMemcpyDeviceToHost,
                                 c->stream));
    }
    unsigned long long short_of = 0;
    if (c->net.ready && c->n > 0) {
        RL_HIP(c, hipMemcpyAsync(&short_of, c->counters + kCtrDelShort, sizeof(short_of), hipMemcpyDeviceToHost,
                                 c->stream));
    }
    RL_HIP(c, hipStreamSynchronize(c->stream));
    if (short_of != 0) {
        // the reference throws here (RandomSynapseDeletionFinder::find_synapses_on_neuron); the
        // deletions that the graph allowed have been made
        return fail(c, RL_EINVAL, "rl_neurons_commit_elements: the network graph holds fewer synapses than the "
                                  "connected counts of the elements to delete");
    }
    return RL_OK;
}

int neurons_get(rl_bh_ctx* c, double* x, double* u, double* ca, uint8_t* fired, double* delta, double* grown,
                uint32_t* connected) {
    Neurons& s = c->neurons;
    if (!s.ready) {
        return fail(c, RL_ESTATE, "rl_neurons_get called before rl_neurons_init");
    }
    const uint64_t n = c->n;
    CopyItem items[kMaxCopies];
    int count = 0;
    auto add = [&](void* dst, const void* src, size_t bytes) {
        if (dst != nullptr && bytes != 0) {
            items[count++] = { dst, src, bytes };
        }
    };
    add(x, s.x, n * sizeof(double));
    add(u, s.u, n * sizeof(double));
    add(ca, s.ca, n * sizeof(double));
    add(fired, s.fired, n);
    add(delta, s.delta, 3 * n * sizeof(double));
    add(grown, s.grown, 3 * n * sizeof(double));
    for (int t = 0; t < 3 && connected != nullptr; t++) {
        add(connected + t * n, c->conn[t], n * sizeof(uint32_t));
    }
    RL_TRY(copy_arrays(c, items, count, hipMemcpyDeviceToHost));
    RL_HIP(c, hipStreamSynchronize(c->stream));
    return RL_OK;
}

}  // namespace rl
