// Grid-wide reductions inside one kernel, for the solvers whose iterations run
// in a single cooperative launch (every workgroup resident at once).
//
// One call adds up to two doubles over all workgroups and is a barrier at the
// same time: each workgroup publishes its sums as the data of a slot, every
// workgroup reads all slots and adds them in the same order, and a slot that
// still holds kSlotEmpty has not arrived. So one store and one load travel
// through memory per call; a counter and a release flag would take two round
// trips. Three sets of slots take turns: once a workgroup has seen all sums
// of call e, every workgroup has finished reading those of call e - 1, and
// it empties its slots of that set, which call e + 2 uses.
//
// Every workgroup publishes into kSlotReplicas copies of the slots (far enough
// apart for other memory channels) and polls the copy of its own XCD: with one
// copy all workgroups poll the same few lines, and a call over 256 workgroups
// took 3.0-3.4 us instead of 2.0 (8 copies; 32 copies 2.3; 16 workgroups
// 1.55, 64 workgroups 1.7 us).
//
// Memory: the slots, and all data that other workgroups read after a call, are
// written with store_shared and read with load_shared: agent scope, past the
// caches of the CU and the XCD, so neither a write-back of the L2 before the
// call (2.4 us) nor an invalidation after it (0.7 us, and it throws out what
// the other workgroups of the XCD still use) is needed. Every wave waits for
// its stores before its workgroup publishes.
//
// Every wait ends: after spin_limit polls (kSpinLimit: at a round trip to memory
// each about 0.1 s, several times the longest launch) the call gives up and returns
// false, and the kernel returns without a result. A workgroup is late by so much
// only where something else holds its CU, for which a solve in separate launches
// need not wait.
#pragma once

#include "common.hpp"
#include "persist_plan.hpp"

namespace {

constexpr uint32_t kGridThreads = kPersistThreads;
constexpr uint32_t kGridWaves = kGridThreads / 64;
constexpr uint32_t kSlotWgs = kPersistWgs;
constexpr uint32_t kSlotReplicas = 8;
constexpr uint32_t kSlotSet = 2 * kSlotWgs;                // two sums per workgroup
constexpr uint32_t kSlotStride = 3 * kSlotSet + 544;       // words between copies: other channels
constexpr size_t kSlotWords = size_t(kSlotReplicas) * kSlotStride;
constexpr unsigned long long kSlotEmpty = 0x7FF8DEADBEEF0001ull;  // a NaN no arithmetic produces
constexpr unsigned long long kSlotNan = 0x7FF8000000000000ull;
constexpr int kSpinLimit = 1 << 17;

struct GridShared
{
    double w[kGridWaves][2];
    double tot[2];
    int ok;
};

template <typename T>
__device__ __forceinline__ void store_shared(T* p, T v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The value at element i of the buffer rs (n values of T), 0 past its end.
template <typename T>
__device__ __forceinline__ T load_shared(__amdgpu_buffer_rsrc_t rs, uint32_t i, uint32_t n)
{
    constexpr int kAgent = 16;  // the sc1 bit: agent scope
    const uint32_t at = i < n ? i * static_cast<uint32_t>(sizeof(T)) : 0xFFFFFFFFu;
    if constexpr (sizeof(T) == 4)
        return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, at, 0, kAgent));
    else
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rs, at, 0, kAgent));
}

// v[0..NV) summed over all threads of all workgroups (NV = 0: a barrier only);
// wg: this workgroup's place in the sums (each of 0..gridDim.x - 1 once).
template <int NV>
__device__ __forceinline__ bool grid_sum(unsigned long long* slots, uint32_t wg, uint32_t& epoch, double (&v)[2],
                                         GridShared& sh, int spin_limit)
{
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const double s = wave_sum(v[j]);
        if (lane == 0) sh.w[wave][j] = s;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's shared stores have arrived
    __syncthreads();
    const uint32_t g = gridDim.x;
    if (wave == 0) {
        constexpr uint32_t kVals = NV == 0 ? 1 : NV;
        const uint32_t cur = (epoch % 3) * kSlotSet, old = ((epoch + 2) % 3) * kSlotSet;
        const uint32_t rep = lane % kSlotReplicas, j = lane / kSlotReplicas;
        bool ok = true;
        double mine = 0.0;
        if (NV > 0 && j < kVals)
#pragma unroll
            for (uint32_t w = 0; w < kGridWaves; ++w) mine += sh.w[w][j];
        if (g > 1) {
            if (j < kVals) {
                unsigned long long bits = __double_as_longlong(mine);
                if (mine != mine) bits = kSlotNan;
                store_shared(slots + rep * kSlotStride + cur + j * kSlotWgs + wg, bits);
            }
            const unsigned long long* my = slots + (blockIdx.x % kSlotReplicas) * kSlotStride + cur;
            unsigned long long s[kVals][kSlotWgs / 64];
            int spin = 0;
            do {
                ok = true;
#pragma unroll
                for (uint32_t q = 0; q < kVals; ++q)
#pragma unroll
                    for (uint32_t u = 0; u < kSlotWgs / 64; ++u) {
                        const uint32_t i = lane + 64 * u;
                        s[q][u] = i < g ? __hip_atomic_load(my + q * kSlotWgs + i, __ATOMIC_RELAXED,
                                                            __HIP_MEMORY_SCOPE_AGENT)
                                        : 0ull;
                    }
#pragma unroll
                for (uint32_t q = 0; q < kVals; ++q)
#pragma unroll
                    for (uint32_t u = 0; u < kSlotWgs / 64; ++u) ok = ok && s[q][u] != kSlotEmpty;
            } while (!ok && ++spin < spin_limit);
#pragma unroll
            for (uint32_t q = 0; q < kVals; ++q) {
                double a = 0.0;
#pragma unroll
                for (uint32_t u = 0; u < kSlotWgs / 64; ++u) a += __longlong_as_double(s[q][u]);
                a = wave_sum(a);
                if (lane == 0) sh.tot[q] = a;
            }
            if (j < 2) store_shared(slots + rep * kSlotStride + old + j * kSlotWgs + wg, kSlotEmpty);
        } else if (rep == 0 && j < kVals) {
            sh.tot[j] = mine;
        }
        const bool good = __all(ok);
        if (lane == 0) sh.ok = good ? 1 : 0;
    }
    __syncthreads();
    ++epoch;
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = sh.tot[j];
    return sh.ok != 0;
}

}  // namespace
