// dyc_wave.hpp -- wave64 helpers shared by the kernel files of libdyc (internal).
#pragma once

#include <type_traits>

#include "dyc_kernels.hpp"

namespace dyc {

constexpr int kWave = 64;

__device__ inline uint64_t lanemask_lt() { return (1ull << __lane_id()) - 1ull; }

__device__ inline uint64_t shfl64(uint64_t v, int src)
{
    uint32_t lo = __shfl((uint32_t)v, src);
    uint32_t hi = __shfl((uint32_t)(v >> 32), src);
    return ((uint64_t)hi << 32) | lo;
}

// 64-bit compare-and-swap at agent scope; on failure `expected` receives the current value.
__device__ inline bool cas_slot(uint64_t *p, uint64_t &expected, uint64_t desired)
{
    return __hip_atomic_compare_exchange_strong(p, &expected, desired, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
}

// 64-bit compare-and-swap at agent scope that returns the value it found (== expected on
// success). Nothing waits for the result until the caller compares it, so several can be in flight.
template <typename Ptr>
__device__ inline uint64_t cas_old(Ptr p, uint64_t expected, uint64_t desired)
{
    __hip_atomic_compare_exchange_strong(p, &expected, desired, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
    return expected;
}

__device__ inline unsigned long long wave_sum(unsigned long long v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += (unsigned long long)shfl64(v, __lane_id() ^ off);
    return v;
}

// This wave's index in the grid, as a wave-uniform (scalar) value.
__device__ inline uint32_t wave_slot()
{
    return __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave);
}

// A wave-uniform pointer as one the compiler knows to be in global memory. A pointer in a kernel
// argument is taken to be global; one read from memory (a directory's descriptor, a chunk record,
// a work item) is generic, and accesses through it become flat ones, which count on the LDS
// counter too: the bucket loads of a group's tile then waited for the shuffles that hand out
// their addresses, one after the other. The empty asm keeps the round trip through the global
// address space from being folded away.
template <typename T>
__device__ inline T *as_global(T *p)
{
    auto q = (__attribute__((address_space(1))) T *)p;
    asm("" : "+s"(q));
    return (T *)q;
}

__device__ inline Desc as_global(Desc D)
{
#pragma unroll
    for (int t = 0; t < kMaxSubtables; ++t) D.sub[t] = as_global(D.sub[t]);
    return D;
}

__device__ inline WideDesc as_global(WideDesc W)
{
    W.D = as_global(W.D);
#pragma unroll
    for (int t = 0; t < kMaxSubtables; ++t) W.val[t] = as_global(W.val[t]);
    return W;
}

__device__ inline ServeItem as_global(ServeItem x)
{
    x.keys = as_global(x.keys);
    x.vals = as_global(x.vals);
    x.out_vals = as_global(x.out_vals);
    x.flags = as_global(x.flags);
    return x;
}

// ---- quads: four lanes share the buckets of their four keys (see the probe tile)
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#define DYC_GLOBAL __attribute__((address_space(1)))

// x of lane KK of each quad, in all of its lanes.
template <int KK>
__device__ inline uint32_t quad_bcast(uint32_t x)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, KK * 0x55, 0xf, 0xf, true);
}
// x of the quad lane whose number differs in bit 0 (XOR = 1) or bit 1 (XOR = 2).
template <int XOR>
__device__ inline uint32_t quad_swap(uint32_t x)
{
    static_assert(XOR == 1 || XOR == 2, "a quad permute");
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, XOR == 1 ? 0xb1 : 0x4e, 0xf, 0xf, true);
}

constexpr uint64_t kQuadLow = 0x1111111111111111ull;  // lane 0 of every quad
// Every lane of each quad that has a lane in m.
__device__ inline uint64_t quad_any(uint64_t m)
{
    m |= m >> 1;
    m = (m | m >> 2) & kQuadLow;
    return (m << 4) - m;
}

template <typename F>
__device__ inline void each_of_quad(F f)
{
    f(std::integral_constant<int, 0>{});
    f(std::integral_constant<int, 1>{});
    f(std::integral_constant<int, 2>{});
    f(std::integral_constant<int, 3>{});
}

// Clears v in the lanes whose slot is not the first match of its quad (copies of one key in slots of
// several lanes: uniform, rare).
__device__ inline uint32_t first_of_quad(uint64_t m, uint64_t any, uint32_t v)
{
    if (__popcll(m) * 4 != __popcll(any)) {
        const uint64_t later = ((m << 1) & ~kQuadLow) | ((m << 2) & (kQuadLow * 0xc)) | ((m << 3) & (kQuadLow * 8));
        if (__builtin_amdgcn_inverse_ballot_w64(later)) v = 0;
    }
    return v;
}

// The OR over the quad of key kk's word v[kk], in lane kk.
__device__ inline uint32_t quad_gather_or(const uint32_t (&v)[4], uint32_t s)
{
    const bool odd = s & 1u, high = s & 2u;
    const uint32_t v01 = (odd ? v[1] : v[0]) | quad_swap<1>(odd ? v[0] : v[1]);
    const uint32_t v23 = (odd ? v[3] : v[2]) | quad_swap<1>(odd ? v[2] : v[3]);
    return (high ? v23 : v01) | quad_swap<2>(high ? v01 : v23);
}

// The lanes of key kk's quads, of a mask of the keys' own lanes.
__device__ inline uint64_t quad_of_key(uint64_t own, int kk)
{
    const uint64_t low = (own >> kk) & kQuadLow;
    return (low << 4) - low;
}

// Add v (from one lane) to the tally `field` (a member of *C) in the stripe of wave slot `slot`.
__device__ inline void tally_add(Counters *C, unsigned long long *field, unsigned long long v, uint32_t slot)
{
    unsigned long long *base = reinterpret_cast<unsigned long long *>(C);
    atomicAdd(base + kTallyStrideWords * (1u + slot % kTallyStripes) + (field - base), v);
}

__device__ inline void wave_tally(Counters *C, unsigned long long *field, unsigned long long v, uint32_t slot)
{
    v = wave_sum(v);
    if (__lane_id() == 0 && v) tally_add(C, field, v, slot);
}

__device__ inline void wave_tally(Counters *C, unsigned long long *field, unsigned long long v)
{
    wave_tally(C, field, v, wave_slot());
}

// The wave's largest v into the tally `field` of the wave's stripe (a field the fold takes the
// maximum of, not the sum).
__device__ inline void wave_tally_max(Counters *C, unsigned long long *field, unsigned long long v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long x = shfl64(v, __lane_id() ^ off);
        v = v > x ? v : x;
    }
    if (__lane_id() == 0 && v) {
        unsigned long long *base = reinterpret_cast<unsigned long long *>(C);
        atomicMax(base + kTallyStrideWords * (1u + wave_slot() % kTallyStripes) + (field - base), v);
    }
}


// Blocks for work_waves waves of work under a launch shape (capped; 0 max_blocks = default_cap).
inline int grid_for(uint64_t work_waves, LaunchShape sh, uint64_t default_cap = 1ull << 20)
{
    const uint64_t wpb = (uint64_t)sh.block_threads / kWave;
    uint64_t blocks = (work_waves + wpb - 1) / wpb;
    if (blocks < 1) blocks = 1;
    const uint64_t cap = sh.max_blocks > 0 ? (uint64_t)sh.max_blocks : default_cap;
    if (blocks > cap) blocks = cap;
    const uint64_t hw_cap = ((1ull << 32) - 1) / (uint64_t)sh.block_threads;
    if (blocks > hw_cap) blocks = hw_cap;
    return (int)blocks;
}

}  // namespace dyc
