// dyc_kernels.hip -- gfx950 kernels of the DyCuckoo hot path.
//
// Wave64 mapping shared by find, erase and update ("probe" kernels): a wave owns a tile of 64
// consecutive keys; lane i loads key i (one coalesced 256 B read) and hashes it, and each quad of
// lanes reads its four keys' buckets (probe_tile). pos2 is read only for keys pos1 did not
// resolve, in the reference order (cuckoo.cu:482-497).
//
// Insert: each lane carries one entry through the eviction chain, its bucket read by the quad as
// in a probe. Lanes are independent: one that finishes takes its next key while the rest of the
// wave keeps kicking, so no lane idles behind a long chain.
#include "dyc_kernels.hpp"
#include "dyc_wave.hpp"

#include <algorithm>

namespace dyc {

namespace {


// Plain (non-atomic) read of two consecutive slots.
__device__ inline void load_slots(const uint64_t *p, uint64_t (&e)[2])
{
    const uint4 v = *reinterpret_cast<const uint4 *>(p);
    e[0] = ((uint64_t)v.y << 32) | v.x;
    e[1] = ((uint64_t)v.w << 32) | v.z;
}

// An input word (key or value). COH: read device-coherently, for a launch that outlives the
// caller's writes to its inputs (a buffer read earlier in the launch may be rewritten and
// handed in again, and this XCD's L2 may still hold the old line).
template <bool COH>
__device__ inline uint32_t load_in(const uint32_t *p)
{
    if constexpr (COH)
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else
        return *p;
}

// A result word or flag. COH: a system-scope store, which leaves no dirty line in this XCD's
// L2, so a launch that keeps running can publish results by waiting for its stores to complete
// (publish_wait) instead of writing the whole L2 back.
template <bool COH, typename T>
__device__ inline void store_out(T *p, T v)
{
    if constexpr (COH)
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    else
        *p = v;
}

// Wait until this wave's earlier memory operations have completed; the compiler keeps memory
// accesses on their side of it. Used after system-scope stores and atomics only, which need no
// cache write-back to be seen by other agents.
__device__ inline void publish_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }


// ---------------------------------------------------------------- find / erase / update
// The probe tile: 64 keys a wave, four lanes a bucket (32 bytes each). Small probes are a chain of
// latencies and probes of lines in the caches come near the rate at which the SIMDs issue, so the
// tile is built to need few instructions:
//   * each lane finds its own key's two bucket addresses once; the quad's lanes take them, and
//     the key, by quad permutes (DPP), which ride on the instruction that uses the result, where a
//     wider group needs an LDS permute with an address of its own;
//   * hit masks are wave masks in scalar registers: which quads have resolved key kk, which lane
//     answers, and the flags are scalar arithmetic;
//   * the values of the quad's four keys are combined by an OR over the quad that leaves key kk's
//     in lane kk (a matching lane holds the value, the others 0), nine instructions for all four.
// Against the same probe with 8 lanes a bucket, LDS permutes and vector hit masks (1178 vector
// instructions a tile, 411 here), a find of 2^10 keys takes 3.5 us (5.9), of 2^17 keys in a table
// of 2^23 5.2 us (7.6), of 2^23 keys 252 us (258: bound by the rate of random lines, 54 G/s), and
// with 16 lanes 8.9, 10.8 and 316 us; so every probe takes this tile, whatever lanes per key the
// caller set.
// A lane's four slots (32 bytes) of a bucket. COH: read device-coherently (agent-scope relaxed
// atomic loads, which skip lines another XCD's writes may have left stale in this XCD's L2), for
// reads that must see exchanges made earlier in the same launch by other waves.
struct QuadSlots {
    u32x4 a, b;
};
template <bool COH>
__device__ inline QuadSlots load_quad_slots(uint32_t lo, uint32_t hi)
{
    const uint64_t at = (uint64_t)hi << 32 | lo;
    QuadSlots e;
    if constexpr (COH) {
        const DYC_GLOBAL uint64_t *p = (const DYC_GLOBAL uint64_t *)at;
        uint64_t x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = __hip_atomic_load(p + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        e.a = u32x4{(uint32_t)x[0], (uint32_t)(x[0] >> 32), (uint32_t)x[1], (uint32_t)(x[1] >> 32)};
        e.b = u32x4{(uint32_t)x[2], (uint32_t)(x[2] >> 32), (uint32_t)x[3], (uint32_t)(x[3] >> 32)};
    } else {
        const DYC_GLOBAL u32x4 *p = (const DYC_GLOBAL u32x4 *)at;
        e.a = p[0];
        e.b = p[1];
    }
    return e;
}
__device__ inline bool slots_hold(const QuadSlots &e, uint32_t k)
{
    return (e.a.y == k) | (e.a.w == k) | (e.b.y == k) | (e.b.w == k);
}
// The value of the first of the lane's slots that holds k, or 0.
__device__ inline uint32_t slots_value(const QuadSlots &e, uint32_t k)
{
    uint32_t v = e.b.w == k ? e.b.z : 0u;
    v = e.b.y == k ? e.b.x : v;
    v = e.a.w == k ? e.a.z : v;
    return e.a.y == k ? e.a.x : v;
}

// Byte offset in the lane's part of the first of its slots that holds k (the last one if none).
__device__ inline uint32_t slots_at(const QuadSlots &e, uint32_t k)
{
    uint32_t o = e.b.y == k ? 16u : 24u;
    o = e.a.w == k ? 8u : o;
    return e.a.y == k ? 0u : o;
}
// Whether two or more of the lane's slots hold k (copies of one key).
__device__ inline bool slots_hold_two(const QuadSlots &e, uint32_t k)
{
    const bool a = e.a.y == k, b = e.a.w == k, c = e.b.y == k, d = e.b.w == k;
    return (a & b) | (c & d) | ((a | b) & (c | d));
}

// One wave probes the 64 keys keys[base, base + 64) clipped to n, in table D. Returns this
// lane's flag for its own key (hit, deleted or updated); all 64 lanes must call it together.
// The first bucket (pos1, then pos2) that holds a key answers. MODE 0 find: vals (optional)
// receives the value of its first matching slot. MODE 1 erase: every copy in that bucket is CAS'd
// to empty, so one of two identical requests deletes a copy. MODE 2 update: those copies are
// CAS'd to the new value vals[i] (an input). The bucket is known once both reads are back, so
// erase and update issue the CASes of all four keys together, after them. COH: read the buckets
// and the inputs device-coherently and write the results with system-scope stores
// (load_quad_slots, load_in, store_out).
template <int MODE, bool COH = false>
__device__ inline uint32_t probe_tile(const Desc &D, const uint32_t *__restrict__ keys, uint32_t *__restrict__ vals,
                                      uint8_t *__restrict__ flags, uint64_t base, uint64_t n)
{
    constexpr bool UPDATE = MODE == 2;
    const uint32_t lane = __lane_id(), s = lane & 3u;
    const uint64_t i = base + lane;
    const bool inb = i < n;
    const uint32_t k = inb ? load_in<COH>(keys + i) : 0u;  // past the end: key 0, which is reserved
    const uint32_t nv = (UPDATE && inb) ? load_in<COH>(vals + i) : 0u;
    const uint32_t p = pair_of(D, k);
    const uint64_t a1 = (uint64_t)bucket_ptr(D, k, pos1(D, p)), a2 = (uint64_t)bucket_ptr(D, k, pos2(D, p));
    // reserved keys read the buckets their hash names like any other and are masked out here
    const uint64_t valid = __ballot(inb && !reserved_key(k));
    const uint32_t off = s * 32u;  // buckets are 128-byte aligned: the lane's part is an OR away
    uint32_t key[4];
    QuadSlots e[4];
    each_of_quad([&](auto q) {
        constexpr int kk = decltype(q)::value;
        key[kk] = quad_bcast<kk>(k);
        e[kk] = load_quad_slots<COH>(quad_bcast<kk>((uint32_t)a1) | off, quad_bcast<kk>((uint32_t)(a1 >> 32)));
    });
    uint64_t done[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) done[kk] = quad_any(__ballot(slots_hold(e[kk], key[kk])));
    // pos2 of the keys pos1 did not resolve; the others keep what they matched
    each_of_quad([&](auto q) {
        constexpr int kk = decltype(q)::value;
        const uint32_t lo = quad_bcast<kk>((uint32_t)a2) | off, hi = quad_bcast<kk>((uint32_t)(a2 >> 32));
        if (!__builtin_amdgcn_inverse_ballot_w64(done[kk])) e[kk] = load_quad_slots<COH>(lo, hi);
    });
    uint32_t v[4];
    uint64_t found = 0;
    if constexpr (MODE == 0) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
            const uint64_t m = __ballot(slots_hold(e[kk], key[kk])), any = quad_any(m);
            v[kk] = first_of_quad(m, any, slots_value(e[kk], key[kk]));
            found |= any & (kQuadLow << kk);
        }
    } else {
        uint64_t got[4];
        uint64_t m[4];
        each_of_quad([&](auto q) {
            constexpr int kk = decltype(q)::value;
            const bool first = __builtin_amdgcn_inverse_ballot_w64(done[kk]);
            v[kk] = slots_value(e[kk], key[kk]);
            const uint32_t lo1 = quad_bcast<kk>((uint32_t)a1), hi1 = quad_bcast<kk>((uint32_t)(a1 >> 32));
            const uint32_t lo2 = quad_bcast<kk>((uint32_t)a2), hi2 = quad_bcast<kk>((uint32_t)(a2 >> 32));
            const uint32_t new_v = UPDATE ? quad_bcast<kk>(nv) : 0u;
            m[kk] = __ballot(slots_hold(e[kk], key[kk])) & quad_of_key(valid, kk);
            const uint64_t at = (uint64_t)(first ? hi1 : hi2) << 32 | ((first ? lo1 : lo2) | off | slots_at(e[kk], key[kk]));
            got[kk] = 0;
            if (__builtin_amdgcn_inverse_ballot_w64(m[kk]))
                got[kk] = cas_old((DYC_GLOBAL uint64_t *)at, pack(key[kk], v[kk]), UPDATE ? pack(key[kk], new_v) : 0ull);
        });
        // The compiler would otherwise turn got == expected into the CAS's own success flag and
        // test it (waiting for the CAS) before the next one issues; an empty asm hides the relation.
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) asm volatile("" : "+v"(got[kk]));
        each_of_quad([&](auto q) {
            constexpr int kk = decltype(q)::value;
            uint64_t ok = __ballot(got[kk] == pack(key[kk], v[kk])) & m[kk];
            // copies of one key in several of a lane's slots: the rest, one at a time (uniform, rare)
            if (__ballot(slots_hold_two(e[kk], key[kk])) & m[kk]) {
                const bool first = __builtin_amdgcn_inverse_ballot_w64(done[kk]);
                const uint32_t lo1 = quad_bcast<kk>((uint32_t)a1), hi1 = quad_bcast<kk>((uint32_t)(a1 >> 32));
                const uint32_t lo2 = quad_bcast<kk>((uint32_t)a2), hi2 = quad_bcast<kk>((uint32_t)(a2 >> 32));
                const uint32_t new_v = UPDATE ? quad_bcast<kk>(nv) : 0u;
                const uint64_t at = (uint64_t)(first ? hi1 : hi2) << 32 | ((first ? lo1 : lo2) | off);
                const uint32_t sk[4] = {e[kk].a.y, e[kk].a.w, e[kk].b.y, e[kk].b.w};
                const uint32_t sv[4] = {e[kk].a.x, e[kk].a.z, e[kk].b.x, e[kk].b.z};
                bool more = false, seen = false;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (sk[j] != key[kk] || !__builtin_amdgcn_inverse_ballot_w64(m[kk])) continue;
                    if (seen) {
                        const uint64_t x = pack(sk[j], sv[j]);
                        more |= cas_old((DYC_GLOBAL uint64_t *)(at + 8 * j), x, UPDATE ? pack(key[kk], new_v) : 0ull) == x;
                    }
                    seen = true;
                }
                ok |= __ballot(more);
            }
            found |= quad_any(ok) & (kQuadLow << kk);
        });
    }
    found &= valid;
    const bool hit = __builtin_amdgcn_inverse_ballot_w64(found);
    if constexpr (MODE == 0) {
        const uint32_t my = quad_gather_or(v, s);
        if (inb && vals) store_out<COH>(vals + i, hit ? my : 0u);
    }
    if (inb && flags) store_out<COH>(flags + i, (uint8_t)hit);
    return hit;
}

// The find of a table that keeps a first-bucket rule (FirstBucket): a stored key is in its first
// bucket, or that bucket had no free slot when the key went elsewhere and none since. So a first
// bucket with a free slot answers alone, hit or miss, and a lookup reads fewer buckets: at fill 0.9
// and 50 % hits 1.40 of them (1.68 in the reference order) over a bulk-filled table. The answer
// is the reference order's: a key whose first bucket is pos2 and full may have a copy in pos1,
// which then counts. 2^28 uniform lookups 10.2 -> 8.65 ms, Zipf 4.65 -> 4.28 ms.
// The keys and results of so many lookups are used once and would push table lines out of L2, so
// their accesses are nontemporal: both finds together 12.98 -> 12.86 ms. (Small calls keep the
// ordinary ones: what follows may still find their lines in L2.)
__device__ inline uint32_t find_tile_first(const Desc &D, FirstBucket rule, const uint32_t *__restrict__ keys,
                                           uint32_t *__restrict__ vals, uint8_t *__restrict__ flags, uint64_t base,
                                           uint64_t n)
{
    const uint32_t lane = __lane_id(), s = lane & 3u;
    const uint64_t i = base + lane;
    const bool inb = i < n;
    const uint32_t k = inb ? __builtin_nontemporal_load(keys + i) : 0u;
    const uint32_t p = pair_of(D, k), ta = pos1(D, p), tb = pos2(D, p);
    const bool from2 = rule == FirstBucket::kFill ? fill_target(D, k, p) == tb : (k & 1u);
    const uint64_t a1 = (uint64_t)bucket_ptr(D, k, from2 ? tb : ta), a2 = (uint64_t)bucket_ptr(D, k, from2 ? ta : tb);
    const uint64_t second = __ballot(from2);
    const uint32_t off = s * 32u;
    uint32_t key[4], v[4];
    QuadSlots e[4];
    each_of_quad([&](auto q) {
        constexpr int kk = decltype(q)::value;
        key[kk] = quad_bcast<kk>(k);
        e[kk] = load_quad_slots<false>(quad_bcast<kk>((uint32_t)a1) | off, quad_bcast<kk>((uint32_t)(a1 >> 32)));
    });
    uint64_t any[4], more[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
        const uint64_t m = __ballot(slots_hold(e[kk], key[kk]));
        any[kk] = quad_any(m);
        v[kk] = first_of_quad(m, any[kk], slots_value(e[kk], key[kk]));
        const uint64_t open = quad_any(__ballot(slots_hold(e[kk], 0u)));
        more[kk] = ~open & (~any[kk] | quad_of_key(second, kk));
    }
    each_of_quad([&](auto q) {
        constexpr int kk = decltype(q)::value;
        const uint32_t lo = quad_bcast<kk>((uint32_t)a2) | off, hi = quad_bcast<kk>((uint32_t)(a2 >> 32));
        if (__builtin_amdgcn_inverse_ballot_w64(more[kk])) e[kk] = load_quad_slots<false>(lo, hi);
    });
    uint64_t found = 0;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
        const uint64_t m = __ballot(slots_hold(e[kk], key[kk])) & more[kk], there = quad_any(m);
        const uint32_t v2 = first_of_quad(m, there, slots_value(e[kk], key[kk]));
        if (__builtin_amdgcn_inverse_ballot_w64(there)) v[kk] = v2;
        found |= (any[kk] | there) & (kQuadLow << kk);
    }
    found &= __ballot(inb && !reserved_key(k));
    const bool hit = __builtin_amdgcn_inverse_ballot_w64(found);
    const uint32_t my = quad_gather_or(v, s);
    if (inb && vals) __builtin_nontemporal_store(hit ? my : 0u, vals + i);
    if (inb && flags) __builtin_nontemporal_store((uint8_t)hit, flags + i);
    return hit;
}

template <int MODE, bool COH = false>
__device__ inline uint32_t pool_probe_at(const Pool &pool, uint64_t np, const uint32_t *keys, uint32_t *vals,
                                         uint8_t *flags, uint64_t n, uint32_t table, uint64_t base, uint32_t f);

// Live entries of a pool (0 for Pool{}: a table without one).
__device__ inline uint64_t pool_size(const Pool &pool)
{
    if (!pool.count) return pool.n < pool.cap ? pool.n : pool.cap;
    const unsigned long long pc = __hip_atomic_load(pool.count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return pc < pool.cap ? pc : pool.cap;
}

// Misses also look in the pool's entries of `table` (a serving table's overflow pool, a single
// table's stash); an empty pool costs nothing.
template <int MODE>
__global__ __launch_bounds__(256) void probe_kernel(Desc D, const uint32_t *__restrict__ keys,
                                                    uint32_t *__restrict__ vals, uint8_t *__restrict__ flags,
                                                    uint64_t n, Counters *__restrict__ C, Pool pool, uint32_t table)
{
    const uint64_t waves = (uint64_t)gridDim.x * (blockDim.x / kWave);
    const uint64_t np = pool_size(pool);
    unsigned long long nhit = 0;
    const uint32_t slot = wave_slot();
    for (uint64_t base = (uint64_t)slot * kWave; base < n; base += waves * kWave) {
        uint32_t f = probe_tile<MODE>(D, keys, vals, flags, base, n);
        if (np) f |= pool_probe_at<MODE>(pool, np, keys, vals, flags, n, table, base, f);
        nhit += f;
    }
    if constexpr (MODE == 1) wave_tally(C, &C->deleted, nhit, slot);
    if constexpr (MODE == 2) wave_tally(C, &C->updated, nhit, slot);
}

__global__ __launch_bounds__(256) void find_first_kernel(Desc D, FirstBucket rule, const uint32_t *__restrict__ keys,
                                                         uint32_t *__restrict__ vals, uint8_t *__restrict__ flags,
                                                         uint64_t n, Pool pool, uint32_t table)
{
    const uint64_t waves = (uint64_t)gridDim.x * (blockDim.x / kWave);
    const uint64_t np = pool_size(pool);
    for (uint64_t base = (uint64_t)wave_slot() * kWave; base < n; base += waves * kWave) {
        const uint32_t f = find_tile_first(D, rule, keys, vals, flags, base, n);
        if (np) (void)pool_probe_at<0>(pool, np, keys, vals, flags, n, table, base, f);
    }
}

// ------------------------------------------------------------------------------- insert
// One lane per in-hand entry, four lanes per bucket read. Per iteration (cuckoo.cu:377-421):
//   t = the other subtable of the entry's pair relative to the previous one; read the bucket;
//   an empty slot takes the entry by CAS; a full bucket gives up a victim: in the first kick_bound
//   iterations the first slot whose resident's pair index differs from t (cuckoo.cu:398-400), else
//   slot (iteration & 15); after them rescue_lane(). The entry is exchanged with the victim, which
//   is carried on (the chain is done if the slot turned out empty).
// With kick_bound 0 (no iteration follows the reference rule) a fresh key whose first bucket is
// full tries the other bucket of its pair before it evicts: at fill 0.8 that saves 0.2 of 1.25
// exchanges a key, and exchanges are what a large insert waits for (18-20 G/s).
// The quad's lanes read the buckets of its four entries as the probe tile does (32 bytes each), so
// a bucket costs two cache accesses a lane and a step about 250 vector instructions; one lane
// reading its whole bucket took eight accesses, each a line of its own, and held its 16 slots in
// registers.
// The buckets are read with plain vector loads. The view may be stale (another XCD's L2 may hold
// a newer line), but no entry is lost or doubled by it: an empty slot is taken by CAS, and a slot
// lost to another entry is not tried again (BucketTries; the bucket is read again, and the view
// may still show the slot empty), so a bucket costs at most 16 lost races and an entry at most
// max_retries before it is pended; a victim is exchanged, which cannot fail.
//
// Input is taken in chunks of 64 indexes: wave w owns chunks w, w + W, w + 2W, ..., loads the next
// one ahead into a register a lane, and hands its entries to idle lanes by ballot rank as they free
// up, so no lane waits for the slowest chain of its wave. Resident waves sweep the input front to
// back together; when the batch was ordered by bucket region (launch_partition), the window they
// work on touches one region's buckets at a time.
struct Hand {
    uint32_t k, v;
    uint64_t idx;  // input index of the key that started the chain
    uint32_t pre, kicks, retries;
    BucketTries tries;  // in the current bucket
    bool fresh;     // not placed or carried yet: its other bucket is still to be tried
    bool active;
};

// A wave's tallies: the counts are wave-uniform, the longest chain is the lane's own.
struct InsertTally {
    unsigned long long kicks = 0, rejected = 0, retries = 0;
    unsigned long long empty = 0;  // zero entries skipped by a from-entries insert
    unsigned long long direct = 0;  // chains that ended with their first exchange
    uint32_t max_chain = 0;
};

// A chain ended (its entry placed or parked): record it for the input index that started it.
__device__ inline void chain_end(Hand &h, const PendSink &sink, InsertTally &tally)
{
    tally.max_chain = tally.max_chain > h.kicks ? tally.max_chain : h.kicks;
    if (sink.chain) sink.chain[h.idx] = h.kicks;
    h.active = false;
}

// Park the in-hand entry on the pending list.
__device__ inline void give_up(Hand &h, Counters *C, const PendSink &sink, uint32_t tag, InsertTally &tally)
{
    chain_end(h, sink, tally);
    const unsigned long long at = atomicAdd(&C->pending, 1ull);
    if (at < sink.cap) {
        sink.pend[at] = pack(h.k, h.v);
        if (sink.tags) sink.tags[at] = tag;
        // rare: publish the entry to every XCD (a serving tick's later finds read the pool
        // within the same launch)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    } else {
        atomicAdd(&C->lost, 1ull);
    }
}

// The slot the reference vote gives up of a full bucket at `at` in subtable t: the first whose
// resident's pair index differs from t. Its slots 0..3 are keys k4 (the quad's first lane read
// them); five in six of them qualify at four subtables, so the others are rarely looked at.
__device__ inline uint32_t vote_slot(const Desc &D, const uint32_t (&k4)[4], uint64_t at, uint32_t t, uint32_t kicks,
                                     bool wanted)
{
    uint32_t slot = kSlots;
#pragma unroll
    for (int j = 3; j >= 0; --j)
        if (vote_victim(D, k4[j], t)) slot = (uint32_t)j;
    const DYC_GLOBAL uint32_t *words = (const DYC_GLOBAL uint32_t *)at;
    for (uint32_t j = 4; j < (uint32_t)kSlots; ++j) {
        if (!__ballot(wanted && slot == (uint32_t)kSlots)) break;
        if (wanted && slot == (uint32_t)kSlots && vote_victim(D, words[2 * j + 1], t)) slot = j;
    }
    return slot < (uint32_t)kSlots ? slot : (kicks & 15u);
}

// At most this many buckets: a wave's lanes meet in one bucket often (64 lanes over 128 buckets: 24
// of them share one) and the insert ranks them. Above it the ranking costs every step 60
// instructions for little (64 over 1024: 4 lanes).
constexpr uint32_t kCrowdedBuckets = 1024;

// A number that tells the buckets of a crowded table apart (12 bits). Lanes of two buckets that share a
// number are ranked together and may pass over an empty slot, which stays open to them. (The first
// subtable stands for all in the choice of crowded tables. Resizes keep subtables within a factor of
// two; loaded images need not, and then more buckets share a number.)
__device__ inline uint32_t bucket_id(const Desc &D, uint64_t at, uint32_t t)
{
    const uint64_t base = (uint64_t)selt(t, D.sub);
    return (t << 9) | ((uint32_t)((at - base) / kBucketBytes) & 511u);
}

// How many lower lanes of `act` hold the same 12-bit number.
__device__ inline uint32_t rank_among_equals(uint64_t act, uint32_t id)
{
    uint64_t same = act;
#pragma unroll
    for (int b = 0; b < 12; ++b) {
        const bool bit = (id >> b) & 1u;
        const uint64_t m = __ballot(bit);
        same &= bit ? m : ~m;
    }
    return (uint32_t)__popcll(same & lanemask_lt());
}

// One eviction-chain iteration of every active lane; all 64 lanes call it together.
__device__ inline void insert_step(const Desc &D, Hand &h, const InsertPolicy &P, Counters *C, const PendSink &sink,
                                   uint32_t tag, InsertTally &tally)
{
    const uint32_t s = __lane_id() & 3u;
    const uint64_t act = __ballot(h.active);
    const uint32_t p = pair_of(D, h.k), ta = pos1(D, p), tb = pos2(D, p);
    const uint32_t t = h.pre == ta || h.pre == kOddStart ? tb : ta;
    const uint64_t at = (uint64_t)bucket_ptr(D, h.k, t);
    const uint32_t off = s * 32u;
    QuadSlots e[4];
    each_of_quad([&](auto q) {
        constexpr int kk = decltype(q)::value;
        const uint32_t lo = quad_bcast<kk>((uint32_t)at) | off, hi = quad_bcast<kk>((uint32_t)(at >> 32));
        const uint64_t low = (act >> kk) & kQuadLow;
        if (__builtin_amdgcn_inverse_ballot_w64((low << 4) - low)) e[kk] = load_quad_slots<false>(lo, hi);
        else e[kk].a = e[kk].b = u32x4{0u, 0u, 0u, 0u};
    });
    // the empty slots of the quad's four buckets, bucket kk's 16-bit mask in lane kk
    uint32_t c[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
        c[kk] = ((e[kk].a.y == 0u ? 1u : 0u) | (e[kk].a.w == 0u ? 2u : 0u) | (e[kk].b.y == 0u ? 4u : 0u) |
                 (e[kk].b.w == 0u ? 8u : 0u))
                << (4u * s);
    const bool odd = s & 1u, high = s & 2u;
    const uint32_t c01 = (odd ? c[1] : c[0]) | quad_swap<1>(odd ? c[0] : c[1]);
    const uint32_t c23 = (odd ? c[3] : c[2]) | quad_swap<1>(odd ? c[2] : c[3]);
    const uint32_t open = h.tries.open((high ? c23 : c01) | quad_swap<2>(high ? c01 : c23));
    const bool full = open == 0u;
    uint32_t slot = BucketTries::aim(open, 0u);
    if (D.nb[0] * D.d <= kCrowdedBuckets) {
        // a table of few buckets: several lanes of the wave want the same bucket's first empty slot,
        // and all but one would lose it; the r-th of them takes the r-th empty slot
        slot = BucketTries::aim(open, rank_among_equals(act, bucket_id(D, at, t)));
    }
    const bool place = h.active && !full;
    const bool swing = h.active && full && h.fresh && P.kick_bound == 0;
    const bool evict = h.active && full && !swing;
    if (__ballot(evict)) {
        uint32_t victim = rescue_lane(h.k, h.kicks);
        const bool vote = evict && h.kicks < P.kick_bound;
        if (__ballot(vote)) {
            uint32_t k4[4];
            auto first_lane = [&](auto get) {  // bucket kk's word from the quad's lane 0, in lane kk
                const uint32_t x0 = quad_bcast<0>(get(e[0])), x1 = quad_bcast<0>(get(e[1]));
                const uint32_t x2 = quad_bcast<0>(get(e[2])), x3 = quad_bcast<0>(get(e[3]));
                return high ? (odd ? x3 : x2) : (odd ? x1 : x0);
            };
            k4[0] = first_lane([](const QuadSlots &x) { return x.a.y; });
            k4[1] = first_lane([](const QuadSlots &x) { return x.a.w; });
            k4[2] = first_lane([](const QuadSlots &x) { return x.b.y; });
            k4[3] = first_lane([](const QuadSlots &x) { return x.b.w; });
            const uint32_t vs = vote_slot(D, k4, at, t, h.kicks, vote);
            victim = vote ? vs : victim;
        }
        slot = evict ? victim : slot;
    }
    DYC_GLOBAL uint64_t *const dst = (DYC_GLOBAL uint64_t *)(at + 8u * (slot & 15u));
    const uint64_t mine = pack(h.k, h.v);
    uint64_t was = 0, out = 0;
    if (place) was = cas_old(dst, 0ull, mine);
    if (evict) out = __hip_atomic_exchange(dst, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool lost = place && was != 0;
    const uint64_t won = __ballot((place && !lost) || evict);
    tally.kicks += __popcll(won);
    tally.direct += __popcll(won & __ballot(h.kicks == 0 && out == 0));
    if (__builtin_amdgcn_inverse_ballot_w64(won)) {
        ++h.kicks;
        if (out == 0) {
            chain_end(h, sink, tally);
        } else {
            h.k = key_of(out);
            h.v = val_of(out);
            h.pre = t;
            h.fresh = false;
            h.tries = {};
            if (h.kicks >= P.kick_bound + P.rescue_kicks) give_up(h, C, sink, tag, tally);
        }
    }
    if (swing) {  // its other bucket next, with nothing exchanged
        h.pre = t;
        h.fresh = false;
        h.tries = {};
    }
    const uint64_t losers = __ballot(lost);
    if (losers) {
        tally.retries += __popcll(losers);
        if (lost) {
            h.tries.lose(slot);
            if (++h.retries > P.max_retries) give_up(h, C, sink, tag, tally);
        }
    }
}

// A wave's way through its input. Input is keys/vals[i], or packed entries[i] (FROM_ENTRIES; a zero
// entry is an empty place). run() inserts the indexes of chunks first, first + stride, ... of 64
// within [begin, end) and returns when every chain has ended; the lanes are idle before and after.
// COH: read the inputs device-coherently (load_in).
template <bool FROM_ENTRIES, bool COH = false>
struct InsertRange {
    const uint32_t *keys, *vals;
    const uint64_t *entries;
    const uint8_t *skip;  // keys: skip[i] != 0 leaves key i out. entries: tile flags (see insert_kernel)
    uint32_t pre_fixed;   // entries: previous table of every entry, kNoTable (the start rule) or kAfterFill
    unsigned long long taken = 0;  // indexes taken in (wave-uniform)

    // input i of the lane (key 0 for an index left out)
    __device__ void load(uint64_t i, bool in, uint32_t &k, uint32_t &v, bool &left_out) const
    {
        k = v = 0;
        left_out = false;
        if (!in) return;
        if constexpr (FROM_ENTRIES) {
            const uint64_t e = entries[i];
            k = key_of(e);
            v = val_of(e);
            left_out = e == 0;
        } else {
            k = load_in<COH>(keys + i);
            v = load_in<COH>(vals + i);
            left_out = skip && skip[i];
        }
    }

    __device__ void run(const Desc &D, uint64_t begin, uint64_t end, uint64_t first, uint64_t stride,
                        const InsertPolicy &P, Counters *C, const PendSink &sink, uint32_t tag, InsertTally &tally)
    {
        const uint32_t lane = __lane_id();
        Hand h{};
        uint32_t bk = 0, bv = 0;        // the chunk being handed out
        uint64_t base = 0;              // its first index
        uint32_t pos = 0, len = 0;      // handed out up to pos of len
        uint32_t nk = 0, nv = 0;        // the chunk loaded ahead
        bool nleft = false;
        uint64_t nbase = begin + first * kWave;
        auto fetch = [&]() {
            if constexpr (FROM_ENTRIES) {
                // a residual list's dead tiles (skip flag 0, a chunk lies inside one tile): find
                // the next live chunk 64 at a time
                while (skip && nbase < end) {
                    const uint64_t b = nbase + (uint64_t)lane * stride * kWave;
                    const uint64_t live = __ballot(b < end && skip[b / kResTileEntries]);
                    if (live) {
                        nbase += (uint64_t)__builtin_ctzll(live) * stride * kWave;
                        break;
                    }
                    nbase += (uint64_t)kWave * stride * kWave;
                }
            }
            load(nbase + lane, nbase + lane < end, nk, nv, nleft);
        };
        if (nbase < end) fetch();
        while (true) {
            while (true) {  // hand entries to idle lanes
                if (pos == len) {
                    if (nbase >= end) break;
                    base = nbase;
                    len = end - base < kWave ? (uint32_t)(end - base) : (uint32_t)kWave;
                    pos = 0;
                    taken += len;
                    bk = nk;
                    bv = nv;
                    const uint64_t left = __ballot(lane < len && nleft);
                    if constexpr (FROM_ENTRIES) tally.empty += __popcll(left);
                    const bool bad = lane < len && !nleft && reserved_key(bk);
                    tally.rejected += __popcll(__ballot(bad));
                    if (sink.chain && lane < len && (nleft || bad)) sink.chain[base + lane] = 0;
                    if (nleft || bad) bk = 0;
                    nbase += stride * kWave;
                    if (nbase < end) fetch();
                }
                const uint64_t idle = __ballot(!h.active);
                if (!idle) break;
                const uint32_t room = (uint32_t)__popcll(idle);
                const uint32_t take = len - pos < room ? len - pos : room;
                const uint32_t rank = (uint32_t)__popcll(idle & lanemask_lt());
                const uint32_t src = (pos + rank) & 63u;
                const uint32_t k = __shfl(bk, src), v = __shfl(bv, src);
                if (!h.active && rank < take && k != 0u) {
                    h.k = k;
                    h.v = v;
                    h.idx = base + src;
                    h.pre = pre_fixed == kAfterFill ? fill_target(D, k, pair_of(D, k)) : pre_fixed;
                    h.fresh = pre_fixed == kNoTable;
                    if (h.fresh && (k & 1u)) h.pre = kOddStart;
                    h.kicks = h.retries = 0;
                    h.tries = {};
                    h.active = true;
                }
                pos += take;
            }
            if (!__ballot(h.active)) break;  // input used up and every lane idle
            insert_step(D, h, P, C, sink, tag, tally);
        }
    }
};

// The wave's tallies into its stripe.
__device__ inline void tally_out(Counters *C, const InsertTally &tally)
{
    const uint32_t slot = wave_slot();
    if (__lane_id() == 0) {
        if (tally.kicks) tally_add(C, &C->kicks, tally.kicks, slot);
        if (tally.rejected) tally_add(C, &C->rejected, tally.rejected, slot);
        if (tally.retries) tally_add(C, &C->retries, tally.retries, slot);
    }
}

// skip (optional): a keys insert leaves out key i where skip[i] != 0; an entries insert reads it
// as the tile flags of a slot-addressed residual list (entries of a tile flagged 0 are empty).
// n_dev (optional): the input ends at *n_dev if that is less than n.
template <bool FROM_ENTRIES>
__global__ __launch_bounds__(256) void insert_kernel(Desc D, const uint32_t *__restrict__ keys,
                                                     const uint32_t *__restrict__ vals,
                                                     const uint64_t *__restrict__ entries, uint64_t n,
                                                     uint32_t pre_fixed, InsertPolicy P, Counters *__restrict__ C,
                                                     PendSink sink, const uint8_t *__restrict__ skip,
                                                     const unsigned long long *__restrict__ n_dev)
{
    static_assert(kResTileEntries % kWave == 0, "a chunk lies inside one residual tile");
    InsertTally tally;
    if (n_dev) n = min((unsigned long long)n, *n_dev);
    InsertRange<FROM_ENTRIES> in{keys, vals, entries, skip, pre_fixed};
    in.run(D, 0, n, wave_slot(), (uint64_t)gridDim.x * (blockDim.x / kWave), P, C, sink, sink.tag, tally);
    if (FROM_ENTRIES && pre_fixed == kAfterFill && __lane_id() == 0 && in.taken > tally.direct)
        tally_add(C, &C->left, in.taken - tally.direct, wave_slot());
    if (sink.count_placed || sink.rejected_at) {
        const unsigned long long skipped = tally.rejected + tally.empty;
        if (__lane_id() == 0) {
            if (sink.count_placed && in.taken > skipped)
                tally_add(C, &C->placed, in.taken - skipped, wave_slot());
            if (sink.rejected_at && tally.rejected) atomicAdd(sink.rejected_at, tally.rejected);
        }
    }
    tally_out(C, tally);
    wave_tally_max(C, &C->max_chain, tally.max_chain);
}

// -------------------------------------------------------------------------- partition
// Orders an insert batch by the region of each key's first bucket (first_region), so that the
// queue-driven insert kernel places one region's keys at a time. Three kernels: a histogram of
// regions (LDS counters per block), an exclusive scan into per-region write cursors, and a
// scatter. The scatter stages each tile of kTile keys in LDS sorted by region (a counting sort:
// LDS histogram, block scan, rank by LDS atomic), claims one global range per region present in
// the tile, and writes each region's run contiguously -- the only LDS use on the insert path is
// this staging of the batch's hashed keys.
constexpr int kPartThreads = 256;
constexpr int kPartPer = 8;
constexpr int kTile = kPartThreads * kPartPer;

__global__ __launch_bounds__(kPartThreads) void partition_count_kernel(Desc D, Regions M,
                                                                       const uint32_t *__restrict__ keys, uint64_t n,
                                                                       unsigned long long *__restrict__ counts)
{
    __shared__ unsigned int hist[kMaxRegions];
    for (uint32_t r = threadIdx.x; r < M.R; r += blockDim.x) hist[r] = 0;
    __syncthreads();
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        atomicAdd(&hist[first_region(D, M, keys[i])], 1u);
    __syncthreads();
    for (uint32_t r = threadIdx.x; r < M.R; r += blockDim.x)
        if (hist[r]) atomicAdd(&counts[r], (unsigned long long)hist[r]);
}

__global__ void partition_scan_kernel(const unsigned long long *__restrict__ counts,
                                      unsigned long long *__restrict__ cursors, uint32_t R)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        unsigned long long acc = 0;
        for (uint32_t r = 0; r < R; ++r) {
            cursors[r] = acc;
            acc += counts[r];
        }
    }
}

__global__ __launch_bounds__(kPartThreads) void partition_scatter_kernel(Desc D, Regions M,
                                                                         const uint32_t *__restrict__ keys,
                                                                         const uint32_t *__restrict__ vals, uint64_t n,
                                                                         unsigned long long *__restrict__ cursors,
                                                                         uint64_t *__restrict__ out)
{
    __shared__ uint64_t stage[kTile];
    __shared__ unsigned short stage_r[kTile];
    __shared__ unsigned int hist[kMaxRegions];
    __shared__ unsigned int lbase[kMaxRegions];
    __shared__ unsigned long long gbase[kMaxRegions];
    __shared__ unsigned int wsum[kPartThreads / kWave];
    const uint32_t R = M.R;
    constexpr uint32_t kPerThread = (kMaxRegions + kPartThreads - 1) / kPartThreads;  // regions per thread in the scan

    for (uint64_t base = (uint64_t)blockIdx.x * kTile; base < n; base += (uint64_t)gridDim.x * kTile) {
        for (uint32_t r = threadIdx.x; r < R; r += kPartThreads) hist[r] = 0;
        __syncthreads();
        uint64_t e[kPartPer];
        uint32_t reg[kPartPer], rank[kPartPer];
#pragma unroll
        for (int j = 0; j < kPartPer; ++j) {
            const uint64_t i = base + (uint64_t)j * kPartThreads + threadIdx.x;
            reg[j] = 0xffffffffu;
            if (i < n) {
                const uint32_t k = keys[i];
                e[j] = pack(k, vals[i]);
                reg[j] = first_region(D, M, k);
                rank[j] = atomicAdd(&hist[reg[j]], 1u);
            }
        }
        __syncthreads();
        // block-wide exclusive scan of hist[0, R): each thread sums kPerThread consecutive
        // regions, the wave scans those sums with shuffles, the waves combine through LDS
        uint32_t mine[kPerThread];
        uint32_t sum = 0;
#pragma unroll
        for (uint32_t q = 0; q < kPerThread; ++q) {
            const uint32_t r = threadIdx.x * kPerThread + q;
            mine[q] = r < R ? hist[r] : 0u;
            sum += mine[q];
        }
        uint32_t incl = sum;
#pragma unroll
        for (int off = 1; off < kWave; off <<= 1) {
            const uint32_t up = __shfl_up(incl, off);
            if (__lane_id() >= off) incl += up;
        }
        if (__lane_id() == kWave - 1) wsum[threadIdx.x / kWave] = incl;
        __syncthreads();
        uint32_t wbase = 0;
        for (uint32_t w = 0; w < threadIdx.x / kWave; ++w) wbase += wsum[w];
        uint32_t run = wbase + incl - sum;
#pragma unroll
        for (uint32_t q = 0; q < kPerThread; ++q) {
            const uint32_t r = threadIdx.x * kPerThread + q;
            if (r < R) {
                lbase[r] = run;
                if (mine[q]) gbase[r] = atomicAdd(&cursors[r], (unsigned long long)mine[q]);
            }
            run += mine[q];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kPartPer; ++j)
            if (reg[j] != 0xffffffffu) {
                const uint32_t at = lbase[reg[j]] + rank[j];
                stage[at] = e[j];
                stage_r[at] = (unsigned short)reg[j];
            }
        __syncthreads();
        const uint64_t cnt = n - base < (uint64_t)kTile ? n - base : (uint64_t)kTile;
        for (uint32_t at = threadIdx.x; at < cnt; at += kPartThreads) {
            const uint32_t r = stage_r[at];
            out[gbase[r] + (at - lbase[r])] = stage[at];
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------- upsize
// cuckoo.cu:600-627: slot i of old bucket j goes to slot i of new bucket h % 2n, which is j or
// j + n. Each group of 8 lanes writes both destination buckets in full (entry or zero), so the
// new subtable needs no separate clearing pass: 8 B read + 16 B written per old slot.
__global__ __launch_bounds__(256) void upsize_kernel(const uint64_t *__restrict__ old, uint32_t old_nb,
                                                     uint64_t *__restrict__ dst, uint32_t t, uint32_t m,
                                                     uint32_t s1, uint32_t s2, Counters *__restrict__ C)
{
    constexpr int G = 8, NG = kWave / G;
    const int lane = __lane_id();
    const int g = lane / G, s = lane % G;
    const uint64_t waves = (uint64_t)gridDim.x * (blockDim.x / kWave);
    const uint32_t nnb = old_nb * 2u;
    unsigned long long bad = 0;
    for (uint64_t tile = ((uint64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave) * NG; tile < old_nb;
         tile += waves * NG) {
        const uint64_t j = tile + g;
        if (j >= old_nb) continue;
        uint64_t e[2];
        load_slots(old + j * kSlots + s * 2, e);
        uint64_t lo[2], hi[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            lo[q] = hi[q] = 0;
            if (e[q]) {
                const uint32_t d = fast_mod(hash_t(key_of(e[q]), t), nnb, m, s1, s2);
                if (d == j)
                    lo[q] = e[q];
                else if (d == j + old_nb)
                    hi[q] = e[q];
                else
                    ++bad;
            }
        }
        *reinterpret_cast<uint4 *>(dst + j * kSlots + s * 2) =
            make_uint4((uint32_t)lo[0], (uint32_t)(lo[0] >> 32), (uint32_t)lo[1], (uint32_t)(lo[1] >> 32));
        *reinterpret_cast<uint4 *>(dst + (j + old_nb) * kSlots + s * 2) =
            make_uint4((uint32_t)hi[0], (uint32_t)(hi[0] >> 32), (uint32_t)hi[1], (uint32_t)(hi[1] >> 32));
    }
    wave_tally(C, &C->misplaced, bad);
}

// ----------------------------------------------------------------------------- downsize
// cuckoo.cu:664-699: new bucket g keeps old bucket g slot-for-slot and fills its empty slots
// from old bucket g+n read back to front (slot i <- slot 15-i). Lane s of a group holds slots
// 2s, 2s+1; their cross partners 15-2s, 14-2s are the two halves of lane 7-s's 16 bytes.
// An entry of bucket g+n that found no hole is a residual. res is slot-addressed: the residual
// from slot i of new bucket g's partner goes to res[g * 16 + i], 0 where there is none, so no
// wave reserves list space (an append index is one address, and atomics to one address are
// serialized: one per wave cost 0.9 ms on a 582,560-bucket downsize). A wave compacts a tile of
// kResTileBuckets buckets; live[tile] says whether it left any residual, and only such tiles
// write their kResTileEntries list entries, so a nearly full table writes almost no list. The
// caller re-inserts the list (launch_insert_entries with live) only after this kernel has
// finished (no race with the plain stores here). Counters::residuals receives their number.
__global__ __launch_bounds__(256) void downsize_kernel(const uint64_t *__restrict__ old, uint32_t new_nb,
                                                       uint64_t *__restrict__ dst, Counters *__restrict__ C,
                                                       uint64_t *__restrict__ res, uint8_t *__restrict__ live)
{
    static_assert(kWave / 8 == (int)kResTileBuckets, "a wave compacts one liveness tile");
    constexpr int G = 8, NG = kWave / G;
    const int lane = __lane_id();
    const int g = lane / G, s = lane % G;
    const uint64_t waves = (uint64_t)gridDim.x * (blockDim.x / kWave);
    const uint32_t slot = wave_slot();
    unsigned long long nres = 0;
    for (uint64_t tile = (uint64_t)slot * NG; tile < new_nb; tile += waves * NG) {
        const uint64_t j = tile + g;
        const bool ok = j < new_nb;
        uint64_t e[2] = {0, 0}, c[2] = {0, 0};
        if (ok) {
            load_slots(old + j * kSlots + s * 2, e);
            uint64_t x[2];
            load_slots(old + (j + new_nb) * kSlots + (7 - s) * 2, x);
            c[0] = x[1];  // slot 15-2s
            c[1] = x[0];  // slot 14-2s
        }
        uint64_t placed[2], r[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            placed[q] = e[q] ? e[q] : c[q];
            r[q] = (placed[q] != c[q] && c[q] != 0) ? c[q] : 0;
            nres += r[q] != 0;
        }
        if (ok)
            *reinterpret_cast<uint4 *>(dst + j * kSlots + s * 2) =
                make_uint4((uint32_t)placed[0], (uint32_t)(placed[0] >> 32), (uint32_t)placed[1],
                           (uint32_t)(placed[1] >> 32));
        const bool any = __ballot(r[0] != 0 || r[1] != 0) != 0;  // wave-uniform
        if (lane == 0) live[tile / NG] = any ? 1 : 0;
        if (any && ok)
            *reinterpret_cast<uint4 *>(res + j * kSlots + s * 2) =
                make_uint4((uint32_t)r[0], (uint32_t)(r[0] >> 32), (uint32_t)r[1], (uint32_t)(r[1] >> 32));
    }
    wave_tally(C, &C->residuals, nres, slot);
}

// Buckets a find reads per key (0 for reserved keys): in the reference order 1 if pos1 holds the key, else
// 2; under a first-bucket rule as find_tile_first. first_hits: keys that the first bucket read holds.
// One thread per key; a diagnostic pass, not on the hot path.
__global__ __launch_bounds__(256) void probe_count_kernel(Desc D, FirstBucket rule, const uint32_t *__restrict__ keys,
                                                          uint64_t n, Counters *__restrict__ C)
{
    unsigned long long probes = 0, first_hits = 0;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const uint32_t k = keys[i];
        if (reserved_key(k)) continue;
        const uint32_t p = pair_of(D, k), tb = pos2(D, p);
        const bool from2 = rule != FirstBucket::kNone &&
                           (rule == FirstBucket::kFill ? fill_target(D, k, p) == tb : (k & 1u) != 0);
        const uint64_t *b = bucket_ptr(D, k, from2 ? tb : pos1(D, p));
        bool hit = false, open = false;
        for (int j = 0; j < kSlots; ++j) {
            hit |= key_of(b[j]) == k;
            open |= key_of(b[j]) == 0;
        }
        probes += (rule != FirstBucket::kNone && open) || (hit && !from2) ? 1 : 2;
        first_hits += hit;
    }
    wave_tally(C, &C->kicks, probes);
    wave_tally(C, &C->occupied, first_hits);
}

// ---------------------------------------------------------------------------- many tables
// One persistent launch serves a batch spread over many tables. The batch is cut into items of
// at most a few thousand keys of one table; wave w takes items w, w + W, w + 2W, ... and loads
// the item's table descriptor from the directory with scalar loads (the item index is
// wave-uniform), so the per-tile code is the single-table code with a different Desc.
__device__ inline uint32_t wave_uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// The kGroupWaves waves of a workgroup share its items: wave w takes the tiles (64 keys) t of the
// workgroup's r-th item with t % kGroupWaves == (w - r) % kGroupWaves, without waiting for the others;
// turning by r spreads items of one tile over the waves. The keys that the waves of an XCD work on
// at a time then span few tables, and its L2 holds their lines: with a whole 4096-key item per
// wave, 2048 tables of 2^8..2^18 keys (77 M lookups) took 1897 us, 80 % of the lines missing L2;
// shared by eight waves 1250 us. Small batches gain too: a table of 200 keys is four tiles at
// once, not in turn.
constexpr int kGroupWaves = kProbeWavesPerBlock;
constexpr int kGroupThreads = kGroupWaves * kWave;

// This wave's first tile of its workgroup's r-th item.
__device__ inline uint32_t group_first_tile(uint32_t r)
{
    return (wave_uniform(threadIdx.x / kWave) - r) % (uint32_t)kGroupWaves;
}

// W: the least waves per SIMD the compiler must leave room for (1: its own choice); the group
// launches take it as an occupancy knob, chosen by measurement.
// MODE 0 find, 1 erase, 3 find of tables that keep a first-bucket rule.
template <int MODE, int W>
__global__ __launch_bounds__(kGroupThreads, W) void group_probe_kernel(const Desc *__restrict__ dir,
                                                          const GroupItem *__restrict__ items, uint32_t n_items,
                                                          const uint32_t *__restrict__ keys,
                                                          uint32_t *__restrict__ vals, uint8_t *__restrict__ flags,
                                                          unsigned long long *__restrict__ table_counts, Pool pool,
                                                          FirstBucket rule)
{
    const uint64_t np = pool_size(pool);
    uint32_t r = 0;
    for (uint32_t it = blockIdx.x; it < n_items; it += gridDim.x, ++r) {
        const GroupItem item = items[it];
        const uint32_t first = group_first_tile(r) * kWave;
        if (first >= item.len) continue;  // wave-uniform: none of its tiles (or an empty slot of a layout by XCD)
        const Desc D = as_global(dir[item.table]);
        const uint64_t end = item.begin + item.len;
        unsigned long long nd = 0;
        for (uint64_t base = item.begin + first; base < end; base += kGroupThreads) {
            uint32_t f;
            if constexpr (MODE == 3) f = find_tile_first(D, rule, keys, vals, flags, base, end);
            else f = probe_tile<MODE>(D, keys, vals, flags, base, end);
            if (np) f |= pool_probe_at<MODE == 1 ? 1 : 0>(pool, np, keys, vals, flags, end, item.table, base, f);
            nd += f;
        }
        if constexpr (MODE == 1) {
            nd = wave_sum(nd);
            if (__lane_id() == 0 && nd) atomicAdd(&table_counts[item.table], nd);
        }
    }
}

// shared: the waves of a workgroup share its items as in the probe, chunk by chunk; else each wave takes
// items of its own (group_insert_item_keys says when). A wave moves on only when all its lanes have
// placed (or pended) their entries.
template <int W>
__global__ __launch_bounds__(kGroupThreads, W) void group_insert_kernel(const Desc *__restrict__ dir,
                                                           const GroupItem *__restrict__ items, uint32_t n_items,
                                                           const uint32_t *__restrict__ keys,
                                                           const uint32_t *__restrict__ vals, InsertPolicy P,
                                                           Counters *__restrict__ C, PendSink sink,
                                                           unsigned long long *__restrict__ table_counts,
                                                           bool shared)
{
    InsertTally tally;
    uint32_t r = 0;
    const uint32_t step = shared ? gridDim.x : gridDim.x * kGroupWaves;
    for (uint32_t it = shared ? blockIdx.x : wave_slot(); it < n_items; it += step, ++r) {
        const GroupItem item = items[it];
        const uint32_t first = shared ? group_first_tile(r) : 0u;
        if (first * kWave >= item.len) continue;  // wave-uniform
        const Desc D = as_global(dir[item.table]);
        const unsigned long long rej0 = tally.rejected;
        InsertRange<false> in{keys, vals, nullptr, nullptr, kNoTable};
        in.run(D, item.begin, item.begin + item.len, first, shared ? kGroupWaves : 1, P, C, sink, item.table, tally);
        const unsigned long long rej = tally.rejected - rej0;
        if (__lane_id() == 0 && in.taken > rej) atomicAdd(&table_counts[item.table], in.taken - rej);
    }
    tally_out(C, tally);
}

// The overflow of a group's bulk fill: small items, each one wave's; there are *n_dev of them if
// that is less than n_items.
__global__ __launch_bounds__(256) void group_overflow_kernel(const Desc *__restrict__ dir,
                                                             const GroupItem *__restrict__ items, uint32_t n_items,
                                                             const unsigned long long *__restrict__ n_dev,
                                                             const uint64_t *__restrict__ ovf, InsertPolicy P,
                                                             Counters *__restrict__ C, PendSink sink,
                                                             unsigned long long *__restrict__ table_counts)
{
    InsertTally tally;
    unsigned long long taken = 0;
    n_items = (uint32_t)min((unsigned long long)n_items, *n_dev);
    const uint32_t waves = gridDim.x * (blockDim.x / kWave);
    for (uint32_t it = wave_slot(); it < n_items; it += waves) {
        const GroupItem item = items[it];
        const Desc D = as_global(dir[item.table]);
        InsertRange<true> in{nullptr, nullptr, ovf, nullptr, kAfterFill};
        in.run(D, item.begin, item.begin + item.len, 0, 1, P, C, sink, item.table, tally);
        taken += in.taken;
        if (__lane_id() == 0) atomicAdd(&table_counts[item.table], (unsigned long long)item.len);
    }
    if (__lane_id() == 0 && taken > tally.direct) tally_add(C, &C->left, taken - tally.direct, wave_slot());
    tally_out(C, tally);
}

// ------------------------------------------------------------------------------ serving
// Items of a serving tick carry their request's own pointers; otherwise the tile code is the
// single-table code. Finds and erases that miss both buckets also look in the server's pool of
// entries that exhausted the eviction bound (normally empty: one scalar load per tile).

// The pool search of one tile's lanes whose key missed both buckets (f = 0). The pool counts as
// one more bucket after pos2. MODE 0 find: vals receives the first matching entry's value.
// MODE 1 erase: every copy is CAS'd to 0. MODE 2 update: every copy is CAS'd to the new value
// vals[i] (an input). Returns this lane's flag, also written to flags when set.
template <int MODE, bool COH>
__device__ inline uint32_t pool_probe_at(const Pool &pool, uint64_t np, const uint32_t *keys, uint32_t *vals,
                                         uint8_t *flags, uint64_t n, uint32_t table, uint64_t base, uint32_t f)
{
    const uint64_t i = base + __lane_id();
    if (i >= n || f) return 0;
    const uint32_t k = keys[i];
    if (reserved_key(k)) return 0;
    const uint32_t nv = MODE == 2 ? vals[i] : 0u;
    uint32_t got = 0;
    for (uint64_t j = 0; j < np; ++j) {
        const uint64_t e = __hip_atomic_load(pool.pend + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (key_of(e) != k ||
            (pool.tags && __hip_atomic_load(pool.tags + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != table))
            continue;
        if constexpr (MODE != 0) {
            uint64_t exp = e;
            got |= (uint32_t)cas_slot(pool.pend + j, exp, MODE == 2 ? pack(k, nv) : 0ull);
        } else {
            if (vals) store_out<COH>(vals + i, val_of(e));
            got = 1;
            break;
        }
    }
    if (got && flags) store_out<COH>(flags + i, (uint8_t)1);
    return got;
}

template <bool ERASE, bool COH = false>
__device__ inline uint32_t pool_probe(const Pool &pool, uint64_t np, const ServeItem &item, uint64_t base, uint32_t f)
{
    return pool_probe_at<ERASE ? 1 : 0, COH>(pool, np, item.keys, item.out_vals, item.flags, item.len, item.table, base,
                                             f);
}

// One item of finds or erases; returns this lane's count of hits (erase: deletions).
template <bool ERASE, bool COH = false>
__device__ inline unsigned long long serve_probe_item(const Desc &D, const ServeItem &item, const Pool &pool,
                                                      uint64_t np)
{
    unsigned long long nd = 0;
    for (uint64_t base = 0; base < item.len; base += kWave) {
        uint32_t f = probe_tile<ERASE ? 1 : 0, COH>(D, item.keys, ERASE ? nullptr : item.out_vals, item.flags, base,
                                                    item.len);
        if (np) f |= pool_probe<ERASE, COH>(pool, np, item, base, f);
        nd += f;
    }
    return nd;
}

// One item of inserts. COH: read the inputs device-coherently (load_in).
template <bool COH = false>
__device__ inline unsigned long long serve_insert_item(const Desc &D, const ServeItem &item, const InsertPolicy &P,
                                                       Counters *C, const PendSink &sink, InsertTally &tally)
{
    const unsigned long long rej0 = tally.rejected;
    InsertRange<false, COH> in{item.keys, item.vals, nullptr, nullptr, kNoTable};
    in.run(D, 0, item.len, 0, 1, P, C, sink, item.table, tally);
    const unsigned long long rej = tally.rejected - rej0;
    return item.len > rej ? item.len - rej : 0;  // entries the item took in (wave-uniform)
}

// A wave's running total for one table, added to that table's word when the wave moves on to
// another table and at the end. Items of one table come in runs, and an atomic per item put
// every item of a busy table on one address (atomics to one address are serialized).
struct WaveTotal {
    uint32_t table = ~0u;
    unsigned long long n = 0;
    __device__ void add(unsigned long long *totals, uint32_t t, unsigned long long v)  // v wave-uniform
    {
        if (t != table) {
            flush(totals);
            table = t;
        }
        n += v;
    }
    __device__ void flush(unsigned long long *totals)
    {
        if (__lane_id() == 0 && table != ~0u && n) atomicAdd(&totals[table], n);
        n = 0;
    }
};


template <bool ERASE>
__global__ __launch_bounds__(256) void serve_probe_kernel(const Desc *__restrict__ dir,
                                                          const ServeItem *__restrict__ items, uint32_t n_items,
                                                          Pool pool, unsigned long long *__restrict__ del_total)
{
    const uint32_t waves = gridDim.x * (blockDim.x / kWave);
    const uint64_t np = pool_size(pool);
    WaveTotal del;
    for (uint32_t it = wave_uniform(blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave); it < n_items;
         it += waves) {
        const ServeItem item = as_global(items[it]);
        const Desc D = as_global(dir[item.table]);
        unsigned long long nd = serve_probe_item<ERASE>(D, item, pool, np);
        if constexpr (ERASE) del.add(del_total, item.table, wave_sum(nd));
    }
    if constexpr (ERASE) del.flush(del_total);
}

__global__ __launch_bounds__(256) void serve_insert_kernel(const Desc *__restrict__ dir,
                                                           const ServeItem *__restrict__ items, uint32_t n_items,
                                                           InsertPolicy P, Counters *__restrict__ C, PendSink sink,
                                                           unsigned long long *__restrict__ ins_total)
{
    InsertTally tally;
    WaveTotal ins;
    const uint32_t waves = gridDim.x * (blockDim.x / kWave);
    for (uint32_t it = wave_uniform(blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave); it < n_items;
         it += waves) {
        const ServeItem item = as_global(items[it]);
        ins.add(ins_total, item.table, serve_insert_item(as_global(dir[item.table]), item, P, C, sink, tally));
    }
    ins.flush(ins_total);
    tally_out(C, tally);
}

// A whole serving tick in one launch. Waves claim items in list order from a counter; an item
// whose stage has a predecessor (the same table's previous round or phase) first waits for the
// stage's ready flag; when a stage's last item finishes it raises the flag of the table's next
// stage. No acquire/release fences: on this chip an agent-scope fence writes back or
// invalidates the whole L2 of the XCD. Table changes are 64-bit exchanges (device-coherent, and
// their results are consumed before the stage count drops), and finds and erases read buckets
// with coherent loads. Items wait only on items earlier in the list, which were claimed by
// running waves, so the earliest unfinished item never waits and the launch always drains. The
// wait is bounded all the same: past spin_cap polls the wave records a stall and goes on (the
// host reports the tick failed).
__global__ __launch_bounds__(256) void serve_tick_kernel(const Desc *__restrict__ dir, const TickItem *__restrict__ items,
                                                         uint32_t n_items, unsigned long long *__restrict__ cursor,
                                                         TickStages stages, InsertPolicy P, Counters *__restrict__ C,
                                                         PendSink sink, Pool pool,
                                                         unsigned long long *__restrict__ ins_total,
                                                         unsigned long long *__restrict__ del_total, uint32_t spin_cap,
                                                         uint32_t max_back)
{
    InsertTally tally;
    WaveTotal ins, del;
    unsigned long long stalls = 0;
    while (true) {
        uint32_t it = 0;
        if (__lane_id() == 0) it = (uint32_t)atomicAdd(cursor, 1ull);
        it = wave_uniform(it);
        if (it >= n_items) break;
        TickItem ti = items[it];
        ti.item = as_global(ti.item);
        if (ti.wait) {
            uint32_t ok = 1;
            if (__lane_id() == 0) {
                uint32_t spins = 0, back = 1;
                const uint32_t *flag = stages.ready + (uint64_t)ti.stage * kReadyStride;
                while (__hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
                    for (uint32_t b = 0; b < back; ++b) __builtin_amdgcn_s_sleep(4);
                    back = back < max_back ? back * 2 : max_back;
                    if (++spins > spin_cap) {
                        ok = 0;
                        break;
                    }
                }
            }
            if (!wave_uniform(ok)) ++stalls;
        }
        const Desc D = as_global(dir[ti.item.table]);
        if (ti.op == 0) {
            ins.add(ins_total, ti.item.table, serve_insert_item(D, ti.item, P, C, sink, tally));
        } else {
            // an item that waited reads what earlier stages of this launch wrote: coherently;
            // a table's first stage reads what earlier launches wrote: through the caches
            unsigned long long nd;
            const uint64_t np = pool_size(pool);
            if (ti.op == 1)
                nd = ti.wait ? serve_probe_item<false, true>(D, ti.item, pool, np)
                             : serve_probe_item<false, false>(D, ti.item, pool, np);
            else
                nd = ti.wait ? serve_probe_item<true, true>(D, ti.item, pool, np)
                             : serve_probe_item<true, false>(D, ti.item, pool, np);
            if (ti.op == 2) del.add(del_total, ti.item.table, wave_sum(nd));
        }
        if (__lane_id() == 0) {
            const uint32_t before =
                __hip_atomic_fetch_sub(stages.left + ti.stage, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (before == 1) {
                const uint32_t nx = stages.next[ti.stage];
                if (nx != ~0u)
                    __hip_atomic_store(stages.ready + (uint64_t)nx * kReadyStride, 1u, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
    ins.flush(ins_total);
    del.flush(del_total);
    tally_out(C, tally);
    if (__lane_id() == 0 && stalls) tally_add(C, &C->stalls, stalls, wave_slot());
}

// ----------------------------------------------------------- device-resident serving loop
// One launch serves requests as the host publishes them (LoopItem). Wave 0 of block 0 is the
// front wave: it polls the control block in host memory and copies the published item count
// into the device word avail. Every other wave claims item indexes from the device cursor in
// order and waits, polling device memory, until its index is published. An item of a table
// whose earlier requests have not finished waits until tbl_done[table] reaches its need. Items
// wait only on items with smaller indexes, which running waves have claimed (the grid is
// resident as a whole), so the earliest unfinished item never waits and every published item
// finishes. A finished item's table writes are atomics whose results it has used: it counts
// itself into its request's progress word at once, and the wave that counts the request's last
// item advances tbl_done. Its results are system-scope stores: it waits for them, then counts
// itself into the request's output count, and the wave that counts the last item writes the
// request's record and appends the request to the completion queue in host memory.
// Every wait is bounded. The front wave ends the launch on the host's stop flag or after
// idle_ticks without new items: it raises quit, and waves waiting for an index past the
// published ones leave. An item gives up waiting for its table after spin_cap polls, or at once
// once the host has given up on the launch (stop = 2 raises abort), and counts as a stall (the
// host fails its request). A ring entry whose stamp does not match after
// spin_cap polls raises the fault flag and quit.
// Tables, inputs and the directory are read device-coherently: the launch outlives the writes
// of resizes and of the caller, and this XCD's L2 may hold lines they made stale.

__device__ inline uint64_t ld_system(const unsigned long long *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ inline uint64_t ld_agent(const unsigned long long *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline uint64_t uniform64(uint64_t v)
{
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (uint64_t)hi << 32 | lo;
}

__device__ inline void sleep_units(uint32_t n)  // n x 256 cycles
{
    for (uint32_t b = 0; b < n; ++b) __builtin_amdgcn_s_sleep(4);
}

// The W words lanes 0..W-1 hold, as one wave-uniform T.
template <int W, typename T>
__device__ inline T wave_gather(uint64_t v)
{
    static_assert(sizeof(T) == W * 8, "T is W words");
    uint64_t w[W];
#pragma unroll
    for (int j = 0; j < W; ++j) {
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, j);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), j);
        w[j] = (uint64_t)hi << 32 | lo;
    }
    T out;
    __builtin_memcpy(&out, w, sizeof(T));
    return out;
}

__device__ inline Desc load_desc_coherent(const Desc *p)
{
    constexpr int W = sizeof(Desc) / 8;
    const unsigned long long *w = reinterpret_cast<const unsigned long long *>(p);
    const uint64_t v = __lane_id() < W ? ld_agent(w + __lane_id()) : 0;
    return wave_gather<W, Desc>(v);
}

__device__ inline void loop_front(const LoopArgs &A)
{
    unsigned long long *avail = A.words + kLoopAvail;
    uint64_t seen = uniform64(ld_agent(avail));
    uint64_t last = __builtin_amdgcn_s_memrealtime();
    while (true) {
        const uint64_t t = uniform64(ld_system(&A.ctl->tail));
        const uint64_t stop = uniform64(ld_system(&A.ctl->stop));
        if (stop) {
            if (stop == 2 && __lane_id() == 0)
                __hip_atomic_store(A.words + kLoopAbort, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
        }
        const uint64_t now = __builtin_amdgcn_s_memrealtime();
        if (t != seen) {
            if (__lane_id() == 0) __hip_atomic_store(avail, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            seen = t;
            last = now;
            continue;
        }
        if (now - last > A.idle_ticks) break;
        __builtin_amdgcn_s_sleep(2);
    }
    if (__lane_id() == 0) __hip_atomic_store(A.words + kLoopQuit, 1ull, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ __launch_bounds__(256) void serve_loop_kernel(LoopArgs A, InsertPolicy P, Counters *__restrict__ C,
                                                         PendSink sink, Pool pool,
                                                         unsigned long long *__restrict__ ins_total,
                                                         unsigned long long *__restrict__ del_total)
{
    if (blockIdx.x == 0 && threadIdx.x < kWave) {
        loop_front(A);
        return;
    }
    InsertTally tally;
    WaveTotal ins, del;
    const int lane = __lane_id();
    unsigned long long *cursor = A.words + kLoopCursor, *avail = A.words + kLoopAvail, *quit = A.words + kLoopQuit;
    while (true) {
        uint64_t idx = 0;
        if (lane == 0) idx = atomicAdd(cursor, 1ull);
        idx = uniform64(idx);
        // wait until the index is published, or the launch ends
        bool go = true;
        for (uint32_t back = 1;;) {
            if (idx < uniform64(ld_agent(avail))) break;
            // the front wave stores avail before quit (a release), and this reload is issued only
            // after quit was read, so it sees the last published count
            if (uniform64(ld_agent(quit))) {
                go = idx < uniform64(ld_agent(avail));
                break;
            }
            sleep_units(back);
            back = back < A.max_back ? back * 2 : A.max_back;
        }
        if (!go) break;
        // the item, 8 words from host memory; its stamp tells that the host finished writing it
        const unsigned long long *src = reinterpret_cast<const unsigned long long *>(A.ring + (idx & A.ring_mask));
        LoopItem it;
        bool ok = false;
        for (uint32_t spins = 0; spins <= A.spin_cap; ++spins) {
            it = wave_gather<8, LoopItem>(lane < 8 ? ld_system(src + lane) : 0ull);
            if (it.stamp == (uint32_t)(idx + 1)) {
                ok = true;
                break;
            }
            sleep_units(1);
        }
        if (!ok) {
            if (lane == 0) {
                __hip_atomic_store(A.words + kLoopFault, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(quit, 1ull, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            }
            break;
        }
        it.item = as_global(it.item);
        const uint32_t table = it.item.table;
        // the descriptor can be read before the wait: a table is resized only while none of its
        // requests is in flight, and the host writes the directory before it publishes items
        const Desc D = as_global(load_desc_coherent(A.dir + table));
        uint32_t stalled = 0;
        if (it.need) {
            uint32_t back = 1, spins = 0;
            while (uniform64(ld_agent(A.tbl_done + table)) < it.need) {
                if (++spins > A.spin_cap || uniform64(ld_agent(A.words + kLoopAbort))) {
                    stalled = 1;
                    break;
                }
                sleep_units(back);
                back = back < A.max_back ? back * 2 : A.max_back;
            }
        }
        unsigned long long acc;
        if (it.op == 0) {
            acc = serve_insert_item<true>(D, it.item, P, C, sink, tally);
            ins.add(ins_total, table, acc);
        } else {
            const uint64_t np = pool_size(pool);
            if (it.op == 1) {
                acc = wave_sum(serve_probe_item<false, true>(D, it.item, pool, np));
            } else {
                acc = wave_sum(serve_probe_item<true, true>(D, it.item, pool, np));
                del.add(del_total, table, acc);
            }
        }
        // Two counts per request. The table's work of the item is done here (its exchanges and
        // erasures are atomics whose results the wave has used; a parked entry was fenced), so
        // the item counts at once towards releasing the table's next requests. Its results are
        // system-scope stores, which it waits for before counting towards the host's completion.
        if (lane == 0) {
            const unsigned long long old = atomicAdd(A.req_word + it.req, (acc << kLoopItemBits) | 1ull);
            if ((old & ((1ull << kLoopItemBits) - 1)) + 1 == it.n_items)
                atomicAdd(A.tbl_done + table, 1ull);  // the table's next requests may start
            if (stalled) atomicAdd(A.req_stall + it.req, 1u);
        }
        publish_wait();
        if (lane == 0) {
            const uint32_t done = atomicAdd(A.req_out + it.req, 1u) + 1;
            if (done == it.n_items) {
                // every item counted into req_word before it counted here
                const unsigned long long total = ld_agent(A.req_word + it.req) >> kLoopItemBits;
                const uint32_t stalls = __hip_atomic_load(A.req_stall + it.req, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(A.req_word + it.req, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(A.req_out + it.req, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(A.req_stall + it.req, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                LoopRec *r = A.rec + it.req;
                __hip_atomic_store(&r->acc, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                __hip_atomic_store(&r->pool, pool.count ? ld_agent(pool.count) : 0ull, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_SYSTEM);
                __hip_atomic_store(&r->lost, ld_agent(&C->lost), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                __hip_atomic_store(&r->stalls, stalls, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                publish_wait();  // the record is in host memory before the queue entry
                const unsigned long long pos = atomicAdd(A.words + kLoopCqTail, 1ull);
                __hip_atomic_store(A.cq + (pos & A.req_mask), ((pos + 1) << 32) | it.req, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_SYSTEM);
            }
        }
    }
    ins.flush(ins_total);
    del.flush(del_total);
    tally_out(C, tally);
}

__global__ void loop_reset_kernel(unsigned long long *words)
{
    words[kLoopCursor] = words[kLoopAvail];
    words[kLoopQuit] = 0;
    words[kLoopFault] = 0;
    words[kLoopAbort] = 0;
}

// Copy between host-pinned and device memory with a kernel instead of a DMA transfer: a
// serving tick moves a few KB each way, where queueing a copy engine costs more than the
// transfer. Up to two (src, dst, words) segments per launch.
struct CopySeg {
    const unsigned long long *src;
    unsigned long long *dst;
    uint64_t words;
};

__global__ __launch_bounds__(256) void copy_kernel(CopySeg a, CopySeg b)
{
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.words; i += stride) a.dst[i] = a.src[i];
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < b.words; i += stride) b.dst[i] = b.src[i];
}

__global__ void zero_kernel(unsigned long long *p, uint64_t words)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = 0;
}

__global__ __launch_bounds__(256) void count_kernel(const uint64_t *__restrict__ sub, uint64_t slots,
                                                    Counters *__restrict__ C)
{
    unsigned long long c = 0;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < slots; i += stride) c += sub[i] != 0;
    wave_tally(C, &C->occupied, c);
}

// Blocks for `work_waves` waves of work. A launch may not exceed 2^32 work-items in total, and
// every kernel here loops grid-stride, so the grid is capped (default_cap when the caller set
// no max_blocks); the rest of the work is taken by the resident waves as they finish.

// Waves hand their chunks' keys to lanes as these finish, and eviction chains vary in length, so a
// grid whose lanes take one key each ends on a tail of late blocks. With no grid from the caller, a lane
// gets at least kInsertKeysPerLane keys, in no fewer than kInsertFloorBlocks blocks (about what the
// device holds) and no more than kInsertDefaultBlocks. Insert into a table at fill 0.8-0.85, by grid:
// 1.7 M keys with eviction bound 15 144 us at 1024 blocks, 156 at 4096 and more (bound 0: 107, 105);
// 2^24 keys 970 us at the default 8192, 974 at 1024, 957 at 65,536 (839, 838, 822); 2^26 keys 3.18 ms at
// the default 32,768, 3.36 at 8192, 3.75 at a block for 256 keys (2.85, 2.91, 3.05). Not everywhere
// the best: 2^22 keys into an empty table take 243 us at 512 blocks, 286 at the default 2048 (302, 352).
constexpr uint64_t kInsertDefaultBlocks = 65536;
constexpr uint64_t kInsertKeysPerLane = 8;
constexpr uint64_t kInsertFloorBlocks = 1024;

inline uint64_t insert_default_cap(uint64_t work_waves, LaunchShape sh)
{
    const uint64_t wpb = (uint64_t)sh.block_threads / kWave;
    const uint64_t work_blocks = (work_waves + wpb - 1) / wpb;
    uint64_t cap = work_blocks / kInsertKeysPerLane;
    if (cap < kInsertFloorBlocks) cap = kInsertFloorBlocks;
    if (cap > kInsertDefaultBlocks) cap = kInsertDefaultBlocks;
    return cap;
}

}  // namespace

hipError_t launch_find(const Desc &D, const uint32_t *keys, uint32_t *vals, uint8_t *hit, uint64_t n, LaunchShape sh,
                       hipStream_t st, const Pool *pool, uint32_t table, FirstBucket rule)
{
    if (n == 0) return hipSuccess;
    const int grid = grid_for((n + kWave - 1) / kWave, sh);
    const Pool p = pool ? *pool : Pool{};
    if (rule != FirstBucket::kNone)
        find_first_kernel<<<grid, sh.block_threads, 0, st>>>(D, rule, keys, vals, hit, n, p, table);
    else
        probe_kernel<0><<<grid, sh.block_threads, 0, st>>>(D, keys, vals, hit, n, nullptr, p, table);
    return hipGetLastError();
}

hipError_t launch_erase(const Desc &D, const uint32_t *keys, uint8_t *deleted, uint64_t n, LaunchShape sh,
                        Counters *C, hipStream_t st, const Pool *pool, uint32_t table)
{
    if (n == 0) return hipSuccess;
    const int grid = grid_for((n + kWave - 1) / kWave, sh);
    const Pool p = pool ? *pool : Pool{};
    probe_kernel<1><<<grid, sh.block_threads, 0, st>>>(D, keys, nullptr, deleted, n, C, p, table);
    return hipGetLastError();
}

template <bool FE>
static hipError_t insert_common(const Desc &D, const uint32_t *keys, const uint32_t *vals, const uint64_t *entries,
                                uint64_t n, uint32_t pre, InsertPolicy pol, LaunchShape sh, Counters *C, PendSink sink,
                                hipStream_t st, const uint8_t *skip, const unsigned long long *n_dev = nullptr)
{
    if (n == 0) return hipSuccess;
    const uint64_t work_waves = (n + kWave - 1) / kWave;
    // Of a bulk fill's batch some 6 % overflow (10 % at fill 0.96): a grid for an eighth of it. For all of it
    // most waves found nothing, and with eviction bound 15 the crowd of short ones cost the rest: 2^28
    // keys' insert 8.4 ms instead of 9.6 (bound 0: 6.77, 6.84), 2^24 into three subtables to 0.94 0.79
    // instead of 0.94 ms (0.54, 0.56).
    const int grid = grid_for(work_waves, sh, insert_default_cap(n_dev ? work_waves / 8 : work_waves, sh));
    insert_kernel<FE><<<grid, sh.block_threads, 0, st>>>(D, keys, vals, entries, n, pre, pol, C, sink, skip, n_dev);
    return hipGetLastError();
}

hipError_t launch_insert(const Desc &D, const uint32_t *keys, const uint32_t *vals, uint64_t n, InsertPolicy pol,
                         LaunchShape sh, Counters *C, PendSink sink, hipStream_t st,
                         const uint8_t *skip)
{
    return insert_common<false>(D, keys, vals, nullptr, n, kNoTable, pol, sh, C, sink, st, skip);
}

hipError_t launch_update(const Desc &D, const uint32_t *keys, const uint32_t *vals, uint8_t *updated, uint64_t n,
                         LaunchShape sh, Counters *C, hipStream_t st, const Pool *pool)
{
    if (n == 0) return hipSuccess;
    const int grid = grid_for((n + kWave - 1) / kWave, sh);
    uint32_t *v = const_cast<uint32_t *>(vals);  // read-only in update mode
    const Pool p = pool ? *pool : Pool{};
    probe_kernel<2><<<grid, sh.block_threads, 0, st>>>(D, keys, v, updated, n, C, p, 0);
    return hipGetLastError();
}

hipError_t launch_insert_entries(const Desc &D, const uint64_t *entries, uint64_t n, uint32_t pre, InsertPolicy pol,
                                 LaunchShape sh, Counters *C, PendSink sink, hipStream_t st,
                                 const uint8_t *live)
{
    return insert_common<true>(D, nullptr, nullptr, entries, n, pre, pol, sh, C, sink, st, live);
}

hipError_t launch_insert_overflow(const Desc &D, const uint64_t *ovf, uint64_t n, InsertPolicy pol, LaunchShape sh,
                                  Counters *C, PendSink sink, hipStream_t st)
{
    return insert_common<true>(D, nullptr, nullptr, ovf, n, kAfterFill, pol, sh, C, sink, st, nullptr, &C->overflow);
}

hipError_t launch_partition(const Desc &D, const Regions &M, const uint32_t *keys, const uint32_t *vals, uint64_t n,
                            unsigned long long *counts, unsigned long long *cursors, uint64_t *out, hipStream_t st)
{
    if (n == 0) return hipSuccess;
    if (M.R == 0 || M.R > kMaxRegions) return hipErrorInvalidValue;
    uint64_t blocks = (n + kTile - 1) / kTile;
    if (blocks > 8192) blocks = 8192;
    partition_count_kernel<<<(int)blocks, kPartThreads, 0, st>>>(D, M, keys, n, counts);
    partition_scan_kernel<<<1, 64, 0, st>>>(counts, cursors, M.R);
    partition_scatter_kernel<<<(int)blocks, kPartThreads, 0, st>>>(D, M, keys, vals, n, cursors, out);
    return hipGetLastError();
}

hipError_t launch_upsize(const uint64_t *old, uint32_t old_nb, uint64_t *dst, uint32_t t, Counters *C,
                         hipStream_t st)
{
    if (old_nb == 0) return hipSuccess;
    const FastDiv f = make_fastdiv(old_nb * 2u);
    const int grid = grid_for((old_nb + 7) / 8, LaunchShape{256, 0});
    upsize_kernel<<<grid, 256, 0, st>>>(old, old_nb, dst, t, f.m, f.s1, f.s2, C);
    return hipGetLastError();
}

hipError_t launch_downsize(const uint64_t *old, uint32_t new_nb, uint64_t *dst, Counters *C, uint64_t *res,
                           uint64_t res_cap, uint8_t *live, hipStream_t st)
{
    if (new_nb == 0) return hipSuccess;
    if (res_cap < (uint64_t)new_nb * kSlots || !live) return hipErrorInvalidValue;
    const int grid = grid_for((new_nb + kResTileBuckets - 1) / kResTileBuckets, LaunchShape{256, 0});
    downsize_kernel<<<grid, 256, 0, st>>>(old, new_nb, dst, C, res, live);
    return hipGetLastError();
}

constexpr int kGroupDefaultBlocks = 2048;  // 8192 waves: 256 CUs x 32 resident waves
constexpr uint32_t kGroupInsertBlocks = 1024;  // as many waves, eight to a workgroup

template <int MODE>
static void group_probe_w(int wpe, int grid, hipStream_t st, const Desc *dir, const GroupItem *items, uint32_t n_items,
                          const uint32_t *keys, uint32_t *vals, uint8_t *flags, unsigned long long *table_counts,
                          const Pool &p, FirstBucket rule = FirstBucket::kNone)
{
    switch (wpe) {
    case 6:
        group_probe_kernel<MODE, 6>
            <<<grid, kGroupThreads, 0, st>>>(dir, items, n_items, keys, vals, flags, table_counts, p, rule);
        break;
    case 8:
        group_probe_kernel<MODE, 8>
            <<<grid, kGroupThreads, 0, st>>>(dir, items, n_items, keys, vals, flags, table_counts, p, rule);
        break;
    default:
        group_probe_kernel<MODE, 1>
            <<<grid, kGroupThreads, 0, st>>>(dir, items, n_items, keys, vals, flags, table_counts, p, rule);
        break;
    }
}

hipError_t launch_group_find(const Desc *dir, const GroupItem *items, uint32_t n_items, const uint32_t *keys,
                             uint32_t *vals, uint8_t *hit, int blocks, hipStream_t st, const Pool *pool,
                             int waves_per_eu, FirstBucket rule)
{
    const Pool p = pool ? *pool : Pool{};
    if (n_items == 0) return hipSuccess;
    const int grid = blocks > 0 ? blocks : group_probe_grid(0, n_items);
    if (rule != FirstBucket::kNone)
        group_probe_w<3>(waves_per_eu, grid, st, dir, items, n_items, keys, vals, hit, nullptr, p, rule);
    else
        group_probe_w<0>(waves_per_eu, grid, st, dir, items, n_items, keys, vals, hit, nullptr, p);
    return hipGetLastError();
}

hipError_t launch_group_erase(const Desc *dir, const GroupItem *items, uint32_t n_items, const uint32_t *keys,
                              uint8_t *deleted, unsigned long long *table_counts, int blocks,
                              hipStream_t st, const Pool *pool, int waves_per_eu)
{
    const Pool p = pool ? *pool : Pool{};
    if (n_items == 0) return hipSuccess;
    const int grid = blocks > 0 ? blocks : group_probe_grid(0, n_items);
    group_probe_w<1>(waves_per_eu, grid, st, dir, items, n_items, keys, nullptr, deleted, table_counts, p);
    return hipGetLastError();
}

hipError_t launch_group_insert(const Desc *dir, const GroupItem *items, uint32_t n_items, const uint32_t *keys,
                               const uint32_t *vals, InsertPolicy pol, int blocks, bool shared, Counters *C,
                               PendSink sink, unsigned long long *table_counts, hipStream_t st, int waves_per_eu)
{
    if (n_items == 0) return hipSuccess;
    const uint32_t most = shared ? n_items : (n_items + kGroupWaves - 1) / kGroupWaves;
    const int grid = blocks > 0 ? blocks : (int)std::min<uint32_t>(kGroupInsertBlocks, most);
    switch (waves_per_eu) {
    case 6:
        group_insert_kernel<6>
            <<<grid, kGroupThreads, 0, st>>>(dir, items, n_items, keys, vals, pol, C, sink, table_counts, shared);
        break;
    case 8:
        group_insert_kernel<8>
            <<<grid, kGroupThreads, 0, st>>>(dir, items, n_items, keys, vals, pol, C, sink, table_counts, shared);
        break;
    default:
        group_insert_kernel<1>
            <<<grid, kGroupThreads, 0, st>>>(dir, items, n_items, keys, vals, pol, C, sink, table_counts, shared);
        break;
    }
    return hipGetLastError();
}

hipError_t launch_group_insert_overflow(const Desc *dir, const GroupItem *items, const unsigned long long *n_items,
                                        uint64_t max_items, const uint64_t *ovf, InsertPolicy pol, int blocks,
                                        Counters *C, PendSink sink, unsigned long long *table_counts, hipStream_t st)
{
    if (max_items == 0) return hipSuccess;
    if (max_items > 0xffffffffull) return hipErrorInvalidValue;
    const int grid = blocks > 0 ? blocks : (int)std::min<uint64_t>(kGroupDefaultBlocks, (max_items + 3) / 4);
    group_overflow_kernel<<<grid, 256, 0, st>>>(dir, items, (uint32_t)max_items, n_items, ovf, pol, C, sink,
                                                table_counts);
    return hipGetLastError();
}

hipError_t launch_copy(const void *src0, void *dst0, uint64_t words0, const void *src1, void *dst1, uint64_t words1,
                       hipStream_t st)
{
    const uint64_t words = std::max(words0, words1);
    if (words == 0) return hipSuccess;
    uint64_t blocks = (words + 255) / 256;
    if (blocks > 256) blocks = 256;
    copy_kernel<<<(int)blocks, 256, 0, st>>>(
        CopySeg{static_cast<const unsigned long long *>(src0), static_cast<unsigned long long *>(dst0), words0},
        CopySeg{static_cast<const unsigned long long *>(src1), static_cast<unsigned long long *>(dst1), words1});
    return hipGetLastError();
}

static int serve_grid(uint32_t n_items, int blocks)
{
    return blocks > 0 ? blocks : std::min<int>(kGroupDefaultBlocks, (int)((n_items + 3) / 4));
}

hipError_t launch_serve_find(const Desc *dir, const ServeItem *items, uint32_t n_items, Pool pool, int blocks,
                             hipStream_t st)
{
    if (n_items == 0) return hipSuccess;
    const int grid = serve_grid(n_items, blocks);
    serve_probe_kernel<false><<<grid, 256, 0, st>>>(dir, items, n_items, pool, nullptr);
    return hipGetLastError();
}

hipError_t launch_serve_erase(const Desc *dir, const ServeItem *items, uint32_t n_items, Pool pool,
                              unsigned long long *del_total, int blocks, hipStream_t st)
{
    if (n_items == 0) return hipSuccess;
    const int grid = serve_grid(n_items, blocks);
    serve_probe_kernel<true><<<grid, 256, 0, st>>>(dir, items, n_items, pool, del_total);
    return hipGetLastError();
}

hipError_t launch_serve_insert(const Desc *dir, const ServeItem *items, uint32_t n_items, InsertPolicy pol, int blocks,
                               Counters *C, PendSink sink, unsigned long long *ins_total, hipStream_t st)
{
    if (n_items == 0) return hipSuccess;
    const int grid = serve_grid(n_items, blocks);
    serve_insert_kernel<<<grid, 256, 0, st>>>(dir, items, n_items, pol, C, sink, ins_total);
    return hipGetLastError();
}

// The lanes have no effect on the kernels; a server that was refused the tick or the loop for them
// still is.
bool serve_tick_supported(int insert_lanes, int find_lanes)
{
    return (insert_lanes == 1 || insert_lanes == 2 || insert_lanes == 4) &&
           (find_lanes == 4 || find_lanes == 8 || find_lanes == 16);
}

hipError_t launch_serve_tick(const Desc *dir, const TickItem *items, uint32_t n_items, unsigned long long *cursor,
                             TickStages done, InsertPolicy pol, int insert_lanes, int find_lanes, int blocks,
                             Counters *C, PendSink sink, Pool pool, unsigned long long *ins_total,
                             unsigned long long *del_total, uint32_t spin_cap, uint32_t max_back, hipStream_t st)
{
    if (n_items == 0) return hipSuccess;
    if (!serve_tick_supported(insert_lanes, find_lanes)) return hipErrorInvalidValue;
    if (max_back == 0) max_back = 1;
    const int grid = serve_grid(n_items, blocks);
    serve_tick_kernel<<<grid, 256, 0, st>>>(dir, items, n_items, cursor, done, pol, C, sink, pool, ins_total, del_total,
                                            spin_cap, max_back);
    return hipGetLastError();
}

hipError_t launch_serve_loop(const LoopArgs &A, InsertPolicy pol, int insert_lanes, int find_lanes, int blocks,
                             Counters *C, PendSink sink, Pool pool, unsigned long long *ins_total,
                             unsigned long long *del_total, hipStream_t st)
{
    if (!serve_tick_supported(insert_lanes, find_lanes) || blocks < 2) return hipErrorInvalidValue;
    serve_loop_kernel<<<blocks, 256, 0, st>>>(A, pol, C, sink, pool, ins_total, del_total);
    return hipGetLastError();
}

hipError_t launch_loop_reset(unsigned long long *words, hipStream_t st)
{
    loop_reset_kernel<<<1, 1, 0, st>>>(words);
    return hipGetLastError();
}

int serve_loop_capacity(int insert_lanes, int find_lanes)
{
    if (!serve_tick_supported(insert_lanes, find_lanes)) return 0;
    int dev = 0, cus = 0, per = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, serve_loop_kernel, 256, 0) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return per * cus;
}

hipError_t launch_zero(unsigned long long *p, uint64_t words, hipStream_t st)
{
    if (words == 0) return hipSuccess;
    uint64_t blocks = (words + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    zero_kernel<<<(int)blocks, 256, 0, st>>>(p, words);
    return hipGetLastError();
}

// One workgroup, a thread per word of every stripe: the sums take one load, two shuffles and one pass
// through LDS, where one wave walking the 64 stripes took 64 loads in turn. The zeroes and the
// words for the host are system-scope stores, complete before seq is stored, so no cache is written back.
// 4.6 -> 2.7 us.
constexpr int kFoldThreads = 16 * kTallyStripes;
__global__ __launch_bounds__(kFoldThreads) void fold_post_kernel(unsigned long long *block, unsigned long long *post,
                                                                 unsigned long long seq)
{
    constexpr int kWords = (int)(sizeof(Counters) / sizeof(unsigned long long));
    static_assert(kWords == 16 && kFoldThreads <= 1024, "16 words a stripe, one workgroup");
    __shared__ unsigned long long part[kFoldThreads / kWave][kWords];
    const int t = threadIdx.x, w = t % kWords, stripe = t / kWords;
    auto join = [&](unsigned long long a, unsigned long long b) {
        return w == kMaxChainWord ? (a > b ? a : b) : a + b;
    };
    unsigned long long *const mine = block + kTallyStrideWords * (1 + stripe) + w;
    unsigned long long v = *mine, base = 0;
    if (t < kWords) base = block[t];
    store_out<true>(mine, 0ull);
    if (t < kWords) store_out<true>(block + t, 0ull);
    v = join(v, shfl64(v, (int)__lane_id() ^ 16));
    v = join(v, shfl64(v, (int)__lane_id() ^ 32));
    if ((int)__lane_id() < kWords) part[t / kWave][w] = v;
    publish_wait();  // the block is zero before seq is posted: the next call may be on another stream
    __syncthreads();
    if (t >= kWave) return;
    if (t < kWords) {
        v = base;
#pragma unroll
        for (int q = 0; q < kFoldThreads / kWave; ++q) v = join(v, part[q][t]);
        store_out<true>(post + 1 + t, v);
    }
    publish_wait();
    if (t == 0) store_out<true>(post, seq);
}

hipError_t launch_fold_post(Counters *C, unsigned long long *post, unsigned long long seq, hipStream_t st)
{
    fold_post_kernel<<<1, kFoldThreads, 0, st>>>(reinterpret_cast<unsigned long long *>(C), post, seq);
    return hipGetLastError();
}

hipError_t launch_probe_count(const Desc &D, const uint32_t *keys, uint64_t n, Counters *C, hipStream_t st,
                              FirstBucket rule)
{
    if (n == 0) return hipSuccess;
    uint64_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    probe_count_kernel<<<(int)blocks, 256, 0, st>>>(D, rule, keys, n, C);
    return hipGetLastError();
}

hipError_t launch_count(const uint64_t *sub, uint64_t slots, Counters *C, hipStream_t st)
{
    uint64_t blocks = (slots + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    if (blocks < 1) blocks = 1;
    count_kernel<<<(int)blocks, 256, 0, st>>>(sub, slots, C);
    return hipGetLastError();
}

}  // namespace dyc
