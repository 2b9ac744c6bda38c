// dyc_part.hpp -- partition of a bulk-fill batch by table chunk (internal to libdyc).
//
// The bulk fill (dyc_bulk.hip, dyc_wide.hip) needs its batch grouped by chunk: every entry of
// chunk c contiguous, and the first index of every chunk. This is a least-significant-digit
// radix partition of the entries by chunk id, at most 8 bits of the chunk id per pass:
//   pack   (in the table's source file): one pass over the batch computes every entry's chunk
//          id -- the hash is the expensive part, so it is done once -- writes the ids in input
//          order and counts the first digit per block;
//   colscan: per digit, the exclusive prefix of the per-block counts over the blocks, and the
//          digit's total;
//   scatter: each block ranks its range tile by tile (stably: by digit, then input index) and
//          writes each tile's entries to their global places, digit run by digit run, so that
//          consecutive lanes store consecutive words. The first pass reads the caller's batch
//          itself; the last writes no chunk ids;
//   count:  the next digit per block, from the chunk ids alone. Before the last pass it also
//          counts every chunk: its input is then sorted by the bits below the last digit, so a
//          block's range holds few of their values and the counts gather in LDS;
//   segment scan: the first index of every chunk from those counts.
// Blocks own fixed contiguous ranges of whole tiles, the same in every launch of a pass, so the
// prefix of block b is final before its scatter starts: no launch waits on another block.
// Chunk ids are carried as 16-bit words when the table has at most 2^16 chunks.
#pragma once

#include <algorithm>
#include <type_traits>

#include "dyc_kernels.hpp"
#include "dyc_wave.hpp"

namespace dyc {

template <int V>
using Int = std::integral_constant<int, V>;
constexpr int kSortThreads = 512;  // threads of a scatter workgroup
constexpr uint32_t kMaxRadixBits = 8;
constexpr uint32_t kMaxRadix = 1u << kMaxRadixBits;
constexpr uint32_t kMaxRadixPasses = 4;
constexpr uint32_t kMaxSortBlocks = 2048;  // colscan gives each of its 256 threads up to 8 blocks
static_assert(kPartialWords == (uint64_t)kMaxSortBlocks * kMaxRadix, "BulkSpace::partial holds every block's counts");
static_assert(kMaxRadixWords == kMaxRadix, "BulkSpace::total holds every digit's total");
// The counting launches (pack, count) stream their block's range with more waves per block
// than the scatter, whose LDS limits it to one to three blocks per CU.
constexpr int kCountThreads = 512;
constexpr int kCountItems = 8;
// Values of the bits below the last digit that one block of the last count bins in LDS; a
// block's entries beyond them (small batches) count with global atomics.
constexpr uint32_t kLowSpan = 8;

struct RadixPass {
    uint32_t shift, bits;  // digit = (cid >> shift) & ((1 << bits) - 1)
};

// Scatter block b of a pass owns tiles [b * per, (b + 1) * per) of the batch, `tile` entries each
// (the last ones may be partial or empty). The counting launches split each block's range into
// `sub` equal parts, one counting block each (their count rows b * sub + s follow the batch's
// order, so the exclusive prefix of row b * sub is scatter block b's): they need more waves than
// the scatter's LDS leaves room for.
struct PartGrid {
    uint64_t n;
    uint32_t blocks, per, tile, sub;
};
constexpr uint32_t kCountBlocks = 1024;  // counting blocks aimed for

// Workgroups of a scatter that fit a CU: its LDS holds a tile's entries, their chunk ids and, at
// most, 10 KiB of counters.
__host__ __device__ constexpr uint32_t sort_blocks_per_cu(size_t entry_bytes, int items)
{
    return std::min<uint32_t>(4, 160 * 1024 / (uint32_t)(kSortThreads * items * entry_bytes + 11 * 1024));
}

template <typename Entry, typename CidT, int ITEMS>
inline PartGrid part_grid(uint64_t n)
{
    constexpr uint32_t tile = kSortThreads * ITEMS;
    constexpr uint32_t max_blocks = 256 * sort_blocks_per_cu(sizeof(Entry) + sizeof(CidT), ITEMS);
    static_assert(max_blocks > 0 && max_blocks <= kMaxSortBlocks, "a tile fits a CU");
    const uint64_t tiles = (n + tile - 1) / tile;
    uint32_t blocks = (uint32_t)std::min<uint64_t>(std::max<uint64_t>(tiles, 1), max_blocks);
    const uint32_t per = (uint32_t)std::max<uint64_t>((tiles + blocks - 1) / blocks, 1);
    blocks = (uint32_t)std::max<uint64_t>((tiles + per - 1) / per, 1);  // no block without a tile
    uint32_t sub = std::max<uint32_t>(1, std::min(kCountBlocks, kMaxSortBlocks) / blocks);
    while (sub > 1 && (tile * per) % sub) --sub;  // equal parts
    return PartGrid{n, blocks, per, tile, sub};
}

// The digit passes of a partition over `bits` bits of chunk id: as few passes as 8-bit digits
// allow, with the bits spread evenly over them (lowest digit first). Returns the pass count.
inline uint32_t radix_passes(uint32_t bits, RadixPass *out)
{
    const uint32_t n = std::max<uint32_t>(1, (bits + kMaxRadixBits - 1) / kMaxRadixBits);
    uint32_t shift = 0;
    for (uint32_t p = 0; p < n; ++p) {
        const uint32_t b = (bits - shift + (n - p) - 1) / (n - p);
        out[p] = RadixPass{shift, std::max<uint32_t>(b, 1)};
        shift += b;
    }
    return n;
}

__device__ inline uint32_t digit_of(uint32_t cid, RadixPass P) { return (cid >> P.shift) & ((1u << P.bits) - 1u); }

// First and one past the last index of scatter block b's range.
__device__ inline uint64_t part_begin(const PartGrid &G, uint32_t b) { return (uint64_t)b * G.per * G.tile; }
__device__ inline uint64_t part_end(const PartGrid &G, uint64_t lo)
{
    const uint64_t hi = lo + (uint64_t)G.per * G.tile;
    return hi < G.n ? hi : G.n;
}
// The same for counting block q (part q % sub of scatter block q / sub).
__device__ inline uint64_t count_begin(const PartGrid &G, uint32_t q) { return (uint64_t)q * (G.per * G.tile / G.sub); }
__device__ inline uint64_t count_end(const PartGrid &G, uint64_t lo)
{
    const uint64_t hi = lo + G.per * G.tile / G.sub;
    return hi < G.n ? hi : G.n;
}

// Where a scatter pass reads its entries: an entry array, or the caller's key and value arrays
// (the first pass of an insert batch). from(i) is the source that starts at entry i.
template <typename Entry>
struct EntrySource {
    const Entry *e;
    __device__ Entry load(uint64_t i) const { return e[i]; }
    __device__ EntrySource from(uint64_t i) const { return {e + i}; }
};
struct KeyValSource {
    const uint32_t *k, *v;
    __device__ uint64_t load(uint64_t i) const { return pack(k[i], v[i]); }
    __device__ KeyValSource from(uint64_t i) const { return {k + i, v + i}; }
};
struct WideKeyValSource {
    const uint64_t *k, *v;
    __device__ WideEntry load(uint64_t i) const { return WideEntry{k[i], v[i]}; }
    __device__ WideKeyValSource from(uint64_t i) const { return {k + i, v + i}; }
};

namespace {

// Exclusive prefix sum over the block's threads (one value each, at most kScanWaves waves);
// *total receives the sum. `tmp` holds kScanWaves words of LDS. Every thread of the block must
// call it.
constexpr int kScanWaves = 16;
__device__ inline uint32_t block_exclusive_scan(uint32_t v, uint32_t *tmp, uint32_t *total)
{
    const uint32_t lane = __lane_id(), w = threadIdx.x / kWave, nw = blockDim.x / kWave;
    uint32_t x = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t y = __shfl_up(x, off);
        if (lane >= (uint32_t)off) x += y;
    }
    if (lane == kWave - 1) tmp[w] = x;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (uint32_t q = 0; q < nw; ++q) {
        const uint32_t s = tmp[q];
        before += q < w ? s : 0u;
        all += s;
    }
    __syncthreads();  // tmp may be reused by the caller
    *total = all;
    return before + x - v;
}

// Per digit d (one block each): partial[b * R + d] := sum of partial[b' * R + d] over b' < b, and
// total[d] := the sum over all blocks.
__global__ __launch_bounds__(256) void part_colscan_kernel(uint32_t *__restrict__ partial, uint32_t blocks, uint32_t R,
                                                           uint32_t *__restrict__ total)
{
    __shared__ uint32_t tmp[kScanWaves];
    const uint32_t d = blockIdx.x;
    constexpr uint32_t kPer = kMaxSortBlocks / 256;
    const uint32_t b0 = threadIdx.x * kPer;
    uint32_t v[kPer], sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) {
        v[j] = b0 + j < blocks ? partial[(uint64_t)(b0 + j) * R + d] : 0u;
        sum += v[j];
    }
    uint32_t all;
    uint32_t run = block_exclusive_scan(sum, tmp, &all);
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) {
        if (b0 + j < blocks) partial[(uint64_t)(b0 + j) * R + d] = run;
        run += v[j];
    }
    if (threadIdx.x == 0) total[d] = all;
}

// Per-block counts of digit P of cid[i] over each block's range: partial[b * R + d]. With
// chunks != nullptr (the last pass, whose input is sorted by the bits of cid below P.shift) it
// also adds every chunk's count to chunks[cid]: a block bins the first kLowSpan values of those
// low bits that its range holds, by (low value, digit), in LDS.
template <typename CidT>
__global__ __launch_bounds__(kCountThreads) void part_count_kernel(const CidT *__restrict__ cid, PartGrid G, RadixPass P,
                                                                   uint32_t *__restrict__ partial,
                                                                   uint32_t *__restrict__ chunks)
{
    __shared__ uint32_t h[kMaxRadix];
    __shared__ uint32_t hc[kLowSpan * kMaxRadix];
    const uint32_t R = 1u << P.bits;
    const uint32_t low_mask = (1u << P.shift) - 1u;
    for (uint32_t d = threadIdx.x; d < R; d += kCountThreads) h[d] = 0;
    if (chunks)
        for (uint32_t x = threadIdx.x; x < kLowSpan * kMaxRadix; x += kCountThreads) hc[x] = 0;
    __syncthreads();
    const uint64_t lo = count_begin(G, blockIdx.x);
    const uint64_t hi = count_end(G, lo);
    const uint32_t l0 = lo < hi ? ((uint32_t)cid[lo] & low_mask) : 0u;
    for (uint64_t i0 = lo + threadIdx.x; i0 < hi; i0 += (uint64_t)kCountThreads * kCountItems) {
        uint32_t c[kCountItems];
#pragma unroll
        for (int u = 0; u < kCountItems; ++u) {
            const uint64_t i = i0 + (uint64_t)u * kCountThreads;
            c[u] = i < hi ? (uint32_t)cid[i] : 0u;
        }
#pragma unroll
        for (int u = 0; u < kCountItems; ++u) {
            if (i0 + (uint64_t)u * kCountThreads >= hi) continue;
            const uint32_t d = digit_of(c[u], P);
            atomicAdd(&h[d], 1u);
            if (chunks) {
                const uint32_t j = (c[u] & low_mask) - l0;  // the input is sorted by these bits
                if (j < kLowSpan) atomicAdd(&hc[j * kMaxRadix + d], 1u);
                else atomicAdd(&chunks[c[u]], 1u);
            }
        }
    }
    __syncthreads();
    for (uint32_t d = threadIdx.x; d < R; d += kCountThreads) partial[(uint64_t)blockIdx.x * R + d] = h[d];
    if (chunks)
        for (uint32_t x = threadIdx.x; x < kLowSpan * kMaxRadix; x += kCountThreads)
            if (hc[x]) atomicAdd(&chunks[((x % kMaxRadix) << P.shift) + l0 + x / kMaxRadix], hc[x]);
}

// start[c] := the first index of chunk c, for c in [0, total], from the chunk counts held in
// start[0, total) (start[total] := their sum). Three launches over segments of kScanSeg counts:
// each segment's sum into seg[], the exclusive prefix of seg[] (one block), then each segment
// rewritten as its prefix plus the running sum of its counts.
constexpr uint32_t kScanSeg = 1024;  // counts per segment: 256 threads x 4
__global__ __launch_bounds__(256) void part_seg_sum_kernel(const uint32_t *__restrict__ start, uint32_t total,
                                                           uint32_t *__restrict__ seg)
{
    __shared__ uint32_t tmp[kScanWaves];
    const uint32_t c0 = blockIdx.x * kScanSeg + threadIdx.x * 4;
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) sum += c0 + j < total ? start[c0 + j] : 0u;
    uint32_t all;
    (void)block_exclusive_scan(sum, tmp, &all);
    if (threadIdx.x == 0) seg[blockIdx.x] = all;
}

__global__ __launch_bounds__(1024) void part_seg_scan_kernel(uint32_t *__restrict__ seg, uint32_t nseg,
                                                             uint32_t *__restrict__ start, uint32_t total)
{
    __shared__ uint32_t tmp[kScanWaves];
    const uint32_t per = (nseg + blockDim.x - 1) / blockDim.x;
    const uint32_t s0 = threadIdx.x * per;
    uint32_t sum = 0;
    for (uint32_t j = 0; j < per; ++j)
        if (s0 + j < nseg) sum += seg[s0 + j];
    uint32_t all;
    uint32_t run = block_exclusive_scan(sum, tmp, &all);
    for (uint32_t j = 0; j < per; ++j) {
        if (s0 + j < nseg) {
            const uint32_t x = seg[s0 + j];
            seg[s0 + j] = run;
            run += x;
        }
    }
    if (threadIdx.x == 0) start[total] = all;
}

__global__ __launch_bounds__(256) void part_seg_write_kernel(uint32_t *__restrict__ start, uint32_t total,
                                                             const uint32_t *__restrict__ seg)
{
    __shared__ uint32_t tmp[kScanWaves];
    const uint32_t c0 = blockIdx.x * kScanSeg + threadIdx.x * 4;
    uint32_t v[4], sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
        v[j] = c0 + j < total ? start[c0 + j] : 0u;
        sum += v[j];
    }
    uint32_t all;
    uint32_t run = seg[blockIdx.x] + block_exclusive_scan(sum, tmp, &all);
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
        if (c0 + j < total) start[c0 + j] = run;
        run += v[j];
    }
}

// The lanes among vm (a ballot) whose digit equals this lane's d, a digit of `bits` bits (BITS if
// it is positive). Per bit: sb = 0 or ~0 (the lane's bit), and the mask keeps the lanes whose bit
// equals it, m &= ~(ballot ^ sb), on the two 32-bit halves.
template <int BITS>
__device__ inline uint64_t match_mask(uint64_t vm, uint32_t d, uint32_t bits)
{
    uint32_t mlo = (uint32_t)vm, mhi = (uint32_t)(vm >> 32);
    auto step = [&](uint32_t b) {
        const uint32_t sb = (uint32_t)((int32_t)(d << (31u - b)) >> 31);
        const uint64_t bb = __ballot(sb != 0u);  // lanes outside vm drop out through the AND
        mlo &= ~((uint32_t)bb ^ sb);
        mhi &= ~((uint32_t)(bb >> 32) ^ sb);
    };
    if constexpr (BITS > 0) {
#pragma unroll
        for (uint32_t b = 0; b < (uint32_t)BITS; ++b) step(b);
    } else {
        for (uint32_t b = 0; b < bits; ++b) step(b);
    }
    return ((uint64_t)mhi << 32) | mlo;
}

// One pass: the entries of each block's range (from src, chunk ids from cid) go to their places
// in ent_out (with CIDS chunk ids to cid_out), ordered by digit P. partial holds the blocks'
// exclusive prefixes per digit and total the digits' totals (part_colscan_kernel).
// What bounds it is how a tile's entries reach memory: a tile writes one run per digit, and the
// first and last line of a run are written in part (4096-entry tiles, 16 entries a run: 35 % more
// bytes than the entries and chunk ids have). So where the batch has tiles enough a tile takes a
// CU's whole LDS, at 8 waves a CU (the caller chooses ITEMS, a thread's entries). The next tile's
// loads are issued when the tile's entries have gone to LDS, ahead of the write-out's stores; all
// of them, and a whole tile's stores, are issued without a branch, so every wait counts the
// younger operations instead of draining the stores.
// 2^28 entries of 8 bytes, first pass 2105 -> 1630 us (3.3 TB/s), last pass 1485 -> 1255 us
// (3.8 TB/s); 2^26 entries of 16 bytes, 675 -> 620 us and 780 -> 505 us.
// Ranking within a wave (BITS):
//   > 0  stably (by digit, then index), with one ballot per digit bit; BITS = P.bits;
//   0    the same with P.bits read at run time;
//   < 0  not stably: each entry's rank is what the workgroup's LDS counter of the digit returned
//        when the entry added itself, in whatever order the lanes' atomics were applied. The
//        first pass of a least-significant-digit partition may do this (its input order means
//        nothing); every later pass must keep the order of the previous digits.
// Where block b's entries lie and where its entries of each digit go (Layout):
//   begin(b), end(b, begin): its input range;
//   base(b, d, R, tmp): the global place of its first entry of digit d (every thread of the block
//   calls it, d = threadIdx.x, and uses the result for d < R; tmp: kScanWaves words of LDS);
//   n: the entry count (no place reaches it).
// PassLayout is a digit pass over the whole batch: fixed block ranges (PartGrid), places from
// the per-block digit counts after part_colscan_kernel and the digit totals.
struct PassLayout {
    PartGrid G;
    const uint32_t *partial, *total;
    uint64_t n;
    __device__ uint64_t begin(uint32_t b) const { return part_begin(G, b); }
    __device__ uint64_t end(uint32_t, uint64_t lo) const { return part_end(G, lo); }
    __device__ uint32_t base(uint32_t b, uint32_t d, uint32_t R, uint32_t *tmp) const
    {
        uint32_t all;
        const uint32_t dbase = block_exclusive_scan(d < R ? total[d] : 0u, tmp, &all);
        return d < R ? dbase + partial[(uint64_t)b * G.sub * R + d] : 0u;
    }
};

// A pass over a batch grouped by table (the group bulk fill): block b covers blocks[b] (one
// table's range) and partial holds the place of its first entry of each local chunk.
struct SegLayout {
    const GroupItem *blocks;
    const uint32_t *partial;
    uint64_t n;
    __device__ uint64_t begin(uint32_t b) const { return blocks[b].begin; }
    __device__ uint64_t end(uint32_t b, uint64_t lo) const { return lo + blocks[b].len; }
    __device__ uint32_t base(uint32_t b, uint32_t d, uint32_t R, uint32_t *) const
    {
        return d < R ? partial[(uint64_t)b * kGroupBulkChunks + d] : 0u;
    }
};

template <typename Entry, typename Src, typename CidT, int ITEMS, int BITS, bool CIDS, typename Layout = PassLayout>
__global__ __launch_bounds__(kSortThreads, 2) void part_scatter_kernel(
    Src src, const CidT *__restrict__ cid, Layout Lay, RadixPass P, Entry *__restrict__ ent_out,
    CidT *__restrict__ cid_out)
{
    constexpr int kWaves = kSortThreads / kWave;
    constexpr uint32_t kTile = kSortThreads * ITEMS;
    static_assert(kSortThreads >= (int)kMaxRadix && kSortThreads % kWave == 0, "one thread per digit");
    __shared__ Entry buf[kTile];
    // what the write-out needs of a chunk id: all of it if it is passed on, else its digit
    using Kept = std::conditional_t<CIDS, CidT, uint8_t>;
    __shared__ Kept cbuf[kTile];
    constexpr int kRows = BITS < 0 ? 1 : kWaves;  // counters: the workgroup's, or per wave
    __shared__ uint32_t wcnt[kRows][kMaxRadix];   // digit counts, then first places in the tile
    __shared__ uint32_t gbase[kMaxRadix];         // global place of the block's next entry of d
    __shared__ uint32_t gdel[kMaxRadix];          // gbase[d] minus the tile's first place of d
    __shared__ uint32_t tmp[kScanWaves];
    const uint32_t R = 1u << P.bits;
    const uint32_t tid = threadIdx.x, lane = __lane_id(), w = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint64_t lo = Lay.begin(blockIdx.x);
    const uint64_t hi = Lay.end(blockIdx.x, lo);
    if (lo >= hi) return;  // block-uniform: nothing to place
    {
        const uint32_t b = Lay.base(blockIdx.x, tid, R, tmp);
        if (tid < R) gbase[tid] = b;
    }
    const uint64_t lanemask = lanemask_lt();
    // wave w holds tile entries w * ITEMS * 64 + u * 64 + lane: stable ranking follows
    // (u, lane) inside the wave, and the waves in order
    const uint32_t wbase = w * ITEMS * kWave;
    Entry e[ITEMS];
    uint32_t c[ITEMS];
    // entries past the range's end are read as its last one and not used
    auto load_tile = [&](uint64_t t0) {
        if (t0 + kTile <= hi) {
            const Src ws = src.from(t0 + wbase);
            const CidT *const wc = cid + t0 + wbase;
#pragma unroll
            for (int u = 0; u < ITEMS; ++u) {
                e[u] = ws.load(u * kWave + lane);
                c[u] = (uint32_t)wc[u * kWave + lane];
            }
        } else {
#pragma unroll
            for (int u = 0; u < ITEMS; ++u) {
                const uint64_t at = t0 + wbase + u * kWave + lane, i = at < hi ? at : hi - 1;
                e[u] = src.load(i);
                c[u] = (uint32_t)cid[i];
            }
        }
    };
    auto tile = [&](uint64_t t0, auto whole) {
        constexpr bool kWhole = decltype(whole)::value;
        const uint32_t tn = kWhole ? kTile : (uint32_t)(hi - t0);
        auto valid = [&](int u) { return kWhole || wbase + u * kWave + lane < tn; };
        for (uint32_t x = tid; x < kRows * kMaxRadix; x += kSortThreads) (&wcnt[0][0])[x] = 0;
        __syncthreads();  // wcnt is zero; the previous tile's output is done with buf and gdel
        uint32_t r[ITEMS];
        if constexpr (BITS < 0) {
#pragma unroll
            for (int u = 0; u < ITEMS; ++u) r[u] = valid(u) ? atomicAdd(&wcnt[0][digit_of(c[u], P)], 1u) : 0u;
        } else {
            // the lanes of one digit in an item (their match mask) take consecutive ranks in lane
            // order after the digit's count so far
            const uint32_t bits = P.bits;
#pragma unroll
            for (int u = 0; u < ITEMS; ++u) {
                const uint32_t d = digit_of(c[u], P);
                const uint64_t m = match_mask<BITS>(__ballot(valid(u)), d, bits);
                const uint32_t below = (uint32_t)__popcll(m & lanemask);
                const uint32_t base = valid(u) ? wcnt[w][d] : 0u;
                r[u] = base + below;
                if (valid(u) && below == 0) wcnt[w][d] = base + (uint32_t)__popcll(m);
            }
        }
        __syncthreads();
        // per digit: the counters' first places in the tile (in their order), and the shift from
        // a tile place to its global place
        {
            uint32_t x[kRows], run = 0;
#pragma unroll
            for (int q = 0; q < kRows; ++q) {
                x[q] = tid < R ? wcnt[q][tid] : 0u;
                run += x[q];
            }
            uint32_t all;
            uint32_t at = block_exclusive_scan(run, tmp, &all);
            if (tid < R) {
                gdel[tid] = gbase[tid] - at;
                gbase[tid] += run;  // read again only after the next tile's offsets are made
#pragma unroll
                for (int q = 0; q < kRows; ++q) {
                    wcnt[q][tid] = at;
                    at += x[q];
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < ITEMS; ++u) {
            if (valid(u)) {
                const uint32_t d = digit_of(c[u], P);
                const uint32_t pos = min(wcnt[BITS < 0 ? 0 : w][d] + r[u], kTile - 1);  // < tn by construction
                buf[pos] = e[u];
                cbuf[pos] = (Kept)(CIDS ? c[u] : d);
            }
        }
        if constexpr (kWhole) load_tile(t0 + kTile);
        __syncthreads();
        auto put = [&](uint32_t q) {
            const uint32_t cq = (uint32_t)cbuf[q];
            const uint64_t g = (uint64_t)(uint32_t)(gdel[CIDS ? digit_of(cq, P) : cq] + q);  // < n by construction
            return g < Lay.n ? g : Lay.n - 1;
        };
        if constexpr (kWhole) {
#pragma unroll
            for (int u = 0; u < ITEMS; ++u) {
                const uint32_t q = tid + u * kSortThreads;
                const uint64_t g = put(q);
                ent_out[g] = buf[q];
                if constexpr (CIDS) cid_out[g] = cbuf[q];
            }
        } else {
            for (uint32_t q = tid; q < tn; q += kSortThreads) {
                const uint64_t g = put(q);
                ent_out[g] = buf[q];
                if constexpr (CIDS) cid_out[g] = cbuf[q];
            }
        }
    };
    uint64_t t0 = lo;
    load_tile(t0);
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0), so the loop's waits count its own operations only
    for (; t0 + kTile <= hi; t0 += kTile) tile(t0, std::true_type{});
    if (t0 < hi) tile(t0, std::false_type{});
}

}  // namespace

// The partition's launches after the pack, which has written the chunk ids of the n entries of
// src0 to cid[0] and the counts of the first digit (passes P[0..np)) of the counting blocks of
// G0 = part_grid<Entry, CidT, ITEMS0>(n) to partial. The first pass (ITEMS0 entries a thread and
// tile) reads src0 and writes ent[0]; each later one (ITEMS1) reads the entry buffer the previous
// one wrote and writes the other. Chunk ids go from cid[p & 1] to cid[(p + 1) & 1], except in the
// last pass. start (chunks + 1 words) receives the first index of every chunk. *out is the entry
// buffer the sorted entries end in.
template <typename Entry, typename Src, typename CidT, int ITEMS0, int ITEMS1>
hipError_t partition_passes(Src src0, Entry *const ent[2], CidT *const cid[2], const PartGrid &G0, const RadixPass *P,
                            uint32_t np, uint32_t *partial, uint32_t *total, uint32_t *start, uint32_t chunks,
                            hipStream_t st, int *out)
{
    int e = 0;
    const PartGrid G1 = part_grid<Entry, CidT, ITEMS1>(G0.n);
    for (uint32_t p = 0; p < np; ++p) {
        const uint32_t R = 1u << P[p].bits;
        const bool last = p + 1 == np;
        const PartGrid &G = p == 0 ? G0 : G1;
        if (last) {  // the chunk counts gather in start[0, chunks) (zeroed as 8-byte words)
            const hipError_t z = launch_zero(reinterpret_cast<unsigned long long *>(start), (chunks + 1) / 2, st);
            if (z != hipSuccess) return z;
        }
        // the first pass's digit counts come with the pack; the last count also counts chunks
        if (p > 0 || last)
            part_count_kernel<CidT><<<G.blocks * G.sub, kCountThreads, 0, st>>>(cid[p & 1], G, P[p], partial,
                                                                                 last ? start : nullptr);
        part_colscan_kernel<<<R, 256, 0, st>>>(partial, G.blocks * G.sub, R, total);
        CidT *const cout = cid[(p + 1) & 1];
        const PassLayout lay{G, partial, total, G.n};
        const EntrySource<Entry> prev{ent[1 - e]};
        auto scatter = [&](auto src, auto items, auto bits, auto cids) {
            part_scatter_kernel<Entry, decltype(src), CidT, decltype(items)::value, decltype(bits)::value,
                                decltype(cids)::value>
                <<<G.blocks, kSortThreads, 0, st>>>(src, cid[p & 1], lay, P[p], ent[e], cout);
        };
        auto stable = [&](auto bits) { scatter(prev, Int<ITEMS1>{}, bits, std::false_type{}); };
        // the first pass ranks by atomics; the later ones stably, the last one's digit bits unrolled
        if (p == 0 && last) scatter(src0, Int<ITEMS0>{}, Int<-1>{}, std::false_type{});
        else if (p == 0) scatter(src0, Int<ITEMS0>{}, Int<-1>{}, std::true_type{});
        else if (!last) {
            if constexpr (sizeof(CidT) > 2) scatter(prev, Int<ITEMS1>{}, Int<0>{}, std::true_type{});
            else return hipErrorInvalidValue;  // 2-byte chunk ids take at most two passes
        } else if (P[p].bits == 4) stable(Int<4>{});
        else if (P[p].bits == 5) stable(Int<5>{});
        else if (P[p].bits == 6) stable(Int<6>{});
        else if (P[p].bits == 7) stable(Int<7>{});
        else if (P[p].bits == 8) stable(Int<8>{});
        else return hipErrorInvalidValue;  // digits are spread evenly: 9 or more bits leave 4 to the last
        if (!last) e = 1 - e;
    }
    const uint32_t nseg = (chunks + kScanSeg - 1) / kScanSeg;  // <= kPartialWords: partial is free now
    part_seg_sum_kernel<<<nseg, 256, 0, st>>>(start, chunks, partial);
    part_seg_scan_kernel<<<1, 1024, 0, st>>>(partial, nseg, start, chunks);
    part_seg_write_kernel<<<nseg, 256, 0, st>>>(start, chunks, partial);
    *out = e;
    return hipGetLastError();
}

}  // namespace dyc
