// Host model of concurrent eviction inserts (waves of 64 lanes over one table) with the library's
// own slot choice (BucketTries). A bucket's view may be old: what a wave read of it earlier in the
// launch, as another XCD's L2 may still hold. Finds of a table that nothing was erased from rely on
// this: a key lies outside its first bucket only if that bucket has no free slot. Counts the keys for
// which that does not hold, and the keys that are lost or doubled.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "dyc_device.hpp"

using namespace dyc;

namespace {

uint64_t g_rng = 88172645463325252ull;
uint32_t rnd()
{
    g_rng ^= g_rng << 13, g_rng ^= g_rng >> 7, g_rng ^= g_rng << 17;
    return (uint32_t)(g_rng >> 32);
}
bool chance(uint32_t percent) { return rnd() % 100u < percent; }

struct Lane {
    uint32_t k = 0, pre = 0, kicks = 0;
    bool fresh = false, active = false;
    BucketTries tries;
};

struct Bucket {
    uint32_t key[kSlots];
};

struct Model {
    Desc D;
    std::vector<Bucket> now;               // every subtable's buckets, one after another
    std::vector<std::vector<Bucket>> old;  // per wave: what it read of each last
    uint32_t first[kMaxSubtables + 1] = {};
    uint32_t kick_bound = 0, old_percent = 0, parked = 0;

    Model(uint32_t d, const std::vector<uint32_t> &nb, uint32_t waves, uint32_t bound, uint32_t percent)
        : kick_bound(bound), old_percent(percent)
    {
        if (!desc_init(D, d)) abort();
        for (uint32_t t = 0; t < d; ++t) {
            desc_set(D, (int)t, nullptr, nb[t]);
            first[t + 1] = first[t] + nb[t];
        }
        now.assign(first[d], Bucket{});
        old.assign(waves, now);
    }
    uint32_t at(uint32_t k, uint32_t t) const { return first[t] + bucket_of(D, k, t); }
    uint32_t start(uint32_t k) const { return (k & 1u) ? pos2(D, pair_of(D, k)) : pos1(D, pair_of(D, k)); }

    // One step of every active lane of a wave, as the kernel's insert_step.
    void step(std::vector<Lane> &wave, uint32_t w)
    {
        struct Aim {
            uint32_t slot, t, b;
            int what;  // 0 nothing, 1 place, 2 swing, 3 evict
        };
        std::vector<Aim> aims(wave.size(), Aim{0, 0, 0, 0});
        std::vector<char> read(now.size(), 0);
        std::vector<uint32_t> id(wave.size(), ~0u);
        for (size_t l = 0; l < wave.size(); ++l) {
            Lane &h = wave[l];
            if (!h.active) continue;
            const uint32_t p = pair_of(D, h.k), ta = pos1(D, p), tb = pos2(D, p);
            const uint32_t t = h.pre == ta || h.pre == kOddStart ? tb : ta, b = at(h.k, t);
            if (!read[b] && !chance(old_percent)) old[w][b] = now[b];
            read[b] = 1;
            id[l] = (t << 9) | ((b - first[t]) & 511u);
            uint32_t view = 0, rank = 0;
            for (uint32_t j = 0; j < (uint32_t)kSlots; ++j)
                if (!old[w][b].key[j]) view |= 1u << j;
            for (size_t q = 0; q < l; ++q) rank += id[q] == id[l];
            const uint32_t open = h.tries.open(view);
            aims[l] = Aim{BucketTries::aim(open, rank), t, b, 1};
            if (open) continue;
            if (h.fresh && kick_bound == 0) {
                aims[l].what = 2;
                continue;
            }
            aims[l].what = 3;
            aims[l].slot = rescue_lane(h.k, h.kicks);
            if (h.kicks < kick_bound)
                for (uint32_t j = 0; j < (uint32_t)kSlots; ++j)
                    if (vote_victim(D, old[w][b].key[j], t)) {
                        aims[l].slot = j;
                        break;
                    }
        }
        const size_t turn = rnd() % wave.size();  // the order in which the lanes' atomics are applied
        for (size_t q = 0; q < wave.size(); ++q) {
            Lane &h = wave[(q + turn) % wave.size()];
            const Aim &a = aims[(q + turn) % wave.size()];
            if (a.what == 0) continue;
            if (a.what == 2) {
                h.pre = a.t;
                h.fresh = false;
                h.tries = {};
                continue;
            }
            uint32_t &slot = now[a.b].key[a.slot];
            if (a.what == 1 && slot != 0) {
                h.tries.lose(a.slot);
                continue;
            }
            const uint32_t out = a.what == 3 ? slot : 0u;
            slot = h.k;
            ++h.kicks;
            if (!out) {
                h.active = false;
                continue;
            }
            h.k = out;
            h.pre = a.t;
            h.fresh = false;
            h.tries = {};
            if (h.kicks >= kick_bound + 128u) {
                h.active = false;
                ++parked;
            }
        }
    }

    void insert(const std::vector<uint32_t> &keys, uint32_t waves)
    {
        std::vector<std::vector<Lane>> wv(waves, std::vector<Lane>(64));
        size_t next = 0;
        for (bool any = true; any;) {
            const uint32_t w = rnd() % waves;
            for (Lane &h : wv[w]) {
                if (h.active || next == keys.size()) continue;
                h = Lane{};
                h.k = keys[next++];
                h.pre = (h.k & 1u) ? kOddStart : kNoTable;
                h.fresh = h.active = true;
            }
            step(wv[w], w);
            any = next < keys.size();
            for (auto &x : wv)
                for (Lane &h : x) any |= h.active;
        }
    }

    // Keys outside a first bucket that has a free slot; *stored counts all keys.
    uint32_t misplaced(uint64_t *stored) const
    {
        uint32_t bad = 0;
        for (size_t b = 0; b < now.size(); ++b)
            for (uint32_t k : now[b].key) {
                if (!k) continue;
                ++*stored;
                const uint32_t home = at(k, start(k));
                if (home == b) continue;
                for (uint32_t other : now[home].key)
                    if (!other) {
                        ++bad;
                        break;
                    }
            }
        return bad;
    }
};

}  // namespace

int main()
{
    struct Shape {
        uint32_t d;
        std::vector<uint32_t> nb;
        int tables;
    };
    // small tables, and one whose first subtable alone makes it crowded (bucket numbers shared)
    const std::vector<Shape> shapes = {{2, {4, 4}, 1500}, {2, {8, 8}, 800}, {4, {2, 2, 2, 2}, 800}, {2, {4, 1100}, 4}};
    unsigned long long bad = 0, keys_in = 0, lost = 0;
    for (const Shape &s : shapes)
        for (uint32_t percent : {0u, 50u, 80u})
            for (uint32_t bound : {0u, 15u})
                for (int i = 0; i < s.tables; ++i) {
                    const uint32_t waves = 3;
                    Model m(s.d, s.nb, waves, bound, percent);
                    const size_t n = (size_t)(0.85 * kSlots * m.now.size());
                    std::vector<uint32_t> keys(n);
                    const uint32_t base = rnd() | 1u;
                    for (size_t j = 0; j < n; ++j) keys[j] = (uint32_t)(j + 1) * 0x9E3779B1u ^ (base << 20 >> 4);
                    for (uint32_t &k : keys)
                        if (reserved_key(k)) k = 12345u;
                    m.insert(keys, waves);
                    uint64_t stored = 0;
                    bad += m.misplaced(&stored);
                    keys_in += n;
                    lost += n - (stored + m.parked);
                }
    printf("keys %llu misplaced %llu lost %llu\n", keys_in, bad, lost);
    return bad != 0 || lost != 0;
}
