// dyc_inflight.hpp -- host state about the device work a table may still have in flight, over the few
// runtime calls it needs (Runtime), so that a host-only build can run it with a stand-in.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <atomic>
#include <mutex>

namespace dyc {

// The bucket of its pair that every stored key was first put to, where a table still keeps the rule:
// a key is elsewhere only if that bucket had no free slot then, and none has become free since (no
// erase, resize or load). kStart: the start rule of the eviction insert (odd keys pos2), kFill: the
// bulk fill's fill_target.
enum class FirstBucket : uint32_t { kNone = 0, kStart = 1, kFill = 2 };

namespace host {

// Which first-bucket rules (FirstBucket) the entries of a table, or of a group's tables, keep, and
// the finds in flight that rely on one. An empty table keeps both; an insert keeps its own; an
// erase, which frees slots, keeps none. A find that relies on a rule records an event (a mark), and the
// erase that drops the rule waits on its own stream for the marks, so it frees no slot under such a
// find on another stream. A stream's handle says which mark its finds share and nothing more: the
// handle may have been another stream's, destroyed with its finds still running. So every mark is
// waited for, whatever its handle, and a mark is recorded again only after a wait for what it
// stood for (both are nothing on the stream that recorded it).
// Finds of fewer than kFirstBucketKeys keys read in the reference order: the mark, and two buckets'
// latencies in turn, cost small calls more than they save (with the mark, in tables of 10 MiB and more:
// 2^18 lookups 0.8-1.1 times as fast, 2^20 0.95-1.2, 2^21 1.03-1.3, 2^22 1.06-1.35). So do finds being captured, which may be replayed after an erase, finds on the per-thread
// stream (one handle for many streams), and those on more than kMarks streams since the last erase or
// clear.
constexpr uint64_t kFirstBucketKeys = 1ull << 22;

// Whether one table's lookups gain from a first-bucket rule. Such a find reads fewer buckets and takes
// 1.3 times the vector and 1.5 times the scalar instructions, so it gains where lookups wait for lines
// from memory and loses where an XCD's L2 (4 MiB) holds most of what they read. Time in the reference
// order over time with the rule, 2^22 uniform lookups, half of them stored: 0.7 in tables of 1 MiB, 0.75 at
// 4, 0.9 at 6, 1.1-1.15 at 8, 1.2-1.3 at 12, 1.3-1.4 at 64 (64-bit keys 0.75, 0.75, 0.85, 1.0, 1.15,
// 1.2); where all are stored 0.9-1.0 at 8 MiB and 1.0-1.15 at 12, so the line is there. Skewed lookups stay
// in L2 longer: Zipf(0.99) 0.75 at 16 MiB, 0.85-0.95 at 64, 1.0-1.15 at 256.
inline bool first_bucket_pays(uint64_t table_bytes) { return table_bytes >= (12ull << 20); }

// The rule a find of 32-bit keys takes where the tables keep `rule`. With two subtables the start rule
// sends every key to subtable 0 first (the pair is the key's parity, and so is the start), whose
// buckets are then full, so almost every lookup goes on to the other one: 0.9-1.03 times as fast at 8
// to 32 MiB and all shares of hits. (The pair of a 64-bit key is its fold's parity: 1.1-1.4.)
inline FirstBucket narrow_rule(FirstBucket rule, uint32_t subtables)
{
    return subtables == 2 && rule == FirstBucket::kStart ? FirstBucket::kNone : rule;
}

// Whether a group's lookups do: table i of tables_n has bytes(i) bytes and the lookups [offsets[i],
// offsets[i + 1]). Large finds lay whole tables out over the 8 XCDs, so what counts is how much of the
// tables an XCD's workgroups read at a time against its L2: the tables that the lookups in flight on it
// span (about 2^18 of them in the grid taken from 2^24 lookups on, 2^19 in the larger one below), and
// no more than its eighth of all. Time in the reference order over time with the rule, 32-bit keys,
// lookups uniform in each table, half of them stored, by that span in MiB (weighted by lookups):
//   2^22 and 2^23 lookups: 1-5 MiB 0.75-0.9, 7-9 0.85-1.15, 12 1.0-1.1, 16 and more 1.05-1.2;
//   2^24 to 2^26: 1-2.5 MiB 0.72-0.95, 4.7 0.92-1.1, 9 and more 1.06-1.26;
//   2^24 to 2^26, fewer than 8 tables (so fewer XCDs than all): 9 MiB 0.8-1.0, 18 1.13-1.2.
// (100 M lookups of 400 tables of 2^14..2^20 keys, 5.2 MiB: 1.11.) 64-bit keys lie nearer to 1 on both
// sides, with the same crossings. Where fewer lookups than two a line come, each line is read from
// memory whatever the L2 holds. Groups of less than 1 MiB a table on average read in the reference
// order at any size.
template <typename Bytes>
bool first_bucket_pays(uint32_t tables_n, const uint64_t *offsets, Bytes bytes)
{
    const uint64_t n = offsets[tables_n];
    const bool narrow_grid = n >= (1ull << 24);
    const double flight = narrow_grid ? 1 << 18 : 1 << 19;
    double all = 0, own = 0, span = 0;  // bytes; bytes of the lookup's own table, and of its span, over the lookups
    for (uint32_t i = 0; i < tables_n; ++i) {
        const double b = (double)bytes(i), m = (double)(offsets[i + 1] - offsets[i]);
        all += b;
        own += b * m;
        span += m == 0 ? 0 : b * (m > flight ? m : flight);
    }
    if (n == 0 || all < tables_n * 1048576.0) return false;
    if ((double)n * 64 <= all) return true;
    const double most = own / (double)n > all / 8 ? own / (double)n : all / 8;
    const double mib = (span / (double)n < most ? span / (double)n : most) / 1048576.0;
    return mib >= (narrow_grid && tables_n >= 8 ? 5 : 10);
}

template <typename Runtime>
class FirstBucketRulesT {
    using Stream = typename Runtime::Stream;
    using Event = typename Runtime::Event;
    using Error = typename Runtime::Error;

  public:
    FirstBucketRulesT() = default;
    FirstBucketRulesT(const FirstBucketRulesT &) = delete;
    FirstBucketRulesT &operator=(const FirstBucketRulesT &) = delete;
    ~FirstBucketRulesT()
    {
        for (Mark &m : marks_)
            if (m.made) Runtime::drop(m.done);
    }
    // Just created.
    void emptied() { restart(kStartBit | kFillBit); }
    // Cleared on s. (A find still in flight would race with the clear itself, so there is nothing left
    // to wait for.) A clear that is being captured empties nothing until it is replayed.
    void cleared(Stream s)
    {
        if (!Runtime::capturing(s)) emptied();
    }
    // launch() clears the table and fills it under `rule`, and has waited for that when it returns. If
    // it fails, the table may still hold what it held before: no rule then.
    template <typename Launch>
    Error refill(FirstBucket rule, Launch launch)
    {
        lost();
        const Error e = launch();
        if (e == Runtime::kOk) restart(bit(rule));
        return e;
    }
    void filled(FirstBucket rule) { keep(bit(rule)); }  // entries are about to be stored under `rule`
    void lost() { keep(0); }                            // resized or loaded
    // Slots are about to be freed on s.
    Error freeing(Stream s)
    {
        std::lock_guard<std::mutex> lk(mu_);
        rules_ = 0;
        for (Mark &m : marks_) {
            if (!m.live) continue;
            const Error e = Runtime::wait(s, m.done);
            if (e != Runtime::kOk) return e;
            m.live = false;
        }
        return Runtime::kOk;
    }
    // Launch a find of n keys on s: launch(rule) with the rule it may rely on. subtables: of tables of
    // 32-bit keys, else 0.
    template <typename Launch>
    Error find(uint64_t n, Stream s, uint32_t subtables, Launch launch)
    {
        last_ = FirstBucket::kNone;
        if (n < kFirstBucketKeys || Runtime::shared(s) || Runtime::capturing(s)) return launch(FirstBucket::kNone);
        std::lock_guard<std::mutex> lk(mu_);
        const FirstBucket kept = rules_ & kFillBit ? FirstBucket::kFill : (rules_ ? FirstBucket::kStart : FirstBucket::kNone);
        const FirstBucket rule = narrow_rule(kept, subtables);
        Mark *m = rule != FirstBucket::kNone ? mark_for(s) : nullptr;
        if (!m || (m->live && Runtime::wait(s, m->done) != Runtime::kOk)) return launch(FirstBucket::kNone);
        last_ = rule;
        Error e = launch(rule);
        if (e == Runtime::kOk && (e = Runtime::record(m->done, s)) != Runtime::kOk)
            (void)Runtime::finish(s);  // no mark: nothing may be in flight
        m->live = true;
        return e;
    }

    // The rule of the last find (tests).
    FirstBucket last() const { return last_; }

  private:
    static constexpr uint32_t kStartBit = 1u, kFillBit = 2u;
    static constexpr int kMarks = 8;
    struct Mark {
        Stream stream{};
        Event done{};
        bool made = false;  // done exists
        bool live = false;  // a find after the last erase relies on a rule
    };
    static uint32_t bit(FirstBucket r)
    {
        return r == FirstBucket::kFill ? kFillBit : (r == FirstBucket::kStart ? kStartBit : 0u);
    }
    void keep(uint32_t bits)
    {
        std::lock_guard<std::mutex> lk(mu_);
        rules_ &= bits;
    }
    void restart(uint32_t bits)
    {
        std::lock_guard<std::mutex> lk(mu_);
        rules_ = bits;
        for (Mark &m : marks_) m.live = false;
    }
    // The mark of stream s: its own, or a free one; nullptr if there is none.
    Mark *mark_for(Stream s)
    {
        for (Mark &m : marks_)
            if (m.live && m.stream == s) return &m;
        for (Mark &m : marks_) {
            if (m.live) continue;
            if (!m.made && !(m.made = Runtime::make(&m.done))) return nullptr;
            m.stream = s;
            return &m;
        }
        return nullptr;
    }
    std::mutex mu_;
    std::atomic<FirstBucket> last_{FirstBucket::kNone};
    uint32_t rules_ = 0;
    Mark marks_[kMarks];
};

// The storage a table's last resize replaced, kept for its next one: a table that grows and shrinks
// around one fill takes the same two sizes in turn, and hipMalloc with the hipFree behind it cost
// many times what the resize's kernels do (to 96 MB and back with a find after each: 3.0 ms, 0.18 ms
// with this). A block fits only a resize to its very size, so a table that keeps growing never
// uses it. Bounded to one block of at most kSpareBlock bytes a table (a downsize is there to give
// memory back, and the larger the block the smaller hipMalloc's share) and to kSpareTotal in the
// process; given back when the next resize leaves another one, when an allocation of the table's
// resizes fails, and with the table.
// hipFree waits for the device, so a replaced block could still be in use by finds and clears in
// flight (every other call waits before it returns, or is waited for by the next one); a block kept
// must not be. So those calls say where they run (used_on). What ran on the null stream has ended
// when a resize on it has, which waits for it. No other handle says as much: the stream may be gone and
// its handle another one's, and captured work is replayed anywhere. After a call on one of those
// nothing is kept. (An event a call would tell, but costs a small find on such a stream 1.1 us of 6.)
constexpr size_t kSpareBlock = 256ull << 20, kSpareTotal = 1ull << 30;
template <typename Runtime>
class SpareBlockT {
    using Stream = typename Runtime::Stream;

  public:
    SpareBlockT() = default;
    SpareBlockT(const SpareBlockT &) = delete;
    SpareBlockT &operator=(const SpareBlockT &) = delete;
    // Work that uses the table's blocks and is not waited for is about to be launched on s. can_keep: the
    // table has a block that a resize could keep (storage that came with the table is never kept).
    void used_on(Stream s, bool can_keep)
    {
        if (can_keep) (Runtime::null(s) ? on_null_ : elsewhere_) = true;
    }
    // The kept block if it has just `bytes` bytes, else nullptr.
    void *take(size_t bytes) { return p_ && bytes_ == bytes ? give_back() : nullptr; }
    // p was replaced by a resize that has waited for s: keep it, and free the block kept before, or
    // free it (on r's thread).
    template <typename Reclaimer>
    void retire(Reclaimer &r, int device, void *p, size_t bytes, Stream s)
    {
        r.defer(device, give_back());
        const bool idle = !elsewhere_ && (!on_null_ || Runtime::null(s));
        if (idle) on_null_ = false;
        if (!idle || bytes > kSpareBlock) return r.defer(device, p);
        if (total().fetch_add(bytes) + bytes > kSpareTotal) {
            total() -= bytes;
            return r.defer(device, p);
        }
        p_ = p;
        bytes_ = bytes;
    }
    // The kept block, no longer kept (nullptr if there is none).
    void *give_back()
    {
        void *const p = p_;
        if (p) total() -= bytes_;
        p_ = nullptr;
        return p;
    }
    size_t kept() const { return p_ ? bytes_ : 0; }

  private:
    static std::atomic<size_t> &total()
    {
        static std::atomic<size_t> bytes{0};
        return bytes;
    }
    std::atomic<bool> on_null_{false};    // work on the null stream may not have ended
    std::atomic<bool> elsewhere_{false};  // work on another stream, or captured: never known to have ended
    void *p_ = nullptr;
    size_t bytes_ = 0;
};

}  // namespace host
}  // namespace dyc
