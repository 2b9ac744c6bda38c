// Host check of dyc_inflight.hpp over a stand-in for the runtime: streams are sets of the work ordered
// before what is next enqueued on them, events copy such a set. Prints "inflight ok".
#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>
#include <vector>

#include "dyc_inflight.hpp"

namespace {

using Work = std::set<int>;
struct Fake {
    using Stream = int;  // a handle; 0 is the null stream
    using Event = int;
    using Error = int;
    static constexpr Error kOk = 0;
    static std::map<int, Work> streams, events;
    static std::set<int> captured;
    static Work finished;
    static bool records_fail, waits_fail;
    static int made, next;
    static bool shared(Stream s) { return s == -1; }
    static bool capturing(Stream s) { return captured.count(s) != 0; }
    static bool make(Event *e)
    {
        *e = ++made;
        return true;
    }
    static void drop(Event e) { events.erase(e); }
    static Error record(Event e, Stream s)
    {
        if (records_fail) return 5;
        events[e] = streams[s];
        return kOk;
    }
    static Error wait(Stream s, Event e)
    {
        if (waits_fail) return 6;
        streams[s].insert(events[e].begin(), events[e].end());
        return kOk;
    }
    static Error finish(Stream s)
    {
        finished.insert(streams[s].begin(), streams[s].end());
        return kOk;
    }
    static bool null(Stream s) { return s == 0; }
    // enqueue a piece of work on s
    static int run(Stream s)
    {
        streams[s].insert(++next);
        return next;
    }
    static bool before(int work, Stream s) { return streams[s].count(work) != 0 || finished.count(work) != 0; }
    // the stream of this handle is destroyed and a new one gets the handle; its work may go on
    static void reuse(Stream s) { streams[s].clear(); }
};
std::map<int, Work> Fake::streams, Fake::events;
std::set<int> Fake::captured;
Work Fake::finished;
bool Fake::records_fail = false, Fake::waits_fail = false;
int Fake::made = 0, Fake::next = 0;

using dyc::FirstBucket;
using Rules = dyc::host::FirstBucketRulesT<Fake>;
constexpr uint64_t kMany = dyc::host::kFirstBucketKeys;

int g_bad = 0;
void check(bool ok, const char *what, int line)
{
    if (ok) return;
    printf("line %d: %s\n", line, what);
    ++g_bad;
}
#define CHECK(x) check((x), #x, __LINE__)

// A find of n keys on s: the rule it was launched with; *work is its place in the stream.
FirstBucket find(Rules &r, int s, int *work = nullptr, uint64_t n = kMany, uint32_t subtables = 4)
{
    FirstBucket used = FirstBucket::kNone;
    const int e = r.find(n, s, subtables, [&](FirstBucket rule) {
        used = rule;
        const int w = Fake::run(s);
        if (work) *work = w;
        return Fake::kOk;
    });
    CHECK(e == Fake::kOk && r.last() == used);
    return used;
}

void rules_kept_and_dropped()
{
    Rules r;
    CHECK(find(r, 1) == FirstBucket::kNone);  // nothing known of the table
    r.emptied();
    CHECK(find(r, 1) == FirstBucket::kFill);
    r.filled(FirstBucket::kStart);
    CHECK(find(r, 1) == FirstBucket::kStart);
    CHECK(find(r, 1, nullptr, kMany - 1) == FirstBucket::kNone);
    CHECK(find(r, 1, nullptr, kMany, 2) == FirstBucket::kNone && find(r, 1, nullptr, kMany, 0) == FirstBucket::kStart);
    CHECK(find(r, -1) == FirstBucket::kNone);
    Fake::captured = {1};
    CHECK(find(r, 1) == FirstBucket::kNone);
    Fake::captured.clear();
    r.filled(FirstBucket::kFill);  // entries under both rules
    CHECK(find(r, 1) == FirstBucket::kNone);
    r.cleared(1);
    CHECK(find(r, 1) == FirstBucket::kFill);
    r.lost();
    CHECK(find(r, 1) == FirstBucket::kNone);
    Fake::captured = {2};
    r.cleared(2);  // the table still holds its entries
    Fake::captured.clear();
    CHECK(find(r, 1) == FirstBucket::kNone);
}

void refill_that_fails_leaves_no_rule()
{
    for (const bool had : {false, true}) {
        Rules r;
        r.emptied();
        r.filled(FirstBucket::kStart);
        if (!had) r.freeing(1);
        CHECK(r.refill(FirstBucket::kFill, [] { return 7; }) == 7);
        CHECK(find(r, 1) == FirstBucket::kNone);
        FirstBucket during = FirstBucket::kFill;
        CHECK(r.refill(FirstBucket::kFill, [&] {
            during = find(r, 1);
            return Fake::kOk;
        }) == Fake::kOk);
        CHECK(during == FirstBucket::kNone);
        CHECK(find(r, 1) == FirstBucket::kFill);
    }
}

void an_erase_comes_after_the_finds_that_rely_on_a_rule()
{
    Rules r;
    r.emptied();
    int a = 0, b = 0, c = 0;
    CHECK(find(r, 1, &a) != FirstBucket::kNone && find(r, 2, &b) != FirstBucket::kNone);
    CHECK(find(r, 2, &c) != FirstBucket::kNone);
    CHECK(r.freeing(3) == Fake::kOk);
    CHECK(Fake::before(a, 3) && Fake::before(b, 3) && Fake::before(c, 3));
    CHECK(find(r, 1) == FirstBucket::kNone);
    // more streams than marks: the rest read in the reference order
    r.emptied();
    int with = 0;
    for (int s = 10; s < 30; ++s) {
        int w = 0;
        if (find(r, s, &w) == FirstBucket::kNone) continue;
        ++with;
    }
    CHECK(with == 8);
}

// Streams 1 and 2 are destroyed with a find running; new streams get their handles.
void a_handle_is_not_a_stream()
{
    Rules r;
    r.emptied();
    int a = 0, b = 0, c = 0;
    CHECK(find(r, 1, &a) != FirstBucket::kNone && find(r, 2, &b) != FirstBucket::kNone);
    Fake::reuse(1);
    Fake::reuse(2);
    CHECK(find(r, 2, &c) != FirstBucket::kNone);  // records stream 2's mark again
    CHECK(r.freeing(1) == Fake::kOk);
    CHECK(Fake::before(a, 1) && Fake::before(b, 1) && Fake::before(c, 1));
}

void runtime_errors()
{
    Rules r;
    r.emptied();
    int a = 0, b = 0;
    CHECK(find(r, 1, &a) != FirstBucket::kNone);
    Fake::waits_fail = true;
    CHECK(r.freeing(2) == 6);  // the erase is not launched
    Fake::waits_fail = false;
    CHECK(find(r, 1) == FirstBucket::kNone);
    CHECK(r.freeing(3) == Fake::kOk && Fake::before(a, 3));
    r.emptied();
    Fake::records_fail = true;
    CHECK(r.find(kMany, 1, 4, [&](FirstBucket) {
        b = Fake::run(1);
        return Fake::kOk;
    }) == 5);
    Fake::records_fail = false;
    CHECK(r.freeing(4) == Fake::kOk && Fake::before(b, 4));
}

// Small tables read in the reference order, whatever the lookups.
void tables_that_gain_from_a_rule()
{
    using dyc::host::first_bucket_pays;
    CHECK(!first_bucket_pays(1 << 15) && !first_bucket_pays(4 << 20) && !first_bucket_pays((12 << 20) - 1));
    CHECK(first_bucket_pays(12 << 20) && first_bucket_pays(1ull << 31));
    using dyc::host::narrow_rule;
    CHECK(narrow_rule(FirstBucket::kStart, 2) == FirstBucket::kNone);
    CHECK(narrow_rule(FirstBucket::kFill, 2) == FirstBucket::kFill);
    CHECK(narrow_rule(FirstBucket::kStart, 3) == FirstBucket::kStart);
    // groups of equal tables: what an XCD reads at a time
    auto group = [](uint32_t tables, double mib, uint64_t n) {
        std::vector<uint64_t> off(tables + 1);
        for (uint32_t i = 0; i <= tables; ++i) off[i] = n * i / tables;
        return first_bucket_pays(tables, off.data(), [mib](uint32_t) { return (uint64_t)(mib * (1 << 20)); });
    };
    const uint64_t few = 1 << 22, many = 1 << 24;
    CHECK(!group(1, 8, few) && group(1, 16, few) && !group(1, 8, many) && group(1, 16, many));
    CHECK(!group(4, 1, few) && !group(4, 4, few) && !group(4, 4, many) && group(4, 16, many));
    CHECK(!group(16, 2, few) && group(16, 16, few) && !group(16, 4, many) && group(16, 8, many));
    CHECK(!group(64, 1, few) && group(64, 2, few) && !group(64, 2, many) && group(64, 8, many));
    CHECK(group(256, 1, few) && !group(256, 1, many) && group(256, 2, many) && !group(256, 2, 4 * many));
    CHECK(group(512, 1, few) && group(512, 1, many) && !group(512, 1, 4 * many));
    CHECK(!group(2048, 0.35, few) && !group(2048, 0.35, 4 * many));
    CHECK(group(8, 4, 1 << 13) && group(8, 4, 1 << 17));  // a small captured step: each line once
    CHECK(!group(8, 4, 0));
    // one large table among small ones takes most lookups
    const uint64_t off[4] = {0, 1000, 1000, 1u << 24};
    CHECK(first_bucket_pays(3, off, [](uint32_t i) { return i == 2 ? 64ull << 20 : 1ull << 16; }));
}

using Spare = dyc::host::SpareBlockT<Fake>;
struct Freed {
    std::set<void *> all;
    void defer(int, void *p)
    {
        if (p) all.insert(p);
    }
};
char g_block[4];

// A resize on s replaces a block: whether it is kept (and then taken).
bool resize_keeps(Spare &sp, int s, size_t bytes = 1 << 20)
{
    Freed r;
    sp.retire(r, 0, g_block, bytes, s);
    CHECK(sp.kept() == (r.all.empty() ? bytes : 0));
    CHECK(sp.take(bytes + 1) == nullptr);
    const bool kept = sp.take(bytes) == g_block;
    CHECK(kept == r.all.empty());
    return kept;
}

void a_block_is_kept_only_when_nothing_uses_it()
{
    for (int on : {0, 1, 2}) {  // nothing in flight
        Spare sp;
        CHECK(resize_keeps(sp, on));
        sp.used_on(1, false);  // a find of a table whose blocks all came with it
        CHECK(resize_keeps(sp, on));
    }
    {  // the null stream, which a resize on it has waited for
        Spare sp;
        sp.used_on(0, true);
        CHECK(!resize_keeps(sp, 2));
        CHECK(resize_keeps(sp, 0));
        sp.used_on(0, true);
        CHECK(resize_keeps(sp, 0));
        CHECK(resize_keeps(sp, 2));
    }
    for (int on : {1, -1}) {  // a handle that may be another stream's by now, or many streams'
        Spare sp;
        sp.used_on(on, true);
        CHECK(!resize_keeps(sp, on) && !resize_keeps(sp, 0) && !resize_keeps(sp, 2));
    }
}

void kept_blocks_are_bounded()
{
    using dyc::host::kSpareBlock;
    using dyc::host::kSpareTotal;
    const size_t fit = kSpareTotal / kSpareBlock;
    std::vector<Spare> sp(fit + 1);
    Freed r;
    CHECK(!resize_keeps(sp[0], 0, kSpareBlock + 1));
    for (size_t i = 0; i < fit; ++i) sp[i].retire(r, 0, g_block, kSpareBlock, 0);
    CHECK(r.all.empty());
    CHECK(!resize_keeps(sp[fit], 0, 1));
    // a table's next block takes the place of the one it kept, which is freed
    sp[0].retire(r, 0, g_block + 1, kSpareBlock, 0);
    CHECK(sp[0].kept() == kSpareBlock && r.all == std::set<void *>{g_block});
    CHECK(sp[0].give_back() == g_block + 1 && sp[0].kept() == 0);
    CHECK(resize_keeps(sp[fit], 0, 1));
    for (Spare &x : sp) (void)x.give_back();
}

}  // namespace

int main()
{
    rules_kept_and_dropped();
    refill_that_fails_leaves_no_rule();
    an_erase_comes_after_the_finds_that_rely_on_a_rule();
    a_handle_is_not_a_stream();
    runtime_errors();
    tables_that_gain_from_a_rule();
    a_block_is_kept_only_when_nothing_uses_it();
    kept_blocks_are_bounded();
    if (!g_bad) printf("inflight ok\n");
    return g_bad != 0;
}
