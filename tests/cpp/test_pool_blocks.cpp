// Randomised check of which block of the device pool a request gets
// (PoolBlocks): a block that an owner retired goes to that owner again or to
// nobody until the owner waited, no block is held twice, segments
// with retired blocks stay, and the byte count follows.  Addresses are
// synthetic (never dereferenced).  Exit status 0 on success.
#include "../../clbool_amd/csrc/pool_blocks.hpp"

#include <cstdio>
#include <cstdlib>
#include <map>
#include <random>

using clb::PoolBlocks;
using u64 = std::uint64_t;

#define CHECK(c)                                                             \
    do {                                                                     \
        if (!(c)) {                                                          \
            std::fprintf(stderr, "check failed at line %d: %s\n", __LINE__, #c); \
            return 1;                                                        \
        }                                                                    \
    } while (0)

int main() {
    constexpr u64 SMALL = 1 << 20, SEG = 2 << 20, BIG = 64ull << 20;
    constexpr int OWNERS = 3;
    std::mt19937_64 rng(7);
    PoolBlocks pool(SMALL, 256, 2 << 20);
    PoolBlocks::Owner ids[OWNERS];
    for (auto &o : ids) pool.enter(&o);
    // what the streams still use: block -> owner that retired it (or none: held)
    std::map<char *, u64> held, in_flight;
    std::map<char *, int> by;
    std::vector<PoolBlocks::Block> mine[OWNERS + 1];
    char *base = reinterpret_cast<char *>(1ull << 40);
    u64 total = 0, held_bytes = 0;
    u64 again = 0, others = 0;
    auto overlaps = [&](const std::map<char *, u64> &m, char *p, u64 n) {
        auto it = m.lower_bound(p);
        if (it != m.end() && it->first < p + n) return true;
        return it != m.begin() && (--it)->first + it->second > p;
    };
    for (int op = 0; op < 200000; ++op) {
        const int o = (int)(rng() % (OWNERS + 1));  // OWNERS: for anyone
        const unsigned what = (unsigned)(rng() % 100);
        if (what < 48) {
            const u64 cap = rng() % 8 ? (1 + rng() % 64) * 256 : (1 + rng() % 8) * (2 << 20);
            const bool in_flight_too = rng() % 2;
            PoolBlocks::Block b = pool.take(cap, o < OWNERS ? &ids[o] : nullptr, in_flight_too);
            if (!b.ptr) {
                const u64 n = cap <= SMALL ? SEG : BIG;
                pool.add_segment(base, n, cap);
                base += n + (1 << 20);
                total += n;
                b = pool.take(cap, nullptr, false);
            }
            CHECK(b.ptr && b.size >= cap);
            CHECK(!overlaps(held, b.ptr, b.size));
            if (overlaps(in_flight, b.ptr, b.size)) {
                // only the block's own owner, and the block as it was
                CHECK(o < OWNERS && in_flight_too && in_flight.count(b.ptr) && by[b.ptr] == o && in_flight[b.ptr] == b.size);
                CHECK(b.size <= cap + cap / 4);
                in_flight.erase(b.ptr);
                ++again;
            } else {
                ++others;
            }
            held[b.ptr] = b.size;
            held_bytes += b.size;
            mine[o].push_back(b);
        } else if (what < 95) {
            if (mine[o].empty()) continue;
            const size_t k = rng() % mine[o].size();
            const PoolBlocks::Block b = mine[o][k];
            mine[o][k] = mine[o].back();
            mine[o].pop_back();
            held.erase(b.ptr);
            held_bytes -= b.size;
            if (o < OWNERS && rng() % 4) {
                pool.retire(b, &ids[o]);
                in_flight[b.ptr] = b.size;
                by[b.ptr] = o;
            } else {
                CHECK(pool.give_back(b.ptr));
            }
        } else if (o < OWNERS) {  // the owner waits for its stream, and retires one more meanwhile
            const u64 began = pool.wait_begins();
            char *late = nullptr;
            if (!mine[o].empty()) {
                const PoolBlocks::Block b = mine[o].back();
                mine[o].pop_back();
                held.erase(b.ptr);
                held_bytes -= b.size;
                pool.retire(b, &ids[o]);
                in_flight[b.ptr] = b.size;
                by[b.ptr] = o;
                late = b.ptr;
            }
            pool.waited(&ids[o], began);
            std::size_t small = 0, large = 0;
            for (auto &r : ids[o].list) (r.size > SMALL ? large : small) += r.epoch == 0;
            CHECK(large == 0 && small <= PoolBlocks::KEEP);
            for (auto it = in_flight.begin(); it != in_flight.end();)
                it = by[it->first] == o && it->first != late ? in_flight.erase(it) : std::next(it);
            if (rng() % 4 == 0) pool.reclaim();
        }
        CHECK(pool.free_bytes() == total - held_bytes);
    }
    CHECK(again > 1000 && others > 1000);
    // segments that hold a retired block stay until it was given back
    for (int o = 0; o <= OWNERS; ++o)
        for (const PoolBlocks::Block &b : mine[o]) CHECK(pool.give_back(b.ptr));
    const PoolBlocks::Block last = pool.take(256, nullptr, false);
    pool.retire(last, &ids[0]);
    std::vector<std::pair<char *, u64>> segs;
    pool.collect_free_segments(segs);
    pool.reclaim();
    for (auto &s : segs) CHECK(!(last.ptr >= s.first && last.ptr < s.first + s.second));
    CHECK(ids[0].list.size() >= 1);
    for (auto &o : ids) pool.leave(&o);
    CHECK(pool.owners().empty());
    pool.collect_free_segments(segs);
    u64 sum = 0;
    for (auto &s : segs) sum += s.second;
    CHECK(sum == total && pool.free_bytes() == 0);
    std::printf("pool blocks: ok (%llu reused by their owner, %llu others)\n", (unsigned long long)again,
                (unsigned long long)others);
    return 0;
}
