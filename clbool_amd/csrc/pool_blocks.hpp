// pool_blocks.hpp -- which free block of the device pool (runtime.hip) a
// request gets, kept free of device calls like block_heap.hpp.
//
// The pool serves every Controls of a GPU, and a Controls releases its
// temporaries on the host while kernels on its stream may still use them.  So a
// released temporary is first retired to its Controls: that Controls may have
// it again at once (its later work comes after on the same stream), anyone else
// only after the Controls has waited for its stream.  Then large blocks go back
// to the heap; small ones stay with the Controls until someone else finds no
// other block, which also spares most calls the heap's bookkeeping.  No wait is
// added to any call.
#pragma once

#include "block_heap.hpp"

#include <cstddef>
#include <utility>
#include <vector>

namespace clb {

class PoolBlocks {
  public:
    using u64 = std::uint64_t;
    struct Block {
        char *ptr = nullptr;
        u64 size = 0;
    };
    struct Retired : Block {
        u64 epoch = 0;  // the clock when it was retired; 0: waited for since
    };
    struct Owner {
        std::vector<Retired> list;
        void *tag = nullptr;  // the user's
    };
    static constexpr std::size_t KEEP = 64;  // small blocks that stay with an owner after a wait

    PoolBlocks(u64 small_max, u64 small_unit, u64 large_unit)
        : small_max_(small_max), large_unit_(large_unit), small_(small_unit), large_(large_unit) {}

    // A block of at least cap bytes (ptr == nullptr: none): the owner's smallest
    // retired one of at most a quarter more (in_flight: also of those that its
    // work may still use), else one of the heap.  owner == nullptr: of the heap.
    Block take(u64 cap, Owner *owner, bool in_flight) {
        if (owner) {
            std::vector<Retired> &l = owner->list;
            std::size_t best = l.size();
            for (std::size_t k = 0; k < l.size(); ++k)
                if (l[k].size >= cap && l[k].size <= cap + cap / 4 && (in_flight || !l[k].epoch) &&
                    (best == l.size() || l[k].size < l[best].size))
                    best = k;
            if (best != l.size()) {
                const Block b = l[best];
                l.erase(l.begin() + (std::ptrdiff_t)best);
                retired_bytes_ -= b.size;
                return b;
            }
        }
        const BlockHeap::Block *b = heap(cap).take(cap);
        return b ? Block{b->ptr, b->size} : Block{};
    }
    // For a small request where there is no memory for a small segment: a large
    // block, which give_back and retire know by its size.
    Block take_large(u64 cap) {
        const BlockHeap::Block *b = large_.take(cap > large_unit_ ? cap : large_unit_);
        return b ? Block{b->ptr, b->size} : Block{};
    }
    void add_segment(char *base, u64 size, u64 cap) { heap(cap).add_segment(base, size); }

    void enter(Owner *o) { owners_.push_back(o); }
    // Nothing uses what the owner retired, and it retires no more.
    void leave(Owner *o) {
        for (const Retired &r : o->list) back(r);
        o->list.clear();
        for (Owner *&x : owners_)
            if (x == o) {
                x = owners_.back();
                owners_.pop_back();
                break;
            }
    }
    const std::vector<Owner *> &owners() const { return owners_; }

    // Work of the owner may still use the block.
    void retire(Block b, Owner *o) {
        Retired r;
        r.ptr = b.ptr;
        r.size = b.size;
        r.epoch = clock_;
        o->list.push_back(r);
        retired_bytes_ += b.size;
    }
    // Before and after the owner waits for its work: what it retired before the
    // wait began is free for anyone.
    u64 wait_begins() { return clock_++; }
    void waited(Owner *o, u64 began) {
        std::vector<Retired> &l = o->list;
        std::size_t excess = l.size() > KEEP ? l.size() - KEEP : 0, n = 0;  // the oldest go first
        for (std::size_t k = 0; k < l.size(); ++k) {
            Retired r = l[k];
            if (r.epoch <= began) {
                r.epoch = 0;
                if (r.size > small_max_ || excess) {
                    excess -= excess ? 1 : 0;
                    back(r);
                    continue;
                }
            }
            l[n++] = r;
        }
        l.resize(n);
    }
    // Gives back what owners keep that was waited for, and of one owner also what
    // it retired before the wait that began at `began` (which has ended).
    void reclaim() {
        for (Owner *o : owners_) reclaim(o, 0);
    }
    void reclaim(Owner *o, u64 began) {
        std::vector<Retired> &l = o->list;
        std::size_t n = 0;
        for (std::size_t k = 0; k < l.size(); ++k) {
            if (l[k].epoch <= began) back(l[k]);
            else l[n++] = l[k];
        }
        l.resize(n);
    }

    // Nothing uses the block any more; false if it is not a live block.
    bool give_back(char *p) { return small_.give_back(p) || large_.give_back(p); }

    void collect_free_segments(std::vector<std::pair<char *, u64>> &out) {
        small_.collect_free_segments(out);
        large_.collect_free_segments(out);
    }
    // The largest free block; retired ones are not among them.
    u64 largest_free() const { return large_.largest_free(); }
    // Bytes that are not in use, retired ones among them.
    u64 free_bytes() const { return small_.free_bytes() + large_.free_bytes() + retired_bytes_; }

  private:
    BlockHeap &heap(u64 cap) { return cap <= small_max_ ? small_ : large_; }
    void back(const Retired &r) {
        retired_bytes_ -= r.size;
        (void)heap(r.size).give_back(r.ptr);
    }
    u64 small_max_, large_unit_;
    BlockHeap small_, large_;
    std::vector<Owner *> owners_;
    u64 retired_bytes_ = 0, clock_ = 1;
};

}  // namespace clb
