// rows.cpp -- host memory of embedding tables (no reference counterpart: the
// reference copies its table into one malloc'd block, HnGPU.cu:1019-1048).
//
// Ordinary memory on huge pages: a table is read on the host, and pinned memory
// is mapped into the process one small page at a time when that first touches it
// (512 MB: 180 ms, after the call), ordinary huge pages while they are written
// (512 MB: 9 ms on four threads).  A table grows in place: realloc moves large
// blocks by their page tables.
#include <sys/mman.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <new>

#include "host.h"

namespace gfsm {

namespace {

struct Head {  // precedes a block's words
    uint64_t bytes;
    uint64_t pad[7];
};
Head *head(uint32_t *p) { return reinterpret_cast<Head *>(p) - 1; }
uint32_t *words(Head *h) { return reinterpret_cast<uint32_t *>(h + 1); }

constexpr size_t kHugePage = 2u << 20;

// Large blocks that results gave back, with their pages, for the next ones (any
// thread, any context): kPoolBytes in all, freed when the last context closes.
// Smaller ones the C library keeps.  (A call returning 1,920,000 rows of seven:
// 1.4 ms with the pool, 2.2 with fresh pages each time.)
constexpr size_t kPoolMin = 4u << 20, kPoolBytes = 256u << 20;
struct Pool {
    std::mutex mu;
    std::vector<Head *> free;
    size_t bytes = 0;
    uint32_t contexts = 0;
};
Pool &pool()
{
    static Pool *p = new Pool;  // never destroyed: results may be freed at exit
    return *p;
}

// The smallest block of the pool that holds `bytes` (and is not far larger, unless
// for a table that grows), or null.
Head *take(size_t bytes, bool grows)
{
    Pool &p = pool();
    std::lock_guard<std::mutex> lk(p.mu);
    size_t best = p.free.size();
    for (size_t i = 0; i < p.free.size(); i++) {
        const uint64_t b = p.free[i]->bytes;
        if (b >= bytes && (grows || b / 4 <= bytes) && (best == p.free.size() || b < p.free[best]->bytes)) best = i;
    }
    if (best == p.free.size()) return nullptr;
    Head *h = p.free[best];
    p.free.erase(p.free.begin() + best);
    p.bytes -= h->bytes;
    return h;
}

void give(Head *h)
{
    if (h->bytes >= kPoolMin) {
        Pool &p = pool();
        std::lock_guard<std::mutex> lk(p.mu);
        if (p.contexts && p.bytes + h->bytes <= kPoolBytes) {
            p.free.push_back(h);
            p.bytes += h->bytes;
            return;
        }
    }
    std::free(h);
}

}  // namespace

void row_pool_open()
{
    Pool &p = pool();
    std::lock_guard<std::mutex> lk(p.mu);
    p.free.reserve(kPoolBytes / kPoolMin);  // give() never allocates
    p.contexts++;
}

void row_pool_close()
{
    Pool &p = pool();
    std::lock_guard<std::mutex> lk(p.mu);
    if (--p.contexts) return;
    for (Head *h : p.free) std::free(h);
    p.free.clear();
    p.bytes = 0;
}

void RowBuf::resize(size_t n)
{
    if (n > cap_) {
        size_t bytes = n * sizeof(uint32_t);
        Head *h = nullptr;
        if (!p_) {
            if (bytes >= kPoolMin) h = take(bytes, false);
            if (!h && (h = static_cast<Head *>(std::malloc(sizeof(Head) + bytes)))) h->bytes = bytes;
        } else {
            // Past what the pool keeps, room is address space that is never touched: a
            // move by page tables splits its huge pages (504 MB in 500 chunks: by
            // halves 270 to 390 ms, by fours 165).
            const size_t had = cap_ * sizeof(uint32_t), more = std::max(bytes, had > kPoolBytes / 2 ? had * 4 : had / 2 * 3);
            if (more >= kPoolMin && (h = take(more, true))) {
                std::memcpy(words(h), p_, n_ * sizeof(uint32_t));
                give(head(p_));
            } else {
                h = static_cast<Head *>(std::realloc(head(p_), sizeof(Head) + more));
                if (h) bytes = more;
                else h = static_cast<Head *>(std::realloc(head(p_), sizeof(Head) + bytes));
                if (h) h->bytes = bytes;
            }
        }
        if (!h) throw std::bad_alloc();
        p_ = words(h);
        cap_ = h->bytes / sizeof(uint32_t);
        const uintptr_t lo = (reinterpret_cast<uintptr_t>(h) + 4095) & ~(uintptr_t)4095;
        const uintptr_t hi = (reinterpret_cast<uintptr_t>(p_) + h->bytes) & ~(uintptr_t)4095;
        if (hi >= lo + kHugePage) (void)madvise(reinterpret_cast<void *>(lo), hi - lo, MADV_HUGEPAGE);
    }
    n_ = n;
}

void RowBuf::clear()
{
    if (p_) give(head(p_));
    p_ = nullptr;
    n_ = cap_ = 0;
}

}  // namespace gfsm
