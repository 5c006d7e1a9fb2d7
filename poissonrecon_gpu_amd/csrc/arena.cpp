// A context's device memory (common.h).
#include <algorithm>

#include "ctx.h"

namespace prg {

namespace {
constexpr size_t kPartAlign = 512;
// Buffers of kOwn bytes and more are allocations of their own, back with the
// device as soon as they are outgrown: of clouds that fill the memory those
// parts would not fit what comes after them.  The line is that high because a
// hipFree slows the copies of pageable memory for several passes (6 M points,
// 72 MB a copy: 21 ms instead of 5 for up to five passes after it), more than
// the whole pass on a cloud whose buffers are smaller.
constexpr size_t kOwn = size_t(1) << 30;
// A new shared allocation holds at least kFirstChunk bytes, half of what the
// shared ones hold already up to kMostSpare, or what is asked for if that is
// more.  Their outgrown parts (each under kOwn) and the last one's rest are
// what a context holds beyond its buffers: over clouds of 1, 2, 4 .. 32 M points
// 13.5 GiB where the last alone takes 11.1 (12.6 and 11.1 when every buffer had
// an allocation of its own).
constexpr size_t kFirstChunk = size_t(32) << 20;
constexpr size_t kMostSpare = size_t(1) << 30;
}  // namespace

Arena*& current_arena() {
    static thread_local Arena* a = nullptr;
    return a;
}

Arena::~Arena() {
    for (const Chunk& c : chunks_)
        if (c.p) (void)hipFree(c.p);
}

// an allocation, or null without room for it
static uint8_t* device_alloc(size_t bytes) {
    void* p = nullptr;
    const hipError_t e = hipMalloc(&p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        return nullptr;
    }
    PRG_HIP(e);
    return static_cast<uint8_t*>(p);
}

bool Arena::add_chunk(size_t bytes) {
    uint8_t* p = device_alloc(bytes);
    if (!p) return false;
    const Part part{p, bytes, false, int(chunks_.size())};
    chunks_.push_back(Chunk{part.p, bytes});
    total_ += bytes;
    free_.insert(std::lower_bound(free_.begin(), free_.end(), part.p, [](const Part& a, const uint8_t* b) { return a.p < b; }),
                 part);
    return true;
}

// shared allocations without a part in use go back to the device
bool Arena::trim() {
    bool freed = false;
    for (size_t i = 0; i < free_.size();) {
        Chunk& c = chunks_[size_t(free_[i].chunk)];
        if (free_[i].p == c.p && free_[i].bytes == c.bytes) {
            (void)hipFree(c.p);  // waits for the device
            total_ -= c.bytes;
            c = Chunk{nullptr, 0};
            free_.erase(free_.begin() + ptrdiff_t(i));
            freed = true;
        } else {
            i++;
        }
    }
    return freed;
}

void* Arena::take(size_t bytes) {
    const size_t want = (bytes + kPartAlign - 1) / kPartAlign * kPartAlign;
    if (want >= kOwn) {
        uint8_t* p = device_alloc(want);
        if (!p && trim()) p = device_alloc(want);
        if (!p) throw Error{PRG_E_NOMEM, "out of device memory (" + std::to_string(bytes) + " bytes)"};
        return p;
    }
    for (int attempt = 0;; attempt++) {
        // the smallest part that holds it, one without queued work if there is one
        size_t best = free_.size();
        for (size_t i = 0; i < free_.size(); i++) {
            const Part& f = free_[i];
            if (f.bytes < want) continue;
            if (best == free_.size() || f.queued < free_[best].queued ||
                (f.queued == free_[best].queued && f.bytes < free_[best].bytes))
                best = i;
        }
        if (best != free_.size()) {
            if (free_[best].queued) {
                for (const hipStream_t* s : streams)
                    if (*s) PRG_HIP(hipStreamSynchronize(*s));
                for (Part& f : free_) f.queued = false;
            }
            Part& f = free_[best];
            void* p = f.p;
            f.p += want;
            f.bytes -= want;
            if (!f.bytes) free_.erase(free_.begin() + ptrdiff_t(best));
            return p;
        }
        if (attempt == 0 &&
            add_chunk(std::max(want, std::max(kFirstChunk, std::min(kMostSpare, total_ / 2)))))
            continue;
        if (attempt <= 1 && add_chunk(want)) {
            attempt = 1;
            continue;
        }
        if (!trim() || !add_chunk(want)) throw Error{PRG_E_NOMEM, "out of device memory (" + std::to_string(bytes) + " bytes)"};
    }
}

void Arena::give(void* p, size_t bytes) {
    Part part{static_cast<uint8_t*>(p), (bytes + kPartAlign - 1) / kPartAlign * kPartAlign, true, -1};
    if (part.bytes >= kOwn) {
        (void)hipFree(p);  // waits for the device
        return;
    }
    for (size_t i = 0; i < chunks_.size(); i++)
        if (chunks_[i].p && part.p >= chunks_[i].p && part.p < chunks_[i].p + chunks_[i].bytes) part.chunk = int(i);
    auto it = std::lower_bound(free_.begin(), free_.end(), part.p, [](const Part& a, const uint8_t* b) { return a.p < b; });
    it = free_.insert(it, part);
    // join with the parts after and before it
    if (it + 1 != free_.end() && (it + 1)->chunk == it->chunk && it->p + it->bytes == (it + 1)->p) {
        it->bytes += (it + 1)->bytes;
        free_.erase(it + 1);
    }
    if (it != free_.begin() && (it - 1)->chunk == it->chunk && (it - 1)->p + (it - 1)->bytes == it->p) {
        (it - 1)->bytes += it->bytes;
        (it - 1)->queued = true;
        free_.erase(it);
    }
}

}  // namespace prg
