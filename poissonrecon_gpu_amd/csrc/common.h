// Internal shared declarations of the MI355X Poisson reconstruction library.
// Everything here is private to libprg.so; the public boundary is include/prg.h.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <map>
#include <string>
#include <vector>

#include "../../include/prg.h"

namespace prg {

constexpr int kMaxDepth = 10;  // 3D key bits must fit in uint32

// A context's pinned read-back area: the solver's part, then counts that
// kernels write there themselves (a copy behind the kernel would cost about
// 10 us): non-empty nodes per depth, the mesh's vertices and triangles, the
// owned corners.
constexpr size_t kCgHostBytes = 8192;
constexpr size_t kCgHostLevels = kCgHostBytes - 64;
constexpr size_t kCgHostMesh = kCgHostBytes - 16;
constexpr size_t kCgHostTopo = kCgHostBytes - 4;
static_assert(kCgHostLevels + 4 * (kMaxDepth + 1) <= kCgHostMesh, "counts overlap");
constexpr int kWeldHost = 56;  // the weld's three counts in sub_host (behind the subdivision's counters)

// ---- errors ------------------------------------------------------------------
struct Error {
    prg_status status;
    std::string msg;
};

#define PRG_HIP(call)                                                                          \
    do {                                                                                       \
        hipError_t e_ = (call);                                                                \
        if (e_ != hipSuccess)                                                                  \
            throw ::prg::Error{e_ == hipErrorOutOfMemory ? PRG_E_NOMEM : PRG_E_HIP,            \
                               std::string(#call) + ": " + hipGetErrorString(e_)};             \
    } while (0)

#define PRG_CHECK_LAUNCH() PRG_HIP(hipGetLastError())

// ---- device buffers ------------------------------------------------------------
// Device memory of one context: buffers (under 1 GiB; larger ones are
// allocations of their own) are parts of a few large allocations, given back to
// the device with the context.  A context's about 170 buffers
// as allocations of their own cost 20 us each to make, and 270 us each to free
// beside other contexts at work (hipFree waits for the whole device).
// A part given back may still be read by work queued on the context's
// streams: it is only handed out again after those streams were waited for.
// Used by one thread at a time, like its context (arena.cpp).
class Arena {
public:
    Arena() = default;
    Arena(const Arena&) = delete;
    Arena& operator=(const Arena&) = delete;
    ~Arena();
    void* take(size_t bytes);
    void give(void* p, size_t bytes);
    std::vector<const hipStream_t*> streams;  // of the context (null ones are not made yet)

private:
    struct Part {
        uint8_t* p;
        size_t bytes;
        bool queued;  // work using it may still be queued
        int chunk;
    };
    struct Chunk {
        uint8_t* p;
        size_t bytes;
    };
    bool add_chunk(size_t bytes);
    bool trim();
    std::vector<Part> free_;  // by address; neighbours of one chunk are joined
    std::vector<Chunk> chunks_;
    size_t total_ = 0;
};

// The arena that buffers reserved by this thread come from (null: allocations
// of their own), for a scope: a context's entry points set theirs.
Arena*& current_arena();
struct ArenaScope {
    Arena* before;
    explicit ArenaScope(Arena* a) : before(current_arena()) { current_arena() = a; }
    ~ArenaScope() { current_arena() = before; }
    ArenaScope(const ArenaScope&) = delete;
    ArenaScope& operator=(const ArenaScope&) = delete;
};

// Owning device buffer that only grows (re-used across calls of a context).
template <class T>
struct DBuf {
    T* p = nullptr;
    size_t n = 0;  // capacity in elements
    Arena* arena = nullptr;  // where p comes from (null: hipMalloc)
    DBuf() = default;
    DBuf(const DBuf&) = delete;
    DBuf& operator=(const DBuf&) = delete;
    ~DBuf() { release(); }
    void release() {
        if (p && arena) arena->give(p, n * sizeof(T));
        else if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    T* reserve(size_t count) {
        if (count <= n && p) return p;
        release();
        size_t c = count ? count : 1;
        arena = current_arena();
        if (arena) p = static_cast<T*>(arena->take(c * sizeof(T)));
        else PRG_HIP(hipMalloc(&p, c * sizeof(T)));
        n = c;
        return p;
    }
    T* get() const { return p; }
};

// A typed view of one slot of a context's buffer pool: grow-only device
// memory kept for the context's lifetime, so a repeated stage allocates
// nothing.  Each function uses its own slot numbers.
template <class T>
struct PoolBuf {
    DBuf<uint8_t>* b;
    T* reserve(size_t count) { return reinterpret_cast<T*>(b->reserve((count ? count : 1) * sizeof(T))); }
    T* get() const { return reinterpret_cast<T*>(b->get()); }
};

// ---- launch helpers --------------------------------------------------------------
inline unsigned grid_for(int64_t n, int block) {
    int64_t g = (n + block - 1) / block;
    if (g < 1) g = 1;
    return unsigned(g);
}

// Per-kernel hipEvent timing (enabled by prg_config.timing).
struct KernelTimer {
    bool enabled = false;
    hipStream_t stream = nullptr;
    struct Rec {
        int64_t launches = 0;
        double total_ms = 0.0;
        double bytes = 0.0;  // algorithmic bytes summed over launches
    };
    std::map<std::string, Rec> recs;
    struct Pending {
        std::string name;
        hipEvent_t a, b;
        double bytes;
    };
    std::vector<Pending> pending;
    std::vector<hipEvent_t> pool;
    hipEvent_t get_event() {
        if (!pool.empty()) {
            hipEvent_t e = pool.back();
            pool.pop_back();
            return e;
        }
        hipEvent_t e;
        PRG_HIP(hipEventCreate(&e));
        return e;
    }
    // Returns an index to pass to end(); -1 if disabled.
    int begin(const char* name, double bytes) {
        if (!enabled) return -1;
        Pending p{name, get_event(), get_event(), bytes};
        PRG_HIP(hipEventRecord(p.a, stream));
        pending.push_back(p);
        return int(pending.size()) - 1;
    }
    void end(int idx) {
        if (idx < 0) return;
        PRG_HIP(hipEventRecord(pending[idx].b, stream));
    }
    // Counts a launch under `name` without timing it (no events: a record
    // that only says which variant ran, beside a timed one).
    void count(const char* name) {
        if (enabled) recs[name].launches++;
    }
    // Files a recorded launch under another name with other algorithmic bytes
    // (e.g. one that found its work already finished and moved nothing), before flush().
    void relabel(int idx, const char* name, double bytes = 0.0) {
        if (idx >= 0 && idx < int(pending.size())) {
            pending[idx].name = name;
            pending[idx].bytes = bytes;
        }
    }
    // Resolves recorded events (synchronises on them).
    void flush() {
        for (auto& p : pending) {
            PRG_HIP(hipEventSynchronize(p.b));
            float ms = 0.0f;
            PRG_HIP(hipEventElapsedTime(&ms, p.a, p.b));
            Rec& r = recs[p.name];
            r.launches++;
            r.total_ms += ms;
            r.bytes += p.bytes;
            pool.push_back(p.a);
            pool.push_back(p.b);
        }
        pending.clear();
    }
    ~KernelTimer() {
        for (auto& p : pending) {
            (void)hipEventDestroy(p.a);
            (void)hipEventDestroy(p.b);
        }
        for (auto e : pool) (void)hipEventDestroy(e);
    }
};

struct TimedScope {
    KernelTimer& t;
    int idx;
    TimedScope(KernelTimer& tm, const char* name, double bytes) : t(tm), idx(tm.begin(name, bytes)) {}
    ~TimedScope() { t.end(idx); }
};

// ---- function-space tables (host-built, funcspace.cpp) -----------------------------
struct FsTables {
    int D = 0;
    int64_t res = 0;
    // baseFunctions[i] as ConfirmedPPolynomial<3,4>: 4 pieces x (start, c0..c3)
    std::vector<float> base_fn;
    // depth-D base function as ConfirmedPPolynomial<2,4>: 4 pieces x (start, c0..c2)
    float base_maxdepth[16] = {};
    // Laplacian stencil per depth, 27 floats each (0 where the reference drops the entry)
    std::vector<float> stencil;
    // divergence weights per node depth d: 3 * 2^(D-d) floats starting at div_off[d]
    std::vector<float> div_table;
    std::vector<int64_t> div_off;
    // per depth: the largest difference, over all grid points of depth D and
    // the three cells around them, between a base function's float value and
    // the quadratic B-spline it stands for (1 at the centre)
    std::vector<float> corner_dev;
};
void build_fs_tables(int D, FsTables* out);

// ---- primitives (primitives.hip) ------------------------------------------------------
struct Scratch;  // grows on demand
// Exclusive scan of n int32 values; writes the total to *d_total (device) if non-null.
// two arrays of the same length (exclusive scans and totals), in one pass each
void scan_exclusive2(const int32_t* a_in, int32_t* a_out, int32_t* a_total, const int32_t* b_in, int32_t* b_out,
                     int32_t* b_total, int64_t n, hipStream_t s, Scratch& scratch, KernelTimer& kt);
// The state of the single-pass scans of one stream, as their kernels take it.
struct LookState {
    uint64_t* words;
    int32_t* error;  // pinned: set by a tile that could not do its part
    uint32_t spins;  // polls before a wait for another tile gives up
};
constexpr uint32_t kLookSpins = 1u << 22;  // seconds: every tile waited for runs already
// ... with room for `words` tiles
LookState look_state(Scratch& scratch, int64_t words, hipStream_t s);
// Where the host has waited for scans of this state on stream s: throws if
// one failed (the state is ready for the next).
void look_check(Scratch& scratch, hipStream_t s);
void scan_exclusive(const int32_t* d_in, int32_t* d_out, int64_t n, int32_t* d_total, hipStream_t s,
                    Scratch& scratch, KernelTimer& kt);
// Stable LSD radix sort of (key, value) pairs on the low `bits` bits of the key.
// Result is in (keys, vals); alt buffers are scratch of the same size.
void radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt, int64_t n,
                      int bits, hipStream_t s, Scratch& scratch, KernelTimer& kt);

struct Scratch {
    DBuf<uint64_t> look;  // the single-pass scans' state (look_state)
    int32_t* look_error = nullptr;
    DBuf<int32_t> b, c;
    DBuf<uint8_t> bytes;
};

}  // namespace prg
