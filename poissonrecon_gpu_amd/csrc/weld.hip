// Optional cross-batch vertex welding.  The reference concatenates the
// leaf-level batch and the subdivision batches without merging the vertices
// they share at the seams (main.cu:3793,4183,4543); this pass merges vertices
// whose three coordinates are bit-identical.  It is not part of the
// reference's output and runs only when asked for.
//
// Result: the first occurrence of each position keeps its place, in the
// original vertex order, so vertices that have no duplicate earlier in the
// list keep their relative order; every triangle entry is renumbered to its
// position's first occurrence.  Triangles are kept as they are (a triangle
// whose corners merge stays, degenerate).
//
// On the GPU: every vertex finds its position's place in a hash table, which
// keeps the smallest index that came there; one pass with a look-back scan
// numbers and compacts the vertices that are their own first occurrence, and
// the triangles are renumbered through the table.  What it moves is 12 B a
// vertex in and out, two table words and the triangles; the copies to and from
// the host take longer.  (As three stable 32-bit sorts and two scans it was 41
// launches: 470 us for 300,000 vertices.)
#include <mutex>
#include <string>

#include "ctx.h"
#include "lookback.h"

namespace prg {
namespace {

constexpr int kBlock = 256;

// The multipliers that fold the three words are the first three 32-bit primes
// of xxHash (Yann Collet); the last four lines are the 32-bit mixer
// "lowbias32" (Chris Wellons, hash-prospector).
__device__ __forceinline__ uint32_t hash_position(uint32_t x, uint32_t y, uint32_t z) {
    uint32_t h = x * 0x9E3779B1u;
    h = ((h << 15) | (h >> 17)) ^ (y * 0x85EBCA77u);
    h = ((h << 13) | (h >> 19)) ^ (z * 0xC2B2AE3Du);
    h ^= h >> 16;
    h *= 0x7FEB352Du;
    h ^= h >> 15;
    h *= 0x846CA68Bu;
    return h ^ (h >> 16);
}

// the table empty, the counts of the call cleared, and `look_words` words of
// the scan's state (none of a context's, whose calls cannot overlap)
__global__ void __launch_bounds__(kBlock) k_weld_init(int32_t* table, int64_t words, int32_t* host_counts,
                                                      uint64_t* look, int look_words) {
    if (blockIdx.x == 0 && threadIdx.x < 3) host_counts[threadIdx.x] = 0;
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < look_words; i += kBlock) look[i] = 0;
    int4* t4 = reinterpret_cast<int4*>(table);  // (a multiple of 4 words)
    for (int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x; i < words / 4; i += int64_t(gridDim.x) * kBlock)
        t4[i] = make_int4(-1, -1, -1, -1);
}

// place[i] = the slot of vertex i's position; table[slot] ends as the smallest
// vertex with it.  The table has twice as many slots as vertices, so a probe
// meets an empty one.  Vertices of one position in a row go in once per wave,
// by the first of them: of 300,000 at a single position, one by one, the
// slot's atomics took most of the call's 2.5 ms (0.42 now).
__global__ void __launch_bounds__(kBlock) k_weld_insert(const float* __restrict__ v, int64_t n, uint32_t mask,
                                                        int32_t* table, uint32_t* __restrict__ place) {
    const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const bool in = i < n;
    if (__ballot(in) == 0) return;  // (wave-uniform)
    const int64_t j = in ? i : n - 1;
    const uint32_t x = __float_as_uint(v[3 * j]), y = __float_as_uint(v[3 * j + 1]), z = __float_as_uint(v[3 * j + 2]);
    const uint32_t px = __shfl_up(x, 1, 64), py = __shfl_up(y, 1, 64), pz = __shfl_up(z, 1, 64);
    const bool head = lane == 0 || x != px || y != py || z != pz;
    uint32_t h = hash_position(x, y, z) & mask;
    // (a lane past the end repeats the last vertex and is no head: lane 0 is in)
    for (uint64_t probe = 0; head && probe <= mask; probe++) {
        int32_t at = __hip_atomic_load(table + h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (at < 0) {
            at = atomicCAS(table + h, -1, int32_t(i));
            if (at < 0) break;
        }
        const int64_t p = 3 * int64_t(at);
        if (__float_as_uint(v[p]) == x && __float_as_uint(v[p + 1]) == y && __float_as_uint(v[p + 2]) == z) {
            if (int32_t(i) < at) atomicMin(table + h, int32_t(i));
            break;
        }
        h = (h + 1) & mask;
    }
    const uint64_t heads = __ballot(head) & (~uint64_t(0) >> (63 - lane));  // at or before this lane
    h = __shfl(h, 63 - int(__builtin_clzll(heads)), 64);
    if (in) place[i] = h;
}

constexpr int kKeepItems = 8;
constexpr int kKeepTile = kBlock * kKeepItems;

// The vertices that are their own first occurrence, numbered in order and
// compacted; number[slot] = the output number of the slot's vertex.  The
// output's vertices, and those of the first n_leaf, go to pinned memory.
__global__ void __launch_bounds__(kBlock) k_weld_compact(const float* __restrict__ v, int64_t n, int64_t n_leaf,
                                                         uint32_t tiles, LookState state,
                                                         const int32_t* __restrict__ table,
                                                         const uint32_t* __restrict__ place,
                                                         int32_t* __restrict__ number, float* __restrict__ out,
                                                         int32_t* host_counts) {
    __shared__ int32_t lds[kBlock / 64];
    __shared__ int32_t s_before;
    const LookTile t = look_begin(state, tiles);
    if (t.tile >= tiles) return;
    const int64_t base = int64_t(t.tile) * kKeepTile + int64_t(threadIdx.x) * kKeepItems;
    uint32_t slot[kKeepItems];
    uint32_t keep = 0;
#pragma unroll
    for (int k = 0; k < kKeepItems; k++) slot[k] = base + k < n ? place[base + k] : 0;
#pragma unroll
    for (int k = 0; k < kKeepItems; k++)
        if (base + k < n && table[slot[k]] == int32_t(base + k)) keep |= 1u << k;
    int32_t total;
    const int32_t ex = block_exclusive_scan(__popc(keep), lds, total);
    if (threadIdx.x < 64) {
        const int32_t b = look_back(state, 0, t, tiles, total);
        if (threadIdx.x == 0) {
            s_before = b;
            if (t.tile == tiles - 1) host_counts[0] = b + total;
        }
    }
    __syncthreads();
    look_end(state, t, tiles);
    int32_t id = s_before + ex;
#pragma unroll
    for (int k = 0; k < kKeepItems; k++) {
        const int64_t i = base + k;
        if (i == n_leaf && i < n) host_counts[1] = id;
        if (!((keep >> k) & 1u)) continue;
        number[slot[k]] = id;
        const int64_t o = 3 * int64_t(id);
        out[o] = v[3 * i];
        out[o + 1] = v[3 * i + 1];
        out[o + 2] = v[3 * i + 2];
        id++;
    }
}

// triangle entries renumbered; one outside [0, n) is reported
__global__ void __launch_bounds__(kBlock) k_weld_triangles(int32_t* t, int64_t m3, int64_t n,
                                                           const uint32_t* __restrict__ place,
                                                           const int32_t* __restrict__ number, int32_t* host_counts) {
    const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= m3) return;
    const int32_t j = t[i];
    if (j < 0 || j >= n) host_counts[2] = 1;
    else t[i] = number[place[j]];
}

// Device arrays of one weld (n vertices, m triangles): the table's slots are
// a power of two, at least twice n.
struct WeldBufs {
    float *V, *out;
    int32_t *table, *number;
    uint32_t* place;
    int32_t* T;
};

uint64_t table_slots(int64_t n) {
    uint64_t h = 4;
    while (h < 2 * uint64_t(n)) h *= 2;
    return h;
}

// The weld proper on device arrays `b`, with the scan's state in `scr`, of
// which the first `look_words` words are cleared first.  The triangles go up
// on the second stream, beside the vertices' kernels.
void weld_core(prg_ctx* c, const WeldBufs& b, Scratch& scr, int look_words, float* vertices, int64_t n,
               int32_t* triangles, int64_t m, int64_t n_leaf, int64_t* n_out, int64_t* n_leaf_out) {
    hipStream_t s = c->stream;
    const uint64_t slots = table_slots(n);
    volatile int32_t* counts = c->sub_host + kWeldHost;  // kept vertices; kept among the first n_leaf; bad triangles
    const uint32_t tiles = uint32_t((n + kKeepTile - 1) / kKeepTile);
    LookState state = look_state(scr, tiles, s);
    state.spins = c->weld_spins;
    PRG_HIP(hipMemcpyAsync(b.V, vertices, size_t(3 * n) * 4, hipMemcpyHostToDevice, s));
    k_weld_init<<<unsigned(std::min<uint64_t>(2048, slots / 1024 + 1)), kBlock, 0, s>>>(
        b.table, int64_t(slots), c->sub_host + kWeldHost, state.words, look_words);
    PRG_CHECK_LAUNCH();
    k_weld_insert<<<grid_for(n, kBlock), kBlock, 0, s>>>(b.V, n, uint32_t(slots - 1), b.table, b.place);
    PRG_CHECK_LAUNCH();
    k_weld_compact<<<tiles, kBlock, 0, s>>>(b.V, n, n_leaf, tiles, state, b.table, b.place, b.number, b.out,
                                            c->sub_host + kWeldHost);
    PRG_CHECK_LAUNCH();
    if (m > 0) {
        // (the last use of T may still run on the context stream)
        PRG_HIP(hipMemcpyAsync(b.T, triangles, size_t(3 * m) * 4, hipMemcpyHostToDevice, c->stream2));
        PRG_HIP(hipEventRecord(c->mesh_ev, c->stream2));
        PRG_HIP(hipStreamWaitEvent(s, c->mesh_ev, 0));
        k_weld_triangles<<<grid_for(3 * m, kBlock), kBlock, 0, s>>>(b.T, 3 * m, n, b.place, b.number,
                                                                    c->sub_host + kWeldHost);
        PRG_CHECK_LAUNCH();
    }
    PRG_HIP(hipStreamSynchronize(s));
    look_check(scr, s);
    if (counts[2]) throw Error{PRG_E_ARG, "triangle index out of range"};  // the mesh is as it was
    const int64_t kept = counts[0];
    if (kept < 1 || kept > n) throw Error{PRG_E_HIP, "weld: inconsistent vertex count"};  // the mesh is as it was
    PRG_HIP(hipMemcpyAsync(vertices, b.out, size_t(3 * kept) * 4, hipMemcpyDeviceToHost, s));
    if (m > 0) PRG_HIP(hipMemcpyAsync(triangles, b.T, size_t(3 * m) * 4, hipMemcpyDeviceToHost, s));
    PRG_HIP(hipStreamSynchronize(s));  // the device arrays are reused or freed after return
    *n_out = kept;
    *n_leaf_out = n_leaf <= 0 ? 0 : (n_leaf < n ? int64_t(counts[1]) : kept);
}

// ---- the weld without allocation ------------------------------------------------------
// Fixed per-device array holding the device copy of the mesh, the weld's
// arrays and its scan and sort temporaries, for up to kNoAllocVertices
// vertices and kNoAllocTriangles triangles.
constexpr int64_t kNoAllocVertices = PRG_WELD_NOALLOC_MAX_VERTICES;
constexpr int64_t kNoAllocTriangles = PRG_WELD_NOALLOC_MAX_TRIANGLES;
constexpr int64_t kAlign = 256;
constexpr int64_t align_up(int64_t b) { return (b + kAlign - 1) / kAlign * kAlign; }
constexpr int64_t kLookWords = kNoAllocVertices / kKeepTile + 1 + kLookHeader;  // the scan's state, 64-bit words
static_assert(2 * align_up(12 * kNoAllocVertices) + 2 * align_up(8 * kNoAllocVertices) + align_up(4 * kNoAllocVertices) +
                      align_up(12 * kNoAllocTriangles) + align_up(8 * kLookWords) <= PRG_WELD_NOALLOC_BYTES,
              "prg.h states the size of the weld's fixed array");
static_assert((kNoAllocVertices & (kNoAllocVertices - 1)) == 0, "the largest table has exactly twice as many slots");
constexpr int64_t kNoAllocBytes = PRG_WELD_NOALLOC_BYTES;

__device__ __align__(256) uint8_t scratch[kNoAllocBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
uint8_t* g_scratch_ptr[kMaxDevices] = {};

}  // namespace

// The device address of `scratch` on `device` (current), looked up once per
// device.  In host code the array's name is only a stand-in for the symbol.
uint8_t* weld_noalloc_scratch(int device) {
    if (device < 0 || device >= kMaxDevices) throw Error{PRG_E_ARG, "device ordinal out of range"};
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        void* p = nullptr;
        PRG_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) throw Error{PRG_E_HIP, "hipGetSymbolAddress(scratch) returned null"};
        g_scratch_ptr[device] = static_cast<uint8_t*>(p);
    }
    return g_scratch_ptr[device];
}

void weld_mesh(prg_ctx* c, float* vertices, int64_t n, int32_t* triangles, int64_t m, int64_t n_leaf,
               int64_t* n_out, int64_t* n_leaf_out) {
    *n_out = n;
    *n_leaf_out = n_leaf < n ? n_leaf : n;
    if (n <= 1) return;
    DBuf<float> V, out;
    DBuf<uint32_t> place;
    DBuf<int32_t> table, number, T;
    const size_t slots = size_t(table_slots(n));
    WeldBufs b{V.reserve(size_t(3 * n)), out.reserve(size_t(3 * n)), table.reserve(slots),
               number.reserve(slots),    place.reserve(size_t(n)),   m > 0 ? T.reserve(size_t(3 * m)) : nullptr};
    weld_core(c, b, c->scratch, 0, vertices, n, triangles, m, n_leaf, n_out, n_leaf_out);
}

void weld_mesh_noalloc(prg_ctx* c, float* vertices, int64_t n, int32_t* triangles, int64_t m, int64_t n_leaf,
                       int64_t* n_out, int64_t* n_leaf_out) {
    if (n > kNoAllocVertices || m > kNoAllocTriangles)
        throw Error{PRG_E_ARG, "mesh exceeds the fixed weld array (" + std::to_string(kNoAllocVertices) +
                                   " vertices, " + std::to_string(kNoAllocTriangles) + " triangles)"};
    *n_out = n;
    *n_leaf_out = n_leaf < n ? n_leaf : n;
    if (n <= 1) return;
    uint8_t* base = weld_noalloc_scratch(c->cfg.device);
    int64_t off = 0;
    auto take = [&](int64_t bytes) {
        uint8_t* p = base + off;
        off += align_up(bytes);
        return p;
    };
    const int64_t N = kNoAllocVertices;
    WeldBufs b{};
    b.V = reinterpret_cast<float*>(take(12 * N));
    b.out = reinterpret_cast<float*>(take(12 * N));
    b.table = reinterpret_cast<int32_t*>(take(8 * N));
    b.number = reinterpret_cast<int32_t*>(take(8 * N));
    b.place = reinterpret_cast<uint32_t*>(take(4 * N));
    b.T = reinterpret_cast<int32_t*>(take(12 * kNoAllocTriangles));
    // the scan's state, lent to a Scratch whose buffer never grows past this
    // capacity (so it is never reallocated or freed).  Calls that overlap on
    // a device race for the array, and what they leave in the state would spoil
    // every later call, so each call clears it (2 KB, in its first kernel).
    Scratch scr;
    struct Lend {
        Scratch& s;
        ~Lend() {
            s.look.p = nullptr;
            s.look.n = 0;
        }
    } lend{scr};
    scr.look.p = reinterpret_cast<uint64_t*>(take(8 * kLookWords));
    scr.look.n = size_t(kLookWords);
    scr.look_error = c->scratch.look_error;
    if (off > kNoAllocBytes) throw Error{PRG_E_HIP, "weld array layout exceeds its size"};
    weld_core(c, b, scr, int(kLookWords), vertices, n, triangles, m, n_leaf, n_out, n_leaf_out);
}

}  // namespace prg
