// Device-wide primitives: exclusive scan of int32 (single-pass, lookback.h) and
// a stable LSD radix sort of (uint32 key, uint32 value) pairs.
//
// Radix sort, one 8-bit digit per pass (3D key bits -> ceil(3D/8) passes):
//   upsweep   - each workgroup counts the digits of its 4096-key tile in LDS
//               and writes a digit-major histogram [256][tiles];
//   scan      - exclusive scan of that histogram gives every (digit, tile)
//               its global output offset;
//   downsweep - each wave ranks its 1024 keys stably with wave64 ballots
//               (peers with the same digit via 8 ballots, rank = popcount of
//               lower peers + running per-wave count), the tile is reordered
//               by digit in LDS, and written out in digit runs so the global
//               stores are contiguous.
// Stability holds because waves own consecutive sub-tiles, items are visited
// in input order and tiles are laid out digit-major in the scan.
#include "lookback.h"

namespace prg {
namespace {

constexpr int kScanItems = 16;  // consecutive elements per thread

// Threads of a scan's workgroups: a tile costs about 50 ns of its own in the
// chain of tiles (the ticket, the look-back), so beyond 2^20 elements a tile is
// four times as large (5.6 M elements: 81 us with 1,359 tiles of 4,096, 51 us
// with a quarter of them; two arrays 55 and 42); below, the smaller ones give
// the chip more workgroups.
constexpr int kScanSmall = 256, kScanLarge = 1024;
int scan_block(int64_t n) { return n > (int64_t(1) << 20) ? kScanLarge : kScanSmall; }

// v[k] = in[base + k], 0 from n on; `wide`: 16-byte loads where all are in range
__device__ __forceinline__ int32_t load_items(const int32_t* __restrict__ in, int64_t base, int64_t n, bool wide,
                                              int32_t v[kScanItems]) {
    if (wide && base + kScanItems <= n) {
#pragma unroll
        for (int k = 0; k < kScanItems; k += 4) *reinterpret_cast<int4*>(v + k) = *reinterpret_cast<const int4*>(in + base + k);
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; k++) v[k] = base + k < n ? in[base + k] : 0;
    }
    int32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) s += v[k];
    return s;
}

__device__ __forceinline__ void store_items(int32_t* __restrict__ out, int64_t base, int64_t n, bool wide, int32_t ex,
                                            int32_t v[kScanItems]) {
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        const int32_t t = v[k];
        v[k] = ex;
        ex += t;
    }
    if (wide && base + kScanItems <= n) {
#pragma unroll
        for (int k = 0; k < kScanItems; k += 4) *reinterpret_cast<int4*>(out + base + k) = *reinterpret_cast<int4*>(v + k);
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; k++)
            if (base + k < n) out[base + k] = v[k];
    }
}

// Exclusive scan of one array, or of two of the same length (TWO), in one
// launch (lookback.h).  Bound by its launch (about 4 us) up to about 10^5
// elements, then by the memory it reads and writes once.
template <bool TWO, int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_scan(const int32_t* in_a, int32_t* out_a, int32_t* total_a,
                                                     const int32_t* in_b, int32_t* out_b, int32_t* total_b, int64_t n,
                                                     uint32_t tiles, bool wide, LookState state) {
    __shared__ int32_t w[BLOCK / 64];
    __shared__ int32_t before[2];
    const LookTile t = look_begin(state, tiles);
    if (t.tile >= tiles) return;  // (uniform)
    const int64_t base = int64_t(t.tile) * (BLOCK * kScanItems) + int64_t(threadIdx.x) * kScanItems;
    int32_t va[kScanItems], vb[kScanItems];
    const int32_t sa = load_items(in_a, base, n, wide, va);
    const int32_t sb = TWO ? load_items(in_b, base, n, wide, vb) : 0;
    int32_t ta, tb = 0;
    const int32_t ea = block_exclusive_scan(sa, w, ta);
    const int32_t eb = TWO ? block_exclusive_scan(sb, w, tb) : 0;
    const int wave = threadIdx.x >> 6;
    if (wave == 0 || (TWO && wave == 1)) {
        const int32_t mine = wave == 0 ? ta : tb;
        const int32_t x = look_back(state, wave, t, tiles, mine);
        if ((threadIdx.x & 63) == 0) {
            before[wave] = x;
            int32_t* total = wave == 0 ? total_a : total_b;
            if (t.tile == tiles - 1 && total) *total = x + mine;
        }
    }
    __syncthreads();
    look_end(state, t, tiles);
    store_items(out_a, base, n, wide, before[0] + ea, va);
    if (TWO) store_items(out_b, base, n, wide, before[1] + eb, vb);
}

// ---- radix sort ------------------------------------------------------------------
constexpr int kSortBlock = 256;           // 4 waves
constexpr int kSortItems = 16;            // keys per thread
constexpr int kSortTile = kSortBlock * kSortItems;
constexpr int kWaveTile = 64 * kSortItems;  // 1024 keys per wave

__global__ void __launch_bounds__(kSortBlock) k_radix_upsweep(const uint32_t* keys, int64_t n, int shift,
                                                                int32_t* hist, int tiles) {
    __shared__ int32_t cnt[256];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    const int64_t base = int64_t(blockIdx.x) * kSortTile;
#pragma unroll
    for (int k = 0; k < kSortItems; k++) {
        int64_t i = base + k * kSortBlock + threadIdx.x;
        if (i < n) atomicAdd(&cnt[(keys[i] >> shift) & 255u], 1);
    }
    __syncthreads();
    hist[int64_t(threadIdx.x) * tiles + blockIdx.x] = cnt[threadIdx.x];
}

__global__ void __launch_bounds__(kSortBlock) k_radix_downsweep(const uint32_t* keys_in, const uint32_t* vals_in,
                                                                  uint32_t* keys_out, uint32_t* vals_out, int64_t n,
                                                                  int shift, const int32_t* offsets, int tiles,
                                                                  bool counts) {
    __shared__ int32_t wcnt[4][256];     // per-wave digit counts, then per-wave digit offsets
    __shared__ int32_t tile_off[256];    // digit start inside the tile
    __shared__ int32_t glob_off[256];    // digit start in the output
    __shared__ uint32_t skeys[kSortTile];
    __shared__ uint32_t svals[kSortTile];
    __shared__ int32_t wsum[4];

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < 4 * 256; i += kSortBlock) (&wcnt[0][0])[i] = 0;
    if (counts) {
        // few tiles: their digit counts instead of the scanned offsets (thread
        // t adds up digit t's)
        int32_t before = 0, all = 0;
        for (int i = 0; i < tiles; i++) {
            const int32_t v = offsets[int64_t(threadIdx.x) * tiles + i];
            before += i < int(blockIdx.x) ? v : 0;
            all += v;
        }
        int32_t tot;
        glob_off[threadIdx.x] = before + block_exclusive_scan(all, wsum, tot);
    } else {
        glob_off[threadIdx.x] = offsets[int64_t(threadIdx.x) * tiles + blockIdx.x];
    }
    __syncthreads();

    const int64_t wbase = int64_t(blockIdx.x) * kSortTile + int64_t(wave) * kWaveTile;
    uint32_t k_reg[kSortItems], v_reg[kSortItems];
    int32_t r_reg[kSortItems];
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
    for (int k = 0; k < kSortItems; k++) {
        const int64_t i = wbase + k * 64 + lane;
        const bool valid = i < n;
        k_reg[k] = valid ? keys_in[i] : 0u;
        v_reg[k] = valid ? vals_in[i] : 0u;
        const uint32_t digit = (k_reg[k] >> shift) & 255u;
        // lanes with the same digit: intersect 8 ballots
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const uint64_t bb = __ballot((digit >> b) & 1u);
            peers &= ((digit >> b) & 1u) ? bb : ~bb;
        }
        int32_t before = 0;
        if (valid) before = wcnt[wave][digit];
        const int32_t rank = before + __popcll(peers & lt_mask);
        // the lowest lane of each peer group advances the running count
        if (valid && (peers & lt_mask) == 0ull) wcnt[wave][digit] = before + __popcll(peers);
        r_reg[k] = valid ? rank : -1;
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // thread t owns digit t: exclusive offsets across waves, tile totals
    {
        const int d = threadIdx.x;
        int32_t run = 0;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            int32_t c = wcnt[w][d];
            wcnt[w][d] = run;
            run += c;
        }
        int32_t tot;
        int32_t ex = block_exclusive_scan(run, wsum, tot);
        tile_off[d] = ex;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kSortItems; k++) {
        if (r_reg[k] < 0) continue;
        const uint32_t digit = (k_reg[k] >> shift) & 255u;
        const int32_t pos = tile_off[digit] + wcnt[wave][digit] + r_reg[k];
        skeys[pos] = k_reg[k];
        svals[pos] = v_reg[k];
    }
    __syncthreads();
    const int64_t tbase = int64_t(blockIdx.x) * kSortTile;
    const int valid_in_tile = int((n - tbase) < kSortTile ? (n - tbase) : kSortTile);
#pragma unroll
    for (int k = 0; k < kSortItems; k++) {
        const int t = k * kSortBlock + threadIdx.x;
        if (t >= valid_in_tile) continue;
        const uint32_t key = skeys[t];
        const uint32_t digit = (key >> shift) & 255u;
        const int64_t dst = int64_t(glob_off[digit]) + (t - tile_off[digit]);
        keys_out[dst] = key;
        vals_out[dst] = svals[t];
    }
}

}  // namespace

// The scan state of a stream for `words` tile words, cleared when it grows.
LookState look_state(Scratch& scratch, int64_t words, hipStream_t s) {
    const size_t want = size_t(words) + kLookHeader;
    if (scratch.look.n < want || !scratch.look.p) {
        scratch.look.reserve(want + want / 4);
        PRG_HIP(hipMemsetAsync(scratch.look.p, 0, scratch.look.n * sizeof(uint64_t), s));
    }
    return LookState{scratch.look.p, scratch.look_error, kLookSpins};
}

void look_check(Scratch& scratch, hipStream_t s) {
    if (!__atomic_load_n(scratch.look_error, __ATOMIC_RELAXED)) return;
    PRG_HIP(hipMemsetAsync(scratch.look.p, 0, scratch.look.n * sizeof(uint64_t), s));
    PRG_HIP(hipStreamSynchronize(s));
    __atomic_store_n(scratch.look_error, 0, __ATOMIC_RELAXED);
    throw Error{PRG_E_HIP, "a scan over many tiles did not finish"};
}

void scan_exclusive(const int32_t* d_in, int32_t* d_out, int64_t n, int32_t* d_total, hipStream_t s,
                    Scratch& scratch, KernelTimer& kt) {
    if (n <= 0) {
        if (d_total) PRG_HIP(hipMemsetAsync(d_total, 0, sizeof(int32_t), s));
        return;
    }
    const int block = scan_block(n), tile = block * kScanItems;
    const int64_t tiles = (n + tile - 1) / tile;
    const LookState state = look_state(scratch, tiles, s);
    const bool wide = ((reinterpret_cast<uintptr_t>(d_in) | reinterpret_cast<uintptr_t>(d_out)) & 15) == 0;
    TimedScope ts(kt, "scan_exclusive", 8.0 * double(n));
    const auto kernel = block == kScanLarge ? k_scan<false, kScanLarge> : k_scan<false, kScanSmall>;
    kernel<<<unsigned(tiles), block, 0, s>>>(d_in, d_out, d_total, nullptr, nullptr, nullptr, n, uint32_t(tiles), wide,
                                             state);
    PRG_CHECK_LAUNCH();
}

void scan_exclusive2(const int32_t* a_in, int32_t* a_out, int32_t* a_total, const int32_t* b_in, int32_t* b_out,
                     int32_t* b_total, int64_t n, hipStream_t s, Scratch& scratch, KernelTimer& kt) {
    if (n <= 0) {
        scan_exclusive(a_in, a_out, n, a_total, s, scratch, kt);
        scan_exclusive(b_in, b_out, n, b_total, s, scratch, kt);
        return;
    }
    const int block = scan_block(n), tile = block * kScanItems;
    const int64_t tiles = (n + tile - 1) / tile;
    const LookState state = look_state(scratch, 2 * tiles, s);
    const bool wide = ((reinterpret_cast<uintptr_t>(a_in) | reinterpret_cast<uintptr_t>(a_out) |
                        reinterpret_cast<uintptr_t>(b_in) | reinterpret_cast<uintptr_t>(b_out)) & 15) == 0;
    TimedScope ts(kt, "scan_exclusive", 16.0 * double(n));
    const auto kernel = block == kScanLarge ? k_scan<true, kScanLarge> : k_scan<true, kScanSmall>;
    kernel<<<unsigned(tiles), block, 0, s>>>(a_in, a_out, a_total, b_in, b_out, b_total, n, uint32_t(tiles), wide,
                                             state);
    PRG_CHECK_LAUNCH();
}

void radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t* keys_alt, uint32_t* vals_alt, int64_t n, int bits,
                      hipStream_t s, Scratch& scratch, KernelTimer& kt) {
    if (n <= 1 || bits <= 0) return;
    const int64_t tiles64 = (n + kSortTile - 1) / kSortTile;
    const int tiles = int(tiles64);
    const int64_t hn = 256 * tiles64;
    int32_t* hist = scratch.b.reserve(size_t(hn));
    int32_t* offs = scratch.c.reserve(size_t(hn));
    uint32_t *ki = keys, *vi = vals, *ko = keys_alt, *vo = vals_alt;
    int passes = 0;
    for (int shift = 0; shift < bits; shift += 8) {
        {
            TimedScope ts(kt, "radix_upsweep", 4.0 * double(n));
            k_radix_upsweep<<<unsigned(tiles), kSortBlock, 0, s>>>(ki, n, shift, hist, tiles);
            PRG_CHECK_LAUNCH();
        }
        // up to 16 tiles (65,536 keys) each workgroup adds up the counts itself:
        // 16 loads per thread cost less than the scan's launch (about 4 us)
        const bool counts = tiles <= 16;
        if (!counts) scan_exclusive(hist, offs, hn, nullptr, s, scratch, kt);
        {
            TimedScope ts(kt, "radix_downsweep", 16.0 * double(n));
            k_radix_downsweep<<<unsigned(tiles), kSortBlock, 0, s>>>(ki, vi, ko, vo, n, shift, counts ? hist : offs,
                                                                     tiles, counts);
            PRG_CHECK_LAUNCH();
        }
        std::swap(ki, ko);
        std::swap(vi, vo);
        passes++;
    }
    if (passes & 1) {
        PRG_HIP(hipMemcpyAsync(keys, ki, size_t(n) * 4, hipMemcpyDeviceToDevice, s));
        PRG_HIP(hipMemcpyAsync(vals, vi, size_t(n) * 4, hipMemcpyDeviceToDevice, s));
    }
}

}  // namespace prg
