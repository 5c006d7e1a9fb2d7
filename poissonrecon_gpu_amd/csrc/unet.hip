// Learned warm start: a 3-D U-Net on the dense grid of one coarse depth
// (G^3 cells, G = 2^depth) mapping the depth's divergence (normalised by its
// root-mean-square) and node mask to the solution on the same scale.  It has
// no counterpart in the reference, whose per-depth solves always start from
// zero (main.cu:1237-1329); CG still runs to the same tolerance, so the
// network can only change the iteration count.
//
// Architecture (4 levels, 16-32-64-64 channels, every 3x3x3 convolution
// followed by ReLU, a 1x1 head):
//   e0: conv 16->16, 16->16 (G)      e1: pool, 16->32, 32->32 (G/2)
//   e2: pool, 32->64, 64->64 (G/4)   b:  pool, 64->64, 64->64 (G/8)
//   d2: up, concat e2, 128->64, 64->64;  d1: up, concat e1, 96->32, 32->32
//   d0: up, concat e0, 48->16, 16->16;   head: 16->1
// Input channels: normalised divergence, node mask, zeros (16 in all).
//
// Convolutions are implicit GEMMs on the BF16 matrix cores
// (v_mfma_f32_16x16x16_bf16, FP32 accumulate): M = voxels, N = output
// channels, K = 27 taps x input channels.  Activations are FP32 in memory
// (channels last) and rounded to BF16 as the fragments load; weights keep an
// FP32 master copy (Adam) and a BF16 copy.  The data gradient is the same
// kernel with the weights flipped and transposed; the weight gradient is a
// GEMM over voxels in fixed chunks whose partials are summed in a fixed
// order, so training is deterministic.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <vector>

#include "../../include/prg_unet.h"
#include "ctx.h"

namespace prg {
namespace {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kT = 256;          // threads per workgroup (4 waves)
constexpr int kWChunk = 2048;    // voxels per weight-gradient partial
constexpr int kMaxBatch = 16;    // samples per launch (training)

__device__ __forceinline__ short bf(float f) {
    const __bf16 h = (__bf16)f;
    return __builtin_bit_cast(short, h);
}

// two values as BF16 in one word, the first in the low half
__device__ __forceinline__ uint32_t bf2(float a, float b) {
    return uint32_t(uint16_t(bf(a))) | (uint32_t(uint16_t(bf(b))) << 16);
}

// Input of a convolution: channels [0, clo) come from `lo` (grid G / 2,
// nearest upsampling), channels [clo, clo + cskip) from `skip` (grid G); clo
// is 0 for a plain input.  Channel counts are 16, 32 or 64 per source.
struct ConvIn {
    const float* lo;
    int clo;
    const float* skip;
    int cskip;
};

// Output of a convolution: channels [0, split) to `lo`, [split, cout) to `hi`,
// each a tensor of its own (split = cout for a plain output).
struct ConvOut {
    float* lo;
    int split;
    float* hi;
};

// The workgroup's sample of a batch (blockIdx.y): tensors hold their samples
// one after another.
__device__ __forceinline__ int64_t sample_offset(int G, int c) { return int64_t(blockIdx.y) * G * G * G * c; }

__device__ __forceinline__ ConvIn sample_of(ConvIn s, int G) {
    s.lo += s.clo ? sample_offset(G >> 1, s.clo) : 0;
    s.skip += sample_offset(G, s.cskip);
    return s;
}

__host__ __device__ __forceinline__ int log2i(int v) { return 31 - __builtin_clz(v); }

// a / d for 0 <= a < 2^20 and 1 <= d < 2^10 (inv = 1.0f / d): the float
// estimate is within one of the quotient and is corrected
__device__ __forceinline__ int small_div(int a, int d, float inv) {
    int q = int(float(a) * inv);
    if (q * d > a) q--;
    if ((q + 1) * d <= a) q++;
    return q;
}

constexpr int kLoadBatch = 8;  // halo loads in flight per thread

// One source of the halo: HX x HY x HZ voxels x c channels into LDS channels
// [choff, choff + c); HALF reads the source at G / 2 (nearest upsampling).
// Each thread issues kLoadBatch independent loads before it converts and
// stores any of them.
template <bool HALF>
__device__ __forceinline__ void load_halo(s4* halo4, int H, int HY, int HZ, const float* __restrict__ src, int c,
                                          int choff, int ox, int oy, int oz, int G) {
    const int shift = log2i(c >> 2);
    const int total = H << shift;
    const int Gs = HALF ? G >> 1 : G;
    const float invz = 1.0f / float(HZ), invy = 1.0f / float(HY);
    for (int base = threadIdx.x; base < total; base += kT * kLoadBatch) {
        float4 v[kLoadBatch];
        int dst[kLoadBatch];
#pragma unroll
        for (int k = 0; k < kLoadBatch; k++) {
            const int it = base + k * kT;
            v[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            dst[k] = -1;
            if (it < total) {
                const int h = it >> shift, c4 = it & ((1 << shift) - 1);
                const int hxy = small_div(h, HZ, invz), hz = h - hxy * HZ;
                const int hx = small_div(hxy, HY, invy), hy = hxy - hx * HY;
                const int gx = ox + hx - 1, gy = oy + hy - 1, gz = oz + hz - 1;
                if (gx >= 0 && gy >= 0 && gz >= 0 && gx < G && gy < G && gz < G) {
                    const int64_t vox = HALF ? (int64_t(gx >> 1) * Gs + (gy >> 1)) * Gs + (gz >> 1)
                                             : (int64_t(gx) * G + gy) * G + gz;
                    v[k] = *reinterpret_cast<const float4*>(src + vox * c + 4 * c4);
                }
                const int ch = choff + 4 * c4;
                dst[k] = ((ch >> 4) * H + h) * 4 + ((ch >> 2) & 3);
            }
        }
#pragma unroll
        for (int k = 0; k < kLoadBatch; k++)
            if (dst[k] >= 0) halo4[dst[k]] = s4{bf(v[k].x), bf(v[k].y), bf(v[k].z), bf(v[k].w)};
    }
}

// out[v, co] = act(bias[co] + sum_t sum_ci bf16(in[v + off_t, ci]) * w[t][co][ci])
// (w as packed_at lays it out)
//
// On grids of 4^3 and 2^3, with 2, 4 or 8 N-tiles (16 output channels each):
// one workgroup per brick of BX x BY x BZ output voxels (x, y, z; z fastest),
// at most 16.  The brick's input halo, (BX + 2)(BY + 2)(BZ + 2) voxels, is
// staged in LDS as BF16, 16-channel slice after slice: lds[s][h][16]; each
// wave loads whole halo rows (contiguous in memory).  The brick's voxels in
// (x, y, z) order are one M-tile; wave w computes it for N-tiles [NA w,
// NA w + NA).
// MFMA lane layout (16x16x16): lane l holds A[l % 16][4 (l / 16) + e],
// B[4 (l / 16) + e][l % 16] and D[4 (l / 16) + e][l % 16], e = 0..3.  K runs
// over slices, then taps; a slice's 27 weight fragments are loaded together.
template <int NA>
__global__ void __launch_bounds__(kT) k_conv3(ConvIn src, const short* __restrict__ w, const float* __restrict__ bias,
                                             int G, int BX, int BY, int BZ, int relu, ConvOut dst, int cout) {
    extern __shared__ s4 halo4[];
    const short* halo = reinterpret_cast<const short*>(halo4);
    const int cin = src.clo + src.cskip;
    src = sample_of(src, G);
    const int HY = BY + 2, HZ = BZ + 2, HYZ = HY * HZ, H = (BX + 2) * HYZ;
    const int nbz = G / BZ, nby = G / BY;
    int b = blockIdx.x;
    const int oz = (b % nbz) * BZ;
    b /= nbz;
    const int oy = (b % nby) * BY;
    const int ox = (b / nby) * BX;
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int i = l & 15, kq = l >> 4;
    const int NT = cout >> 4, S = cin >> 4, nvox = BX * BY * BZ;
    const bool active = (wave + 1) * NA <= NT;
    // the first slice's weight fragments are in flight while the halo loads
    const short* wl = w + ((active ? wave : 0) * NA * 16 + i) * 16 + 4 * kq;
    s4 wr[27][NA];
#pragma unroll
    for (int t = 0; t < 27; t++)
#pragma unroll
        for (int n = 0; n < NA; n++) wr[t][n] = *reinterpret_cast<const s4*>(wl + (t * cout + n * 16) * 16);
    if (src.clo) load_halo<true>(halo4, H, HY, HZ, src.lo, src.clo, 0, ox, oy, oz, G);
    load_halo<false>(halo4, H, HY, HZ, src.skip, src.cskip, src.clo, ox, oy, oz, G);
    __syncthreads();
    if (!active) return;  // idle wave; no barrier follows
    // lanes past the brick's voxels (2^3 grids) read the brick's first voxel,
    // whose 27 neighbours are all in the halo, and use zeros
    const bool ok = i < nvox;
    const int hb = ok ? (i / (BY * BZ) + 1) * HYZ + ((i / BZ) % BY + 1) * HZ + i % BZ + 1 : HYZ + HZ + 1;
    // three partial sums over alternating taps keep independent MFMAs in flight
    f4 acc[3][NA];
#pragma unroll
    for (int x = 0; x < 3; x++)
#pragma unroll
        for (int n = 0; n < NA; n++) acc[x][n] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    const s4 zero4 = s4{0, 0, 0, 0};
    for (int sl = 0; sl < S; sl++) {
        const short* hs = halo + sl * H * 16 + 4 * kq;
        // next slice's weights (the last slice re-reads its own: in bounds, unused)
        const int nsl = sl + 1 < S ? sl + 1 : sl;
#pragma unroll
        for (int g = 0; g < 3; g++) {
            // the nine taps with dx = g - 1: their A fragments first, then the MFMAs
            s4 a[9];
#pragma unroll
            for (int j = 0; j < 9; j++) {
                const int toff = (g - 1) * HYZ + (j / 3 - 1) * HZ + (j % 3 - 1);
                a[j] = *reinterpret_cast<const s4*>(hs + (hb + toff) * 16);
            }
#pragma unroll
            for (int j = 0; j < 9; j++) a[j] = ok ? a[j] : zero4;
#pragma unroll
            for (int j = 0; j < 9; j++) {
                const int t = 9 * g + j;
#pragma unroll
                for (int n = 0; n < NA; n++) {
                    acc[j % 3][n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[j], wr[t][n], acc[j % 3][n], 0, 0, 0);
                    wr[t][n] = *reinterpret_cast<const s4*>(wl + ((nsl * 27 + t) * cout + n * 16) * 16);
                }
            }
        }
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int q = 4 * kq + e;
        if (q >= nvox) continue;
        const int gx = ox + q / (BY * BZ), gy = oy + (q / BZ) % BY, gz = oz + q % BZ;
        const int64_t v = (int64_t(gx) * G + gy) * G + gz;
#pragma unroll
        for (int n = 0; n < NA; n++) {
            const int co = (wave * NA + n) * 16 + i;
            const bool hi = co >= dst.split;
            const int oc = hi ? cout - dst.split : dst.split;
            float* o = (hi ? dst.hi : dst.lo) + sample_offset(G, oc) + v * oc + co - (hi ? dst.split : 0);
            float val = (acc[0][n][e] + acc[1][n][e]) + acc[2][n][e];
            if (bias) val = val + bias[co];
            if (relu) val = val > 0.0f ? val : 0.0f;
            *o = val;
        }
    }
}

// The same sums, in the same order, on grids of 8^3 and more, where a tile is
// a run of voxels: ZL = 16 voxels of a z row, or two rows of 8.
//
// A workgroup of 4 waves, WX x WY in space by WN in output channels (16
// each); a wave computes RX x RY tiles.  The halo lies in LDS one 16-channel
// slice at a time (the next slice loads while this one is used), a slice as
// four planes of 4 channels, so the 16 voxels of a fragment read are
// consecutive 8-byte words (no bank conflict).  A fragment, shifted in z by a
// tap, serves every tile it lies next to: 48 reads instead of 108 for the 27
// taps of 2 x 2 tiles.  All 27 weight fragments of a slice sit in registers;
// each is replaced by the next slice's after its last use.  The weights are
// the MFMA's first operand, so a lane ends with 4 channels of one voxel and
// stores 16 bytes.
// Sizes known at compile time keep the index arithmetic to shifts and
// constants; it had bounded these convolutions (3300 vector instructions a
// wave against 108 MFMAs of 16 -> 16 channels).
template <int LZ, int RX, int RY, int WX, int WY, int WN>
struct ConvTile {
    static constexpr int ZL = 1 << LZ, YS = 16 >> LZ;  // a tile: YS rows of ZL voxels
    static constexpr int BX = WX * RX, BY = WY * RY * YS;
    static constexpr int HX = BX + 2, HY = BY + 2, HZ = ZL + 2, H = HX * HY * HZ;
    // words (of 4 channels) per plane, 160 bytes past a multiple of 256: the
    // staging's writes of a half-wave, 8 voxels in 4 planes, meet no bank
    // more often than their 256 bytes need
    static constexpr int P = H + ((20 - H % 32) + 32) % 32;
    static constexpr int L = (4 * H + kT - 1) / kT;  // staging loads per thread
};

template <int LZ, int RX, int RY, int WX, int WY, int WN, bool MULTI>
__global__ void __launch_bounds__(kT, RX * RY > 1 ? (MULTI ? 2 : 4) : (MULTI ? 3 : 5)) k_conv3_rows(
    ConvIn src, const short* __restrict__ w, const float* __restrict__ bias, int G, int relu, ConvOut dst, int cout,
    int ntg) {
    using C = ConvTile<LZ, RX, RY, WX, WY, WN>;
    static_assert(WX * WY * WN * 64 == kT, "one wave per part");
    constexpr int FY = C::YS * (RY - 1) + 3;
    __shared__ s4 halo[(MULTI ? 2 : 1) * 4 * C::P];
    const int cin = src.clo + src.cskip;
    src = sample_of(src, G);
    const int nbz = G >> LZ, nby = G / C::BY;
    // workgroups are dealt to the 8 XCDs in turn: each XCD takes one
    // contiguous range of bricks, whose halos meet in its L2
    int b = blockIdx.x;
    if ((gridDim.x & 7) == 0) b = (b & 7) * int(gridDim.x >> 3) + (b >> 3);
    const int oz = (b & (nbz - 1)) << LZ;  // (both counts are powers of two)
    b >>= log2i(nbz);
    const int oy = (b & (nby - 1)) * C::BY, ox = (b >> log2i(nby)) * C::BX;
    const int tid = threadIdx.x, l = tid & 63, i = l & 15, kq = l >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wx = wave % WX, wy = (wave / WX) % WY, wn = wave / (WX * WY);
    const int S = cin >> 4, Q = S * (ntg / WN);
    int nt = blockIdx.z * ntg + wn, sl = 0;

    // staging: this thread's words, word k of halo voxel (tid + k kT) / 4
    const int c4 = tid & 3;
    int vox[C::L];
    float4 st[C::L];
    auto stage_load = [&](int slice) {
        const bool lo = slice * 16 < src.clo;
        if (slice == 0 || slice * 16 == src.clo) {
            // voxel indices in this source (-1 outside the grid)
#pragma unroll
            for (int k = 0; k < C::L; k++) {
                const int h = (tid + k * kT) >> 2;
                const int hxy = h / C::HZ, hz = h - hxy * C::HZ, hx = hxy / C::HY, hy = hxy - hx * C::HY;
                const int gx = ox + hx - 1, gy = oy + hy - 1, gz = oz + hz - 1;
                const bool in = h < C::H && uint32_t(gx) < uint32_t(G) && uint32_t(gy) < uint32_t(G) &&
                                uint32_t(gz) < uint32_t(G);
                const int sh = lo ? 1 : 0, Gs = G >> sh;
                vox[k] = in ? ((gx >> sh) * Gs + (gy >> sh)) * Gs + (gz >> sh) : -1;
            }
        }
        const int c = lo ? src.clo : src.cskip;
        const float* p = (lo ? src.lo + slice * 16 : src.skip + (slice * 16 - src.clo)) + 4 * c4;
#pragma unroll
        for (int k = 0; k < C::L; k++) {
            st[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (vox[k] >= 0) st[k] = *reinterpret_cast<const float4*>(p + int64_t(vox[k]) * c);
        }
    };
    auto stage_store = [&](int buf) {
        s4* d = halo + (buf * 4 + c4) * C::P + (tid >> 2);
#pragma unroll
        for (int k = 0; k < C::L; k++)
            if (4 * C::H % kT == 0 || k + 1 < C::L || tid + k * kT < 4 * C::H)
                d[k * (kT / 4)] = s4{bf(st[k].x), bf(st[k].y), bf(st[k].z), bf(st[k].w)};
    };
    const int tstep = cout * 16;
    auto weights = [&](int ntile, int slice) { return w + (slice * 27 * cout + ntile * 16 + i) * 16 + 4 * kq; };
    s4 wr[27];
    {
        const short* wl = weights(nt, 0);
#pragma unroll
        for (int t = 0; t < 27; t++) wr[t] = *reinterpret_cast<const s4*>(wl + t * tstep);
    }
    stage_load(0);
    stage_store(0);
    const int vy = i >> LZ, vz = i & (C::ZL - 1);  // the lane's voxel of a tile
    const int frag0 = kq * C::P + ((wx * RX) * C::HY + wy * RY * C::YS + vy) * C::HZ + vz;
    // three partial sums, one per dz, keep independent MFMAs in flight
    f4 acc[3][RX][RY];
    for (int q = 0;; q++) {
        const bool more = MULTI && q + 1 < Q;
        const int nsl = sl + 1 < S ? sl + 1 : 0, nnt = sl + 1 < S ? nt : nt + WN;
        const bool restage = more && S > 1;
        if (restage) stage_load(nsl);
        if (q == 0 || S > 1) __syncthreads();
        const short* wnext = weights(more ? nnt : nt, more ? nsl : sl);  // (the last re-reads its own: unused)
        if (sl == 0)
#pragma unroll
            for (int z = 0; z < 3; z++)
#pragma unroll
                for (int x = 0; x < RX; x++)
#pragma unroll
                    for (int y = 0; y < RY; y++) acc[z][x][y] = f4{0.0f, 0.0f, 0.0f, 0.0f};
        const s4* frag = halo + (MULTI && S > 1 ? (q & 1) * 4 * C::P : 0) + frag0;
#pragma unroll
        for (int fx = 0; fx < RX + 2; fx++)
#pragma unroll
            for (int fy = 0; fy < FY; fy++)
#pragma unroll
                for (int z = 0; z < 3; z++) {
                    const s4 a = frag[(fx * C::HY + fy) * C::HZ + z];
#pragma unroll
                    for (int x = 0; x < RX; x++)
#pragma unroll
                        for (int y = 0; y < RY; y++) {
                            const int dx = fx - x, dy = fy - C::YS * y;
                            if (dx < 0 || dx > 2 || dy < 0 || dy > 2) continue;
                            const int t = (dx * 3 + dy) * 3 + z;
                            acc[z][x][y] =
                                __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wr[t], a, acc[z][x][y], 0, 0, 0);
                        }
                    if (MULTI) {
                        const int dx = fx - (RX - 1), dy = fy - C::YS * (RY - 1);
                        if (dx >= 0 && dy >= 0) {
                            const int t = (dx * 3 + dy) * 3 + z;
                            wr[t] = *reinterpret_cast<const s4*>(wnext + t * tstep);
                        }
                    }
                }
        if (sl == S - 1) {
            const bool hi = nt * 16 >= dst.split;
            const int oc = hi ? cout - dst.split : dst.split;
            float* out = (hi ? dst.hi - dst.split : dst.lo) + sample_offset(G, oc) + nt * 16 + 4 * kq;
            float4 bv = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (bias) bv = *reinterpret_cast<const float4*>(bias + nt * 16 + 4 * kq);
#pragma unroll
            for (int x = 0; x < RX; x++)
#pragma unroll
                for (int y = 0; y < RY; y++) {
                    const int gx = ox + wx * RX + x, gy = oy + (wy * RY + y) * C::YS + vy, gz = oz + vz;
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        v[e] = (acc[0][x][y][e] + acc[1][x][y][e]) + acc[2][x][y][e];
                        const float be = e == 0 ? bv.x : e == 1 ? bv.y : e == 2 ? bv.z : bv.w;
                        if (bias) v[e] = v[e] + be;
                        if (relu) v[e] = v[e] > 0.0f ? v[e] : 0.0f;
                    }
                    *reinterpret_cast<float4*>(out + (int64_t(gx * G + gy) * G + gz) * oc) =
                        make_float4(v[0], v[1], v[2], v[3]);
                }
        }
        if (!more) break;
        if (restage) stage_store((q + 1) & 1);
        sl = nsl;
        nt = nnt;
    }
}

// dW partials: part[ch][t][co][ci] = sum over the chunk's voxels v of
// bf16(g[v, co]) * bf16(in[v + off_t, ci]), 16 voxels per MFMA in voxel order.
//
// On grids of 8^3 and more (k_wgrad_rows): one workgroup per (chunk, dx, co
// tile, ci tile), one wave per dy, the three dz of a wave's taps in three
// accumulators.  The chunk passes through LDS in stages of 512 voxels, the
// gradient and the input's rows (one more on either side) as BF16, channel by
// channel with z innermost, so a lane's four voxels of one channel are one
// 8-byte read; the fragments shifted by dz = -1 and 1 are funnel shifts of it
// and the two words beside it.  Rows carry zeros on both ends in z, rows
// outside the grid in x are staged as zeros and rows outside in y are
// replaced by zeros.  The channel strides are 4 words past a multiple of 32
// (no bank conflict beyond the two cycles a half-wave's 256 bytes need).
// What bounds it is the staging (each element is read for 3 dx and per tile
// of the other operand), not the matrix cores; a stage's loads are in flight
// during the products of the one before.  One wave per (chunk, tap,
// tiles) with scalar loads straight from memory and 64-bit divisions per
// element took 440 us for 16 -> 16 channels on 64^3 and 990 us for 48 -> 16.
constexpr int kWStage = 512;  // voxels per stage

template <int LG>
__global__ void __launch_bounds__(192) k_wgrad_rows(ConvIn src, const float* __restrict__ g, int cout, int nchunk,
                                                   float* __restrict__ part) {
    constexpr int G = 1 << LG, V = G * G * G, R = kWStage / G, ROWS = R + 2, RS = G + 8;
    constexpr int CW0 = ROWS * RS / 2, CW = CW0 + ((4 - CW0) & 31);  // words per input channel
    constexpr int GW = kWStage / 2 + 4;                               // words per gradient channel
    __shared__ __align__(16) uint32_t si[16 * CW];
    __shared__ __align__(16) uint32_t sg[16 * GW];
    const int cin = src.clo + src.cskip;
    src = sample_of(src, G);
    g += sample_offset(G, cout);
    part += int64_t(blockIdx.y) * nchunk * 27 * cout * cin;
    const int ntc = cout >> 4, nti = cin >> 4;
    int b = blockIdx.x;
    const int ch = b % nchunk;  // fastest: workgroups of one chunk meet on few XCDs
    b /= nchunk;
    const int cit = b % nti;
    b /= nti;
    const int cot = b % ntc;
    const int dx = b / ntc - 1;
    const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63;
    const int i = l & 15, kq = l >> 4, dy = wave - 1;
    const bool lo = cit * 16 < src.clo;
    const int sc = lo ? src.clo : src.cskip;  // channels of the source tensor
    const float* sp = lo ? src.lo + cit * 16 : src.skip + (cit * 16 - src.clo);
    const float* gp = g + cot * 16;
    // the zeros beyond both ends of every row
    for (int t = tid; t < 16 * ROWS; t += 192) {
        uint32_t* r = si + (t / ROWS) * CW + (t % ROWS) * (RS / 2);
        r[1] = 0;
        r[G / 2 + 2] = 0;
    }
    f4 acc[3];
#pragma unroll
    for (int z = 0; z < 3; z++) acc[z] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    const int v0 = ch * kWChunk, v1 = v0 + kWChunk < V ? v0 + kWChunk : V;
    // a stage's loads: pairs of voxels along z, four channels each
    constexpr int NI = (ROWS * G * 2 + 191) / 192, NG = (kWStage * 2 + 191) / 192;
    float4 ia[NI], ib[NI], ga[NG], gb[NG];
    const int zstep = lo ? 0 : sc;  // to the second voxel (upsampled: the same)
    auto load_stage = [&](int vs) {
        const int row0 = vs >> LG;  // first row (x G + y) of the stage
#pragma unroll
        for (int k = 0; k < NI; k++) {
            const int t = tid + k * 192, cq = t & 3, zp = (t >> 2) & (G / 2 - 1), r = t >> (LG + 1);
            const int row = row0 - 1 + r, x = (row >> LG) + dx, y = row & (G - 1);
            ia[k] = ib[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (r < ROWS && row >= 0 && row < G * G && x >= 0 && x < G) {
                const int vox = lo ? (((x >> 1) << (LG - 1)) + (y >> 1)) * (G / 2) + zp : ((x << LG) + y) * G + 2 * zp;
                const float* q = sp + int64_t(vox) * sc + 4 * cq;
                ia[k] = *reinterpret_cast<const float4*>(q);
                ib[k] = *reinterpret_cast<const float4*>(q + zstep);
            }
        }
#pragma unroll
        for (int k = 0; k < NG; k++) {
            const int t = tid + k * 192, cq = t & 3, vp = t >> 2;
            const float* q = gp + int64_t(vs + 2 * (vp < kWStage / 2 ? vp : 0)) * cout + 4 * cq;
            ga[k] = *reinterpret_cast<const float4*>(q);
            gb[k] = *reinterpret_cast<const float4*>(q + cout);
        }
    };
    load_stage(v0);
    for (int vs = v0; vs < v1; vs += kWStage) {
        __syncthreads();  // the previous stage's reads
        const int row0 = vs >> LG;
#pragma unroll
        for (int k = 0; k < NI; k++) {
            const int t = tid + k * 192, cq = t & 3, zp = (t >> 2) & (G / 2 - 1), r = t >> (LG + 1);
            if (r >= ROWS) continue;
            uint32_t* d = si + 4 * cq * CW + r * (RS / 2) + 2 + zp;
            d[0] = bf2(ia[k].x, ib[k].x);
            d[CW] = bf2(ia[k].y, ib[k].y);
            d[2 * CW] = bf2(ia[k].z, ib[k].z);
            d[3 * CW] = bf2(ia[k].w, ib[k].w);
        }
#pragma unroll
        for (int k = 0; k < NG; k++) {
            const int t = tid + k * 192, cq = t & 3, vp = t >> 2;
            if (vp >= kWStage / 2) continue;
            uint32_t* d = sg + 4 * cq * GW + vp;
            d[0] = bf2(ga[k].x, gb[k].x);
            d[GW] = bf2(ga[k].y, gb[k].y);
            d[2 * GW] = bf2(ga[k].z, gb[k].z);
            d[3 * GW] = bf2(ga[k].w, gb[k].w);
        }
        __syncthreads();
        if (vs + kWStage < v1) load_stage(vs + kWStage);  // in flight during the products
#pragma unroll 4
        for (int st = 0; st < kWStage / 16; st++) {
            const int v = st * 16 + 4 * kq;  // the lane's first voxel in the stage
            const int r = v >> LG, z = v & (G - 1), y = (row0 + r) & (G - 1);
            const uint2 gv = *reinterpret_cast<const uint2*>(sg + i * GW + (v >> 1));
            const uint32_t* q = si + i * CW + (r + 1 + dy) * (RS / 2) + 2 + (z >> 1);
            uint2 m = *reinterpret_cast<const uint2*>(q);
            uint32_t w0 = q[-1], w3 = q[2];
            if (y + dy < 0 || y + dy >= G) m.x = m.y = w0 = w3 = 0;
            const uint32_t s0 = __builtin_amdgcn_alignbit(m.x, w0, 16), s1 = __builtin_amdgcn_alignbit(m.y, m.x, 16),
                           s2 = __builtin_amdgcn_alignbit(w3, m.y, 16);
            const s4 av = __builtin_bit_cast(s4, gv);
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, __builtin_bit_cast(s4, make_uint2(s0, s1)), acc[0],
                                                               0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, __builtin_bit_cast(s4, m), acc[1], 0, 0, 0);
            acc[2] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(av, __builtin_bit_cast(s4, make_uint2(s1, s2)), acc[2],
                                                               0, 0, 0);
        }
    }
#pragma unroll
    for (int z = 0; z < 3; z++) {
        const int t = 9 * (dx + 1) + 3 * (dy + 1) + z;
        float* dst = part + (int64_t(ch) * 27 + t) * cout * cin;
#pragma unroll
        for (int e = 0; e < 4; e++) dst[int64_t(cot * 16 + 4 * kq + e) * cin + cit * 16 + i] = acc[z][e];
    }
}

// The same on grids under 8^3 (at most 64 voxels, which need not fill an
// MFMA): one wave per (tap, co tile, ci tile).
__global__ void __launch_bounds__(kT) k_wgrad_small(ConvIn src, const float* __restrict__ g, int cout, int G,
                                                   float* __restrict__ part) {
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
    const int cin = src.clo + src.cskip;
    src = sample_of(src, G);
    g += sample_offset(G, cout);
    part += int64_t(blockIdx.y) * 27 * cout * cin;
    const int ntc = cout / 16, nti = cin / 16;
    const int job = int(blockIdx.x) * 4 + wave;
    if (job >= 27 * ntc * nti) return;
    const int cit = job % nti, cot = (job / nti) % ntc, t = job / (nti * ntc);
    const int V = G * G * G;
    const int i = l & 15, kq = l >> 4;
    const int co = cot * 16 + i, ci = cit * 16 + i;
    f4 acc = f4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int vb = 0; vb < V; vb += 16) {
        s4 a, b;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int v = vb + 4 * kq + e;
            float ga = 0.0f, xb = 0.0f;
            if (v < V) {
                ga = g[v * cout + co];
                const int x = v / (G * G) + t / 9 - 1, y = (v / G) % G + (t / 3) % 3 - 1, z = v % G + t % 3 - 1;
                if (x >= 0 && y >= 0 && z >= 0 && x < G && y < G && z < G)
                    xb = ci < src.clo ? src.lo[(((x >> 1) * (G / 2) + (y >> 1)) * (G / 2) + (z >> 1)) * src.clo + ci]
                                      : src.skip[((x * G + y) * G + z) * src.cskip + (ci - src.clo)];
            }
            a[e] = bf(ga);
            b[e] = bf(xb);
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
    }
    float* dst = part + int64_t(t) * cout * cin;
#pragma unroll
    for (int e = 0; e < 4; e++) dst[int64_t(cot * 16 + 4 * kq + e) * cin + ci] = acc[e];
}

// ---- sums over a sample's voxels in one fixed order ----
// A bias or head gradient is a sum over all voxels in float, and a training
// step amplifies its rounding (Adam divides small gradients by their own
// size), so its order is part of the results: kChains running sums, chain t
// over the voxels t, t + kChains, .. in order, then a binary tree over the
// chains.  A group of workgroup-wide loads feeds the running sums through
// LDS: the voxels of kSteps steps are read (and their other work done) by all
// threads, kStepLanes lanes a step, and kStepLanes lanes then add them up step
// by step.  (One workgroup per channel, each thread following its own chain
// in memory, took 325 us for 16 channels on 64^3.)
constexpr int kChains = 256;
constexpr int kSumT = 512;        // threads
constexpr int kStepLanes = 32;    // lanes of a step: kStepLanes / (C / 4) chains of C channels
constexpr int kSteps = 32;        // steps in LDS at a time
constexpr int kStepLoads = kSteps * kStepLanes / kSumT;  // of each thread

// the tree over the chains' sums of one column, by one wave (every lane)
__device__ __forceinline__ float chain_tree(const float* __restrict__ bp, int cols, int col) {
    const int l = threadIdx.x & 63;
    float v0 = bp[int64_t(l) * cols + col], v1 = bp[int64_t(l + 64) * cols + col];
    const float v2 = bp[int64_t(l + 128) * cols + col], v3 = bp[int64_t(l + 192) * cols + col];
    v0 += v2;
    v1 += v3;
    v0 += v1;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v0 += __shfl_down(v0, o, 64);
    return __shfl(v0, 0, 64);
}

// For each of B samples in turn, grad[k] += sum over its chunks (in order) of
// part[b][ch][k], k < n, and in the workgroups past those db[c] += the tree
// over its chains' sums bp[b][t][c], one wave per channel
__global__ void __launch_bounds__(kT) k_grad_finish(const float* __restrict__ part, int nchunk, int64_t n,
                                                   float* __restrict__ grad, const float* __restrict__ bp, int C,
                                                   float* __restrict__ db, int B) {
    const int64_t nb = (n + kT - 1) / kT;
    if (int64_t(blockIdx.x) < nb) {
        const int64_t k = int64_t(blockIdx.x) * kT + threadIdx.x;
        if (k >= n) return;
        float total = grad[k];
        for (int b = 0; b < B; b++) {
            float s = 0.0f;
#pragma unroll 16
            for (int c = 0; c < nchunk; c++) s += part[(int64_t(b) * nchunk + c) * n + k];
            total += s;
        }
        grad[k] = total;
    } else {
        const int c = int(int64_t(blockIdx.x) - nb) * (kT / 64) + (threadIdx.x >> 6);
        if (c >= C) return;
        float total = db[c];
        for (int b = 0; b < B; b++) total += chain_tree(bp + int64_t(b) * kChains * C, C, c);
        if ((threadIdx.x & 63) == 0) db[c] = total;
    }
}

// Where the weight of tap t, output channel co and input channel ci lies in a
// convolution's BF16 weights, [ci / 16][t][co][ci % 16]: a wave's fragment of
// 16 output by 16 input channels is 512 consecutive bytes (with all input
// channels of a row together it was 32 bytes each of 16 lines).
__device__ __forceinline__ int64_t packed_at(int t, int co, int ci, int cout) {
    return ((int64_t(ci >> 4) * 27 + t) * cout + co) * 16 + (ci & 15);
}

struct PackJobs {
    int64_t woff[14];
    int32_t cin[14], cout[14];
    short *wb[14], *wf[14];
};

// The BF16 weights of every convolution (blockIdx.y) and of its data gradient:
// wb holds w[t][co][ci], wf the flipped and transposed w[26 - t][ci][co].
__global__ void __launch_bounds__(kT) k_pack(const float* __restrict__ params, PackJobs J) {
    const int k = blockIdx.y, cin = J.cin[k], cout = J.cout[k];
    const int64_t j = int64_t(blockIdx.x) * kT + threadIdx.x;
    if (j >= int64_t(27) * cout * cin) return;
    const int ci = int(j % cin), co = int((j / cin) % cout), t = int(j / (int64_t(cin) * cout));
    const short h = bf(params[J.woff[k] + j]);
    J.wb[k][packed_at(t, co, ci, cout)] = h;
    J.wf[k][packed_at(26 - t, ci, co, cin)] = h;
}

// g[v, c] *= (y[v, c] > 0), after adding the gradient pg of the output's
// average pooling (grid G / 2; null: none), and the bias gradient's running
// sums bp[t][c]: one pass over g and y for all three (the pooling's as a pass
// of its own took 130 us for 8 samples).
__global__ void __launch_bounds__(kSumT) k_relu_bias(float* __restrict__ g, const float* __restrict__ y,
                                                    const float* __restrict__ pg, int lg, int C,
                                                    float* __restrict__ bp) {
    __shared__ float4 buf[2][kSteps][kStepLanes];
    const int G = 1 << lg;
    const int64_t V = int64_t(1) << (3 * lg);
    g += int64_t(blockIdx.y) * V * C;
    y += int64_t(blockIdx.y) * V * C;
    pg += pg ? sample_offset(G >> 1, C) : 0;
    bp += int64_t(blockIdx.y) * kChains * C;
    const int lq = log2i(C) - 2, l = threadIdx.x & (kStepLanes - 1), sl = threadIdx.x / kStepLanes;
    const int q = l & ((1 << lq) - 1), t = (int(blockIdx.x) * kStepLanes + l) >> lq;  // this lane's chain
    const int nsteps = int((V + kChains - 1) / kChains);
    float4 a[kStepLoads], b[kStepLoads];
    auto load = [&](int kb) {
#pragma unroll
        for (int u = 0; u < kStepLoads; u++) {
            const int64_t v = t + int64_t(kChains) * (kb + sl + u * (kSumT / kStepLanes));
            a[u] = b[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (v >= V) continue;
            a[u] = *(reinterpret_cast<const float4*>(y + v * C) + q);
            b[u] = *(reinterpret_cast<const float4*>(g + v * C) + q);
            if (pg) {
                const int z = int(v) & (G - 1), yy = int(v >> lg) & (G - 1), x = int(v >> (2 * lg));
                const int64_t w = (((int64_t(x >> 1) << (lg - 1)) + (yy >> 1)) << (lg - 1)) + (z >> 1);
                const float4 h = *(reinterpret_cast<const float4*>(pg + w * C) + q);
                b[u].x = b[u].x + h.x * 0.125f;
                b[u].y = b[u].y + h.y * 0.125f;
                b[u].z = b[u].z + h.z * 0.125f;
                b[u].w = b[u].w + h.w * 0.125f;
            }
        }
    };
    load(0);
    float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int kb = 0, cur = 0; kb < nsteps; kb += kSteps, cur ^= 1) {
#pragma unroll
        for (int u = 0; u < kStepLoads; u++) {
            const int k = sl + u * (kSumT / kStepLanes);
            const int64_t v = t + int64_t(kChains) * (kb + k);
            if (!(a[u].x > 0.0f)) b[u].x = 0.0f;
            if (!(a[u].y > 0.0f)) b[u].y = 0.0f;
            if (!(a[u].z > 0.0f)) b[u].z = 0.0f;
            if (!(a[u].w > 0.0f)) b[u].w = 0.0f;
            if (v < V) *(reinterpret_cast<float4*>(g + v * C) + q) = b[u];
            buf[cur][k][l] = b[u];
        }
        __syncthreads();
        if (kb + kSteps < nsteps) load(kb + kSteps);  // in flight during the sums
        if (threadIdx.x < kStepLanes) {
            // (steps past the last voxel hold +0, which changes no sum that is not -0)
#pragma unroll 8
            for (int k = 0; k < kSteps; k++) {
                const float4 x = buf[cur][k][l];
                s.x += x.x;
                s.y += x.y;
                s.z += x.z;
                s.w += x.w;
            }
        }
    }
    if (threadIdx.x < kStepLanes) *(reinterpret_cast<float4*>(bp + int64_t(t) * C) + q) = s;
}

// a 2x2x2 cell's eight voxels summed in order, four channels per thread: out
// (G / 2) = f * sum.  Channels C = 2^lc, G = 2^lg.
__device__ __forceinline__ void sum_cells(const float* __restrict__ in, int lc, int lg, float f,
                                          float* __restrict__ out) {
    const int lh = lg - 1, G = 1 << lg, C = 1 << lc;
    const int64_t k = int64_t(blockIdx.x) * kT + threadIdx.x;
    if (k >= int64_t(1) << (3 * lh + lc - 2)) return;
    in += sample_offset(G, C);
    out += sample_offset(G >> 1, C);
    const int q = int(k) & ((C >> 2) - 1);
    const int64_t v = k >> (lc - 2);
    const int z = int(v) & ((1 << lh) - 1), y = int(v >> lh) & ((1 << lh) - 1), x = int(v >> (2 * lh));
    float4 a[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int64_t u = (((int64_t(2 * x + (j >> 2)) << lg) + 2 * y + ((j >> 1) & 1)) << lg) + 2 * z + (j & 1);
        a[j] = reinterpret_cast<const float4*>(in)[(u << (lc - 2)) + q];
    }
    float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int j = 0; j < 8; j++) {
        s.x += a[j].x;
        s.y += a[j].y;
        s.z += a[j].z;
        s.w += a[j].w;
    }
    reinterpret_cast<float4*>(out)[k] = make_float4(s.x * f, s.y * f, s.z * f, s.w * f);
}

// average pooling 2x2x2 (its gradient is added by k_relu_bias)
__global__ void __launch_bounds__(kT) k_pool(const float* in, int lc, int lg, float* out) {
    sum_cells(in, lc, lg, 0.125f, out);
}

// gradient of nearest upsampling
__global__ void __launch_bounds__(kT) k_up_back(const float* g, int lc, int lg, float* glo) {
    sum_cells(g, lc, lg, 1.0f, glo);
}

// head: pred[v] = f * (b + sum_c w[c] * in[v, c]) (float, c = 0..15 in order)
__global__ void __launch_bounds__(kT) k_head(const float* __restrict__ in, const float* __restrict__ w, int64_t V,
                                            float f, float* __restrict__ pred) {
    const int64_t v = int64_t(blockIdx.x) * kT + threadIdx.x;
    if (v >= V) return;
    float a[16];
#pragma unroll
    for (int c = 0; c < 16; c += 4) *reinterpret_cast<float4*>(a + c) = *reinterpret_cast<const float4*>(in + v * 16 + c);
    float s = 0.0f;
#pragma unroll
    for (int c = 0; c < 16; c++) s += w[c] * a[c];
    pred[v] = (s + w[16]) * f;
}

// Two doubles per thread summed over the workgroup (a fixed tree).
template <int kThreads = kT>
__device__ __forceinline__ void pair_sum(double& a, double& b, double* ra, double* rb) {
    const int t = threadIdx.x;
    ra[t] = a;
    rb[t] = b;
    __syncthreads();
    for (int o = kThreads / 2; o > 0; o >>= 1) {
        if (t < o) {
            ra[t] += ra[t + o];
            rb[t] += rb[t + o];
        }
        __syncthreads();
    }
    a = ra[0];
    b = rb[0];
}

constexpr int kLossVox = 2048;  // voxels per workgroup of k_loss_part
constexpr int kHeadCols = 33;   // its partials: head weights (16), head bias, d0b's bias (16)

// masked MSE: per-workgroup partials of sum_v m and sum_v m (p - t)^2 (double)
__global__ void __launch_bounds__(kT) k_loss_part(const float* __restrict__ pred, const float* __restrict__ tgt,
                                                 const float* __restrict__ mask, int64_t V, double* __restrict__ lp) {
    __shared__ double r1[kT], r2[kT];
    pred += int64_t(blockIdx.y) * V;
    tgt += int64_t(blockIdx.y) * V;
    mask += int64_t(blockIdx.y) * V;
    lp += 2 * int64_t(blockIdx.y) * gridDim.x;
    const int64_t v0 = int64_t(blockIdx.x) * kLossVox, v1 = v0 + kLossVox < V ? v0 + kLossVox : V;
    double sm = 0.0, sl = 0.0;
#pragma unroll 4
    for (int64_t v = v0 + threadIdx.x; v < v1; v += kT) {
        const double m = mask[v], d = double(pred[v]) - double(tgt[v]);
        sm += m;
        sl += m * d * d;
    }
    pair_sum(sm, sl, r1, r2);
    if (threadIdx.x == 0) {
        lp[2 * blockIdx.x] = sm;
        lp[2 * blockIdx.x + 1] = sl;
    }
}

// The loss, sum_v m (p - t)^2 / sum_v m, from the nl partials (each workgroup
// sums them in the same order), its gradient gp = 2 m (p - t) / sum m at each
// voxel, and through the head to the last convolution's pre-activation:
// gin[v, c] = gp w[c] where in[v, c] > 0, else 0.  hp[t][..]: the running sums
// of the head's weight and bias gradients and of that convolution's bias
// gradient.  (The loss in one workgroup took 530 us on 64^3 and the head's
// weight gradient in 17 took 350 us.)
__global__ void __launch_bounds__(kSumT) k_loss_back(const float* __restrict__ pred, const float* __restrict__ tgt,
                                                    const float* __restrict__ mask, const float* __restrict__ in,
                                                    const float* __restrict__ w, int64_t V,
                                                    const double* __restrict__ lp, int nl, double* __restrict__ loss,
                                                    float* __restrict__ gin, float* __restrict__ hp) {
    __shared__ double r1[kSumT], r2[kSumT];
    __shared__ float4 bw[2][kSteps][kStepLanes], bb[2][kSteps][kStepLanes];
    __shared__ float bg[2][kSteps][kStepLanes / 4];
    pred += int64_t(blockIdx.y) * V;
    tgt += int64_t(blockIdx.y) * V;
    mask += int64_t(blockIdx.y) * V;
    in += int64_t(blockIdx.y) * V * 16;
    gin += int64_t(blockIdx.y) * V * 16;
    lp += 2 * int64_t(blockIdx.y) * nl;
    hp += int64_t(blockIdx.y) * kChains * kHeadCols;
    double sm = 0.0, sl2 = 0.0;
    for (int k = threadIdx.x; k < nl; k += kSumT) {
        sm += lp[2 * k];
        sl2 += lp[2 * k + 1];
    }
    pair_sum<kSumT>(sm, sl2, r1, r2);
    const double msum = sm;
    if (blockIdx.x == 0 && threadIdx.x == 0) loss[blockIdx.y] = msum > 0.0 ? sl2 / msum : 0.0;
    const int l = threadIdx.x & (kStepLanes - 1), sl = threadIdx.x / kStepLanes;
    const int q = l & 3, t = (int(blockIdx.x) * kStepLanes + l) >> 2;
    const float4 wq = make_float4(w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]);
    const int nsteps = int((V + kChains - 1) / kChains);
    float4 a[kStepLoads];
    float m[kStepLoads], p[kStepLoads], tg[kStepLoads];
    auto load = [&](int kb) {
#pragma unroll
        for (int u = 0; u < kStepLoads; u++) {
            const int64_t v = t + int64_t(kChains) * (kb + sl + u * (kSumT / kStepLanes));
            a[u] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            m[u] = p[u] = tg[u] = 0.0f;
            if (v >= V) continue;
            a[u] = *(reinterpret_cast<const float4*>(in + v * 16) + q);
            m[u] = mask[v];
            p[u] = pred[v];
            tg[u] = tgt[v];
        }
    };
    load(0);
    float4 sw = make_float4(0.0f, 0.0f, 0.0f, 0.0f), sb = sw;
    float sg = 0.0f;
    for (int kb = 0, cur = 0; kb < nsteps; kb += kSteps, cur ^= 1) {
#pragma unroll
        for (int u = 0; u < kStepLoads; u++) {
            const int k = sl + u * (kSumT / kStepLanes);
            const int64_t v = t + int64_t(kChains) * (kb + k);
            const float gp = msum > 0.0 ? float(2.0 * m[u] * (double(p[u]) - double(tg[u])) / msum) : 0.0f;
            const float4 b = make_float4(a[u].x > 0.0f ? gp * wq.x : 0.0f, a[u].y > 0.0f ? gp * wq.y : 0.0f,
                                         a[u].z > 0.0f ? gp * wq.z : 0.0f, a[u].w > 0.0f ? gp * wq.w : 0.0f);
            if (v < V) *(reinterpret_cast<float4*>(gin + v * 16) + q) = b;
            bw[cur][k][l] = make_float4(gp * a[u].x, gp * a[u].y, gp * a[u].z, gp * a[u].w);
            bb[cur][k][l] = b;
            if (q == 0) bg[cur][k][l >> 2] = gp;
        }
        __syncthreads();
        if (kb + kSteps < nsteps) load(kb + kSteps);
        // the head's weights and bias in one wave, the convolution's bias in another
        if (threadIdx.x < kStepLanes) {
#pragma unroll 8
            for (int k = 0; k < kSteps; k++) {
                const float4 x = bw[cur][k][l];
                sw.x += x.x;
                sw.y += x.y;
                sw.z += x.z;
                sw.w += x.w;
                sg += bg[cur][k][l >> 2];
            }
        } else if (threadIdx.x >= 64 && threadIdx.x < 64 + kStepLanes) {
#pragma unroll 8
            for (int k = 0; k < kSteps; k++) {
                const float4 x = bb[cur][k][l];
                sb.x += x.x;
                sb.y += x.y;
                sb.z += x.z;
                sb.w += x.w;
            }
        }
    }
    float* dst = hp + int64_t(t) * kHeadCols;
    if (threadIdx.x < kStepLanes) {
        dst[4 * q] = sw.x;
        dst[4 * q + 1] = sw.y;
        dst[4 * q + 2] = sw.z;
        dst[4 * q + 3] = sw.w;
        if (q == 0) dst[16] = sg;
    } else if (threadIdx.x >= 64 && threadIdx.x < 64 + kStepLanes) {
        dst[17 + 4 * q] = sb.x;
        dst[17 + 4 * q + 1] = sb.y;
        dst[17 + 4 * q + 2] = sb.z;
        dst[17 + 4 * q + 3] = sb.w;
    }
}

// the head's gradients (dw: 16 weights, bias) and the last convolution's bias
// gradient from k_loss_back's running sums, sample by sample; one wave per column
__global__ void __launch_bounds__(kT) k_head_finish(const float* __restrict__ hp, float* __restrict__ dw,
                                                   float* __restrict__ db, int B) {
    const int c = int(blockIdx.x) * (kT / 64) + (threadIdx.x >> 6);
    if (c >= kHeadCols) return;
    float* dst = c < 17 ? dw + c : db + (c - 17);
    float total = *dst;
    for (int b = 0; b < B; b++) total += chain_tree(hp + int64_t(b) * kChains * kHeadCols, kHeadCols, c);
    if ((threadIdx.x & 63) == 0) *dst = total;
}

// Adam (beta1 0.9, beta2 0.999, eps 1e-8) on the FP32 master parameters
__global__ void k_adam(float* p, const float* g, float* m, float* v, int64_t n, float lr, float c1, float c2,
                       float gscale) {
    const int64_t k = int64_t(blockIdx.x) * kT + threadIdx.x;
    if (k >= n) return;
    const float gk = g[k] * gscale;
    m[k] = 0.9f * m[k] + 0.1f * gk;
    v[k] = 0.999f * v[k] + 0.001f * gk * gk;
    p[k] = p[k] - lr * (m[k] / c1) / (sqrtf(v[k] / c2) + 1e-8f);
}

// input tensor: channel 0 = divergence / scale, channel 1 = mask, others 0;
// one thread per voxel, inv[sample] = 1 / scale
__global__ void __launch_bounds__(kT) k_input(const float* __restrict__ b, const float* __restrict__ mask,
                                             const float* __restrict__ inv, int64_t V, float* __restrict__ x) {
    const int64_t v = int64_t(blockIdx.x) * kT + threadIdx.x;
    if (v >= V) return;
    const int64_t u = int64_t(blockIdx.y) * V + v;
    float4* o = reinterpret_cast<float4*>(x + u * 16);
    o[0] = make_float4(b[u] * inv[blockIdx.y], mask[u], 0.0f, 0.0f);
    o[1] = o[2] = o[3] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

// a[v] *= f[sample] (V values per sample)
__global__ void __launch_bounds__(kT) k_scale(float* a, int64_t V, const float* f) {
    const int64_t v = int64_t(blockIdx.x) * kT + threadIdx.x;
    if (v >= V) return;
    a[int64_t(blockIdx.y) * V + v] *= f[blockIdx.y];
}

// ---- dense grids of one depth of a context ----
// cell of node i at depth d: its key's per-axis offsets
__device__ __forceinline__ uint32_t compact3u(uint32_t x) {
    x &= 0x09249249u;
    x = (x ^ (x >> 2)) & 0x030c30c3u;
    x = (x ^ (x >> 4)) & 0x0300f00fu;
    x = (x ^ (x >> 8)) & 0xff0000ffu;
    x = (x ^ (x >> 16)) & 0x000003ffu;
    return x;
}

__device__ __forceinline__ int64_t node_cell(uint32_t k, int d, int D) {
    const int64_t G = int64_t(1) << d;
    const int64_t x = compact3u(k >> 2) >> (D - d), y = compact3u(k >> 1) >> (D - d), z = compact3u(k) >> (D - d);
    return (x * G + y) * G + z;
}

// grid[cell(i)] = val[i] (and mask = 1) for the n nodes of one depth
__global__ void k_scatter_nodes(const uint32_t* key, const float* val, int64_t n, int d, int D, float* grid,
                                float* mask) {
    const int64_t i = int64_t(blockIdx.x) * kT + threadIdx.x;
    if (i >= n) return;
    const int64_t v = node_cell(key[i], d, D);
    if (grid) grid[v] = val[i];
    if (mask) mask[v] = 1.0f;
}

// out[0] = sum of val^2 (double, one workgroup, fixed order); out[1] = n
__global__ void k_sumsq(const float* val, int64_t n, double* out) {
    __shared__ double red[kT];
    double s = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += kT) s += double(val[i]) * double(val[i]);
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = kT / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = red[0];
        out[1] = double(n);
    }
}

__device__ __forceinline__ float rms_of(const double* ss) {
    const double r = ss[1] > 0.0 ? sqrt(ss[0] / ss[1]) : 0.0;
    return r > 0.0 ? float(r) : 1.0f;
}

__global__ void k_input_dev(const float* b, const float* mask, const double* ss, int64_t V, float* x) {
    const int64_t k = int64_t(blockIdx.x) * kT + threadIdx.x;
    if (k >= V * 16) return;
    const int c = int(k % 16);
    const int64_t v = k / 16;
    x[k] = c == 0 ? b[v] * (1.0f / rms_of(ss)) : (c == 1 ? mask[v] : 0.0f);
}

// x[i] = pred[cell(i)] * scale for the n nodes of one depth (times `extra`,
// a test setting that is 1 otherwise)
__global__ void k_gather_nodes(const uint32_t* key, const float* pred, const double* ss, int64_t n, int d, int D,
                               float extra, float* x) {
    const int64_t i = int64_t(blockIdx.x) * kT + threadIdx.x;
    if (i >= n) return;
    x[i] = pred[node_cell(key[i], d, D)] * rms_of(ss) * extra;
}

unsigned blocks(int64_t n) { return unsigned((n + kT - 1) / kT); }

}  // namespace

// ---- the network object -------------------------------------------------------------
struct UNetConv {
    int cin, cout, G;
    int64_t woff, boff;
    const float* lo;  // decoder convolutions: the upsampled part of the input (clo channels, grid G / 2)
    int clo;          // 0 for a plain input
    const float* skip;
    float* out;
    DBuf<short> wb, wf;
};

}  // namespace prg

struct prg_unet {
    int device = 0;
    int G = 64;
    hipStream_t stream = nullptr;
    hipStream_t copy_stream = nullptr;  // the targets' upload, made when first used
    hipEvent_t copied = nullptr;
    std::string err;
    int64_t nparams = 0;
    prg::DBuf<float> params, grads, adam_m, adam_v;
    int64_t adam_t = 0;
    prg::UNetConv conv[14];  // the convolutions, encoder to decoder
    // activations
    prg::DBuf<float> x0, p1, p2, p3, pred, target, mask, bgrid;
    prg::DBuf<float> act[14];
    // gradients
    prg::DBuf<float> ga, gb, ge0, ge1, ge2, part, bpart;
    prg::DBuf<float> inv;  // 1 / scale of each sample
    float inv_host[prg::kMaxBatch];
    prg::DBuf<double> loss, lpart;
    int batch_cap = 0;  // samples the buffers hold
    // test knob (PRG_UNET_FAIL_CALL at creation): the first call that uploads
    // targets fails behind the upload
    bool fail_call = false;
};

namespace prg {
namespace {

const int kConvDef[14][3] = {{16, 16, 0}, {16, 16, 0}, {16, 32, 1}, {32, 32, 1}, {32, 64, 2}, {64, 64, 2}, {64, 64, 3},
                             {64, 64, 3}, {128, 64, 2}, {64, 64, 2}, {96, 32, 1}, {32, 32, 1}, {48, 16, 0}, {16, 16, 0}};

bool pow2_channels(int c) { return c == 16 || c == 32 || c == 64; }

// Tiles of 16 voxels and 16 channels from which a wave takes 2 x 2 of them
// (below: one, for the waves that fill the chip).  Four at a time over one at a
// time, over the convolutions and data gradients of grids of 16^3 to 128^3 with
// 1 to 16 samples: 1.42 of the time with 1,024 tiles (64 -> 64 channels on 16^3:
// 12.1 and 8.7 us), 1.01 with 2,048, 0.71 with 4,096 (32 -> 32 on 32^3: 9.0 and
// 14.6 us), 0.5 from 8,192 on (64 -> 64 on 32^3: 19.5 and 40.6 us).
constexpr int64_t kConvManyTiles = 4096;

template <int LZ, int RX, int RY, int WX, int WY, int WN>
void launch_conv_rows(hipStream_t s, ConvIn src, const short* w, const float* bias, int G, int relu, ConvOut out,
                      int cout, int B) {
    using C = ConvTile<LZ, RX, RY, WX, WY, WN>;
    const int NT = cout / 16, S = (src.clo + src.cskip) / 16;
    if (NT % WN || G % C::BX || G % C::BY || G % C::ZL) throw Error{PRG_E_ARG, "convolution tile does not divide"};
    // one slice: its halo is staged once for all N-tiles
    const int ntg = S == 1 ? NT : WN;
    const dim3 grid(unsigned((G / C::BX) * (G / C::BY) * (G / C::ZL)), unsigned(B), unsigned(NT / ntg));
    if (S * (ntg / WN) > 1)
        k_conv3_rows<LZ, RX, RY, WX, WY, WN, true><<<grid, kT, 0, s>>>(src, w, bias, G, relu, out, cout, ntg);
    else
        k_conv3_rows<LZ, RX, RY, WX, WY, WN, false><<<grid, kT, 0, s>>>(src, w, bias, G, relu, out, cout, ntg);
    PRG_CHECK_LAUNCH();
}

template <int LZ>
void launch_conv_grid(hipStream_t s, ConvIn src, const short* w, const float* bias, int G, int relu, ConvOut out,
                      int cout, int B) {
    const int NT = cout / 16;
    const bool many = int64_t(B) * G * G * G / 16 * NT >= kConvManyTiles;
    if (NT % 4 == 0) {
        if (many) launch_conv_rows<LZ, 2, 2, 1, 1, 4>(s, src, w, bias, G, relu, out, cout, B);
        else launch_conv_rows<LZ, 1, 1, 1, 1, 4>(s, src, w, bias, G, relu, out, cout, B);
    } else if (NT % 2 == 0) {
        if (many) launch_conv_rows<LZ, 2, 2, 2, 1, 2>(s, src, w, bias, G, relu, out, cout, B);
        else launch_conv_rows<LZ, 1, 1, 1, 2, 2>(s, src, w, bias, G, relu, out, cout, B);
    } else {
        if (many) launch_conv_rows<LZ, 2, 2, 2, 2, 1>(s, src, w, bias, G, relu, out, cout, B);
        else launch_conv_rows<LZ, 1, 1, 2, 2, 1>(s, src, w, bias, G, relu, out, cout, B);
    }
}

void launch_conv(hipStream_t s, ConvIn src, const short* w, const float* bias, int G, int relu, ConvOut out, int cout,
                 int B) {
    const int cin = src.clo + src.cskip;
    if (!pow2_channels(src.cskip) || (src.clo && !pow2_channels(src.clo)) || cout % 16 || cout <= 0 ||
        (src.clo && G < 2))
        throw Error{PRG_E_ARG, "unsupported convolution channels"};
    if (G >= 16) return launch_conv_grid<4>(s, src, w, bias, G, relu, out, cout, B);
    if (G == 8) return launch_conv_grid<3>(s, src, w, bias, G, relu, out, cout, B);
    // 4^3 in bricks of 1 x 4 x 4 voxels, 2^3 whole; a wave per N-tile, or two
    // with eight of them (the grids under 8^3 are the levels of 32 and 64
    // channels and of their concatenation)
    const int NT = cout / 16, BX = G == 4 ? 1 : G;
    if ((G != 4 && G != 2) || (NT != 2 && NT != 4 && NT != 8)) throw Error{PRG_E_ARG, "unsupported convolution"};
    const size_t lds = size_t(BX + 2) * (G + 2) * (G + 2) * cin * 2;  // at most 27 KB
    const dim3 grid(unsigned(G / BX), unsigned(B));
    const auto kernel = NT == 8 ? k_conv3<2> : k_conv3<1>;
    kernel<<<grid, kT, lds, s>>>(src, w, bias, G, BX, G, G, relu, out, cout);
    PRG_CHECK_LAUNCH();
}

void pack_all(prg_unet* n) {
    PackJobs J{};
    int64_t most = 0;
    for (int k = 0; k < 14; k++) {
        auto& L = n->conv[k];
        J.woff[k] = L.woff;
        J.cin[k] = L.cin;
        J.cout[k] = L.cout;
        J.wb[k] = L.wb.get();
        J.wf[k] = L.wf.get();
        most = std::max(most, int64_t(27) * L.cout * L.cin);
    }
    k_pack<<<dim3(blocks(most), 14), kT, 0, n->stream>>>(n->params.get(), J);
    PRG_CHECK_LAUNCH();
}

// prediction of the B samples in x0, times f
void forward(prg_unet* n, int B, float f = 1.0f) {
    hipStream_t s = n->stream;
    const int G = n->G;
    auto& C = n->conv;
    auto run = [&](int k) {
        auto& L = C[k];
        launch_conv(s, ConvIn{L.lo, L.clo, L.skip, L.cin - L.clo}, L.wb.get(), n->params.get() + L.boff, L.G, 1,
                    ConvOut{L.out, L.cout, nullptr}, L.cout, B);
    };
    auto pool = [&](const float* in, int g, int c, float* out) {
        const int64_t h = g / 2;
        k_pool<<<dim3(blocks(h * h * h * c / 4), unsigned(B)), kT, 0, s>>>(in, log2i(c), log2i(g), out);
        PRG_CHECK_LAUNCH();
    };
    run(0);
    run(1);
    pool(C[1].out, G, 16, n->p1.get());
    run(2);
    run(3);
    pool(C[3].out, G / 2, 32, n->p2.get());
    run(4);
    run(5);
    pool(C[5].out, G / 4, 64, n->p3.get());
    run(6);
    run(7);
    run(8);
    run(9);
    run(10);
    run(11);
    run(12);
    run(13);
    const int64_t V = int64_t(G) * G * G * B;
    k_head<<<blocks(V), kT, 0, s>>>(C[13].out, n->params.get() + (n->nparams - 17), V, f, n->pred.get());
    PRG_CHECK_LAUNCH();
}

// Gradient of conv k for incoming gradient g (in place: the pooled gradient
// `pg` of its output added, then the ReLU mask; unless `masked`: g has both
// and the bias gradient is accumulated).  Writes the input gradient to gin
// unless it is null (of a concatenated input: the upsampled channels to gin,
// the skip's to gskip); accumulates dW and db.
void conv_back(prg_unet* n, int B, int k, float* g, float* gin, float* gskip = nullptr, const float* pg = nullptr,
               bool masked = false) {
    hipStream_t s = n->stream;
    auto& L = n->conv[k];
    const int64_t V = int64_t(L.G) * L.G * L.G;
    if (!masked) {
        k_relu_bias<<<dim3(unsigned(kChains * L.cout / 4 / kStepLanes), unsigned(B)), kSumT, 0, s>>>(
            g, L.out, pg, log2i(L.G), L.cout, n->bpart.get());
        PRG_CHECK_LAUNCH();
    }
    const int nchunk = int((V + kWChunk - 1) / kWChunk);
    const int64_t nw = int64_t(27) * L.cout * L.cin;
    const ConvIn src{L.lo, L.clo, L.skip, L.cin - L.clo};
    const dim3 jobs(unsigned(nchunk * 3 * (L.cout / 16) * (L.cin / 16)), unsigned(B));
    switch (L.G) {
        case 128: k_wgrad_rows<7><<<jobs, 192, 0, s>>>(src, g, L.cout, nchunk, n->part.get()); break;
        case 64: k_wgrad_rows<6><<<jobs, 192, 0, s>>>(src, g, L.cout, nchunk, n->part.get()); break;
        case 32: k_wgrad_rows<5><<<jobs, 192, 0, s>>>(src, g, L.cout, nchunk, n->part.get()); break;
        case 16: k_wgrad_rows<4><<<jobs, 192, 0, s>>>(src, g, L.cout, nchunk, n->part.get()); break;
        case 8: k_wgrad_rows<3><<<jobs, 192, 0, s>>>(src, g, L.cout, nchunk, n->part.get()); break;
        default:  // 4 or 2
            k_wgrad_small<<<dim3((9 * jobs.x + 3) / 4, unsigned(B)), kT, 0, s>>>(src, g, L.cout, L.G, n->part.get());
    }
    PRG_CHECK_LAUNCH();
    k_grad_finish<<<blocks(nw) + (masked ? 0 : L.cout / (kT / 64)), kT, 0, s>>>(
        n->part.get(), nchunk, nw, n->grads.get() + L.woff, n->bpart.get(), L.cout,
        n->grads.get() + L.boff, B);
    PRG_CHECK_LAUNCH();
    if (gin)
        launch_conv(s, ConvIn{nullptr, 0, g, L.cout}, L.wf.get(), nullptr, L.G, 0,
                    gskip ? ConvOut{gin, L.clo, gskip} : ConvOut{gin, L.cin, nullptr}, L.cin, B);
}

// the losses of the B samples `forward` ran on, and their gradients for every
// parameter, added sample after sample
void backward(prg_unet* n, int B) {
    hipStream_t s = n->stream;
    const int G = n->G;
    const int64_t V0 = int64_t(G) * G * G, V1 = V0 / 8, V2 = V1 / 8;
    auto& C = n->conv;
    float* ga = n->ga.get();
    float* gb = n->gb.get();
    // loss, head and the last ReLU
    const int nl = int((V0 + kLossVox - 1) / kLossVox);
    const int64_t head = n->nparams - 17;
    k_loss_part<<<dim3(unsigned(nl), unsigned(B)), kT, 0, s>>>(n->pred.get(), n->target.get(), n->mask.get(), V0,
                                                               n->lpart.get());
    PRG_CHECK_LAUNCH();
    k_loss_back<<<dim3(unsigned(kChains * 4 / kStepLanes), unsigned(B)), kSumT, 0, s>>>(
        n->pred.get(), n->target.get(), n->mask.get(), C[13].out, n->params.get() + head, V0, n->lpart.get(), nl,
        n->loss.get(), ga, n->bpart.get());
    PRG_CHECK_LAUNCH();
    k_head_finish<<<(kHeadCols + 3) / 4, kT, 0, s>>>(n->bpart.get(), n->grads.get() + head,
                                                     n->grads.get() + C[13].boff, B);
    PRG_CHECK_LAUNCH();
    auto up_back = [&](const float* g, int c, int g1, float* glo) {
        const int64_t h = g1 / 2;
        k_up_back<<<dim3(blocks(h * h * h * c / 4), unsigned(B)), kT, 0, s>>>(g, log2i(c), log2i(g1), glo);
        PRG_CHECK_LAUNCH();
    };
    float *ge0 = n->ge0.get(), *ge1 = n->ge1.get(), *ge2 = n->ge2.get();
    // d0
    conv_back(n, B, 13, ga, gb, nullptr, nullptr, true);
    conv_back(n, B, 12, gb, ga, ge0);  // ga: gradient of d1's output upsampled (G, 32)
    up_back(ga, 32, G, gb);
    // d1 (gb: gradient of d1 output, G/2, 32 channels)
    conv_back(n, B, 11, gb, ga);
    conv_back(n, B, 10, ga, gb, ge1);  // gb: gradient of d2's output upsampled (G/2, 64)
    up_back(gb, 64, G / 2, ga);
    // d2 (ga: gradient of d2 output, G/4, 64)
    conv_back(n, B, 9, ga, gb);
    conv_back(n, B, 8, gb, ga, ge2);  // ga: gradient of the bottleneck's output upsampled (G/4, 64)
    up_back(ga, 64, G / 4, gb);
    // bottleneck (gb: G/8, 64)
    conv_back(n, B, 7, gb, ga);
    conv_back(n, B, 6, ga, gb);  // gb: gradient of p3 (G/8, 64)
    // e2
    conv_back(n, B, 5, ge2, ga, nullptr, gb);
    conv_back(n, B, 4, ga, gb);  // gb: gradient of p2 (G/4, 32)
    // e1
    conv_back(n, B, 3, ge1, ga, nullptr, gb);
    conv_back(n, B, 2, ga, gb);  // gb: gradient of p1 (G/2, 16)
    // e0
    conv_back(n, B, 1, ge0, ga, nullptr, gb);
    conv_back(n, B, 0, ga, nullptr);
}

void upload(prg_unet* n, float* dst, const float* src, int64_t count) {
    PRG_HIP(hipMemcpyAsync(dst, src, size_t(count) * 4, hipMemcpyHostToDevice, n->stream));
}

// B samples' inputs (divergence and mask grids), normalised by their scales
void load_samples(prg_unet* n, const float* bgrid, const float* mask, const float* scale, int B) {
    const int64_t V = int64_t(n->G) * n->G * n->G;
    for (int b = 0; b < B; b++) n->inv_host[b] = 1.0f / scale[b];
    upload(n, n->inv.get(), n->inv_host, B);
    upload(n, n->bgrid.get(), bgrid, V * B);
    upload(n, n->mask.get(), mask, V * B);
    k_input<<<dim3(blocks(V), unsigned(B)), kT, 0, n->stream>>>(n->bgrid.get(), n->mask.get(), n->inv.get(), V,
                                                               n->x0.get());
    PRG_CHECK_LAUNCH();
}

// Their targets, normalised likewise: up on a stream of their own, beside the
// forward pass queued before (0.3 ms of a training step of 8 at 64^3).
// Nothing queued uses the buffer: every step and gradient call ends with a
// synchronisation, failed ones in unet_guard.
void load_targets(prg_unet* n, const float* target, int B) {
    const int64_t V = int64_t(n->G) * n->G * n->G;
    if (!n->copy_stream) {
        PRG_HIP(hipStreamCreateWithFlags(&n->copy_stream, hipStreamNonBlocking));
        PRG_HIP(hipEventCreateWithFlags(&n->copied, hipEventDisableTiming));
    }
    PRG_HIP(hipMemcpyAsync(n->target.get(), target, size_t(V * B) * 4, hipMemcpyHostToDevice, n->copy_stream));
    PRG_HIP(hipEventRecord(n->copied, n->copy_stream));
    PRG_HIP(hipStreamWaitEvent(n->stream, n->copied, 0));
    k_scale<<<dim3(blocks(V), unsigned(B)), kT, 0, n->stream>>>(n->target.get(), V, n->inv.get());
    PRG_CHECK_LAUNCH();
    if (n->fail_call) {
        n->fail_call = false;
        throw Error{PRG_E_HIP, "failed as PRG_UNET_FAIL_CALL asks"};
    }
}

// Buffers for B samples at a time (they only grow) and the convolutions'
// input and output tensors in them.
void reserve_batch(prg_unet* n, int B) {
    if (B <= n->batch_cap) return;
    PRG_HIP(hipStreamSynchronize(n->stream));
    n->batch_cap = 0;  // until every buffer has grown
    const int G = n->G;
    const size_t V0 = size_t(G) * G * G * B;
    auto& C = n->conv;
    size_t pc = 0;
    for (int k = 0; k < 14; k++) {
        auto& L = C[k];
        const size_t V = size_t(L.G) * L.G * L.G;
        L.out = n->act[k].reserve(V * L.cout * B);
        pc = std::max(pc, ((V + kWChunk - 1) / kWChunk) * 27 * L.cin * L.cout * B);
    }
    n->x0.reserve(V0 * 16);
    n->p1.reserve(V0 / 8 * 16);
    n->p2.reserve(V0 / 64 * 32);
    n->p3.reserve(V0 / 512 * 64);
    for (auto* g : {&n->pred, &n->target, &n->mask, &n->bgrid}) g->reserve(V0);
    n->ga.reserve(V0 * 48);
    n->gb.reserve(V0 * 48);
    n->ge0.reserve(V0 * 16);
    n->ge1.reserve(V0 / 8 * 32);
    n->ge2.reserve(V0 / 64 * 64);
    n->part.reserve(pc);
    n->bpart.reserve(size_t(kChains) * 64 * B);
    n->lpart.reserve(2 * ((V0 + size_t(kLossVox) * B) / kLossVox));
    n->loss.reserve(B);
    n->inv.reserve(B);
    // inputs: the previous output, or a pooled one at the encoder's levels
    for (int k = 0; k < 14; k++) {
        C[k].lo = nullptr;
        C[k].clo = 0;
        C[k].skip = k ? C[k - 1].out : n->x0.get();
    }
    C[2].skip = n->p1.get();
    C[4].skip = n->p2.get();
    C[6].skip = n->p3.get();
    // decoder inputs: concat(upsampled coarser output, encoder skip)
    const int dec[3][3] = {{8, 7, 5}, {10, 9, 3}, {12, 11, 1}};
    for (int j = 0; j < 3; j++) {
        auto& L = C[dec[j][0]];
        L.lo = C[dec[j][1]].out;
        L.clo = C[dec[j][1]].cout;
        L.skip = C[dec[j][2]].out;
    }
    n->batch_cap = B;
}

template <class F>
prg_status unet_guard(prg_unet* n, F&& f) {
    if (!n) return PRG_E_ARG;
    // what a failed call has queued ends before it returns: it reads the
    // caller's arrays, and the next call's uploads are ordered behind nothing
    auto quiet = [&] {
        for (hipStream_t x : {n->stream, n->copy_stream})
            if (x) (void)hipStreamSynchronize(x);
    };
    try {
        PRG_HIP(hipSetDevice(n->device));
        return f();
    } catch (const Error& e) {
        quiet();
        n->err = e.msg;
        return e.status;
    } catch (const std::bad_alloc&) {
        quiet();
        n->err = "host allocation failed";
        return PRG_E_NOMEM;
    }
}

}  // namespace

void unet_warm_start(prg_ctx* c, int depth, hipStream_t s) {
    const ArenaScope scope(nullptr);  // the network's buffers outlive the context
    prg_unet* n = c->warm_net;
    if (!n || (int64_t(1) << depth) != n->G) throw Error{PRG_E_STATE, "warm-start network does not match the depth"};
    if (n->device != c->cfg.device) throw Error{PRG_E_ARG, "warm-start network is on another device"};
    reserve_batch(n, 1);  // (nothing to do unless an earlier growth failed)
    hipStream_t keep = n->stream;
    n->stream = s;  // the network's kernels run in the order of the chain that solves `depth`
    try {
        const int64_t V = int64_t(n->G) * n->G * n->G, cnt = c->counts[depth], base = c->bases[depth];
        PRG_HIP(hipMemsetAsync(n->bgrid.get(), 0, size_t(V) * 4, s));
        PRG_HIP(hipMemsetAsync(n->mask.get(), 0, size_t(V) * 4, s));
        PoolBuf<double> ss{&c->pool[96]};
        ss.reserve(2);
        k_scatter_nodes<<<blocks(cnt), kT, 0, s>>>(c->key.get() + base, c->div.get() + base, cnt, depth, c->D,
                                                   n->bgrid.get(), n->mask.get());
        PRG_CHECK_LAUNCH();
        k_sumsq<<<1, kT, 0, s>>>(c->div.get() + base, cnt, ss.get());
        PRG_CHECK_LAUNCH();
        k_input_dev<<<blocks(V * 16), kT, 0, s>>>(n->bgrid.get(), n->mask.get(), ss.get(), V, n->x0.get());
        PRG_CHECK_LAUNCH();
        {
            TimedScope ts(c->kt, "unet_forward", 0.0);
            forward(n, 1);
        }
        k_gather_nodes<<<blocks(cnt), kT, 0, s>>>(c->key.get() + base, n->pred.get(), ss.get(), cnt, depth, c->D,
                                                  c->warm_scale, c->x.get() + base);
        PRG_CHECK_LAUNCH();
    } catch (...) {
        n->stream = keep;
        throw;
    }
    n->stream = keep;
}

}  // namespace prg

extern "C" {

prg_status prg_unet_create(prg_unet** out, int32_t device, int32_t grid, uint64_t seed) {
    if (!out) return PRG_E_ARG;
    *out = nullptr;
    if (grid < 16 || grid > 128 || (grid & (grid - 1))) return PRG_E_ARG;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= device || device < 0) return PRG_E_NODEVICE;
    prg_unet* n = new prg_unet();
    n->device = device;
    n->G = grid;
    if (const char* fc = std::getenv("PRG_UNET_FAIL_CALL")) n->fail_call = std::atoi(fc) != 0;
    const prg_status st = prg::unet_guard(n, [&]() {
        PRG_HIP(hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking));
        int64_t off = 0;
        for (int k = 0; k < 14; k++) {
            auto& L = n->conv[k];
            L.cin = prg::kConvDef[k][0];
            L.cout = prg::kConvDef[k][1];
            L.G = grid >> prg::kConvDef[k][2];
            L.woff = off;
            off += int64_t(27) * L.cin * L.cout;
            L.boff = off;
            off += L.cout;
            L.wb.reserve(size_t(27) * L.cin * L.cout);
            L.wf.reserve(size_t(27) * L.cin * L.cout);
        }
        off += 17;  // head: 16 weights, bias
        n->nparams = off;
        prg::reserve_batch(n, 1);
        auto& C = n->conv;
        // He-normal initial weights (splitmix64 + Box-Muller), zero biases
        std::vector<float> h(size_t(n->nparams), 0.0f);
        uint64_t st = seed;
        auto next = [&]() {
            st += 0x9E3779B97F4A7C15ull;
            uint64_t z = st;
            z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
            z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
            return z ^ (z >> 31);
        };
        auto gauss = [&]() {
            const double u1 = (double((next() >> 11) + 1)) * (1.0 / 9007199254740993.0);
            const double u2 = double(next() >> 11) * (1.0 / 9007199254740992.0);
            return std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2);
        };
        for (auto& L : C) {
            const double sd = std::sqrt(2.0 / (27.0 * L.cin));
            for (int64_t k = 0; k < int64_t(27) * L.cin * L.cout; k++) h[size_t(L.woff + k)] = float(gauss() * sd);
        }
        for (int c = 0; c < 16; c++) h[size_t(n->nparams - 17 + c)] = float(gauss() * 0.25);
        n->params.reserve(n->nparams);
        n->grads.reserve(n->nparams);
        n->adam_m.reserve(n->nparams);
        n->adam_v.reserve(n->nparams);
        PRG_HIP(hipMemcpyAsync(n->params.get(), h.data(), size_t(n->nparams) * 4, hipMemcpyHostToDevice, n->stream));
        PRG_HIP(hipMemsetAsync(n->adam_m.get(), 0, size_t(n->nparams) * 4, n->stream));
        PRG_HIP(hipMemsetAsync(n->adam_v.get(), 0, size_t(n->nparams) * 4, n->stream));
        prg::pack_all(n);
        PRG_HIP(hipStreamSynchronize(n->stream));
        return PRG_OK;
    });
    if (st != PRG_OK) {
        prg_unet_destroy(n);
        return st;
    }
    *out = n;
    return PRG_OK;
}

void prg_unet_destroy(prg_unet* n) {
    if (!n) return;
    (void)hipSetDevice(n->device);
    if (n->copy_stream) {
        (void)hipStreamSynchronize(n->copy_stream);
        (void)hipStreamDestroy(n->copy_stream);
    }
    if (n->copied) (void)hipEventDestroy(n->copied);
    if (n->stream) {
        (void)hipStreamSynchronize(n->stream);
        (void)hipStreamDestroy(n->stream);
    }
    delete n;
}

const char* prg_unet_last_error(prg_unet* n) { return n ? n->err.c_str() : "null network"; }

int64_t prg_unet_num_params(prg_unet* n) { return n ? n->nparams : -1; }

int32_t prg_unet_grid(prg_unet* n) { return n ? n->G : -1; }

prg_status prg_unet_get_params(prg_unet* n, float* out, int64_t count) {
    return prg::unet_guard(n, [&]() {
        if (!out || count != n->nparams) return PRG_E_ARG;
        PRG_HIP(hipMemcpyAsync(out, n->params.get(), size_t(count) * 4, hipMemcpyDeviceToHost, n->stream));
        PRG_HIP(hipStreamSynchronize(n->stream));
        return PRG_OK;
    });
}

prg_status prg_unet_set_params(prg_unet* n, const float* in, int64_t count) {
    return prg::unet_guard(n, [&]() {
        if (!in || count != n->nparams) return PRG_E_ARG;
        PRG_HIP(hipMemcpyAsync(n->params.get(), in, size_t(count) * 4, hipMemcpyHostToDevice, n->stream));
        prg::pack_all(n);
        PRG_HIP(hipStreamSynchronize(n->stream));
        return PRG_OK;
    });
}

prg_status prg_unet_predict(prg_unet* n, const float* bgrid, const float* mask, float scale, float* out) {
    return prg::unet_guard(n, [&]() {
        if (!bgrid || !mask || !out || !(scale > 0.0f)) return PRG_E_ARG;
        const int64_t V = int64_t(n->G) * n->G * n->G;
        prg::reserve_batch(n, 1);
        prg::load_samples(n, bgrid, mask, &scale, 1);
        prg::forward(n, 1, scale);
        PRG_HIP(hipMemcpyAsync(out, n->pred.get(), size_t(V) * 4, hipMemcpyDeviceToHost, n->stream));
        PRG_HIP(hipStreamSynchronize(n->stream));
        return PRG_OK;
    });
}

prg_status prg_unet_gradients(prg_unet* n, const float* bgrid, const float* mask, const float* target, float scale,
                              float* grads, double* loss) {
    return prg::unet_guard(n, [&]() {
        if (!bgrid || !mask || !target || !grads || !loss || !(scale > 0.0f)) return PRG_E_ARG;
        PRG_HIP(hipMemsetAsync(n->grads.get(), 0, size_t(n->nparams) * 4, n->stream));
        prg::reserve_batch(n, 1);
        prg::load_samples(n, bgrid, mask, &scale, 1);
        prg::forward(n, 1);
        prg::load_targets(n, target, 1);
        prg::backward(n, 1);
        PRG_HIP(hipMemcpyAsync(grads, n->grads.get(), size_t(n->nparams) * 4, hipMemcpyDeviceToHost, n->stream));
        PRG_HIP(hipMemcpyAsync(loss, n->loss.get(), 8, hipMemcpyDeviceToHost, n->stream));
        PRG_HIP(hipStreamSynchronize(n->stream));
        return PRG_OK;
    });
}

prg_status prg_unet_train_step(prg_unet* n, const float* bgrids, const float* masks, const float* targets,
                               const float* scales, int32_t batch, float lr, double* mean_loss) {
    return prg::unet_guard(n, [&]() {
        if (!bgrids || !masks || !targets || !scales || batch < 1 || !(lr > 0.0f)) return PRG_E_ARG;
        const int64_t V = int64_t(n->G) * n->G * n->G;
        PRG_HIP(hipMemsetAsync(n->grads.get(), 0, size_t(n->nparams) * 4, n->stream));
        // several samples per launch, as many as 2^21 voxels hold: the coarse
        // levels of one sample are a few workgroups, and a launch costs about
        // 4 us whatever it does (8 samples on 64^3 one by one: 14.6 ms)
        int sub = int(std::min<int64_t>({batch, prg::kMaxBatch, std::max<int64_t>(1, (int64_t(1) << 21) / V)}));
        for (;; sub /= 2) {
            try {
                prg::reserve_batch(n, sub);
                break;
            } catch (const prg::Error& e) {
                // fewer at a time where the device has no room for them
                if (e.status != PRG_E_NOMEM || sub == 1) throw;
                (void)hipGetLastError();
            }
        }
        double total = 0.0;
        for (int b0 = 0; b0 < batch; b0 += sub) {
            const int B = std::min(sub, batch - b0);
            prg::load_samples(n, bgrids + b0 * V, masks + b0 * V, scales + b0, B);
            prg::forward(n, B);
            prg::load_targets(n, targets + b0 * V, B);
            prg::backward(n, B);
            double l[prg::kMaxBatch];
            PRG_HIP(hipMemcpyAsync(l, n->loss.get(), size_t(B) * 8, hipMemcpyDeviceToHost, n->stream));
            PRG_HIP(hipStreamSynchronize(n->stream));
            for (int b = 0; b < B; b++) total += l[b];
        }
        n->adam_t++;
        const float c1 = float(1.0 - std::pow(0.9, double(n->adam_t)));
        const float c2 = float(1.0 - std::pow(0.999, double(n->adam_t)));
        prg::k_adam<<<prg::blocks(n->nparams), prg::kT, 0, n->stream>>>(n->params.get(), n->grads.get(),
                                                                        n->adam_m.get(), n->adam_v.get(),
                                                                        n->nparams, lr, c1, c2, 1.0f / batch);
        PRG_CHECK_LAUNCH();
        prg::pack_all(n);
        PRG_HIP(hipStreamSynchronize(n->stream));
        if (mean_loss) *mean_loss = total / batch;
        return PRG_OK;
    });
}

prg_status prg_dense_grid(prg_ctx* c, int32_t depth, int32_t which, float* grid, float* div_rms) {
    if (!c) return PRG_E_ARG;
    try {
        if (!c->have_tree) return PRG_E_STATE;
        if (depth < 1 || depth > c->D || depth > 7 || which < 0 || which > 2 || !grid) return PRG_E_ARG;
        if (which == 0 && !c->have_div) return PRG_E_STATE;
        if (which == 1 && !c->have_x) return PRG_E_STATE;
        PRG_HIP(hipSetDevice(c->cfg.device));
        hipStream_t s = c->stream;
        const int64_t G = int64_t(1) << depth, V = G * G * G, cnt = c->counts[depth], base = c->bases[depth];
        prg::DBuf<float> g;
        prg::DBuf<double> ss;
        g.reserve(V);
        ss.reserve(2);
        PRG_HIP(hipMemsetAsync(g.get(), 0, size_t(V) * 4, s));
        const float* src = which == 0 ? c->div.get() : c->x.get();
        prg::k_scatter_nodes<<<prg::blocks(cnt), prg::kT, 0, s>>>(c->key.get() + base,
                                                                  which == 2 ? nullptr : src + base, cnt, depth,
                                                                  c->D, which == 2 ? nullptr : g.get(),
                                                                  which == 2 ? g.get() : nullptr);
        PRG_CHECK_LAUNCH();
        double h[2] = {0.0, 0.0};
        if (div_rms && c->have_div) {
            prg::k_sumsq<<<1, prg::kT, 0, s>>>(c->div.get() + base, cnt, ss.get());
            PRG_CHECK_LAUNCH();
            PRG_HIP(hipMemcpyAsync(h, ss.get(), 16, hipMemcpyDeviceToHost, s));
        }
        PRG_HIP(hipMemcpyAsync(grid, g.get(), size_t(V) * 4, hipMemcpyDeviceToHost, s));
        PRG_HIP(hipStreamSynchronize(s));
        if (div_rms) *div_rms = (h[1] > 0.0 && h[0] > 0.0) ? float(std::sqrt(h[0] / h[1])) : 1.0f;
        return PRG_OK;
    } catch (const prg::Error& e) {
        return e.status;
    }
}

prg_status prg_set_warm_start_net(prg_ctx* c, prg_unet* n) {
    if (!c) return PRG_E_ARG;
    c->warm_net = n;
    return PRG_OK;
}

prg_status prg_warm_start_info(prg_ctx* c, int32_t* depth, int32_t* rejected) {
    if (!c || !depth || !rejected) return PRG_E_ARG;
    *depth = c->warm_depth_used;
    *rejected = c->warm_rejected;
    return PRG_OK;
}

}  // extern "C"
