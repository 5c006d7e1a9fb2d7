// Coarse-leaf subdivision (reference: ProcessLeafNodesAtOtherDepth / ifSubdivide
// main.cu:2957-2992; the face array :2827-2955 and its surface marks
// :2734-2755; the virtual subtrees, their neighbours and marching cubes
// :1500-2222, 2328-2442, 2481-2825, 3114-3217; driver :3799-4561).
//
// A leaf above the leaf level is refined virtually down to depth D when its
// corner values change sign or one of its faces carries a leaf-level surface
// crossing.  The reference builds one array of virtual nodes per group (each
// root shallower than depth 3 alone, then all roots of one depth together),
// finds neighbours through the parents with the parent's child pointer
// redirected to the virtual root, and runs marching cubes over the virtual
// leaves, one mesh batch per group.
//
// Here no virtual tree is built.  A virtual leaf is (root, Morton offset inside
// the root); its key is the root's key with the offset in the low bits.  The
// combined tree of a group has exactly these facts:
//   - a depth-D cell is virtual iff its ancestor at the root depth r is the
//     root itself or (roots at depth >= 3) another root of depth r;
//   - a real node below depth r is reached from one of the root's 27 real
//     neighbours by its key bits; a coarse leaf (in the group or not) has no
//     real descendants.
// Corners and edges are owned by the smallest-key virtual leaf sharing them
// (real leaves never own, main.cu:1541-1545); vertex values sum the real
// neighbours of the owner's virtual ancestors (virtual coefficients are 0) and
// then the root's real ancestor chain (main.cu:2346-2380).  Leaves are
// numbered in root order, Morton order inside a root: the reference's batch
// order, so one scan numbers every batch's vertices and triangles.
//
// Work is split into bricks: Morton-contiguous blocks of up to 8^3 virtual
// leaves of one root (the whole root when it is smaller).  Certificates settle
// the 8^3 bricks without a sign change, one wavefront each; for the others
//   values    the 9^3 corner values, each from its owner's point of view (the
//             owner fixes the summation order)
//   cubes     per leaf: cube index and owned crossing edges, into per-brick
//             tables, and the brick's vertex and triangle counts
//   vertices  the vertices, numbered by scans of the counts
//   triangles triangle entries, a vertex owned by a leaf of another brick
//             found through that brick's tables
// Memory grows with the number of bricks (about 1 M for 506 M virtual
// leaves) and with the bricks that carry output, never with the virtual leaves.
// Roots of 2^3 and 4^3 leaves (one brick each) take a path of their own, with
// several roots to a wave and no certificates (k_small_values and on).
#include <algorithm>
#include <vector>

#include "ctx.h"
#include "lookback.h"
#include "mc_common.h"
#include "tile.h"

namespace prg {
namespace {

constexpr int kBlockS = 256;
constexpr int kFinerDepth = 3;  // main.cu:3894: shallower roots go one at a time

// parentFaceKind (MarchingCubes.cuh:708-717), indexed [sonKey][face] literally
__constant__ int8_t c_parent_face[8][6] = {{0, -1, 2, -1, 4, -1}, {-1, 1, 2, -1, 4, -1}, {0, -1, -1, 3, 4, -1},
                                           {-1, 1, -1, 3, 4, -1}, {0, -1, 2, -1, -1, 5}, {-1, 1, 2, -1, -1, 5},
                                           {0, -1, -1, 3, -1, 5}, {0, 1, -1, 3, -1, 5}};
// faceEdges (MarchingCubes.cuh:734-741) as bit masks of edge kinds
constexpr uint16_t kFaceEdges[6] = {(1 << 4) | (1 << 6) | (1 << 8) | (1 << 10), (1 << 5) | (1 << 7) | (1 << 9) | (1 << 11),
                                    (1 << 0) | (1 << 2) | (1 << 8) | (1 << 9),  (1 << 1) | (1 << 3) | (1 << 10) | (1 << 11),
                                    (1 << 0) | (1 << 1) | (1 << 4) | (1 << 5),  (1 << 2) | (1 << 3) | (1 << 6) | (1 << 7)};
// Faces of a leaf cube touched by its triangles' edges, per cube
// configuration: bit j when an edge of face j (kFaceEdges) is an edge of one
// of the configuration's triangles.  Built at compile time from the
// marching-cubes triangle table.
struct CubeFaces {
    uint8_t f[256];
};
constexpr CubeFaces make_cube_faces() {
    constexpr int8_t tri[256][16] = {PRG_MC_TRIANGLE_TABLE_DATA};
    CubeFaces t{};
    for (int cube = 0; cube < 256; cube++) {
        uint32_t em = 0;
        for (int k = 0; k < 15 && tri[cube][k] >= 0; k++) em |= 1u << tri[cube][k];
        uint8_t f = 0;
        for (int j = 0; j < 6; j++)
            if (em & kFaceEdges[j]) f = uint8_t(f | (1u << j));
        t.f[cube] = f;
    }
    return t;
}
__constant__ CubeFaces c_cube_faces = make_cube_faces();
// childrenVertexKind (MarchingCubes.cuh:720-723), used literally
__constant__ int8_t c_children_vertex_kind[8] = {0, 1, 3, 2, 4, 5, 7, 6};

// slots of the device counter array; the cells of 2^k leaves a side listed at
// kCntCells + k
enum { kCntCoarse = 0, kCntCorners = 1, kCntRoots = 2, kCntBricks = 3, kCntVerts = 4, kCntTris = 5, kCntLeaves = 6,
       kCntErr = 7, kCntDense = 8, kCntExact = 9, kCntSmall1 = 11, kCntSmall2 = 12,
       kCntGroup = 13, kCntCells = 16, kCntSlots = 32 };
static_assert(kCntSlots * 4 <= 256 && kCntCells + kMaxDepth < kCntSlots && kCntSlots <= kWeldHost,
              "the pinned counter copy holds 64 ints");

__device__ __forceinline__ int depth_of(int64_t i, const Levels& L, int D) {
    int d = 0;
#pragma unroll
    for (int k = 1; k <= kMaxDepth; k++) d += k <= D && i >= L.base[k] ? 1 : 0;
    return d;
}

__device__ __forceinline__ int nidx(int dx, int dy, int dz) { return 9 * (dx + 1) + 3 * (dy + 1) + (dz + 1); }

// Neighbour j = nidx(dx, dy, dz) of node i at depth d, or -1 (computeNeighbor,
// main.cu:492-509): child LUTchild[s][j] of the parent's neighbour
// LUTparent[s][j], read from the sibling block's parent-neighbour row (the
// level-local child base of each of the parent's 27 neighbours).  Nodes of a
// depth come in sibling blocks of 8 in child order, so the slot s is the
// node's level-local index mod 8.  The root's only neighbour is itself.
__device__ __forceinline__ int32_t neighbour_of(const int32_t* __restrict__ pnt, const Levels& L, int d, int64_t i,
                                                int j) {
    if (d == 0) return j == 13 ? int32_t(i) : -1;
    const int64_t loc = i - L.base[d];
    int entry, child;
    tile_neighbour(int(loc & 7), j, entry, child);
    const int32_t cb = pnt[27 * (L.pnt_off[d] + (loc >> 3)) + entry];
    return cb < 0 ? -1 : int32_t(L.base[d] + cb + child);
}

// The face record holding face j of node X at depth d (initFaceArray /
// maintainFaceNodePointer, main.cu:2827-2955): owned by the smaller key of X
// and its neighbour across the face, numbered (owner, kind seen from the owner).
__device__ __forceinline__ int64_t face_rec(int64_t X, int d, int j, const uint32_t* __restrict__ key,
                                            const int32_t* __restrict__ pnt, const Levels& L) {
    const int o = j >> 1, dl = (j & 1) ? 1 : -1;
    const int32_t nb = neighbour_of(pnt, L, d, X, nidx(o == 0 ? dl : 0, o == 1 ? dl : 0, o == 2 ? dl : 0));
    if (nb != -1 && key[nb] < key[X]) return 6 * int64_t(nb) + (j ^ 1);
    return 6 * X + j;
}

// hasSurfaceIntersection marks from the leaf-level triangles (generateTrianglePos,
// main.cu:2734-2755): every face of a leaf-level node touched by one of its
// triangle edges, and the faces up the parent chain while the face record
// has a parent face.  The reference walks each chain from its leaf-level
// node; here the walk goes level by level.  A node's face j is visited when a
// chain reaches (node, j); the chain moves on to (parent, j) when the face's
// record has a parent face (hasParentFace, MarchingCubes.cuh:708-717, on the
// record's owner and kind).  So the leaf pass marks its own faces and ORs the
// continuing faces into the parent's byte of `up`; each coarser depth, after
// the finer one, does the same for the faces its byte collected.  The set of
// marked records is the reference's.
__device__ __forceinline__ void face_visit(int64_t Y, uint32_t faces, const uint32_t* __restrict__ key,
                                           const int32_t* __restrict__ pnt, const Levels& L,
                                           const int32_t* __restrict__ parent, int d, int D, uint8_t* inter,
                                           uint32_t* up) {
    // the face record (face_rec): owned by the smaller key of Y and its
    // neighbour across the face, both at depth d.  The six neighbours' loads
    // go out together, then their keys'.
    const uint32_t ky = key[Y];
    const int64_t loc = Y - L.base[d];
    const int s = int(loc & 7);
    const int32_t* row = pnt + 27 * (L.pnt_off[d] + (loc >> 3));
    int32_t nb[6];
    uint32_t kn[6];
#pragma unroll
    for (int j = 0; j < 6; j++) {
        const int o3 = j >> 1, dl = (j & 1) ? 1 : -1;
        int entry, child;
        tile_neighbour(s, nidx(o3 == 0 ? dl : 0, o3 == 1 ? dl : 0, o3 == 2 ? dl : 0), entry, child);
        // (the tree's root has no neighbour and no row)
        const int32_t cb = d > 0 && ((faces >> j) & 1u) ? row[entry] : -1;
        nb[j] = cb < 0 ? -1 : int32_t(L.base[d] + cb + child);
    }
#pragma unroll
    for (int j = 0; j < 6; j++) kn[j] = nb[j] < 0 ? 0xffffffffu : key[nb[j]];
    uint32_t cont = 0;
#pragma unroll
    for (int j = 0; j < 6; j++) {
        if (!((faces >> j) & 1u)) continue;
        const bool far = nb[j] >= 0 && kn[j] < ky;
        const int64_t owner = far ? nb[j] : Y;
        const int kind = far ? j ^ 1 : j;
        inter[6 * owner + kind] = 1;
        // only the root (depth 0) has no parent
        if (d > 0 && c_parent_face[((far ? kn[j] : ky) >> (3 * (D - d))) & 7u][kind] != -1) cont |= 1u << j;
    }
    if (cont) {
        const int64_t P = parent[Y];
        atomicOr(up + (P >> 2), cont << (8 * (P & 3)));
    }
}

// (cubes: the leaf-level cube indices the marching cubes pass stored)
__global__ void __launch_bounds__(kBlockS) k_face_marks(const uint8_t* cubes, int64_t MD, int64_t baseD,
                                                        const uint32_t* key, const int32_t* pnt, Levels L,
                                                        const int32_t* parent, int D, uint8_t* inter, uint32_t* up) {
    const int64_t t = int64_t(blockIdx.x) * kBlockS + threadIdx.x;
    if (t >= MD) return;
    const uint32_t faces = c_cube_faces.f[cubes[t]];
    if (faces) face_visit(baseD + t, faces, key, pnt, L, parent, D, D, inter, up);
}

// the faces the chains carried up to the nodes of depth d (nodes base .. base + n)
__global__ void __launch_bounds__(kBlockS) k_face_marks_up(int64_t base, int64_t n, int d, const uint32_t* key,
                                                           const int32_t* pnt, Levels L, const int32_t* parent,
                                                           int D, uint8_t* inter, uint32_t* up) {
    const int64_t t = int64_t(blockIdx.x) * kBlockS + threadIdx.x;
    if (t >= n) return;
    const int64_t Y = base + t;
    const uint32_t faces = (up[Y >> 2] >> (8 * (Y & 3))) & 0xffu;
    if (faces) face_visit(Y, faces, key, pnt, L, parent, d, D, inter, up);
}

// The same for depths ds .. 0, of at most kSmallUp nodes each, by one
// workgroup: a launch per depth costs about 4 us whatever it does.  The
// faces of a depth are ORed in L2, and the loads read them there.
constexpr int kUpBlock = 1024;
constexpr int64_t kSmallUp = 4096;
__global__ void __launch_bounds__(kUpBlock) k_face_marks_up_small(int ds, const uint32_t* key, const int32_t* pnt,
                                                                  Levels L, const int32_t* parent, int D,
                                                                  uint8_t* inter, uint32_t* up) {
    for (int d = ds; d >= 0; d--) {
        for (int64_t Y = L.base[d] + threadIdx.x; Y < L.base[d + 1]; Y += kUpBlock) {
            const uint32_t w = __hip_atomic_load(up + (Y >> 2), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint32_t faces = (w >> (8 * (Y & 3))) & 0xffu;
            if (faces) face_visit(Y, faces, key, pnt, L, parent, d, D, inter, up);
        }
        // (the waits complete the ORs in L2, where one workgroup's are ordered
        // without a device-scope fence, which writes the L2 back)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
    }
}

// bytes of a buffer set to a repeated value, by a whole grid (16-byte stores, then the tail)
__device__ __forceinline__ void fill_bytes(void* p, int64_t bytes, uint32_t v, int64_t gid, int64_t gsize) {
    uint4* q = static_cast<uint4*>(p);
    const int64_t n16 = bytes >> 4;
    for (int64_t i = gid; i < n16; i += gsize) q[i] = uint4{v, v, v, v};
    uint8_t* b = static_cast<uint8_t*>(p) + 16 * n16;
    if (gid < (bytes & 15)) b[gid] = uint8_t(v);
}

// Everything the subdivision starts cleared: counters, face marks, the up
// bytes, the needed corners; root_of to -1.
__global__ void __launch_bounds__(kBlockS) k_sub_init(int32_t* cnt, uint8_t* inter, uint32_t* up, uint8_t* need,
                                                      int32_t* root_of, int64_t M, int64_t baseD) {
    const int64_t gid = int64_t(blockIdx.x) * kBlockS + threadIdx.x, gsize = int64_t(gridDim.x) * kBlockS;
    fill_bytes(cnt, kCntSlots * 4, 0, gid, gsize);
    fill_bytes(inter, 6 * M, 0, gid, gsize);
    fill_bytes(up, 4 * ((M + 3) / 4), 0, gid, gsize);
    fill_bytes(need, 8 * baseD, 0, gid, gsize);
    fill_bytes(root_of, 4 * M, 0xffffffffu, gid, gsize);
}

constexpr int kSelItems = 16;
// Beyond 2^20 elements a tile is four times as large: each costs about 50 ns of
// its own in the chain of tiles (12.4 M marks: 164 us with 3,021 tiles of 4,096,
// 52 us with a quarter of them; 1.5 M nodes 15 and 12).
constexpr int kSelSmall = kBlockS, kSelLarge = 4 * kBlockS;
int select_block(int64_t n) { return n > (int64_t(1) << 20) ? kSelLarge : kSelSmall; }

// In one launch (lookback.h), the list of the i < n with a mark, in order:
// LEAF: the coarse leaves (no children; the root is none), from child_base;
// else: the bytes of `marks` that are not 0, and each one's place in nid.
template <bool LEAF, int BLOCK>
__global__ void __launch_bounds__(BLOCK) k_select(const int32_t* __restrict__ child_base,
                                                    const uint8_t* __restrict__ marks, int64_t n, uint32_t tiles,
                                                    LookState state, int32_t* __restrict__ list,
                                                    int32_t* __restrict__ nid, int32_t* count) {
    __shared__ int32_t lds[BLOCK / 64];
    __shared__ int32_t s_before;
    const LookTile t = look_begin(state, tiles);
    if (t.tile >= tiles) return;
    const int64_t base = int64_t(t.tile) * (BLOCK * kSelItems) + int64_t(threadIdx.x) * kSelItems;
    uint32_t m = 0;
    if (LEAF) {
        int32_t v[kSelItems];
        if (base + kSelItems <= n) {
#pragma unroll
            for (int j = 0; j < kSelItems; j += 4)
                *reinterpret_cast<int4*>(v + j) = *reinterpret_cast<const int4*>(child_base + base + j);
        } else {
#pragma unroll
            for (int j = 0; j < kSelItems; j++) v[j] = base + j < n ? child_base[base + j] : 0;
        }
#pragma unroll
        for (int j = 0; j < kSelItems; j++) m |= (v[j] < 0 && base + j >= 1) ? 1u << j : 0u;
    } else {
        uint8_t v[kSelItems];
        if (base + kSelItems <= n) {
            *reinterpret_cast<uint4*>(v) = *reinterpret_cast<const uint4*>(marks + base);
        } else {
#pragma unroll
            for (int j = 0; j < kSelItems; j++) v[j] = base + j < n ? marks[base + j] : 0;
        }
#pragma unroll
        for (int j = 0; j < kSelItems; j++) m |= v[j] ? 1u << j : 0u;
    }
    int32_t total;
    const int32_t ex = block_exclusive_scan(__popc(m), lds, total);
    if (threadIdx.x < 64) {
        const int32_t b = look_back(state, 0, t, tiles, total);
        if (threadIdx.x == 0) {
            s_before = b;
            if (t.tile == tiles - 1) *count = b + total;
        }
    }
    __syncthreads();
    look_end(state, t, tiles);
    int32_t at = s_before + ex;
    for (; m; m &= m - 1) {
        const int64_t i = base + __builtin_ctz(m);
        list[at] = int32_t(i);
        if (!LEAF) nid[i] = at;
        at++;
    }
}

// Corner owners of the coarse leaves' corners among the same-depth nodes
// (initVertexOwner, main.cu:1438-1498); marks each (owner, corner) needed.
// ncl (device) coarse leaves in cl.
__global__ void __launch_bounds__(kBlockS) k_coarse_corner_owner(const int32_t* cl, const int32_t* ncl,
                                                                 const uint32_t* key, const int32_t* pnt, Levels L,
                                                                 int D, int32_t* oref, uint8_t* need) {
    const int64_t g = int64_t(blockIdx.x) * kBlockS + threadIdx.x;
    if (g >= 8 * int64_t(*ncl)) return;
    const int64_t X = cl[g >> 3];
    const int dX = depth_of(X, L, D);
    const int j = int(g & 7);
    const int cx = j & 1, cy = (j >> 1) & 1, cz = (j >> 2) & 1;
    uint32_t best = key[X];
    int64_t owner = X;
    int jo = j;
    for (int a = 0; a < 2; a++)
        for (int b = 0; b < 2; b++)
            for (int e = 0; e < 2; e++) {
                if (!(a | b | e)) continue;
                const int32_t nb = neighbour_of(pnt, L, dX, X, nidx(a ? 2 * cx - 1 : 0, b ? 2 * cy - 1 : 0, e ? 2 * cz - 1 : 0));
                if (nb == -1) continue;
                if (key[nb] < best) {
                    best = key[nb];
                    owner = nb;
                    jo = j ^ (a | (b << 1) | (e << 2));
                }
            }
    oref[g] = int32_t(8 * owner + jo);
    need[8 * owner + jo] = 1;
}

// computeVertexImplicitFunctionValue (main.cu:2259-2326) for a corner of a
// node above the leaf level: the owner's ancestor chain, then the descent
// through children[childrenVertexKind[corner]] down to D.
// chain_value for lanes that start on different nodes at different depths
// (the owners of coarse-leaf corners, in node order).  Each lane adds its
// depths d, d - 1, ..., 1 in that order, then the root, as chain_value does.
// The deepest lanes step first, so the wave's lanes reach each depth
// together; once every walking lane stands on the same node the rest of the
// chain runs on one wave-uniform index (its row and coefficients come through
// the scalar cache once per wave).  A node with leaf-level slots below it
// (dnum > 0) has a coarse row, whose sum is level_contrib's (row_sum); the
// others gather through the parent-neighbour rows.
__device__ __forceinline__ float coarse_chain_value(int64_t nd, int d, bool valid, float px, float py, float pz,
                                                    const uint32_t* __restrict__ key, const int32_t* __restrict__ pnt,
                                                    const Levels& L, const int32_t* __restrict__ parent,
                                                    const int32_t* __restrict__ dnum, const float* __restrict__ x,
                                                    const float* __restrict__ bf, int D, const float* __restrict__ rows,
                                                    int rows_depth) {
    float val = 0.0f;
    int dm = 0;  // the deepest walking lane's depth
    for (int t = kMaxDepth; t >= 1; t--)
        if (__builtin_amdgcn_ballot_w64(valid && d == t) != 0) {
            dm = t;
            break;
        }
    for (; dm > 0; dm--) {
        const bool walking = valid && d > 0;
        const uint64_t wl = __builtin_amdgcn_ballot_w64(walking);
        const int first = int(__builtin_ctzll(wl));  // (wl != 0 while dm > 0)
        const int64_t n0 = __builtin_amdgcn_readlane(int32_t(nd), first);
        if (__builtin_amdgcn_ballot_w64(walking && (d != dm || nd != n0)) == 0) break;
        if (walking && d == dm) {
            if (dm <= rows_depth && dnum[nd] > 0) {
                const float* R = rows + kRowFloats * (nd - L.base[1]);
                float bx[3], by[3], bz[3];
                node_basis(nd, dm, px, py, pz, key, bf, D, bx, by, bz);
                val = row_sum(R, bx, by, bz, val);
            } else {
                val = level_contrib(nd, dm, px, py, pz, key, pnt, L, x, bf, D, val);
            }
            nd = parent[nd];
            d--;
        }
    }
    if (dm > 0) {  // every walking lane on node u at depth dm
        const uint64_t wl = __builtin_amdgcn_ballot_w64(valid && d > 0);
        int32_t u = __builtin_amdgcn_readlane(int32_t(nd), int(__builtin_ctzll(wl)));
        for (; dm > 0; dm--) {
            const bool row = dm <= rows_depth && dnum[u] > 0;
            float bx[3], by[3], bz[3];
            if (valid) {
                if (row) {
                    node_basis(u, dm, px, py, pz, key, bf, D, bx, by, bz);
                    val = row_sum(rows + kRowFloats * (int64_t(u) - L.base[1]), bx, by, bz, val);
                } else {
                    val = level_contrib(u, dm, px, py, pz, key, pnt, L, x, bf, D, val);
                }
            }
            u = __builtin_amdgcn_readfirstlane(parent[u]);
        }
    }
    float tt = x[0] * basis_value(bf, 0, px);
    tt = tt * basis_value(bf, 0, py);
    tt = tt * basis_value(bf, 0, pz);
    return val + tt;
}

// (five waves per SIMD: 95 VGPRs without spills, 7% faster than four)
__global__ void __launch_bounds__(kBlockS, 5) k_coarse_corner_value(const int32_t* list, const int32_t* n_dev,
                                                                 const uint32_t* key, const int32_t* pnt, Levels L,
                                                                 const int32_t* parent, const int32_t* child_base,
                                                                 const int32_t* dnum, const float* x, const float* bf,
                                                                 const float* rows, int rows_depth, int D,
                                                                 const float* iso, float* out) {
    const int64_t i = int64_t(blockIdx.x) * kBlockS + threadIdx.x;
    const bool valid = i < *n_dev;
    if (__builtin_amdgcn_ballot_w64(valid) == 0) return;  // (wave-uniform)
    int64_t O = 0;
    int jo = 0, d = 0;
    float px = 0.5f, py = 0.5f, pz = 0.5f;
    if (valid) {
        O = list[i] >> 3;
        jo = list[i] & 7;
        d = depth_of(O, L, D);
        float c[3];
        node_center(key[O], d, D, c);
        const float hw = 1.0f / float(1 << (d + 1));
        px = c[0] + float(2 * (jo & 1) - 1) * hw;
        py = c[1] + float(2 * ((jo & 2) >> 1) - 1) * hw;
        pz = c[2] + float(2 * ((jo & 4) >> 2) - 1) * hw;
    }
    // (every lane of the wave takes part in the chain walk's wave votes)
    float f = coarse_chain_value(O, d, valid, px, py, pz, key, pnt, L, parent, dnum, x, bf, D, rows, rows_depth);
    if (!valid) return;
    const int ex = c_children_vertex_kind[jo];
    int64_t nd = O;
    for (int dd = d + 1; dd <= D; dd++) {
        const int32_t cb = child_base[nd];
        if (cb < 0) break;
        nd = cb + ex;
        f = level_contrib(nd, dd, px, py, pz, key, pnt, L, x, bf, D, f);
    }
    out[i] = f - *iso;
}

// hasTriangle || hasIntersection for each coarse leaf (ProcessLeafNodesAtOtherDepth
// + ifSubdivide, main.cu:2957-2992).
__global__ void __launch_bounds__(kBlockS) k_coarse_select(const int32_t* cl, const int32_t* ncl, const int32_t* oref,
                                                           const int32_t* nid, const float* cv, const uint32_t* key,
                                                           const int32_t* pnt, Levels L, int D, const uint8_t* inter,
                                                           uint8_t* rflag) {
    const int64_t c = int64_t(blockIdx.x) * kBlockS + threadIdx.x;
    if (c >= *ncl) return;
    const int64_t X = cl[c];
    // vertices[0] is the (0,0,0) corner in either numbering
    const float v0 = cv[nid[oref[8 * c]]];
    const float sign = (v0 < 0) ? -1.0f : 1.0f;
    bool tri = false;
    for (int j = 1; j < 8; j++)
        if (sign * cv[nid[oref[8 * c + j]]] < 0) tri = true;
    bool hit = false;
    const int dX = depth_of(X, L, D);
    for (int j = 0; j < 6; j++)
        if (inter[face_rec(X, dX, j, key, pnt, L)]) hit = true;
    rflag[c] = (tri || hit) ? 1 : 0;
}

// ---- roots and bricks ---------------------------------------------------------------
constexpr int kWave = 64;
constexpr int kBrickLog = 3;  // bricks of up to 8^3 virtual leaves
constexpr int kBrickLeaves = 1 << (3 * kBrickLog);
constexpr int kBrickPts = ((1 << kBrickLog) + 1) * ((1 << kBrickLog) + 1) * ((1 << kBrickLog) + 1);

// The place in a list (its length in *counter) of each lane with `want`: one
// atomic per wave, lanes in order.
__device__ __forceinline__ int32_t wave_append(bool want, int32_t* counter) {
    const uint64_t m = __builtin_amdgcn_ballot_w64(want);
    if (m == 0) return 0;
    const int lane = threadIdx.x & 63, first = int(__builtin_ctzll(m));
    int32_t at = 0;
    if (lane == first) at = atomicAdd(counter, int32_t(__popcll(m)));
    at = __shfl(at, first, 64);
    return at + int32_t(__popcll(m & ((uint64_t(1) << lane) - 1)));
}

constexpr int kRootBlock = 320;  // one wave per look-back
constexpr int kRootItems = 16;
constexpr int kRootTile = kRootBlock * kRootItems;

// The roots, in order, from the marked coarse leaves, in one launch
// (lookback.h): each root's real index and first brick, its number at its
// node (root_of), and the roots of 2^3 and of 4^3 leaves in lists of their
// own with each one's place in its list (sidx).  The last tile leaves the
// counts in cnt and in pinned memory.  (As flags, compaction, sizes, two
// scans and an append these were five launches over the upper bound n.)
__global__ void __launch_bounds__(kRootBlock) k_list_all_roots(const int32_t* __restrict__ cl,
                                                               const uint8_t* __restrict__ rflag, LookState state,
                                                               Levels L, int D,
                                                               int32_t* __restrict__ roots, int32_t* __restrict__ boff,
                                                               int32_t* __restrict__ root_of,
                                                               int32_t* __restrict__ list1,
                                                               int32_t* __restrict__ list2, int32_t* __restrict__ sidx,
                                                               int32_t* cnt, int32_t* host_cnt) {
    __shared__ int32_t lds[kRootBlock / 64];
    __shared__ int32_t s_before[5];
    const int64_t n = cnt[kCntCoarse];
    // (the launch is sized for the upper bound)
    const uint32_t tiles = n > 0 ? uint32_t((n + kRootTile - 1) / kRootTile) : 1;
    if (blockIdx.x >= tiles) return;
    const LookTile t = look_begin(state, tiles);
    if (t.tile >= tiles) return;
    const int64_t base = int64_t(t.tile) * kRootTile + int64_t(threadIdx.x) * kRootItems;
    uint32_t m = 0;
    if (base < n) {
        uint8_t v[kRootItems];
        // (whole 16-byte words lie inside the array, which is sized for the upper bound)
        *reinterpret_cast<uint4*>(v) = *reinterpret_cast<const uint4*>(rflag + base);
#pragma unroll
        for (int j = 0; j < kRootItems; j++) m |= (base + j < n && v[j]) ? 1u << j : 0u;
    }
    int32_t bricks = 0, leaves = 0, n1 = 0, n2 = 0;
    for (uint32_t w = m; w; w &= w - 1) {
        const int kb = D - depth_of(cl[base + __builtin_ctz(w)], L, D);
        bricks += 1 << (3 * (kb - min(kb, kBrickLog)));
        leaves += 1 << (3 * kb);
        n1 += kb == 1;
        n2 += kb == 2;
    }
    int32_t tot[5];
    int32_t q = block_exclusive_scan(__popc(m), lds, tot[0]);
    int32_t b = block_exclusive_scan(bricks, lds, tot[1]);
    (void)block_exclusive_scan(leaves, lds, tot[2]);
    int32_t a1 = block_exclusive_scan(n1, lds, tot[3]);
    int32_t a2 = block_exclusive_scan(n2, lds, tot[4]);
    const int wave = threadIdx.x >> 6;
    const int32_t mine = wave == 0 ? tot[0] : wave == 1 ? tot[1] : wave == 2 ? tot[2] : wave == 3 ? tot[3] : tot[4];
    const int32_t x = look_back(state, wave, t, tiles, mine);
    if ((threadIdx.x & 63) == 0) {
        s_before[wave] = x;
        if (t.tile == tiles - 1) {
            const int slot = wave == 0 ? kCntRoots : wave == 1 ? kCntBricks : wave == 2 ? kCntLeaves
                             : wave == 3 ? kCntSmall1 : kCntSmall2;
            cnt[slot] = x + mine;
            host_cnt[slot] = x + mine;
        }
    }
    __syncthreads();
    look_end(state, t, tiles);
    q += s_before[0];
    b += s_before[1];
    a1 += s_before[3];
    a2 += s_before[4];
    for (; m; m &= m - 1) {
        const int32_t rho = cl[base + __builtin_ctz(m)];
        const int kb = D - depth_of(rho, L, D);
        roots[q] = rho;
        boff[q] = b;
        root_of[rho] = q;
        if (kb == 1) {
            list1[a1] = q;
            sidx[q] = a1++;
        }
        if (kb == 2) {
            list2[a2] = q;
            sidx[q] = a2++;
        }
        b += 1 << (3 * (kb - min(kb, kBrickLog)));
        q++;
    }
}

// counts and signs of n bricks to 0, no brick listed for evaluation
__global__ void __launch_bounds__(kBlockS) k_clear_bricks(int32_t* bnv, int32_t* bnt, int8_t* sign, int32_t* didx,
                                                          int64_t n) {
    const int64_t i = int64_t(blockIdx.x) * kBlockS + threadIdx.x;
    if (i >= n) return;
    bnv[i] = 0;
    bnt[i] = 0;
    sign[i] = 0;
    didx[i] = -1;
}

struct SubArgs {
    const uint32_t* key;
    const int32_t* child_base;
    const int32_t* parent;
    const int32_t* pnt;
    Levels L;
    const float* x;
    const float* bf;
    const float4* btab;  // corner basis table (corner_basis_entry)
    const float* rows;   // coarse rows of depths 1 .. D - 1
    int D;
    const float* iso;
    const int32_t* roots;
    const int32_t* boff;     // first brick of each root
    const int32_t* root_of;  // per real node: its root number, or -1
    const int32_t* cnt;      // device counters
    const int32_t* bmap;     // root number of each brick
    const int32_t* rec;      // per root: its record (kRecWords words, root_record)
    // per depth: the largest corner value of sum |x_k b_x b_y b_z| over 27
    // neighbours for coefficients up to 1, and the largest difference between
    // the evaluation's value and the spline's there (depth_bounds)
    float big[kMaxDepth + 1], dev[kMaxDepth + 1];
};

// Per-root record, built once per root and loaded by each of its bricks in
// one coalesced read: the root's 27 neighbours, their child bases and root
// numbers (group), its ancestor chain's neighbour values (27 per depth
// 0..r), the root's index, depth and key; for roots of 8^3 leaves and more the
// chain's values over the root as one polynomial (27 Bezier control values)
// and the bound of what the evaluation's chain sum differs from it.
constexpr int kRecWords = 416;
constexpr int kRecNB = 0, kRecNBK = 27, kRecNBR = 54, kRecX = 81, kRecRho = 378, kRecR = 379, kRecKey = 380;
constexpr int kRecPoly = 384, kRecErr = 411;

// A brick and its root (wave-uniform).
struct Brick {
    int32_t q, rho, r, kb;
    int32_t R[3];     // root coordinates at depth r
    int32_t R0[3];    // first depth-D cell of the root
    int32_t Sr;       // root side in depth-D cells
    int32_t org[3];   // first depth-D cell of the brick
    uint32_t bkey;    // key of the brick's first leaf
    bool deep;        // a neighbour of the root has children (real nodes below depth r)
    uint32_t kids;    // bit j: neighbour j (j != 13) has children
};

constexpr int kP = (1 << kBrickLog) + 1;  // grid points per brick side (at most)

// Blocks of the real nodes below the root that a brick's corner owners see:
// at most (D - 3 - r) blocks of 4^3 cells and blocks of 5^3, 7^3 and 11^3
// cells at the three finest depths.
constexpr int kXBlk = 2304;
constexpr int kXBlkScreen = 768;        // and in the screens' LDS: of cells of 16^3 leaves and more,
constexpr int kXBlkScreenBrick = 2176;  // and of bricks

// LDS of one brick's wave: the root's neighbourhood, the brick's basis
// tables and blocks (BrickCore).
// One basis table entry of the brick (the owner's three values along one
// axis): 12 bytes, the corner basis table's fourth float is never read.
struct BasisT {
    float x, y, z;
};

struct BrickCore {
    // per depth d, axis a and grid coordinate i: the corner basis table entry
    // of the owner (own_cell) of grid coordinate org[a] + i, (d, a, i) at
    // d * 3 kP + a kP + i
    BasisT T[(kMaxDepth + 1) * 3 * kP];
    float X[(kMaxDepth + 1) * 27];     // the root's chain: neighbour values at depths 0..r
    float XB[kXBlk];                   // per depth below the root: its block (xb_off)
    int32_t xb_off[kMaxDepth + 1];     // start of depth dd's block in XB, or -1 (no real node in it)
    // child bases of a block's cells while the blocks are filled, at depths
    // D, D - 2, .. and D - 1, D - 3, ..: up to 5^3 and 7^3 cells
    int32_t CB0[125], CB1[343];
    int32_t NB[27], NBK[27], NBR[27];  // the root's neighbours, their child bases, their root numbers (group)
};

// A screened cell's: the chain's polynomial and blocks of up to FLOATS
// coefficients and 7^3 cells above depth D (a cell that needs more is not
// settled).
template <int FLOATS>
struct CellLds {
    float P[27];
    float XB[FLOATS];
    int32_t xb_off[kMaxDepth + 1];
    int32_t CB0[343], CB1[343];
    int32_t NBK[27], NBR[27];
};

// A brick's for the per-corner certificate: a cell's, with the basis table
// entries (BrickCore's T) of the three finest depths, (e, a, i) for depth
// D - kBrickLog + 1 + e.
struct CertLds : CellLds<kXBlk> {
    BasisT T[kBrickLog * 3 * kP];
};

__device__ __forceinline__ void decode_cell(uint32_t k, int32_t c[3]) {
    c[0] = int32_t(compact3(k >> 2));
    c[1] = int32_t(compact3(k >> 1));
    c[2] = int32_t(compact3(k));
}

// ---- the implicit function over a cell as a polynomial ----
// Depth d's functions are quadratic B-splines of the depth's cell width (1 at
// the node's centre, 4/3 summed over the three that overlap a point), whose
// pieces meet at the depth's cell faces.  Over a cell of depth c, the sum of
// all depths up to c is therefore one polynomial, quadratic along each axis;
// its 27 Bezier control values bound it on the cell, and they are linear in
// the depths' coefficients, so the depths add up (and cancel) before any
// bound is taken.

// Weights of the Bernstein control values of [0, 1] in control value i (0, 1,
// 2) of the interval [t0, t0 + h]: the blossom at (t0, t0), (t0, t1), (t1, t1).
__device__ __forceinline__ void bernstein_weights(float t0, float h, int i, float w[3]) {
    const float s = i < 2 ? t0 : t0 + h, t = i < 1 ? t0 : t0 + h;
    w[0] = (1.0f - s) * (1.0f - t);
    w[1] = s * (1.0f - t) + t * (1.0f - s);
    w[2] = s * t;
}

// Weights of the coefficients of a depth's three cells around cell A (A - 1,
// A, A + 1) in control value i of the cell at coordinate c, `up` depths below
// A: the spline's control values over A are (2/3)(x- + x), (4/3) x,
// (2/3)(x + x+).
__device__ __forceinline__ void spline_weights(int32_t c, int up, int i, float w[3]) {
    const float h = 1.0f / float(1 << up), t0 = float(c & ((1 << up) - 1)) * h;
    float b[3];
    bernstein_weights(t0, h, i, b);
    w[0] = (2.0f / 3.0f) * b[0];
    w[1] = (2.0f / 3.0f) * (b[0] + b[2]) + (4.0f / 3.0f) * b[1];
    w[2] = (2.0f / 3.0f) * b[2];
}

// sum over m, n, l of w[0][m] w[1][n] w[2][l] X[sx m + sy n + l]
__device__ __forceinline__ float sum27(const float* X, int sx, int sy, const float w[3][3]) {
    float v = 0.0f;
#pragma unroll
    for (int m = 0; m < 3; m++) {
        float y = 0.0f;
#pragma unroll
        for (int n = 0; n < 3; n++) {
            float z = 0.0f;
#pragma unroll
            for (int l = 0; l < 3; l++) z = __builtin_fmaf(X[sx * m + sy * n + l], w[2][l], z);
            y = __builtin_fmaf(z, w[1][n], y);
        }
        v = __builtin_fmaf(y, w[0][m], v);
    }
    return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, kWave));
    return v;
}

// The records of roots 2 w and 2 w + 1, half a wave each: following a root's
// ancestors row by row is a chain of dependent loads, so the waves' number is
// what counts (one root per wave: 324 us for 294,344 roots).
__global__ void __launch_bounds__(kWave) k_root_records(SubArgs A, int32_t nr, int32_t* rec) {
    const int D = A.D, lane = threadIdx.x & 31;
    const int32_t q = 2 * blockIdx.x + (threadIdx.x >> 5);
    __shared__ float Xs[2][(kMaxDepth + 1) * 27];
    float* X = Xs[threadIdx.x >> 5];
    const bool in = q < nr;
    const int32_t rho = A.roots[in ? q : 0];
    const int r = depth_of(rho, A.L, D);
    int32_t* R = rec + int64_t(q) * kRecWords;
    const bool use = in && lane < 27;
    const int l27 = lane < 27 ? lane : 0;
    if (use) {
        const int32_t nb = neighbour_of(A.pnt, A.L, r, rho, lane);
        R[kRecNB + lane] = nb;
        R[kRecNBK + lane] = nb < 0 ? -1 : A.child_base[nb];
        R[kRecNBR + lane] = (nb < 0 || r < kFinerDepth) ? -1 : A.root_of[nb];
        const float xv = nb < 0 ? 0.0f : A.x[nb];
        R[kRecX + 27 * r + lane] = __float_as_int(xv);
        X[27 * r + lane] = xv;
    }
    // ancestors' rows (their 27 neighbour values, then the parent), depths r-1 .. 1
    int32_t a = A.parent[rho];
    for (int d = r - 1; d >= 1; d--) {
        const float* Row = A.rows + kRowFloats * (int64_t(a) - A.L.base[1]);
        const float xv = Row[l27];
        a = __float_as_int(Row[27]);
        if (use) {
            R[kRecX + 27 * d + lane] = __float_as_int(xv);
            X[27 * d + lane] = xv;
        }
    }
    if (in && lane == 0) {
        R[kRecX] = __float_as_int(A.x[0]);
        R[kRecRho] = rho;
        R[kRecR] = r;
        R[kRecKey] = int32_t(A.key[rho]);
    }
    const bool cells = in && D - r >= kBrickLog;  // cells to screen
    if (__builtin_amdgcn_ballot_w64(cells) == 0) return;
    if (lane < 27) X[lane] = lane == 13 ? A.x[0] : 0.0f;  // depth 0: the tree's root has no neighbours
    __syncthreads();
    if (!cells) return;  // (no barrier follows; a half's shuffles stay inside it)
    int32_t rc[3];
    decode_cell(A.key[rho], rc);
    float val = 0.0f, err = 0.0f;
    for (int d = 0; d <= r; d++) {
        float w[3][3];
#pragma unroll
        for (int a3 = 0; a3 < 3; a3++)
            spline_weights(rc[a3] >> (D - r), r - d, a3 == 0 ? l27 / 9 : a3 == 1 ? (l27 / 3) % 3 : l27 % 3, w[a3]);
        val += sum27(X + 27 * d, 9, 3, w);
        float m = fabsf(X[27 * d + l27]);
#pragma unroll
        for (int o = 16; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 32));
        err += A.dev[d] * m;
    }
    if (use) R[kRecPoly + lane] = __float_as_int(val);
    if (lane == 0) R[kRecErr] = __float_as_int(err);
}

// bmap[b] = the root of brick b (binary search of the brick offsets).
__global__ void __launch_bounds__(kBlockS) k_brick_map(const int32_t* boff, const int32_t* cnt, int64_t nb,
                                                       int32_t* bmap) {
    const int64_t b = int64_t(blockIdx.x) * kBlockS + threadIdx.x;
    if (b >= nb) return;
    int32_t lo = 0, hi = cnt[kCntRoots] - 1;
    while (lo < hi) {
        const int32_t mid = (lo + hi + 1) >> 1;
        if (boff[mid] <= b) lo = mid;
        else hi = mid - 1;
    }
    bmap[b] = lo;
}

// The geometry of the cell of 2^kb leaves a side (a brick, or one of a root's
// cells above) whose first brick is b, in a root with record R.
__device__ __forceinline__ void cell_geometry(const SubArgs& A, int32_t b, int kb, const int32_t* R, Brick& B) {
    const int D = A.D;
    B.rho = __builtin_amdgcn_readfirstlane(R[kRecRho]);
    B.r = __builtin_amdgcn_readfirstlane(R[kRecR]);
    const uint32_t rkey = uint32_t(__builtin_amdgcn_readfirstlane(R[kRecKey]));
    B.kb = kb;
    B.Sr = 1 << (D - B.r);
    B.bkey = rkey | (uint32_t(b - A.boff[B.q]) << (3 * kBrickLog));
    int32_t rc[3];
    decode_cell(rkey, rc);
    decode_cell(B.bkey, B.org);
    for (int a = 0; a < 3; a++) {
        B.R[a] = rc[a] >> (D - B.r);
        B.R0[a] = rc[a];
    }
}

template <class L>
__device__ __forceinline__ void set_kids(Brick& B, const L& S) {
    const int lane = threadIdx.x & 63;
    const uint64_t kids = __builtin_amdgcn_ballot_w64(lane < 27 && lane != 13 && S.NBK[lane < 27 ? lane : 0] >= 0);
    B.kids = uint32_t(kids);
    B.deep = B.kids != 0;
}

// Loads the root record of brick b (8^3 leaves) into LDS (its neighbours and
// its chain's values) and sets the brick's geometry.
template <int kThreads, class L>
__device__ __forceinline__ void brick_setup(const SubArgs& A, int32_t b, Brick& B, L& S) {
    B.q = __builtin_amdgcn_readfirstlane(A.bmap[b]);
    const int32_t* R = A.rec + int64_t(B.q) * kRecWords;
    cell_geometry(A, b, kBrickLog, R, B);
    for (int w = threadIdx.x; w < kRecX; w += kThreads) {
        const int32_t v = R[w];
        if (w < kRecNBK) S.NB[w] = v;
        else if (w < kRecNBR) S.NBK[w - kRecNBK] = v;
        else S.NBR[w - kRecNBR] = v;
    }
    for (int w = threadIdx.x; w < 27 * (B.r + 1); w += kThreads) S.X[w] = __int_as_float(R[kRecX + w]);
    __syncthreads();
    set_kids(B, S);
}

// Loads a screened cell's part of its root's record into LDS and sets the
// cell's geometry.  q_loaded: the root whose record S already holds (the
// previous cell's, in a kernel that walks a list), or -1.
template <class L>
__device__ __forceinline__ void cell_setup(const SubArgs& A, int32_t b, int k, Brick& B, L& S, int32_t q_loaded) {
    const int lane = threadIdx.x;
    B.q = __builtin_amdgcn_readfirstlane(A.bmap[b]);
    const int32_t* R = A.rec + int64_t(B.q) * kRecWords;
    cell_geometry(A, b, k, R, B);
    if (B.q != q_loaded && lane < 27) {
        S.NBK[lane] = R[kRecNBK + lane];
        S.NBR[lane] = R[kRecNBR + lane];
        S.P[lane] = __int_as_float(R[kRecPoly + lane]);
    }
    __syncthreads();
    set_kids(B, S);
}

// Whether the depth-D cell c (inside the root's 3x3x3 neighbourhood) is a
// virtual leaf of the brick's group; *q receives its root's neighbour slot
// (13 for the brick's own root).
template <class L>
__device__ __forceinline__ bool cell_virtual(const Brick& B, const L& S, int D, const int32_t c[3], int* slot) {
    const int W = 1 << D;
    if (c[0] < 0 || c[1] < 0 || c[2] < 0 || c[0] >= W || c[1] >= W || c[2] >= W) return false;
    const int sh = D - B.r;
    const int ax = (c[0] >> sh) - B.R[0], ay = (c[1] >> sh) - B.R[1], az = (c[2] >> sh) - B.R[2];
    const int j = nidx(ax, ay, az);
    *slot = j;
    if (j == 13) return true;
    return S.NBR[j] >= 0;
}

// Width in cells of the block at depth dd: the owners' ancestors (the cells
// the brick spans, and one more below for owners in the lower brick) +-1.
__device__ __forceinline__ int block_width(int D, int kb, int dd) {
    const int e = dd - (D - kb);
    return (e > 0 ? (1 << e) : 1) + 3;
}

// Along one axis of grid coordinate g, the owner cell for a root whose owners
// are all its own leaves: the smaller of the two cells around g that lies in
// the root (Morton keys grow with each coordinate).
__device__ __forceinline__ int32_t own_cell(int32_t g, int32_t R0) { return g == R0 ? g : g - 1; }

// Loads the brick's basis table entries (S.T) for owners inside its root.
// The smallest-key leaf around a grid point, when it is a leaf of the
// brick's own root, is own_cell along every axis, so every corner the
// brick's root owns reads its three basis values per depth from S.T.
template <int kThreads, class L>
__device__ __forceinline__ void brick_tables(const SubArgs& A, const Brick& B, L& S) {
    const int D = A.D, P = (1 << B.kb) + 1;
    constexpr int TP = kP;
    for (int e = threadIdx.x; e < (D + 1) * TP; e += kThreads) {
        const int d = e / TP, i = e % TP;
        if (i >= P) continue;
#pragma unroll
        for (int ax = 0; ax < 3; ax++) {  // constant indices keep B in registers
            const int32_t g = B.org[ax] + i, o = own_cell(g, B.R0[ax]);
            const float4 t = A.btab[((int64_t(d) << D) + o) * 2 + (g - o)];
            S.T[3 * TP * d + TP * ax + i] = BasisT{t.x, t.y, t.z};
        }
    }
}

// Whether v holds in any thread of the workgroup.
template <int kThreads>
__device__ __forceinline__ bool any_thread(bool v) {
    if (kThreads == kWave) return __builtin_amdgcn_ballot_w64(v) != 0;
    return __syncthreads_or(v) != 0;
}

// Fills the brick's blocks (depths r+1..D), level by level: each cell's
// coefficient, 0 where it is virtual or absent.  The cells of depth r+1 come
// from the neighbours' child bases, each deeper cell from its parent's, which
// lies in the block one depth up; a cell's coefficient and child base load
// together.  The levels end where no cell of a block has children: most
// bricks of a large root see real nodes of the first depths below it only,
// and blocks of 5^3, 7^3 and 11^3 empty cells neither take time nor fill the
// LDS (109,000 of the 160,000 bricks that a screen with all the blocks left were
// left for those alone).
// A depth whose block holds no nonzero coefficient gets none.  Returns false
// when the caller's LDS cannot hold the blocks.
// (kThreads: of the workgroup, all of which take part.)
template <int kThreads = kWave, class L>
__device__ __forceinline__ bool brick_blocks(const SubArgs& A, const Brick& B, L& S) {
    constexpr int kCap = int(sizeof(S.XB) / sizeof(float));
    constexpr int kBatch = kThreads == kWave ? 3 : 1;
    constexpr int kCapC[2] = {int(sizeof(S.CB0) / sizeof(int32_t)), int(sizeof(S.CB1) / sizeof(int32_t))};
    const int D = A.D, lane = threadIdx.x;
    bool on = B.deep;  // (uniform) the next depth may have real cells
    int total = 0;
    if (lane <= kMaxDepth) S.xb_off[lane] = -1;
#pragma unroll 1
    for (int dd = B.r + 1; dd <= D && on; dd++) {  // (unrolled, its code came from memory at every launch)
        const int W = block_width(D, B.kb, dd), sh = D - dd, n = W * W * W;
        // child bases of depth dd - 1 in one buffer, of dd in the other
        const bool odd = (sh & 1) != 0;
        if (total + n > kCap || (dd < D && n > kCapC[odd ? 1 : 0])) return false;
        const int32_t* CBp = odd ? S.CB0 : S.CB1;
        int32_t* CBn = odd ? S.CB1 : S.CB0;
        const uint32_t rw = (65536u + uint32_t(W) - 1u) / uint32_t(W);
        const int32_t lo[3] = {(B.org[0] >> sh) - 2, (B.org[1] >> sh) - 2, (B.org[2] >> sh) - 2};
        const int32_t width = 1 << dd;
        const int Wp = dd > B.r + 1 ? block_width(D, B.kb, dd - 1) : 0;
        const int32_t plo[3] = {(B.org[0] >> (sh + 1)) - 2, (B.org[1] >> (sh + 1)) - 2, (B.org[2] >> (sh + 1)) - 2};
        bool kids = false, nz = false;
        // kBatch cells per thread at a time: their loads go out together
        for (int e0 = lane; e0 < n; e0 += kBatch * kThreads) {
            int32_t node[kBatch], ck[kBatch];
            float xv[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; u++) {
                // e / W and e / W^2 for e < W^3 <= 1331 by a 16-bit reciprocal (exact: e / W
                // has a fractional part of at most (W-1)/W, the reciprocal's excess adds < 0.03)
                const int e = e0 + u * kThreads;
                const int q1 = int((uint32_t(e) * rw) >> 16), q2 = int((uint32_t(q1) * rw) >> 16);
                const int32_t c[3] = {lo[0] + q2, lo[1] + (q1 - q2 * W), lo[2] + (e - q1 * W)};
                int32_t cb = -1;
                if (e < n && uint32_t(c[0]) < uint32_t(width) && uint32_t(c[1]) < uint32_t(width) &&
                    uint32_t(c[2]) < uint32_t(width)) {
                    if (dd == B.r + 1) {
                        const int ox = (c[0] >> 1) - B.R[0], oy = (c[1] >> 1) - B.R[1], oz = (c[2] >> 1) - B.R[2];
                        cb = (ox | oy | oz) ? S.NBK[nidx(ox, oy, oz)] : -1;
                    } else {
                        cb = CBp[(((c[0] >> 1) - plo[0]) * Wp + ((c[1] >> 1) - plo[1])) * Wp + ((c[2] >> 1) - plo[2])];
                    }
                }
                node[u] = cb < 0 ? -1 : cb + (((c[0] & 1) << 2) | ((c[1] & 1) << 1) | (c[2] & 1));
            }
#pragma unroll
            for (int u = 0; u < kBatch; u++) {
                xv[u] = node[u] < 0 ? 0.0f : A.x[node[u]];
                ck[u] = node[u] < 0 || dd >= D ? -1 : A.child_base[node[u]];
            }
#pragma unroll
            for (int u = 0; u < kBatch; u++) {
                const int e = e0 + u * kThreads;
                if (e >= n) continue;
                S.XB[total + e] = xv[u];
                if (dd < D) CBn[e] = ck[u];
                nz = nz || xv[u] != 0.0f;
                kids = kids || ck[u] >= 0;
            }
        }
        const bool any = any_thread<kThreads>(nz);
        on = any_thread<kThreads>(kids);
        if (any && lane == 0) S.xb_off[dd] = total;
        total += n;
        __syncthreads();  // this depth's child bases are read by the next
    }
    __syncthreads();
    return true;
}

// deep_sum for an owner leaf o of the brick's own root (the owner of grid
// point org + gi), reading the blocks and S.T.  Every one of the 27 terms is
// added: a neighbour that is virtual, absent or outside the domain
// contributes +-0 (its coefficient or its basis value is 0), which leaves a
// float sum that started at +0 unchanged, so the result is deep_sum's bit
// for bit.
template <class L>
__device__ __forceinline__ float deep_sum_lds(const SubArgs& A, const Brick& B, const L& S, const int32_t o[3], const int gi[3]) {
    const int D = A.D;
    float f = 0.0f;
    for (int dd = D; dd > B.r; dd--) {
        const int slot = S.xb_off[dd];
        if (slot < 0) continue;
        const int up = dd - B.r, sh = D - dd;
        const int32_t ax = o[0] >> sh, ay = o[1] >> sh, az = o[2] >> sh;
        const int32_t ext = (1 << up) - 1;
        const int32_t lx = B.R[0] << up, ly = B.R[1] << up, lz = B.R[2] << up;
        if (ax - 1 >= lx && ax + 1 <= lx + ext && ay - 1 >= ly && ay + 1 <= ly + ext && az - 1 >= lz &&
            az + 1 <= lz + ext)
            continue;
        const int W = block_width(D, B.kb, dd);
        const int bx0 = ax - 1 - ((B.org[0] >> sh) - 2), by0 = ay - 1 - ((B.org[1] >> sh) - 2),
                  bz0 = az - 1 - ((B.org[2] >> sh) - 2);
        const BasisT tx = S.T[3 * kP * dd + gi[0]];
        const BasisT ty = S.T[3 * kP * dd + kP + gi[1]];
        const BasisT tz = S.T[3 * kP * dd + 2 * kP + gi[2]];
        const float bx[3] = {tx.x, tx.y, tx.z}, by[3] = {ty.x, ty.y, ty.z}, bz[3] = {tz.x, tz.y, tz.z};
        const float* Xb = S.XB + slot;
#pragma unroll
        for (int k = 0; k < 27; k++) {
            const float xv = Xb[((bx0 + k / 9) * W + (by0 + (k / 3) % 3)) * W + (bz0 + k % 3)];
            float tt = xv * bx[k / 9];
            tt = tt * by[(k / 3) % 3];
            tt = tt * bz[k % 3];
            f = f + tt;
        }
    }
    return f;
}

// Sum over the real nodes below depth r (virtual coefficients are 0) for the
// corner of owner leaf o on sides s, in the reference's order: depth D up to
// r + 1, neighbours j = 0..26 of the owner's virtual ancestor
// (computeSubdivideVertexImplicitFunctionValue, main.cu:2346-2372).  R is the
// owner's root at depth r; kids(j) the child base of its neighbour j.  All 27
// neighbours descend together, one level's loads in flight at once: walking
// them one after another took a memory round trip per neighbour and level,
// 0.4 ms for the one brick per wave that a small cloud leaves to evaluate.
template <class KidsFn>
__device__ __forceinline__ float deep_sum(const SubArgs& A, int r, const int32_t R[3], const int32_t o[3], const int s[3],
                          KidsFn kids) {
    const int D = A.D;
    float f = 0.0f;
    for (int dd = D; dd > r; dd--) {
        const int up = dd - r, sh = D - dd;
        const int32_t ax = o[0] >> sh, ay = o[1] >> sh, az = o[2] >> sh;
        const int32_t ext = (1 << up) - 1;
        const int32_t lx = R[0] << up, ly = R[1] << up, lz = R[2] << up;
        // all 27 neighbours inside the root: virtual, nothing to add
        if (ax - 1 >= lx && ax + 1 <= lx + ext && ay - 1 >= ly && ay + 1 <= ly + ext && az - 1 >= lz &&
            az + 1 <= lz + ext)
            continue;
        const float4 tx = A.btab[((int64_t(dd) << D) + o[0]) * 2 + s[0]];
        const float4 ty = A.btab[((int64_t(dd) << D) + o[1]) * 2 + s[1]];
        const float4 tz = A.btab[((int64_t(dd) << D) + o[2]) * 2 + s[2]];
        const float bx[3] = {tx.x, tx.y, tx.z}, by[3] = {ty.x, ty.y, ty.z}, bz[3] = {tz.x, tz.y, tz.z};
        const int32_t width = 1 << dd;
        // the node of each neighbour, from the child base one level up; -1
        // where it is outside the domain, inside the root (virtual), absent
        // or below a coarse leaf
        int32_t cur[27];
#pragma unroll
        for (int k = 0; k < 27; k++) {
            const int32_t nx = ax + (k / 9 - 1), ny = ay + ((k / 3) % 3 - 1), nz = az + (k % 3 - 1);
            const int cx = (nx >> up) - R[0], cy = (ny >> up) - R[1], cz = (nz >> up) - R[2];
            const bool in = nx >= 0 && ny >= 0 && nz >= 0 && nx < width && ny < width && nz < width && (cx | cy | cz);
            cur[k] = in ? kids(nidx(cx, cy, cz)) : -1;
        }
        for (int l = r + 1; l <= dd; l++) {
            const int s2 = dd - l;
#pragma unroll
            for (int k = 0; k < 27; k++) {
                const int32_t nx = ax + (k / 9 - 1), ny = ay + ((k / 3) % 3 - 1), nz = az + (k % 3 - 1);
                const int oct = (((nx >> s2) & 1) << 2) | (((ny >> s2) & 1) << 1) | ((nz >> s2) & 1);
                cur[k] = cur[k] < 0 ? -1 : cur[k] + oct;
            }
            if (l < dd) {
#pragma unroll
                for (int k = 0; k < 27; k++) cur[k] = cur[k] < 0 ? -1 : A.child_base[cur[k]];
            }
        }
        float xv[27];
#pragma unroll
        for (int k = 0; k < 27; k++) xv[k] = cur[k] < 0 ? 0.0f : A.x[cur[k]];
#pragma unroll
        for (int k = 0; k < 27; k++) {
            float tt = xv[k] * bx[k / 9];
            tt = tt * by[(k / 3) % 3];
            tt = tt * bz[k % 3];
            f = cur[k] < 0 ? f : f + tt;
        }
    }
    return f;
}

// The root's chain from LDS (chain_value's order: depth r down to 1, then the
// root of the tree), continuing from f, for the owner of grid point org + gi
// in the brick's own root.
template <class L>
__device__ __forceinline__ float chain_lds(const L& S, int r, const int gi[3], float f) {
    for (int d = r; d >= 1; d--) {
        const BasisT tx = S.T[3 * kP * d + gi[0]];
        const BasisT ty = S.T[3 * kP * d + kP + gi[1]];
        const BasisT tz = S.T[3 * kP * d + 2 * kP + gi[2]];
        const float bx[3] = {tx.x, tx.y, tx.z}, by[3] = {ty.x, ty.y, ty.z}, bz[3] = {tz.x, tz.y, tz.z};
        const float* X = S.X + 27 * d;
#pragma unroll
        for (int j = 0; j < 27; j++) {
            float tt = X[j] * bx[j / 9];
            tt = tt * by[(j / 3) % 3];
            tt = tt * bz[j % 3];
            f = f + tt;
        }
    }
    const float b0x = S.T[gi[0]].y, b0y = S.T[kP + gi[1]].y, b0z = S.T[2 * kP + gi[2]].y;
    float tt = S.X[0] * b0x;
    tt = tt * b0y;
    tt = tt * b0z;
    return f + tt;
}

// The owner of grid point g (depth-D corner coordinates) of the brick's root
// cell: the smallest-key virtual leaf of the group around g.  Returns its
// root's neighbour slot (13: the brick's own root) and its cell in o.
template <class L>
__device__ __forceinline__ int corner_owner(const Brick& B, const L& S, int D, const int32_t g[3],
                                            int32_t o[3]) {
    uint32_t best = 0xffffffffu;
    int slot = 13;
    for (int t = 0; t < 8; t++) {
        const int32_t c[3] = {g[0] - 1 + (t & 1), g[1] - 1 + ((t >> 1) & 1), g[2] - 1 + (t >> 2)};
        int sl;
        if (!cell_virtual(B, S, D, c, &sl)) continue;
        const uint32_t k = cell_key(uint32_t(c[0]), uint32_t(c[1]), uint32_t(c[2]));
        if (k < best) {
            best = k;
            slot = sl;
            for (int a = 0; a < 3; a++) o[a] = c[a];
        }
    }
    return slot;
}

// f - iso at grid point g (depth-D corner coordinates) of the brick's root cell,
// computed by its owner: the smallest-key virtual leaf around it.
template <class L>
__device__ __forceinline__ float grid_value(const SubArgs& A, const Brick& B, const L& S, const int32_t g[3]) {
    const int D = A.D;
    int32_t o[3];
    int side[3];
    int slot = 13;
    const bool interior = g[0] > B.R0[0] && g[0] < B.R0[0] + B.Sr && g[1] > B.R0[1] && g[1] < B.R0[1] + B.Sr &&
                          g[2] > B.R0[2] && g[2] < B.R0[2] + B.Sr;
    if (interior) {
        // all 8 cells around are leaves of this root; (g - 1) has the smallest key
        for (int a = 0; a < 3; a++) {
            o[a] = g[a] - 1;
            side[a] = 1;
        }
    } else {
        slot = corner_owner(B, S, D, g, o);
        for (int a = 0; a < 3; a++) side[a] = g[a] - o[a];
    }
    if (slot == 13) {
        // o is own_cell along every axis: S.T holds its basis values
        const int gi[3] = {g[0] - B.org[0], g[1] - B.org[1], g[2] - B.org[2]};
        const float f = B.deep ? deep_sum_lds(A, B, S, o, gi) : 0.0f;
        return chain_lds(S, B.r, gi, f) - *A.iso;
    }
    // owned by a leaf of another root of the group: that root's record (its
    // neighbours, their child bases, its chain's values: what the neighbour
    // planes and chain_value would read), with the owner's basis values from
    // the corner basis table
    const int32_t* R2 = A.rec + int64_t(S.NBR[slot]) * kRecWords;
    const int32_t RC[3] = {B.R[0] + slot / 9 - 1, B.R[1] + (slot / 3) % 3 - 1, B.R[2] + slot % 3 - 1};
    float f = deep_sum(A, B.r, RC, o, side, [&](int j) { return R2[kRecNBK + j]; });
    for (int d = B.r; d >= 1; d--) {
        const float4 tx = A.btab[((int64_t(d) << D) + o[0]) * 2 + side[0]];
        const float4 ty = A.btab[((int64_t(d) << D) + o[1]) * 2 + side[1]];
        const float4 tz = A.btab[((int64_t(d) << D) + o[2]) * 2 + side[2]];
        const float bx[3] = {tx.x, tx.y, tx.z}, by[3] = {ty.x, ty.y, ty.z}, bz[3] = {tz.x, tz.y, tz.z};
        const int32_t* X = R2 + kRecX + 27 * d;
#pragma unroll
        for (int j = 0; j < 27; j++) {
            float tt = __int_as_float(X[j]) * bx[j / 9];
            tt = tt * by[(j / 3) % 3];
            tt = tt * bz[j % 3];
            f = f + tt;
        }
    }
    const float b0x = A.btab[o[0] * 2 + side[0]].y, b0y = A.btab[o[1] * 2 + side[1]].y, b0z = A.btab[o[2] * 2 + side[2]].y;
    float tt = __int_as_float(R2[kRecX]) * b0x;
    tt = tt * b0y;
    tt = tt * b0z;
    return f + tt - *A.iso;
}

// Owner of edge e of leaf v among the virtual leaves sharing it
// (initSubdivideEdgeArray, main.cu:1867-2019): its cell and the edge kind seen
// from it.
template <class L>
__device__ __forceinline__ void edge_owner(const Brick& B, const L& S, int D, const int32_t v[3], int e,
                                           int32_t ow[3], int* eo) {
    const int o = e >> 2;
    const int a1 = (o == 0) ? 1 : 0, a2 = (o == 2) ? 1 : 2;
    const int b1 = e & 1, b2 = (e >> 1) & 1;
    uint32_t best = cell_key(uint32_t(v[0]), uint32_t(v[1]), uint32_t(v[2]));
    for (int a = 0; a < 3; a++) ow[a] = v[a];
    *eo = e;
    for (int u = 0; u < 2; u++)
        for (int w = 0; w < 2; w++) {
            if (!(u | w)) continue;
            int32_t n[3] = {v[0], v[1], v[2]};
            if (u) n[a1] += 2 * b1 - 1;
            if (w) n[a2] += 2 * b2 - 1;
            int sl;
            if (!cell_virtual(B, S, D, n, &sl)) continue;
            const uint32_t kk = cell_key(uint32_t(n[0]), uint32_t(n[1]), uint32_t(n[2]));
            if (kk < best) {
                best = kk;
                for (int a = 0; a < 3; a++) ow[a] = n[a];
                *eo = (o << 2) | ((b2 ^ w) << 1) | (b1 ^ u);
            }
        }
}

// Cube index and owned crossing edges of leaf l of the brick
// (generateSubdivideVexNums, main.cu:2481-2531; generateTriNums, :2562-2582).
// (G: the brick's corner values, (i, j, k) at (k kStride + j) kStride + i)
template <int kStride = kP, class L>
__device__ __forceinline__ void leaf_cube(const Brick& B, const L& S, const float* G, int D, int l, int32_t v[3],
                                          float cv[8], int* cube, int* emask) {
    const int lx = int(compact3(uint32_t(l) >> 2)), ly = int(compact3(uint32_t(l) >> 1)), lz = int(compact3(uint32_t(l)));
    v[0] = B.org[0] + lx;
    v[1] = B.org[1] + ly;
    v[2] = B.org[2] + lz;
    int cb = 0;
#pragma unroll
    for (int q = 0; q < 8; q++) {
        const int y = (q >> 1) & 1, xx = (q & 1) ^ y, z = q >> 2;
        cv[q] = G[((lz + z) * kStride + (ly + y)) * kStride + (lx + xx)];
        if (cv[q] < 0) cb |= 1 << q;
    }
    *cube = cb;
    // a leaf not on its root's boundary owns exactly its edges on the high side
    // of both other axes (kinds 3, 7, 11): its 26 neighbours are all in the root
    bool inner = true;
    for (int a = 0; a < 3; a++) inner = inner && v[a] > B.R0[a] && v[a] < B.R0[a] + B.Sr - 1;
    int m = 0;
#pragma unroll
    for (int e = 0; e < 12; e++) {
        const float f1 = cv[c_edge_vertex_h[e][0]], f2 = cv[c_edge_vertex_h[e][1]];
        if (!(f1 * f2 <= 0)) continue;
        bool own;
        if (inner) {
            own = (e & 3) == 3;
        } else {
            int32_t ow[3];
            int eo;
            edge_owner(B, S, D, v, e, ow, &eo);
            own = ow[0] == v[0] && ow[1] == v[1] && ow[2] == v[2];
        }
        if (own) m |= 1 << e;
    }
    *emask = m;
}

// The function over a cell from the depths up to its own (c = D - kb), lane i
// < 27 returning control value i of its polynomial: the chain's (restricted
// from the root's) plus, per depth r + 1 .. c, the spline of the block's three
// cells per axis around the cell's ancestor.  A corner's owner may be a leaf
// of the cell below along an axis; its 27 neighbours then reach one cell
// further down and one less up, and the spline of the cell left out is 0
// there.  The corners' float values differ from it by at most *slack: dev[d]
// times the largest |x| per depth (depth_bounds, the rounding of all sums
// included).  *finite: false in a lane that saw a coefficient that is not (a
// maximum passes over NaN; it also makes every control value NaN).
template <class L>
__device__ __forceinline__ float cell_polynomial(const SubArgs& A, const Brick& B, const L& S, float* slack,
                                                 bool* finite) {
    const int D = A.D, lane = threadIdx.x, c = D - B.kb;
    const int l27 = lane < 27 ? lane : 0;
    const int i3[3] = {l27 / 9, (l27 / 3) % 3, l27 % 3};
    float w[3][3];
    const float inv = 1.0f / float(B.Sr);
#pragma unroll
    for (int a = 0; a < 3; a++)
        bernstein_weights(float(B.org[a] - B.R0[a]) * inv, float(1 << B.kb) * inv, i3[a], w[a]);
    float val = sum27(S.P, 9, 3, w);
    *slack = __int_as_float(__builtin_amdgcn_readfirstlane(A.rec[int64_t(B.q) * kRecWords + kRecErr]));
    for (int d = B.r + 1; d <= c; d++) {
        const int o = S.xb_off[d];  // (uniform)
        if (o < 0) continue;
        const float x = fabsf(S.XB[o + lane]);  // 4^3 cells
        *finite = *finite && x < INFINITY;
#pragma unroll
        for (int a = 0; a < 3; a++) spline_weights(B.org[a] >> B.kb, c - d, i3[a], w[a]);
        val += sum27(S.XB + o + 21, 16, 4, w);  // slots 1..3 along each axis
        *slack += A.dev[d] * wave_max(x);
    }
    *finite = *finite && fabsf(val) < INFINITY;
    return val;
}

// A sign for every corner of the cell that its root owns: the polynomial's
// range lies between the smallest and the largest control value; the depths
// below the cell's add at most their largest |x| times big[d] each.  The cell
// is settled when all of that is clear of iso.
template <class L>
__device__ __forceinline__ int cell_sign(const SubArgs& A, const Brick& B, const L& S) {
    const int D = A.D, lane = threadIdx.x, c = D - B.kb;
    bool finite = true;
    float slack;
    const float val = cell_polynomial(A, B, S, &slack, &finite);
    for (int d = c + 1; d <= D; d++) {
        const int o = S.xb_off[d];  // (uniform)
        if (o < 0) continue;
        const int W = block_width(D, B.kb, d), n = W * W * W;
        float m = 0.0f;
        for (int e = lane; e < n; e += kWave) {
            const float x = fabsf(S.XB[o + e]);
            m = fmaxf(m, x);
            finite = finite && x < INFINITY;
        }
        slack += (A.big[d] + A.dev[d]) * wave_max(m);
    }
    if (__builtin_amdgcn_ballot_w64(!finite) != 0) return 0;
    const float hi = wave_max(val), lo = -wave_max(-val);
    const float iso = *A.iso;
    const float margin = 1.001f * slack + 1.2e-7f * (fabsf(lo) + fabsf(hi) + 2.0f * fabsf(iso)) + 1e-15f;
    if (lo - iso > margin) return 1;
    if (hi - iso < -margin) return -1;
    return 0;
}

// The offsets (bit nidx(delta)) of the bricks holding the owners of the
// brick's corners that leaves of other roots of the group own.
template <class L>
__device__ __forceinline__ uint32_t brick_group_deps(const Brick& B, const L& S, int D) {
    const int Sb = 1 << B.kb, P = Sb + 1;
    uint32_t deps = 0;
    for (int p = threadIdx.x; p < kBrickPts; p += kWave) {
        const int i = p % kP, j = (p / kP) % kP, k = p / (kP * kP);
        if (i >= P || j >= P || k >= P) continue;
        const int32_t g[3] = {B.org[0] + i, B.org[1] + j, B.org[2] + k};
        bool interior = true;
        for (int a = 0; a < 3; a++) interior = interior && g[a] > B.R0[a] && g[a] < B.R0[a] + B.Sr;
        if (interior) continue;
        int32_t o[3];
        if (corner_owner(B, S, D, g, o) == 13) continue;
        int dv[3];
        for (int a = 0; a < 3; a++) dv[a] = o[a] < B.org[a] ? -1 : (o[a] >= B.org[a] + Sb ? 1 : 0);
        deps |= 1u << nidx(dv[0], dv[1], dv[2]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) deps |= uint32_t(__shfl_xor(int(deps), o, kWave));
    return deps;
}

// Whether the brick touches a face, edge or corner its root shares with
// another root of the group (whose leaves may own corners of the brick).
template <class L>
__device__ __forceinline__ bool brick_in_group(const Brick& B, const L& S) {
    const int Sb = 1 << B.kb;
    bool lo[3], hi[3];
    for (int a = 0; a < 3; a++) {
        lo[a] = B.org[a] == B.R0[a];
        hi[a] = B.org[a] + Sb == B.R0[a] + B.Sr;
    }
    bool group = false;
    for (int j = 0; j < 27; j++) {
        if (j == 13 || S.NBR[j] < 0) continue;
        const int dv[3] = {j / 9 - 1, (j / 3) % 3 - 1, j % 3 - 1};
        bool touches = true;
        for (int a = 0; a < 3; a++)
            if (dv[a] != 0) touches = touches && (dv[a] < 0 ? lo[a] : hi[a]);
        group = group || touches;
    }
    return group;
}

// Proves, when it can, that every corner value of the 8^3 brick has one strict
// sign, so the brick has no crossing edge and no triangle.  Each lane owns the
// column of grid points (*, j, k).  The depths up to D - 3, whose cell holds
// the whole brick, are one polynomial (cell_polynomial), contracted over z and
// y to three values per column and then evaluated at its nine points.  At the
// three finer depths d, where the brick spans several cells, the sum
// S(g) = sum_k x_k b_x b_y b_z over the corner owner's 27 neighbours is formed
// from the same float coefficients and basis table entries the evaluation
// reads, contracted over z and y per x slot of the block and added to the
// points whose owners see the slot.  The float value the evaluation computes,
// a sum of n <= 27 (D + 1) + 1 products of three roundings each, differs from
// S(g) by at most (n + 3) 2^-24 A(g) with A(g) = sum_k |x_k b_x b_y b_z|
// (recursive summation bound); the contraction's own rounding adds less than
// 60 2^-24 A(g), and A(g) is at most the block's sum of |x| times the cube of
// the largest |basis value| among the entries: 560 2^-24 of that covers both
// (float sums of non-negative terms are within 0.1%).  The polynomial's share
// of the distance is cell_polynomial's slack, its evaluation here less than 40
// roundings of its largest control value.  The brick is certified when the
// distance to iso exceeds all of it with one sign at every corner its root
// owns.  A corner on the root's boundary may be owned by a leaf of another
// root of the group: its value is the one that root's brick holding the owner
// computes for its own corner (the same owner, table entries and order), so
// the sign is compared with that brick's afterwards (k_group_check).  Returns
// +1 or -1 (every corner the brick's root owns has this sign) or 0 (not
// proven).  Depth by depth over the columns, all from the tables, this took
// 33 ns a brick; the list was half as long again.
__device__ __forceinline__ int brick_certify(const SubArgs& A, const Brick& B, const CertLds& S, bool group) {
    const int D = A.D, lane = threadIdx.x, c = D - kBrickLog;
    const float iso = *A.iso;
    bool finite = true;
    float slack;
    const float val = cell_polynomial(A, B, S, &slack, &finite);
    float fine = 0.0f;
    for (int d = c + 1; d <= D; d++) {
        const int o = S.xb_off[d];  // (uniform)
        if (o < 0) continue;
        const int W = block_width(D, kBrickLog, d), n = W * W * W;
        float sx = 0.0f;
        for (int e = lane; e < n; e += kWave) sx += fabsf(S.XB[o + e]);
#pragma unroll
        for (int h = 32; h > 0; h >>= 1) sx += __shfl_xor(sx, h, kWave);
        const BasisT t = S.T[3 * kP * (d - c - 1) + (lane < 3 * kP ? lane : 0)];
        const float tm = wave_max(fmaxf(fabsf(t.x), fmaxf(fabsf(t.y), fabsf(t.z))));
        fine += sx * (tm * tm * tm);
    }
    finite = finite && fine < INFINITY;
    if (__builtin_amdgcn_ballot_w64(!finite) != 0) return 0;
    const float margin0 = 1.001f * slack + 1.001f * (560.0f * 5.9604645e-8f) * fine +
                          2.4e-6f * wave_max(fabsf(val)) + 1e-15f;
    float Q[27];  // the control values, uniform
#pragma unroll
    for (int q = 0; q < 27; q++) Q[q] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(val), q));
    bool ok = true, pos = false, neg = false;
    for (int pp = lane; pp < kP * kP; pp += kWave) {
        const int j = pp % kP, k = pp / kP;
        const float tj = float(j) * 0.125f, tk = float(k) * 0.125f;
        const float wj[3] = {(1.0f - tj) * (1.0f - tj), 2.0f * tj * (1.0f - tj), tj * tj};
        const float wk[3] = {(1.0f - tk) * (1.0f - tk), 2.0f * tk * (1.0f - tk), tk * tk};
        float Y[3];
#pragma unroll
        for (int m = 0; m < 3; m++) {
            float y = 0.0f;
#pragma unroll
            for (int n = 0; n < 3; n++) {
                float z = 0.0f;
#pragma unroll
                for (int l = 0; l < 3; l++) z = __builtin_fmaf(Q[9 * m + 3 * n + l], wk[l], z);
                y = __builtin_fmaf(wj[n], z, y);
            }
            Y[m] = y;
        }
        float v[kP];
#pragma unroll
        for (int i = 0; i < kP; i++) {
            const float t = float(i) * 0.125f;  // (constants: i is unrolled)
            v[i] = __builtin_fmaf(t * t, Y[2], __builtin_fmaf(2.0f * t * (1.0f - t), Y[1], (1.0f - t) * (1.0f - t) * Y[0]));
        }
        // the finer depths, where the brick spans several cells: per x slot m
        // of the block, Y_m = sum over the lane's 3 y and 3 z slots, then
        // each point adds its owner's three x slots' Y (the slots a point's
        // owner sees follow from grid coordinates alone: uniform per i)
        for (int d = c + 1; d <= D; d++) {
            const int slot = S.xb_off[d];
            if (slot < 0) continue;
            const int sh = D - d, W = block_width(D, kBrickLog, d);
            const BasisT* T = S.T + 3 * kP * (d - c - 1);
            const int b1 = (own_cell(B.org[1] + j, B.R0[1]) >> sh) - 1 - ((B.org[1] >> sh) - 2);
            const int b2 = (own_cell(B.org[2] + k, B.R0[2]) >> sh) - 1 - ((B.org[2] >> sh) - 2);
            const BasisT ty = T[kP + j], tz = T[2 * kP + k];
            const float by[3] = {ty.x, ty.y, ty.z}, bz[3] = {tz.x, tz.y, tz.z};
            int b0[kP];
            float bx[kP][3];
#pragma unroll
            for (int i = 0; i < kP; i++) {
                b0[i] = (own_cell(B.org[0] + i, B.R0[0]) >> sh) - 1 - ((B.org[0] >> sh) - 2);
                const BasisT tx = T[i];
                bx[i][0] = tx.x;
                bx[i][1] = tx.y;
                bx[i][2] = tx.z;
            }
#pragma unroll
            for (int m = 0; m < 11; m++) {  // W <= 11
                if (m >= W || m < b0[0] || m > b0[kP - 1] + 2) continue;  // (uniform) a slot no point sees
                const float* Xm = S.XB + slot + m * W * W;
                float y = 0.0f;
#pragma unroll
                for (int n = 0; n < 3; n++) {
                    float z = 0.0f;
#pragma unroll
                    for (int l = 0; l < 3; l++) z = __builtin_fmaf(Xm[(b1 + n) * W + (b2 + l)], bz[l], z);
                    y = __builtin_fmaf(by[n], z, y);
                }
#pragma unroll
                for (int i = 0; i < kP; i++) {
                    const int q = m - b0[i];  // uniform
                    if (q >= 0 && q <= 2) v[i] = __builtin_fmaf(q == 0 ? bx[i][0] : q == 1 ? bx[i][1] : bx[i][2], y, v[i]);
                }
            }
        }
        const bool jk_inner = B.org[1] + j > B.R0[1] && B.org[1] + j < B.R0[1] + B.Sr && B.org[2] + k > B.R0[2] &&
                              B.org[2] + k < B.R0[2] + B.Sr;
#pragma unroll
        for (int i = 0; i < kP; i++) {
            const int32_t gx = B.org[0] + i;
            if (group && !(jk_inner && gx > B.R0[0] && gx < B.R0[0] + B.Sr)) {
                // on the root's boundary: is the owner a leaf of another root?
                const int32_t g[3] = {gx, B.org[1] + j, B.org[2] + k};
                int32_t o[3];
                if (corner_owner(B, S, D, g, o) != 13) continue;
            }
            const float dist = v[i] - iso;
            const float margin = margin0 + 1.2e-7f * (fabsf(v[i]) + fabsf(iso));
            ok = ok && fabsf(dist) > margin;
            pos = pos || dist > 0;
            neg = neg || dist < 0;
        }
    }
    const bool lane_good = ok && !(pos && neg);
    const uint64_t good = __builtin_amdgcn_ballot_w64(lane_good);
    const uint64_t anypos = __builtin_amdgcn_ballot_w64(pos), anyneg = __builtin_amdgcn_ballot_w64(neg);
    return (good == ~uint64_t(0) && !(anypos && anyneg)) ? (anypos ? 1 : -1) : 0;
}

// The roots of 8^3 leaves and more: each is the first cell of its size to be
// screened (lists: the cells of 2^k leaves a side at lists.at[k], as the
// number of their first brick).
struct CellLists {
    int32_t* at[kMaxDepth + 1];
};

__global__ void __launch_bounds__(kBlockS) k_list_roots(const int32_t* roots, const int32_t* boff, int64_t nr, Levels L,
                                                        int D, CellLists lists, int32_t* cnt) {
    const int64_t q = int64_t(blockIdx.x) * kBlockS + threadIdx.x;
    const int kb = q < nr ? D - depth_of(roots[q], L, D) : 0;
#pragma unroll
    for (int k = kBrickLog; k <= kMaxDepth; k++) {
        if (k >= D) break;
        const int32_t at = wave_append(kb == k, cnt + kCntCells + k);
        if (kb == k) lists.at[k][at] = boff[q];
    }
}

// Entries a wave has found for a list, in LDS until there are kWaveList: one
// atomic on the list's counter for all of them.  (An atomic per entry, and one
// per few entries taken from the input list, was most of the screens' and the
// certificate's time: thousands of waves on one counter wait for each other,
// 43 us a cell in k_cell_screen.)
constexpr int kWaveList = 128;
struct WaveList {
    int32_t e[kWaveList];
};

// Appends the n buffered entries times `each` (entry j * each + i: e[j] + (i << shift)).
__device__ __forceinline__ void wave_flush(const WaveList& L, int32_t n, int32_t each, int shift, int32_t* counter,
                                           int32_t* list) {
    __syncthreads();  // (one wave: the buffered entries are in LDS)
    int32_t at = 0;
    if (threadIdx.x == 0 && n > 0) at = atomicAdd(counter, n * each);
    at = __shfl(at, 0, kWave);
    for (int32_t j = threadIdx.x; j < n * each; j += kWave) {
        const int32_t q = each == 1 ? j : j >> 3, i = each == 1 ? 0 : j & 7;  // (each is 1 or 8)
        list[at + j] = L.e[q] + (i << shift);
    }
    __syncthreads();
}

// Buffers v of the lanes with `want` (uniform n), flushing before it is full.
__device__ __forceinline__ int32_t wave_push(WaveList& L, int32_t n, bool want, int32_t v, int32_t* counter,
                                             int32_t* list) {
    const uint64_t m = __builtin_amdgcn_ballot_w64(want);
    if (m == 0) return n;
    if (n + kWave > kWaveList) {
        wave_flush(L, n, 1, 0, counter, list);
        n = 0;
    }
    if (want) L.e[n + int32_t(__popcll(m & ((uint64_t(1) << threadIdx.x) - 1)))] = v;
    return n + int32_t(__popcll(m));
}

// Pass 0: screens the listed cells of 2^k leaves a side, one wave each (a
// resident grid strides over the list).  A settled cell gives its bricks its
// sign (their counts stay 0), and lists those that touch another root of the
// group for k_group_check; of the others, a cell of more than one brick lists
// its eight parts for the next size and a brick goes to the per-corner
// certificate.  Most of the refined volume is far from the surface and settles
// in large cells.  All passes of the screens, 2 M points at depth 10
// (1,036,945 bricks): 1333 us with shared counters for the list's next entries
// and for each entry found, 925 us without.
template <int FLOATS>
__global__ void __launch_bounds__(kWave, FLOATS > kXBlkScreen ? 3 : 5) k_cell_screen(SubArgs A, int k, const int32_t* list, int32_t* parts,
                                                       int32_t* xlist, int8_t* sign, int32_t* glist, int32_t* cnt,
                                                       int certify) {
    __shared__ CellLds<FLOATS> S;
    __shared__ WaveList left, group;
    const int lane = threadIdx.x;
    const int32_t n = cnt[kCntCells + k];
    const bool brick = k == kBrickLog;
    int32_t* const next = brick ? xlist : parts;
    int32_t* const next_cnt = cnt + (brick ? int(kCntExact) : kCntCells + k - 1);
    const int32_t each = brick ? 1 : 8;
    const int shift = brick ? 0 : 3 * (k - 1 - kBrickLog);
    int32_t q_loaded = -1, nleft = 0, ngroup = 0;
    for (int32_t it = blockIdx.x; it < n; it += int32_t(gridDim.x)) {
        const int32_t b = list[it];
        Brick B;
        __syncthreads();  // the previous cell's LDS reads are done
        cell_setup(A, b, k, B, S, q_loaded);
        q_loaded = B.q;
        int s = 0;
        if (certify && brick_blocks(A, B, S)) s = cell_sign(A, B, S);
        if (s == 0) {
            if (nleft == kWaveList) {
                wave_flush(left, nleft, each, shift, next_cnt, next);
                nleft = 0;
            }
            if (lane == 0) left.e[nleft] = b;
            nleft++;
            continue;
        }
        // the cell's bricks; those on a face, edge or corner shared with the group
        const uint64_t in_group = __builtin_amdgcn_ballot_w64(lane < 27 && lane != 13 && S.NBR[lane < 27 ? lane : 0] >= 0);
        const uint32_t gm = uint32_t(in_group);
        const bool touches = gm && brick_in_group(B, S);
        const int32_t nbk = 1 << (3 * (k - kBrickLog));
        for (int32_t i0 = 0; i0 < nbk; i0 += kWave) {
            const int32_t i = i0 + lane;
            const bool in = i < nbk;
            if (in) sign[b + i] = int8_t(s);
            if (touches) {
                int32_t o[3];
                decode_cell(uint32_t(i), o);
                uint32_t m[3];
#pragma unroll
                for (int a = 0; a < 3; a++) {
                    // neighbour slots with offset -1, 0, +1 along axis a
                    const uint32_t z = a == 0 ? 0x000001ffu : a == 1 ? 0x001c0e07u : 0x01249249u;
                    const int step = a == 0 ? 9 : a == 1 ? 3 : 1;
                    const int32_t g = B.org[a] + (o[a] << kBrickLog);
                    m[a] = z << step;
                    if (g == B.R0[a]) m[a] |= z;
                    if (g + (1 << kBrickLog) == B.R0[a] + B.Sr) m[a] |= z << (2 * step);
                }
                const bool want = in && (m[0] & m[1] & m[2] & gm) != 0;
                ngroup = wave_push(group, ngroup, want, b + i, cnt + kCntGroup, glist);
            }
        }
    }
    wave_flush(left, nleft, each, shift, next_cnt, next);
    wave_flush(group, ngroup, 1, 0, cnt + kCntGroup, glist);
}

// Pass 0b: the per-corner certificate (brick_certify) for the bricks the
// screen left (a resident grid strides over them); the bricks it does not
// settle are listed for the evaluation.
// Bound by the length of a wave's work, not by memory: 5,800 vector and as
// many scalar instructions a brick, half of the cycles spent waiting on the
// chain of block levels and LDS reads; 0.39 ms for the 13,508 bricks of 2 M
// points at depth 10.  Three waves a brick (one per finest depth and per
// three points of a column) shorten the chain but repeat the set-up: 5% less
// there, 3% more on the 5,000 bricks of a torus at depth 9.
__global__ void __launch_bounds__(kWave, 3) k_brick_exact(SubArgs A, const int32_t* xlist, int8_t* sign, int32_t* list,
                                                       int32_t* glist, int32_t* cnt, int certify) {
    __shared__ CertLds S;
    __shared__ WaveList left, group;
    const int lane = threadIdx.x;
    const int32_t n = cnt[kCntExact];
    int32_t q_loaded = -1, nleft = 0, ngroup = 0;
    for (int32_t it = blockIdx.x; it < n; it += int32_t(gridDim.x)) {
        const int32_t b = xlist[it];
        Brick B;
        __syncthreads();  // the previous brick's LDS reads are done
        cell_setup(A, b, kBrickLog, B, S, q_loaded);
        q_loaded = B.q;
        if (lane < kBrickLog * kP) {
            const int d = A.D - kBrickLog + 1 + lane / kP, i = lane % kP;
#pragma unroll
            for (int ax = 0; ax < 3; ax++) {
                const int32_t g = B.org[ax] + i, o = own_cell(g, B.R0[ax]);
                const float4 t = A.btab[((int64_t(d) << A.D) + o) * 2 + (g - o)];
                S.T[3 * kP * (lane / kP) + kP * ax + i] = BasisT{t.x, t.y, t.z};
            }
        }
        const bool fits = brick_blocks(A, B, S);
        const bool in_group = brick_in_group(B, S);
        const int s = certify && fits ? brick_certify(A, B, S, in_group) : 0;
        if (lane == 0) sign[b] = int8_t(s);
        nleft = wave_push(left, nleft, lane == 0 && s == 0, b, cnt + kCntDense, list);
        ngroup = wave_push(group, ngroup, lane == 0 && s != 0 && in_group, b, cnt + kCntGroup, glist);
    }
    wave_flush(left, nleft, 1, 0, cnt + kCntDense, list);
    wave_flush(group, ngroup, 1, 0, cnt + kCntGroup, glist);
}

// The corner values of the bricks the certificates left (grid_value): gv at
// kBrickPts per listed brick.  A value is a serial chain of LDS reads and
// sums, so what counts is the waves in flight; a brick's tables and blocks are
// 16 KB of LDS, which held them to 2.5 per SIMD as one wave per brick (532 us
// for 3,338 bricks of 150,000 points at depth 10; 277 us with four, for 3,418).  `slices` workgroups share the rounds
// of a brick (each sets up its own tables and blocks): a list shorter than the
// chip leaves each of them one round instead of all three.
constexpr int kValThreads = 256;
constexpr int kValRounds = (kBrickPts + kValThreads - 1) / kValThreads;
__global__ void __launch_bounds__(kValThreads, 5) k_brick_values(SubArgs A, const int32_t* list, int slices, float* gv) {
    __shared__ BrickCore S;
    const int32_t it = int32_t(blockIdx.x) / slices;
    const int per = kValRounds / slices, first = (int(blockIdx.x) % slices) * per;
    Brick B;
    brick_setup<kValThreads>(A, list[it], B, S);
    brick_tables<kValThreads>(A, B, S);
    brick_blocks<kValThreads>(A, B, S);
    float* out = gv + int64_t(it) * kBrickPts;
    for (int t = first; t < first + per; t++) {
        const int p = threadIdx.x + kValThreads * t;
        if (p >= kBrickPts) break;
        const int32_t g[3] = {B.org[0] + p % kP, B.org[1] + (p / kP) % kP, B.org[2] + p / (kP * kP)};
        out[p] = grid_value(A, B, S, g);
    }
}

// The vertices of the leaf with key k on the edges of mask em, from its corner
// values (interpolatePoint and generateSubdivideIntersectionPoint,
// main.cu:2584-2597, 2629-2697); returns their number.
__device__ __forceinline__ int emit_leaf_vertices(uint32_t k, int D, int em, const float cv[8], float* out) {
    float c[3];
    node_center(k, D, D, c);
    const float hw = 1.0f / float(1 << (D + 1));
    int n = 0;
#pragma unroll
    for (int e = 0; e < 12; e++) {
        if (!(em & (1 << e))) continue;
        const int q1 = c_edge_vertex_h[e][0], q2 = c_edge_vertex_h[e][1];
        float p1[3], p2[3];
        {
            const int y = (q1 >> 1) & 1, xx = (q1 & 1) ^ y, z = q1 >> 2;
            p1[0] = c[0] + float(2 * xx - 1) * hw;
            p1[1] = c[1] + float(2 * y - 1) * hw;
            p1[2] = c[2] + float(2 * z - 1) * hw;
        }
        {
            const int y = (q2 >> 1) & 1, xx = (q2 & 1) ^ y, z = q2 >> 2;
            p2[0] = c[0] + float(2 * xx - 1) * hw;
            p2[1] = c[1] + float(2 * y - 1) * hw;
            p2[2] = c[2] + float(2 * z - 1) * hw;
        }
        const float f1 = cv[q1], f2 = cv[q2];
        const int dim = e >> 2;
        float o3[3] = {p1[0], p1[1], p1[2]};
        const float pivot = f1 / (f1 - f2);
        const float another = 1 - pivot;
        const float s1 = p2[dim] * pivot;
        const float s2 = p1[dim] * another;
        o3[dim] = s1 + s2;
        out[3 * n + 0] = o3[0];
        out[3 * n + 1] = o3[1];
        out[3 * n + 2] = o3[2];
        n++;
    }
    return n;
}

// The vertex of edge e of leaf v: its owner leaf's place (root number q2, -1
// if none, and Morton offset mort in the root) and the edge kind seen there.
// root_of_slot(j): the root number of the brick's root's neighbour j.
template <class L, class RootFn>
__device__ __forceinline__ int32_t edge_vertex_place(const Brick& B, const L& S, int D, const int32_t v[3], int e,
                                                     RootFn root_of_slot, uint32_t* mort, int* eo) {
    int32_t ow[3];
    edge_owner(B, S, D, v, e, ow, eo);
    int sl = 13;
    cell_virtual(B, S, D, ow, &sl);
    const int sh = 3 * (D - B.r);
    const uint32_t rmask = sh >= 32 ? 0xffffffffu : ((1u << sh) - 1u);
    *mort = cell_key(uint32_t(ow[0]), uint32_t(ow[1]), uint32_t(ow[2])) & rmask;
    return sl == 13 ? B.q : root_of_slot(sl);
}

// Per-leaf tables (the evaluated bricks': place in the list x 512 + leaf; the
// small roots': place x leaves + leaf): owned crossing edges, first vertex
// within the brick, cube index.
struct LeafTabs {
    uint16_t* emask;
    uint16_t* lofs;
    uint8_t* cube;
};

// The group's roots around a root as a bit mask, for the owner tests (which
// only ask whether a neighbour is in the group).
struct GroupMask {
    struct {
        uint32_t m;
        __device__ __forceinline__ int32_t operator[](int j) const { return ((m >> j) & 1u) ? 0 : -1; }
    } NBR;
};

// An 8^3 brick's geometry and group, for passes without its root's record in
// LDS (every wave for itself).
__device__ __forceinline__ void brick_geometry(const SubArgs& A, int32_t b, Brick& B, GroupMask& S) {
    const int lane = threadIdx.x & 63;
    B.q = __builtin_amdgcn_readfirstlane(A.bmap[b]);
    const int32_t* R = A.rec + int64_t(B.q) * kRecWords;
    cell_geometry(A, b, kBrickLog, R, B);
    S.NBR.m = uint32_t(__builtin_amdgcn_ballot_w64(lane < 27 && R[kRecNBR + (lane < 27 ? lane : 0)] >= 0));
}

// The settled bricks with corners that leaves of other roots of the group
// own: settled only when every brick holding such an owner carries the same
// sign; the others are listed for the evaluation.  The bricks around it in
// other roots of the group include all of those, and mostly agree, so the
// owners themselves are looked up only when one does not.
__global__ void __launch_bounds__(kWave) k_group_check(SubArgs A, const int32_t* glist, const int8_t* sign,
                                                       int32_t* list, int32_t* cnt) {
    __shared__ WaveList left;
    const int lane = threadIdx.x, D = A.D;
    const int32_t n = cnt[kCntGroup];
    int32_t nleft = 0;
    for (int32_t it = blockIdx.x; it < n; it += int32_t(gridDim.x)) {
        const int32_t b = glist[it];
        Brick B;
        GroupMask S;
        brick_geometry(A, b, B, S);
        // the brick at offset nidx = lane, when another root of the group holds it
        bool other = false, differs = false;
        if (lane < 27) {
            int32_t cc[3];
            int ro[3];
            const int sh = D - B.r;
            for (int a = 0; a < 3; a++) {
                const int dv = (a == 0 ? lane / 9 : a == 1 ? (lane / 3) % 3 : lane % 3) - 1;
                cc[a] = B.org[a] + (dv << kBrickLog);
                ro[a] = (cc[a] >> sh) - B.R[a];
            }
            const int slot = nidx(ro[0], ro[1], ro[2]);
            const int32_t q2 = slot == 13 ? -1 : A.rec[int64_t(B.q) * kRecWords + kRecNBR + slot];
            if (q2 >= 0) {
                const uint32_t rmask = 3 * sh >= 32 ? 0xffffffffu : ((1u << (3 * sh)) - 1u);
                const uint32_t mort = cell_key(uint32_t(cc[0]), uint32_t(cc[1]), uint32_t(cc[2])) & rmask;
                other = true;
                differs = sign[A.boff[q2] + int32_t(mort >> (3 * kBrickLog))] != sign[b];
            }
        }
        const uint64_t bad = __builtin_amdgcn_ballot_w64(differs);
        if (bad == 0) continue;
        const uint64_t around = __builtin_amdgcn_ballot_w64(other);
        const uint32_t deps = brick_group_deps(B, S, D);
        // (an owner in a brick outside the group's roots cannot be)
        const bool listed = (deps & uint32_t(bad)) || (deps & ~uint32_t(around));
        nleft = wave_push(left, nleft, lane == 0 && listed, b, cnt + kCntDense, list);
    }
    wave_flush(left, nleft, 1, 0, cnt + kCntDense, list);
}

// Exclusive sum of v over the workgroup's 512 threads, and the total.
__device__ __forceinline__ int block_excl_scan(int v, int* total) {
    __shared__ int sums[kBrickLeaves / kWave];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int inc = v;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int t = __shfl_up(inc, o, kWave);
        if (lane >= o) inc += t;
    }
    __syncthreads();
    if (lane == kWave - 1) sums[wave] = inc;
    __syncthreads();
    int base = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kBrickLeaves / kWave; w++) {
        if (w < wave) base += sums[w];
        all += sums[w];
    }
    *total = all;
    return base + inc - v;
}

// Cube indices and owned crossing edges of the evaluated bricks' leaves, the
// bricks' vertex and triangle counts, and their places in the list (didx).
__global__ void __launch_bounds__(kBrickLeaves) k_brick_cubes(SubArgs A, const int32_t* list, const float* gv,
                                                              LeafTabs T, int32_t* bnv, int32_t* bnt, int32_t* didx) {
    __shared__ float G[kBrickPts];
    const int32_t it = blockIdx.x, b = list[it], l = threadIdx.x;
    for (int p = l; p < kBrickPts; p += kBrickLeaves) G[p] = gv[int64_t(it) * kBrickPts + p];
    Brick B;
    GroupMask S;
    brick_geometry(A, b, B, S);
    __syncthreads();
    int32_t v[3];
    float cv[8];
    int cube, em;
    leaf_cube(B, S, G, A.D, l, v, cv, &cube, &em);
    int nv, nt;
    const int ofs = block_excl_scan(__popc(uint32_t(em)), &nv);
    (void)block_excl_scan(tri_count(cube), &nt);
    const int64_t at = int64_t(it) * kBrickLeaves + l;
    T.emask[at] = uint16_t(em);
    T.lofs[at] = uint16_t(ofs);
    T.cube[at] = uint8_t(cube);
    if (l == 0) {
        bnv[b] = nv;
        bnt[b] = nt;
        didx[b] = it;
    }
}

// The vertices of the evaluated bricks.
__global__ void __launch_bounds__(kBrickLeaves) k_brick_vertices(SubArgs A, const int32_t* list, const float* gv,
                                                                 LeafTabs T, const int32_t* bnv, const int32_t* bvoff,
                                                                 float* out_v) {
    __shared__ float G[kBrickPts];
    const int32_t it = blockIdx.x, b = list[it], l = threadIdx.x;
    if (bnv[b] == 0) return;
    for (int p = l; p < kBrickPts; p += kBrickLeaves) G[p] = gv[int64_t(it) * kBrickPts + p];
    __syncthreads();
    const int64_t at = int64_t(it) * kBrickLeaves + l;
    const int em = T.emask[at];
    if (!em) return;
    const int32_t q = A.bmap[b];
    const uint32_t key = uint32_t(A.rec[int64_t(q) * kRecWords + kRecKey]) |
                         (uint32_t(b - A.boff[q]) << (3 * kBrickLog)) | uint32_t(l);
    const int lx = int(compact3(uint32_t(l) >> 2)), ly = int(compact3(uint32_t(l) >> 1)), lz = int(compact3(uint32_t(l)));
    float cv[8];
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const int y = (c >> 1) & 1, xx = (c & 1) ^ y, z = c >> 2;
        cv[c] = G[((lz + z) * kP + (ly + y)) * kP + (lx + xx)];
    }
    emit_leaf_vertices(key, A.D, em, cv, out_v + 3 * (int64_t(bvoff[b]) + T.lofs[at]));
}

// Triangle entries of the evaluated bricks (generateSubdivideTrianglePos,
// main.cu:2759-2825).  A vertex owned by a leaf of another brick (of this
// root or of another root of the group) is found through that brick's tables.
__global__ void __launch_bounds__(kBrickLeaves) k_brick_triangles(SubArgs A, const int32_t* list, const int32_t* didx,
                                                                  LeafTabs T, const int32_t* bnt, const int32_t* bvoff,
                                                                  const int32_t* btoff, int64_t vbase, int32_t* out_t,
                                                                  int32_t* err) {
    const int32_t it = blockIdx.x, b = list[it], l = threadIdx.x;
    if (bnt[b] == 0) return;
    Brick B;
    GroupMask S;
    brick_geometry(A, b, B, S);
    const int cube = T.cube[int64_t(it) * kBrickLeaves + l];
    const int nt = tri_count(cube);
    int total;
    const int first = block_excl_scan(nt, &total);
    if (!nt) return;
    int32_t* out = out_t + 3 * (int64_t(btoff[b]) + first);
    const int32_t v[3] = {B.org[0] + int32_t(compact3(uint32_t(l) >> 2)), B.org[1] + int32_t(compact3(uint32_t(l) >> 1)),
                          B.org[2] + int32_t(compact3(uint32_t(l)))};
    const int32_t* NBR = A.rec + int64_t(B.q) * kRecWords + kRecNBR;
    for (int k = 0; k < 3 * nt; k++) {
        uint32_t mort;
        int eo;
        const int32_t q2 = edge_vertex_place(B, S, A.D, v, c_tri[cube][k], [&](int j) { return NBR[j]; }, &mort, &eo);
        const int32_t b2 = q2 < 0 ? 0 : A.boff[q2] + int32_t(mort >> (3 * kBrickLog));
        const int32_t at = q2 < 0 ? -1 : didx[b2];
        const int64_t t = at < 0 ? 0 : int64_t(at) * kBrickLeaves + (mort & (kBrickLeaves - 1));
        const uint32_t em = at < 0 ? 0 : T.emask[t];
        int32_t id = 0;
        if (!((em >> eo) & 1u)) {
            err[0] = 1;  // a crossing edge whose owner has no vertex on it: inconsistent counts
        } else {
            id = int32_t(vbase + bvoff[b2] + T.lofs[t] + __popc(em & ((1u << eo) - 1u)));
        }
        out[k] = id;
    }
}

// ---- small roots -----------------------------------------------------------------------
// A root of 2^3 (KB = 1) or 4^3 leaves (KB = 2) is one brick of 27 or 125
// corner values.  Such roots lie at the surface: certificates settle few of
// them (on a sparse 150,000-point cloud at depth 10, 2% of 235,000), and a
// certificate costs about what the values cost.  So every small root is
// evaluated.  A wave of its own per root left 37 of 64 lanes idle in each of
// three rounds (27 points strewn over an 8^3 brick's numbering); here a wave
// takes two 2^3 roots or two rounds of a 4^3 root.  Corners that a leaf of another
// root of the group owns are not evaluated at all: the roots of a group have
// one depth, so the owner's root is small too and computes the value as its
// own corner (the same owner, table entries and order); gref says where.
// Bound by the exact sums' issue: 27 products in the reference's order per
// depth and corner.  A whole pass over
// 150,000 points at depth 10 (294,344 roots, 282,635 of them small) went from
// 35.8 to 14.2 ms, over 35,947 points at depth 8 from 5.4 to 3.9 ms.
template <int KB>
struct SmallRoots {
    static constexpr int kS = 1 << KB, kPts1 = kS + 1, kPts = kPts1 * kPts1 * kPts1;
    static constexpr int kLanes = KB == 1 ? 32 : 64, kPerWave = kWave / kLanes;  // value pass
    static constexpr int kLeaves = 1 << (3 * KB), kLeafRoots = kWave / kLeaves;  // leaf passes
};

template <int KB>
struct SmallLds {
    // the chain's neighbour values, 28 floats per depth (16-byte reads)
    alignas(16) float X[(kMaxDepth + 1) * 28];
    BasisT T[(kMaxDepth + 1) * 3 * SmallRoots<KB>::kPts1];  // per depth and axis, each grid coordinate's owner's
    // coefficients of the real cells around the root: 4^3 at depth r + 1 and,
    // for 4^3 leaves, 6^3 at depth D (0 where virtual or absent)
    float XB[KB == 1 ? 64 : 64 + 216];
    int32_t CB[KB == 1 ? 1 : 64];  // child bases of the depth r + 1 cells
    int32_t NBK[27], NBR[27];
};

// Adds the 27 terms of one block depth (W cells a side, the owner's low
// neighbour at cx, cy, cz) in the reference's order.
template <int W>
__device__ __forceinline__ float small_block_sum(const float* Xb, int cx, int cy, int cz, BasisT tx, BasisT ty,
                                                 BasisT tz, float f) {
    const float bx[3] = {tx.x, tx.y, tx.z}, by[3] = {ty.x, ty.y, ty.z}, bz[3] = {tz.x, tz.y, tz.z};
    const float* X0 = Xb + (cx * W + cy) * W + cz;
    float xv[27];
#pragma unroll
    for (int k = 0; k < 27; k++) xv[k] = X0[((k / 9) * W + (k / 3) % 3) * W + k % 3];
#pragma unroll
    for (int k = 0; k < 27; k++) {
        float tt = xv[k] * bx[k / 9];
        tt = tt * by[(k / 3) % 3];
        tt = tt * bz[k % 3];
        f = f + tt;
    }
    return f;
}

// A small root's geometry (Brick's fields that the owner tests read).
__device__ __forceinline__ void small_brick(Brick& B, const int32_t* R, int32_t q, int D, int kb) {
    B.q = q;
    B.r = D - kb;
    B.kb = kb;
    B.bkey = uint32_t(R[kRecKey]);
    B.Sr = 1 << kb;
    decode_cell(B.bkey, B.org);
    for (int a = 0; a < 3; a++) {
        B.R[a] = B.org[a] >> kb;
        B.R0[a] = B.org[a];
    }
}

// The corner values its own leaves own, of every small root: gv[slot kPts + p]
// (f - iso at grid point p = (k kPts1 + j) kPts1 + i), and for every corner
// where its value is (gref).
template <int KB>
__global__ void __launch_bounds__(kWave) k_small_values(SubArgs A, const int32_t* slist, int32_t ns,
                                                        const int32_t* sidx, float* gv, int32_t* gref) {
    using C = SmallRoots<KB>;
    constexpr int P = C::kPts1, LP = C::kLanes;
    __shared__ SmallLds<KB> SS[C::kPerWave];
    const int D = A.D, r = D - KB, lane = threadIdx.x, l = lane % LP;
    SmallLds<KB>& S = SS[lane / LP];
    const int32_t slot = int32_t(blockIdx.x) * C::kPerWave + lane / LP;
    const bool live = slot < ns;
    const int32_t q = slist[live ? slot : ns - 1];
    const int32_t* R = A.rec + int64_t(q) * kRecWords;
    Brick B;
    small_brick(B, R, q, D, KB);
    if (l < 27) {
        S.NBK[l] = R[kRecNBK + l];
        S.NBR[l] = R[kRecNBR + l];
#pragma unroll
        for (int d = 0; d <= kMaxDepth; d++)
            if (d <= r) S.X[28 * d + l] = __int_as_float(R[kRecX + 27 * d + l]);
    }
    for (int e = l; e < (D + 1) * 3 * P; e += LP) {
        const int d = e / (3 * P), a = (e / P) % 3, i = e % P;
        const int32_t g = (a == 0 ? B.org[0] : a == 1 ? B.org[1] : B.org[2]) + i;
        const int32_t o = i == 0 ? g : g - 1;  // own_cell
        const float4 t = A.btab[((int64_t(d) << D) + o) * 2 + (g - o)];
        S.T[e] = BasisT{t.x, t.y, t.z};
    }
    __syncthreads();
    // depth r + 1: the root's 2^3 cells (virtual) and one more on every side
    bool kids = false;
#pragma unroll
    for (int e = l; e < 64; e += LP) {
        const int x = e >> 4, y = (e >> 2) & 3, z = e & 3;
        const int ox = x == 0 ? -1 : x == 3, oy = y == 0 ? -1 : y == 3, oz = z == 0 ? -1 : z == 3;
        const int32_t cb = (ox | oy | oz) ? S.NBK[nidx(ox, oy, oz)] : -1;
        // (the root's first cell is even along every axis)
        const int32_t node = cb < 0 ? -1 : cb + ((((x + 1) & 1) << 2) | (((y + 1) & 1) << 1) | ((z + 1) & 1));
        S.XB[e] = node < 0 ? 0.0f : A.x[node];
        if constexpr (KB == 2) {
            const int32_t c2 = node < 0 ? -1 : A.child_base[node];
            S.CB[e] = c2;
            kids = kids || c2 >= 0;
        }
    }
    if constexpr (KB == 2) {  // depth D: the children of those cells around the 4^3 leaves
        kids = __builtin_amdgcn_ballot_w64(kids) != 0;
        __syncthreads();
        if (kids) {
            for (int e = l; e < 216; e += kWave) {
                const int x = e / 36, y = (e / 6) % 6, z = e % 6;
                const int32_t cb = S.CB[(((x + 1) >> 1) * 4 + ((y + 1) >> 1)) * 4 + ((z + 1) >> 1)];
                const int32_t node = cb < 0 ? -1 : cb + ((((x + 1) & 1) << 2) | (((y + 1) & 1) << 1) | ((z + 1) & 1));
                S.XB[64 + e] = node < 0 ? 0.0f : A.x[node];
            }
        }
    }
    __syncthreads();
    const float iso = *A.iso;
    for (int p = l; p < C::kPts; p += LP) {
        const int gi[3] = {p % P, (p / P) % P, p / (P * P)};
        const int32_t g[3] = {B.org[0] + gi[0], B.org[1] + gi[1], B.org[2] + gi[2]};
        int32_t o[3] = {0, 0, 0};
        const int sl = corner_owner(B, S, D, g, o);
        int32_t ref = slot * C::kPts + p;
        if (sl != 13) {
            const int li = gi[0] - (sl / 9 - 1) * C::kS, lj = gi[1] - ((sl / 3) % 3 - 1) * C::kS,
                      lk = gi[2] - (sl % 3 - 1) * C::kS;
            ref = sidx[S.NBR[sl]] * C::kPts + (lk * P + lj) * P + li;
        } else {
            // the owner is own_cell along every axis; its cell in the root
            const int c[3] = {gi[0] - (gi[0] > 0), gi[1] - (gi[1] > 0), gi[2] - (gi[2] > 0)};
            const BasisT* Tx = S.T + gi[0];
            const BasisT* Ty = S.T + P + gi[1];
            const BasisT* Tz = S.T + 2 * P + gi[2];
            // real nodes below the root, depth D up to r + 1 (a virtual,
            // absent or outside neighbour adds +-0, which leaves a float sum
            // that started at +0 unchanged)
            float f = 0.0f;
            if constexpr (KB == 2) {
                if (kids) f = small_block_sum<6>(S.XB + 64, c[0], c[1], c[2], Tx[3 * P * D], Ty[3 * P * D], Tz[3 * P * D], f);
            }
            f = small_block_sum<4>(S.XB, c[0] >> (KB - 1), c[1] >> (KB - 1), c[2] >> (KB - 1), Tx[3 * P * (r + 1)],
                                   Ty[3 * P * (r + 1)], Tz[3 * P * (r + 1)], f);
            // the root's chain (chain_lds's order)
            for (int d = r; d >= 1; d--) {
                const BasisT tx = Tx[3 * P * d], ty = Ty[3 * P * d], tz = Tz[3 * P * d];
                const float bx[3] = {tx.x, tx.y, tx.z}, by[3] = {ty.x, ty.y, ty.z}, bz[3] = {tz.x, tz.y, tz.z};
                float xv[28];
#pragma unroll
                for (int j = 0; j < 7; j++)
                    *reinterpret_cast<float4*>(xv + 4 * j) = *reinterpret_cast<const float4*>(S.X + 28 * d + 4 * j);
#pragma unroll
                for (int j = 0; j < 27; j++) {
                    float tt = xv[j] * bx[j / 9];
                    tt = tt * by[(j / 3) % 3];
                    tt = tt * bz[j % 3];
                    f = f + tt;
                }
            }
            float tt = S.X[0] * Tx[0].y;
            tt = tt * Ty[0].y;
            tt = tt * Tz[0].y;
            f = f + tt;
            if (live) gv[ref] = f - iso;
        }
        if (live) gref[int64_t(slot) * C::kPts + p] = ref;
    }
}

// The leaf passes' lanes: kLeafRoots roots to a wave, one leaf per lane.  Sets
// the lane's root geometry and group.
template <int KB>
__device__ __forceinline__ void small_leaf_setup(const SubArgs& A, int32_t q, Brick& B, GroupMask& S) {
    constexpr int LV = SmallRoots<KB>::kLeaves;
    const int32_t* R = A.rec + int64_t(q) * kRecWords;
    small_brick(B, R, q, A.D, KB);
    const int l = threadIdx.x % LV;
    uint32_t m = 0;
#pragma unroll
    for (int j = l; j < 27; j += LV)
        if (R[kRecNBR + j] >= 0) m |= 1u << j;
#pragma unroll
    for (int o = 1; o < (LV < 32 ? LV : 32); o <<= 1) m |= uint32_t(__shfl_xor(int(m), o, kWave));
    if constexpr (LV == 64) m |= uint32_t(__shfl_xor(int(m), 32, kWave));
    S.NBR.m = m;
}

// Exclusive sums of v over the leaves of the lane's root, and the total.
template <int LV>
__device__ __forceinline__ int leaf_excl_scan(int v, int* total) {
    int inc = v;
#pragma unroll
    for (int o = 1; o < LV; o <<= 1) {
        const int t = __shfl_up(inc, o, LV);
        if (int(threadIdx.x % LV) >= o) inc += t;
    }
    *total = __shfl(inc, LV - 1, LV);
    return inc - v;
}

// The corner values of the wave's roots into LDS.
template <int KB>
__device__ __forceinline__ void small_corner_values(int32_t s0, int32_t ns, const float* gv, const int32_t* gref,
                                                    float* G) {
    using C = SmallRoots<KB>;
    const int n = std::min(int(ns - s0), C::kLeafRoots) * C::kPts;
    const int32_t* gr = gref + int64_t(s0) * C::kPts;
#pragma unroll
    for (int t = threadIdx.x; t < C::kLeafRoots * C::kPts; t += kWave) G[t] = t < n ? gv[gr[t]] : 1.0f;
    __syncthreads();
}

// Cube indices and owned crossing edges of every small root's leaves, and the
// root's vertex and triangle counts.
template <int KB>
__global__ void __launch_bounds__(kWave) k_small_cubes(SubArgs A, const int32_t* slist, int32_t ns, const float* gv,
                                                       const int32_t* gref, LeafTabs T, int32_t* bnv, int32_t* bnt) {
    using C = SmallRoots<KB>;
    constexpr int LV = C::kLeaves;
    __shared__ float G[C::kLeafRoots * C::kPts];
    const int lane = threadIdx.x, l = lane % LV;
    const int32_t s0 = int32_t(blockIdx.x) * C::kLeafRoots, slot = s0 + lane / LV;
    const bool live = slot < ns;
    const int32_t q = slist[live ? slot : ns - 1];
    Brick B;
    GroupMask S;
    small_leaf_setup<KB>(A, q, B, S);
    small_corner_values<KB>(s0, ns, gv, gref, G);
    int32_t v[3];
    float cv[8];
    int cube, em;
    leaf_cube<C::kPts1>(B, S, G + (lane / LV) * C::kPts, A.D, l, v, cv, &cube, &em);
    int nv, nt;
    const int ofs = leaf_excl_scan<LV>(__popc(uint32_t(em)), &nv);
    (void)leaf_excl_scan<LV>(tri_count(cube), &nt);
    if (!live) return;
    const int64_t at = int64_t(slot) * LV + l;
    T.emask[at] = uint16_t(em);
    T.lofs[at] = uint16_t(ofs);
    T.cube[at] = uint8_t(cube);
    if (l == 0) {
        const int32_t b = A.boff[q];
        bnv[b] = nv;
        bnt[b] = nt;
    }
}

template <int KB>
__global__ void __launch_bounds__(kWave) k_small_vertices(SubArgs A, const int32_t* slist, int32_t ns, const float* gv,
                                                          const int32_t* gref, LeafTabs T, const int32_t* bvoff,
                                                          float* out_v) {
    using C = SmallRoots<KB>;
    constexpr int LV = C::kLeaves, P = C::kPts1;
    __shared__ float Gs[C::kLeafRoots * C::kPts];
    const int lane = threadIdx.x, l = lane % LV;
    const int32_t s0 = int32_t(blockIdx.x) * C::kLeafRoots, slot = s0 + lane / LV;
    const int64_t at = int64_t(slot) * LV + l;
    const int em = slot < ns ? T.emask[at] : 0;
    if (__builtin_amdgcn_ballot_w64(em != 0) == 0) return;
    small_corner_values<KB>(s0, ns, gv, gref, Gs);
    if (!em) return;
    const int32_t q = slist[slot];
    const uint32_t key = uint32_t(A.rec[int64_t(q) * kRecWords + kRecKey]) | uint32_t(l);
    const int lx = int(compact3(uint32_t(l) >> 2)), ly = int(compact3(uint32_t(l) >> 1)), lz = int(compact3(uint32_t(l)));
    const float* G = Gs + (lane / LV) * C::kPts;
    float cv[8];
#pragma unroll
    for (int c = 0; c < 8; c++) {
        const int y = (c >> 1) & 1, xx = (c & 1) ^ y, z = c >> 2;
        cv[c] = G[((lz + z) * P + (ly + y)) * P + (lx + xx)];
    }
    (void)emit_leaf_vertices(key, A.D, em, cv, out_v + 3 * (int64_t(bvoff[A.boff[q]]) + T.lofs[at]));
}

template <int KB>
__global__ void __launch_bounds__(kWave) k_small_triangles(SubArgs A, const int32_t* slist, int32_t ns,
                                                           const int32_t* sidx, LeafTabs T, const int32_t* bvoff,
                                                           const int32_t* btoff, int64_t vbase, int32_t* out_t,
                                                           int32_t* err) {
    using C = SmallRoots<KB>;
    constexpr int LV = C::kLeaves;
    const int lane = threadIdx.x, l = lane % LV;
    const int32_t slot = int32_t(blockIdx.x) * C::kLeafRoots + lane / LV;
    const bool live = slot < ns;
    const int cube = live ? T.cube[int64_t(slot) * LV + l] : 0;
    const int nt = tri_count(cube);
    if (__builtin_amdgcn_ballot_w64(nt != 0) == 0) return;
    const int32_t q = slist[live ? slot : ns - 1];
    Brick B;
    GroupMask S;
    small_leaf_setup<KB>(A, q, B, S);
    int total;
    const int first = leaf_excl_scan<LV>(nt, &total);
    if (!nt) return;
    int32_t* out = out_t + 3 * (int64_t(btoff[A.boff[q]]) + first);
    const int32_t v[3] = {B.org[0] + int32_t(compact3(uint32_t(l) >> 2)), B.org[1] + int32_t(compact3(uint32_t(l) >> 1)),
                          B.org[2] + int32_t(compact3(uint32_t(l)))};
    const int32_t* NBR = A.rec + int64_t(q) * kRecWords + kRecNBR;
    for (int k = 0; k < 3 * nt; k++) {
        uint32_t mort;
        int eo;
        const int32_t q2 = edge_vertex_place(B, S, A.D, v, c_tri[cube][k], [&](int j) { return NBR[j]; }, &mort, &eo);
        const int64_t t = q2 < 0 ? 0 : int64_t(sidx[q2]) * LV + mort;
        const uint32_t em = q2 < 0 ? 0 : T.emask[t];
        int32_t id = 0;
        if (!((em >> eo) & 1u)) {
            err[0] = 1;  // the owner has no vertex on the edge
        } else {
            id = int32_t(vbase + bvoff[A.boff[q2]] + T.lofs[t] + __popc(em & ((1u << eo) - 1u)));
        }
        out[k] = id;
    }
}

}  // namespace

// Per depth, with the coefficients bounded by 1: the basis functions of three
// cells sum to 4/3 along an axis, and a table value differs from the spline's
// by at most t = corner_dev[d], so 27 products sum to at most
// big = (4/3 + 3 t)^3 in absolute value, and differ from the spline's products
// by at most 3 (3 t) (4/3 + 3 t)^2 in all.  A corner's float sum of
// n <= 27 (D + 1) + 1 products of three roundings lies within (n + 3) 2^-24 of
// its terms' absolute sum; the polynomial's own float sums within 300 of that
// unit: 700 covers both.
static void depth_bounds(const FsTables& fs, SubArgs* A) {
    for (int d = 0; d <= kMaxDepth; d++) {
        const double t = d <= fs.D ? double(fs.corner_dev[d]) : 0.0, m = 4.0 / 3.0 + 3.0 * t;
        A->big[d] = float(1.001 * m * m * m);
        A->dev[d] = float(1.001 * (9.0 * t * m * m + 700.0 * 5.9604645e-8 * m * m * m));
    }
}

// the coarse rows of the current solution (mc.hip)
int ensure_coarse_rows(prg_ctx* c, hipStream_t s);

void extract_subdivision(prg_ctx* c) {
    ensure_tables(c);
    StageTimer st(c, PRG_STAGE_SUBDIVIDE);
    hipStream_t s = c->stream;
    const int D = c->D;
    const int64_t M = c->M, MD = c->MD(), baseD = c->bases[D];
    KernelTimer& kt = c->kt;
    const Levels Lv = levels_of(c);
    c->sub_nv = c->sub_nt = 0;
    c->sub_v_copied = false;
    c->sub_roots = c->sub_leaves = 0;
    c->sub_bricks = c->sub_exact = c->sub_evaluated = 0;
    if (baseD <= 1) return;
    if (8 * baseD >= (int64_t(1) << 31)) throw Error{PRG_E_ARG, "too many nodes above the leaf level for subdivision"};
    const int rd = ensure_coarse_rows(c, s);
    if (rd < D - 1) throw Error{PRG_E_STATE, "coarse rows missing"};

    // pool slots 97..159
    PoolBuf<uint8_t> inter{&c->pool[97]}, need{&c->pool[103]}, rflag{&c->pool[107]};
    PoolBuf<int32_t> cnt{&c->pool[98]}, cl{&c->pool[101]}, oref{&c->pool[102]}, nid{&c->pool[104]},
        clist{&c->pool[105]}, roots{&c->pool[110]}, boff{&c->pool[112]}, root_of{&c->pool[115]};
    PoolBuf<uint32_t> up{&c->pool[140]};
    PoolBuf<float> cv{&c->pool[106]};
    int32_t* C = cnt.reserve(kCntSlots);
    int32_t* H = c->sub_host;  // pinned; the counts that kernels write there, and copies of C
    std::fill(H, H + kCntSlots, 0);
    inter.reserve(6 * M);
    up.reserve((M + 3) / 4);
    need.reserve(8 * baseD);
    root_of.reserve(M);
    k_sub_init<<<unsigned(std::min<int64_t>(4 * std::max(1, c->num_cu), grid_for(M, kBlockS))), kBlockS, 0, s>>>(
        C, inter.get(), up.get(), need.get(), root_of.get(), M, baseD);
    PRG_CHECK_LAUNCH();

    // faces touched by the leaf-level surface, and up the parent chains
    {
        // bytes: the cube index of each leaf-level node and the face byte of
        // each coarser node, read once (the face visits' gathers come on top)
        TimedScope ts(kt, "face_marks", double(M));
        // the leaf-level cube indices of the marching cubes pass that ran just before
        PoolBuf<uint8_t> cubes{&c->pool[94]};
        k_face_marks<<<grid_for(MD, kBlockS), kBlockS, 0, s>>>(cubes.get(), MD, baseD, c->key.get(), c->pnt.get(),
                                                                Lv, c->parent.get(), D, inter.get(), up.get());
        PRG_CHECK_LAUNCH();
        int d = D - 1;
        for (; c->counts[d] > kSmallUp; d--) {
            k_face_marks_up<<<grid_for(c->counts[d], kBlockS), kBlockS, 0, s>>>(
                c->bases[d], c->counts[d], d, c->key.get(), c->pnt.get(), Lv, c->parent.get(), D, inter.get(),
                up.get());
            PRG_CHECK_LAUNCH();
        }
        k_face_marks_up_small<<<1, kUpBlock, 0, s>>>(d, c->key.get(), c->pnt.get(), Lv, c->parent.get(), D, inter.get(),
                                                     up.get());
        PRG_CHECK_LAUNCH();
    }
    // coarse leaves (counts stay on the device; launches are sized by upper bounds)
    cl.reserve(baseD);
    auto select_tiles = [&](int64_t n, int tile) { return uint32_t((n + tile - 1) / tile); };
    {
        const int block = select_block(baseD);
        const uint32_t tiles = select_tiles(baseD, block * kSelItems);
        const LookState state = look_state(c->scratch, tiles, s);
        (block == kSelLarge ? k_select<true, kSelLarge> : k_select<true, kSelSmall>)<<<tiles, block, 0, s>>>(
            c->child_base.get(), nullptr, baseD, tiles, state, cl.get(), nullptr, C + kCntCoarse);
        PRG_CHECK_LAUNCH();
    }
    // their corner values
    oref.reserve(8 * baseD);
    nid.reserve(8 * baseD);
    clist.reserve(8 * baseD);
    cv.reserve(8 * baseD);
    k_coarse_corner_owner<<<grid_for(8 * baseD, kBlockS), kBlockS, 0, s>>>(cl.get(), C + kCntCoarse, c->key.get(),
                                                                            c->pnt.get(), Lv, D, oref.get(), need.get());
    PRG_CHECK_LAUNCH();
    {
        const int block = select_block(8 * baseD);
        const uint32_t tiles = select_tiles(8 * baseD, block * kSelItems);
        const LookState state = look_state(c->scratch, tiles, s);
        (block == kSelLarge ? k_select<false, kSelLarge> : k_select<false, kSelSmall>)<<<tiles, block, 0, s>>>(
            nullptr, need.get(), 8 * baseD, tiles, state, clist.get(), nid.get(), C + kCntCorners);
        PRG_CHECK_LAUNCH();
    }
    {
        TimedScope ts(kt, "coarse_corner_value", 24.0 * double(baseD));
        k_coarse_corner_value<<<grid_for(8 * baseD, kBlockS), kBlockS, 0, s>>>(
            clist.get(), C + kCntCorners, c->key.get(), c->pnt.get(), Lv, c->parent.get(), c->child_base.get(),
            c->dnum.get(), c->x.get(), c->d_base_fn.get(), c->coarse_rows.get(), rd, D, c->iso_dev.get(), cv.get());
        PRG_CHECK_LAUNCH();
    }
    // roots, their bricks and virtual leaves
    rflag.reserve(baseD + 16);
    roots.reserve(baseD);
    boff.reserve(baseD);
    k_coarse_select<<<grid_for(baseD, kBlockS), kBlockS, 0, s>>>(cl.get(), C + kCntCoarse, oref.get(), nid.get(),
                                                                  cv.get(), c->key.get(), c->pnt.get(), Lv, D,
                                                                  inter.get(), rflag.get());
    PRG_CHECK_LAUNCH();
    PoolBuf<int32_t> slist1{&c->pool[144]}, slist2{&c->pool[145]}, sidx{&c->pool[146]};
    slist1.reserve(baseD);
    slist2.reserve(baseD);
    sidx.reserve(baseD);
    {
        const uint32_t tiles = select_tiles(baseD, kRootTile);
        const LookState state = look_state(c->scratch, 5 * int64_t(tiles), s);
        k_list_all_roots<<<tiles, kRootBlock, 0, s>>>(cl.get(), rflag.get(), state, Lv, D, roots.get(),
                                                      boff.get(), root_of.get(), slist1.get(), slist2.get(),
                                                      sidx.get(), C, H);
        PRG_CHECK_LAUNCH();
    }
    PRG_HIP(hipStreamSynchronize(s));
    look_check(c->scratch, s);
    const int64_t nr = H[kCntRoots], nb = H[kCntBricks];
    c->sub_roots = nr;
    c->sub_leaves = H[kCntLeaves];
    if (nr == 0) return;
    if (nb <= 0 || H[kCntLeaves] <= 0) throw Error{PRG_E_HIP, "subdivision: inconsistent brick counts"};

    PoolBuf<float> btab{&c->pool[91]};
    SubArgs A{c->key.get(),
                    c->child_base.get(), c->parent.get(), c->pnt.get(),
                    Lv,                c->x.get(),      c->d_base_fn.get(),
                    reinterpret_cast<const float4*>(btab.get()), c->coarse_rows.get(), D,
                    c->iso_dev.get(),  roots.get(),     boff.get(),
                    root_of.get(),     C,               nullptr,
                    nullptr,           {},              {}};

    depth_bounds(*c->fs, &A);
    // per-root records and the brick -> root map
    PoolBuf<int32_t> rec{&c->pool[127]}, bmap{&c->pool[128]};
    rec.reserve(size_t(nr) * kRecWords);
    bmap.reserve(size_t(nb));
    A.rec = rec.get();
    A.bmap = bmap.get();
    k_root_records<<<unsigned((nr + 1) / 2), kWave, 0, s>>>(A, int32_t(nr), rec.get());
    PRG_CHECK_LAUNCH();
    k_brick_map<<<grid_for(nb, kBlockS), kBlockS, 0, s>>>(boff.get(), C, nb, bmap.get());
    PRG_CHECK_LAUNCH();

    // pass 1: counts per brick
    PoolBuf<int32_t> bnv{&c->pool[116]}, bnt{&c->pool[117]}, bvoff{&c->pool[118]}, btoff{&c->pool[119]};
    bnv.reserve(nb);
    bnt.reserve(nb);
    bvoff.reserve(nb);
    btoff.reserve(nb);
    // pass 0: certificates; pass 1: counts of the bricks left
    PoolBuf<int32_t> dlist{&c->pool[129]}, glist{&c->pool[130]}, xlist{&c->pool[133]}, cells{&c->pool[136]};
    PoolBuf<int8_t> bsign{&c->pool[132]};
    dlist.reserve(nb);
    xlist.reserve(nb);
    glist.reserve(nb);
    bsign.reserve(nb);
    PoolBuf<int32_t> didx{&c->pool[135]};
    didx.reserve(nb);
    k_clear_bricks<<<grid_for(nb, kBlockS), kBlockS, 0, s>>>(bnv.get(), bnt.get(), bsign.get(), didx.get(), nb);
    PRG_CHECK_LAUNCH();
    // the small roots: values, cubes and counts
    const int32_t n1 = H[kCntSmall1], n2 = H[kCntSmall2];
    const int64_t nb3 = nb - n1 - n2;  // 8^3 bricks
    PoolBuf<float> gv1{&c->pool[147]}, gv2{&c->pool[148]};
    PoolBuf<int32_t> gref1{&c->pool[149]}, gref2{&c->pool[150]};
    PoolBuf<uint16_t> semask{&c->pool[151]}, slofs{&c->pool[152]};
    PoolBuf<uint8_t> scube{&c->pool[153]};
    using Small1 = SmallRoots<1>;
    using Small2 = SmallRoots<2>;
    if (int64_t(n1) * Small1::kPts >= (int64_t(1) << 31) || int64_t(n2) * Small2::kPts >= (int64_t(1) << 31))
        throw Error{PRG_E_NOMEM, "too many small subdivision roots"};
    const size_t tab2 = size_t(n1) * Small1::kLeaves, tabn = tab2 + size_t(n2) * Small2::kLeaves;
    semask.reserve(tabn);
    slofs.reserve(tabn);
    scube.reserve(tabn);
    const LeafTabs T1{semask.get(), slofs.get(), scube.get()};
    const LeafTabs T2{semask.get() + tab2, slofs.get() + tab2, scube.get() + tab2};
    const unsigned lw1 = grid_for(n1, Small1::kLeafRoots), lw2 = grid_for(n2, Small2::kLeafRoots);
    {
        TimedScope ts(kt, "subdivide_small_values", 0.0);  // issue-bound: no byte figure
        if (n1) {
            gv1.reserve(size_t(n1) * Small1::kPts);
            gref1.reserve(size_t(n1) * Small1::kPts);
            k_small_values<1><<<grid_for(n1, Small1::kPerWave), kWave, 0, s>>>(A, slist1.get(), n1, sidx.get(),
                                                                               gv1.get(), gref1.get());
            PRG_CHECK_LAUNCH();
            k_small_cubes<1><<<lw1, kWave, 0, s>>>(A, slist1.get(), n1, gv1.get(), gref1.get(), T1, bnv.get(),
                                                   bnt.get());
            PRG_CHECK_LAUNCH();
        }
        if (n2) {
            gv2.reserve(size_t(n2) * Small2::kPts);
            gref2.reserve(size_t(n2) * Small2::kPts);
            k_small_values<2><<<grid_for(n2, Small2::kPerWave), kWave, 0, s>>>(A, slist2.get(), n2, sidx.get(),
                                                                               gv2.get(), gref2.get());
            PRG_CHECK_LAUNCH();
            k_small_cubes<2><<<lw2, kWave, 0, s>>>(A, slist2.get(), n2, gv2.get(), gref2.get(), T2, bnv.get(),
                                                   bnt.get());
            PRG_CHECK_LAUNCH();
        }
    }
    if (nb3 > 0) {
        TimedScope ts(kt, "subdivide_screen", 0.0);  // latency- and issue-bound: no byte figure
        // per size, at most as many cells as the bricks fill
        CellLists lists{};
        int64_t total = 0;
        for (int k = kBrickLog; k < D; k++) total += (nb3 >> (3 * (k - kBrickLog))) + 1;
        int32_t* at = cells.reserve(total);
        for (int k = kBrickLog; k < D; k++) {
            lists.at[k] = at;
            at += (nb3 >> (3 * (k - kBrickLog))) + 1;
        }
        k_list_roots<<<grid_for(nr, kBlockS), kBlockS, 0, s>>>(roots.get(), boff.get(), nr, Lv, D, lists, C);
        PRG_CHECK_LAUNCH();
        // resident grids: every workgroup walks its share
        auto resident = [&](const void* kernel, int64_t most) {
            int per_cu = 0;
            PRG_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kWave, 0));
            return unsigned(std::max<int64_t>(1, std::min<int64_t>(most, int64_t(std::max(1, per_cu)) * c->num_cu)));
        };
        // largest root: no cell is larger
        int kmax = D - 1;
        while (kmax > kBrickLog && (int64_t(1) << (3 * (kmax - kBrickLog))) > nb3) kmax--;
        for (int k = kmax; k >= kBrickLog; k--) {
            const auto screen = k == kBrickLog ? k_cell_screen<kXBlkScreenBrick> : k_cell_screen<kXBlkScreen>;
            screen<<<resident(reinterpret_cast<const void*>(screen), (nb3 >> (3 * (k - kBrickLog))) + 1),
                            kWave, 0, s>>>(A, k, lists.at[k], k > kBrickLog ? lists.at[k - 1] : nullptr, xlist.get(),
                                           bsign.get(), glist.get(), C, int(c->sub_certify));
            PRG_CHECK_LAUNCH();
        }
        k_brick_exact<<<resident(reinterpret_cast<const void*>(k_brick_exact), nb3), kWave, 0, s>>>(
            A, xlist.get(), bsign.get(), dlist.get(), glist.get(), C, int(c->sub_certify));
        PRG_CHECK_LAUNCH();
        k_group_check<<<resident(reinterpret_cast<const void*>(k_group_check), nb3), kWave, 0, s>>>(
            A, glist.get(), bsign.get(), dlist.get(), C);
        PRG_CHECK_LAUNCH();
    }
    if (nb3 > 0) {
        PRG_HIP(hipMemcpyAsync(H, C, kCntSlots * 4, hipMemcpyDeviceToHost, s));
        PRG_HIP(hipStreamSynchronize(s));
    }
    const int64_t ndense = nb3 > 0 ? H[kCntDense] : 0;
    PoolBuf<float> gvals{&c->pool[134]};
    PoolBuf<uint16_t> lofs_tab{&c->pool[124]}, emask_tab{&c->pool[125]};
    PoolBuf<uint8_t> cube_tab{&c->pool[126]};
    LeafTabs T3{};
    if (ndense > 0) {
        gvals.reserve(size_t(ndense) * kBrickPts);
        T3.lofs = lofs_tab.reserve(size_t(ndense) * kBrickLeaves);
        T3.emask = emask_tab.reserve(size_t(ndense) * kBrickLeaves);
        T3.cube = cube_tab.reserve(size_t(ndense) * kBrickLeaves);
        TimedScope ts(kt, "subdivide_count", 0.0);
        // one workgroup per round while that fills no more than the chip
        const int slices = ndense * kValRounds <= 4 * std::max(1, c->num_cu) ? kValRounds : 1;
        k_brick_values<<<unsigned(ndense * slices), kValThreads, 0, s>>>(A, dlist.get(), slices, gvals.get());
        PRG_CHECK_LAUNCH();
        k_brick_cubes<<<unsigned(ndense), kBrickLeaves, 0, s>>>(A, dlist.get(), gvals.get(), T3, bnv.get(), bnt.get(),
                                                                didx.get());
        PRG_CHECK_LAUNCH();
    }
    scan_exclusive2(bnv.get(), bvoff.get(), H + kCntVerts, bnt.get(), btoff.get(), H + kCntTris, nb, s, c->scratch,
                    kt);
    PRG_HIP(hipStreamSynchronize(s));
    look_check(c->scratch, s);
    const int64_t snv = H[kCntVerts], snt = H[kCntTris];
    c->sub_bricks = nb;
    c->sub_exact = int64_t(H[kCntExact]) + n1 + n2;
    c->sub_evaluated = int64_t(H[kCntDense]) + n1 + n2;
    if (snv < 0 || snt < 0) throw Error{PRG_E_NOMEM, "subdivision mesh exceeds int32 counts"};
    if (c->mesh_nv + snv >= (int64_t(1) << 31)) throw Error{PRG_E_NOMEM, "mesh vertex count exceeds int32 indices"};
    if (snv == 0 && snt == 0) return;

    // the vertices and triangles of the small roots and the evaluated bricks
    float* SV = c->sub_v.reserve(size_t(3) * snv + 3);
    int32_t* ST = c->sub_t.reserve(size_t(3) * snt + 3);
    {
        TimedScope ts(kt, "subdivide_vertices", 12.0 * double(snv));
        if (n1) {
            k_small_vertices<1><<<lw1, kWave, 0, s>>>(A, slist1.get(), n1, gv1.get(), gref1.get(), T1, bvoff.get(), SV);
            PRG_CHECK_LAUNCH();
        }
        if (n2) {
            k_small_vertices<2><<<lw2, kWave, 0, s>>>(A, slist2.get(), n2, gv2.get(), gref2.get(), T2, bvoff.get(), SV);
            PRG_CHECK_LAUNCH();
        }
        if (ndense > 0) {
            k_brick_vertices<<<unsigned(ndense), kBrickLeaves, 0, s>>>(A, dlist.get(), gvals.get(), T3, bnv.get(),
                                                                       bvoff.get(), SV);
            PRG_CHECK_LAUNCH();
        }
    }
    // into the caller's buffers, when they hold the whole mesh, the vertices go
    // on the second stream while the triangles are emitted
    const bool direct = c->out_copied && c->out_async && 3 * (c->mesh_nv + snv) <= c->out_vcap &&
                        3 * (c->mesh_nt + snt) <= c->out_tcap && snv > 0;
    if (direct) PRG_HIP(hipEventRecord(c->mesh_ev2, s));
    {
        TimedScope ts(kt, "subdivide_triangles", 12.0 * double(snt));
        if (n1) {
            k_small_triangles<1><<<lw1, kWave, 0, s>>>(A, slist1.get(), n1, sidx.get(), T1, bvoff.get(), btoff.get(),
                                                       c->mesh_nv, ST, H + kCntErr);
            PRG_CHECK_LAUNCH();
        }
        if (n2) {
            k_small_triangles<2><<<lw2, kWave, 0, s>>>(A, slist2.get(), n2, sidx.get(), T2, bvoff.get(), btoff.get(),
                                                       c->mesh_nv, ST, H + kCntErr);
            PRG_CHECK_LAUNCH();
        }
        if (ndense > 0) {
            k_brick_triangles<<<unsigned(ndense), kBrickLeaves, 0, s>>>(A, dlist.get(), didx.get(), T3, bnt.get(),
                                                                        bvoff.get(), btoff.get(), c->mesh_nv, ST,
                                                                        H + kCntErr);
            PRG_CHECK_LAUNCH();
        }
    }
    if (direct) {
        PRG_HIP(hipStreamWaitEvent(c->stream2, c->mesh_ev2, 0));
        PRG_HIP(hipMemcpyAsync(c->out_v + 3 * c->mesh_nv, SV, size_t(3 * snv) * 4, hipMemcpyDeviceToHost, c->stream2));
        PRG_HIP(hipEventRecord(c->mesh_ev, c->stream2));
        c->sub_v_copied = true;
    }
    PRG_HIP(hipStreamSynchronize(s));
    if (H[kCntErr]) throw Error{PRG_E_HIP, "subdivision: a triangle edge has no owner vertex"};
    c->sub_nv = snv;
    c->sub_nt = snt;
}

}  // namespace prg
