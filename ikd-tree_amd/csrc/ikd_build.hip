// ikd_build.hip — level-synchronous GPU build of one or more subtrees.
//
// Restates BuildTree (ikd_Tree.cpp:573-622) for the device.  Every segment
// [l, r] of a level is split exactly as the reference splits it:
//   axis = longest extent of the segment (strict '>', ties go to the lower
//          axis, cpp:594-595),
//   node = element of rank mid-l on that axis with mid = (l+r)>>1 (cpp:581,
//          599-614),
//   left = the mid-l smaller elements, right = the rest (cpp:616-617).
// The three coordinate orders are sorted once (stable, so equal keys keep
// their input order); each level then stably partitions all three lists
// around the pivot, so the segment's bbox is always its first and last
// element per list and the rank-(mid-l) element is read directly.  For keys
// without ties on the split axis the resulting tree is the reference's tree;
// with ties the placement of equal keys is deterministic (input order) where
// the reference's depends on libstdc++'s nth_element.
//
// Nodes are written top-down: a segment's node gets its point, axis, size and
// depth, and its subtree AABB (the segment bbox) goes into the parent's child
// box slot.  Children are allocated as sibling pairs in segment order, so
// the layout is deterministic.
#include "ikd_internal.h"

namespace ikd {

__global__ void k_build_keys(const float4* __restrict__ pts, const int* __restrict__ seg_of, int m, int axis,
                             unsigned long long* __restrict__ keys, uint32_t* __restrict__ vals) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    float4 p = pts[i];
    float c = axis == 0 ? p.x : (axis == 1 ? p.y : p.z);
    keys[i] = ((unsigned long long)(uint32_t)seg_of[i] << 32) | float_key(c);
    vals[i] = (uint32_t)i;
}

// one segment: the coordinate alone
__global__ void k_build_keys32(const float4* __restrict__ pts, int m, int axis, uint32_t* __restrict__ keys,
                               uint32_t* __restrict__ vals) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    float4 p = pts[i];
    keys[i] = float_key(axis == 0 ? p.x : (axis == 1 ? p.y : p.z));
    vals[i] = (uint32_t)i;
}

__global__ void k_build_init_sid(const unsigned long long* __restrict__ k0, int m, int* __restrict__ sid) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m) return;
    sid[i] = (int)(k0[i] >> 32);
}

// ---- stable sort of up to RANK_SORT_MAX keys in two launches ---------------
// Tiles of 2048 keys are sorted in registers (bitonic network over (key,
// index), so the order is stable), then every key finds its final place in one
// pass: its place in its own tile plus, for every other tile, how many of that
// tile's keys come before it (equal keys of earlier tiles do).  A workgroup's
// 256 keys are neighbours in their tile's order, so they search one short
// stretch of every other tile, found once per workgroup.  Several lists of
// the same length are sorted by the same two launches (grid y).
//
// At these sizes a sort is a chain of dependent launches: the library's merge
// sort takes one per doubling (29k keys: 8 launches, about 75 us with their
// gaps; here 18 + 33 us for three lists at once), and the build ran three of
// them behind one another.  The searches grow with the square of the length, so
// longer lists go to the library: a Build of 30k points takes 383 us for 452,
// one of 65536 459 for 516.
constexpr int TILE_SB = 512, TILE_E = 4, TILE_KEYS = TILE_SB * TILE_E;
constexpr int MERGE_SB = 256;
static_assert(RANK_SORT_MAX % TILE_KEYS == 0 && TILE_KEYS % MERGE_SB == 0, "whole tiles");

// lane ^ M's value; the exchanges inside 16 lanes are register moves
template <int M>
__device__ __forceinline__ int lane_xor(int v) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (M == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xf, 0xf, true);   // quad_perm 1,0,3,2
    if constexpr (M == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xf, 0xf, true);   // quad_perm 2,3,0,1
    if constexpr (M == 4)  // row_half_mirror is ^ 7, quad_perm 3,2,1,0 is ^ 3
        return __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(v, 0x141, 0xf, 0xf, true), 0x1B, 0xf, 0xf, true);
    if constexpr (M == 8) return __builtin_amdgcn_mov_dpp(v, 0x128, 0xf, 0xf, true);  // row_ror:8
#endif
    return __shfl_xor(v, M);
}
__device__ __forceinline__ bool pair_less(unsigned long long ka, uint32_t va, unsigned long long kb, uint32_t vb) {
    return ka < kb || (ka == kb && va < vb);
}

// One stage of the network: every entry and its partner (index ^ J) are put in
// order, ascending where the bit KK of the index is clear.  Entry 4 t + e is
// in k[e], v[e] of thread t: partners are in the thread's registers (J < 4),
// in its wavefront (J < 256), or exchanged through LDS.
template <int KK, int J>
__device__ __forceinline__ void sort_stage(unsigned long long (&k)[TILE_E], uint32_t (&v)[TILE_E],
                                           unsigned long long* xk, uint32_t* xv) {
    const int t = threadIdx.x;
    if constexpr (J < TILE_E) {
#pragma unroll
        for (int e = 0; e < TILE_E; ++e) {
            if (e & J) continue;
            const bool up = (((TILE_E * t + e) & KK) == 0);
            if (pair_less(k[e | J], v[e | J], k[e], v[e]) == up) {
                const unsigned long long tk = k[e];
                const uint32_t tv = v[e];
                k[e] = k[e | J];
                v[e] = v[e | J];
                k[e | J] = tk;
                v[e | J] = tv;
            }
        }
    } else {
        unsigned long long ok[TILE_E];
        uint32_t ov[TILE_E];
        if constexpr (J < 64 * TILE_E) {
#pragma unroll
            for (int e = 0; e < TILE_E; ++e) {
                const unsigned lo = (unsigned)lane_xor<J / TILE_E>((int)(unsigned)k[e]);
                const unsigned hi = (unsigned)lane_xor<J / TILE_E>((int)(unsigned)(k[e] >> 32));
                ok[e] = ((unsigned long long)hi << 32) | lo;
                ov[e] = (uint32_t)lane_xor<J / TILE_E>((int)v[e]);
            }
        } else {
            __syncthreads();
#pragma unroll
            for (int e = 0; e < TILE_E; ++e) {
                xk[e * TILE_SB + t] = k[e];
                xv[e * TILE_SB + t] = v[e];
            }
            __syncthreads();
#pragma unroll
            for (int e = 0; e < TILE_E; ++e) {
                ok[e] = xk[e * TILE_SB + (t ^ (J / TILE_E))];
                ov[e] = xv[e * TILE_SB + (t ^ (J / TILE_E))];
            }
        }
        const bool keep_min = ((TILE_E * t) & J) == 0 ? ((TILE_E * t) & KK) == 0 : ((TILE_E * t) & KK) != 0;
#pragma unroll
        for (int e = 0; e < TILE_E; ++e) {
            if (pair_less(ok[e], ov[e], k[e], v[e]) == keep_min) {
                k[e] = ok[e];
                v[e] = ov[e];
            }
        }
    }
}
template <int KK, int J>
__device__ __forceinline__ void sort_stages(unsigned long long (&k)[TILE_E], uint32_t (&v)[TILE_E],
                                            unsigned long long* xk, uint32_t* xv) {
    sort_stage<KK, J>(k, v, xk, xv);
    if constexpr (J > 1) sort_stages<KK, J / 2>(k, v, xk, xv);
    else if constexpr (KK < TILE_KEYS) sort_stages<2 * KK, KK>(k, v, xk, xv);
}

// keys: the list itself, or null for the build's keys (segment, coordinate of
// axis blockIdx.y).  okey, oval: lists of n entries one behind the other.
__global__ __launch_bounds__(TILE_SB) void k_tile_sort(const unsigned long long* __restrict__ keys,
                                                       const float4* __restrict__ pts,
                                                       const int* __restrict__ seg_of, int n,
                                                       unsigned long long* __restrict__ okey,
                                                       uint32_t* __restrict__ oval) {
    __shared__ unsigned long long xk[TILE_KEYS];
    __shared__ uint32_t xv[TILE_KEYS];
    const int axis = blockIdx.y, first = blockIdx.x * TILE_KEYS + TILE_E * (int)threadIdx.x;
    unsigned long long k[TILE_E];
    uint32_t v[TILE_E];
#pragma unroll
    for (int e = 0; e < TILE_E; ++e) {
        const int i = first + e;
        v[e] = (uint32_t)i;
        k[e] = ~0ull;  // padding ranks last
        if (i < n) {
            if (keys) {
                k[e] = keys[i];
            } else {
                const float4 p = pts[i];
                k[e] = ((unsigned long long)(uint32_t)seg_of[i] << 32) |
                       float_key(axis == 0 ? p.x : (axis == 1 ? p.y : p.z));
            }
        }
    }
    sort_stages<2, 1>(k, v, xk, xv);
    const size_t off = (size_t)blockIdx.y * n;
#pragma unroll
    for (int e = 0; e < TILE_E; ++e) {
        if (first + e < n) {
            okey[off + first + e] = k[e];
            oval[off + first + e] = v[e];
        }
    }
}

// The number of keys below k in the ascending key[lo, hi), plus lo.
__device__ __forceinline__ int key_bound(const unsigned long long* __restrict__ key, int lo, int hi,
                                         unsigned long long k) {
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (key[mid] < k) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// val_out[l]: list l's order; key_out (nullable): the sorted keys of list 0;
// seg_out (nullable): their upper halves.
struct RankOut {
    uint32_t* val[3];
    unsigned long long* key;
    int* seg;
};
__global__ __launch_bounds__(MERGE_SB) void k_rank_merge(const unsigned long long* __restrict__ keys,
                                                        const uint32_t* __restrict__ vals, int n, RankOut out) {
    constexpr int TILES = RANK_SORT_MAX / TILE_KEYS;
    static_assert(2 * TILES <= MERGE_SB, "two searches per tile");
    __shared__ int lo[TILES], hi[TILES];
    const size_t off = (size_t)blockIdx.y * n;
    const unsigned long long* __restrict__ key = keys + off;
    const int t = threadIdx.x, first = blockIdx.x * MERGE_SB, last = min(first + MERGE_SB, n) - 1;
    const int tiles = (n + TILE_KEYS - 1) / TILE_KEYS, own = first / TILE_KEYS;
    if (t < 2 * tiles) {
        const int q = t >> 1, a = q * TILE_KEYS, b = min(a + TILE_KEYS, n);
        // keys are below 2^64 - 1: k + 1 does not wrap
        const int at = q == own ? a : key_bound(key, a, b, (t & 1) ? key[last] + 1 : key[first]);
        if (t & 1) hi[q] = at;
        else lo[q] = at;
    }
    __syncthreads();
    const int i = first + t;
    if (i > last) return;
    const unsigned long long k = key[i];
    int rank = i - own * TILE_KEYS;
    // four tiles at a time (their searches do not wait for each other; eight measured 21 us for 18)
    constexpr int W = 4;
    for (int j = 0; j < tiles; j += W) {
        int at[W], len[W], any = 0;
        unsigned long long kj[W];
#pragma unroll
        for (int u = 0; u < W; ++u) {
            const int q = min(j + u, tiles - 1);
            const bool use = j + u < tiles && q != own;
            at[u] = use ? lo[q] : q * TILE_KEYS;
            len[u] = use ? hi[q] - lo[q] : 0;
            kj[u] = k + (q < own ? 1 : 0);  // an earlier tile's equal keys come first
            rank -= q * TILE_KEYS;
            any |= len[u];
        }
        while (any != 0) {
            any = 0;
#pragma unroll
            for (int u = 0; u < W; ++u) {
                const int half = len[u] >> 1;
                const bool below = len[u] > 0 && key[at[u] + half] < kj[u];
                at[u] = below ? at[u] + half + 1 : at[u];
                len[u] = below ? len[u] - half - 1 : half;
                any |= len[u];
            }
        }
#pragma unroll
        for (int u = 0; u < W; ++u) rank += at[u];
    }
    out.val[blockIdx.y][rank] = vals[off + i];
    if (blockIdx.y == 0) {
        if (out.key) out.key[rank] = k;
        if (out.seg) out.seg[rank] = (int)(k >> 32);
    }
}

static inline int tiles_for(int n, int per) { return (n + per - 1) / per; }

void launch_rank_sort(const unsigned long long* keys, int n, unsigned long long* tmp_key, uint32_t* tmp_val,
                      unsigned long long* key_out, uint32_t* val_out, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_tile_sort, dim3(tiles_for(n, TILE_KEYS)), dim3(TILE_SB), 0, s, keys, (const float4*)nullptr,
                       (const int*)nullptr, n, tmp_key, tmp_val);
    RankOut out{{val_out, nullptr, nullptr}, key_out, nullptr};
    hipLaunchKernelGGL(k_rank_merge, dim3(tiles_for(n, MERGE_SB)), dim3(MERGE_SB), 0, s, tmp_key, tmp_val, n, out);
}
void launch_build_sort3(const float4* pts, const int* seg_of, int n, unsigned long long* tmp_key, uint32_t* tmp_val,
                        uint32_t* const (&perm)[3], int* sid, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_tile_sort, dim3(tiles_for(n, TILE_KEYS), 3), dim3(TILE_SB), 0, s,
                       (const unsigned long long*)nullptr, pts, seg_of, n, tmp_key, tmp_val);
    RankOut out{{perm[0], perm[1], perm[2]}, nullptr, sid};
    hipLaunchKernelGGL(k_rank_merge, dim3(tiles_for(n, MERGE_SB), 3), dim3(MERGE_SB), 0, s, tmp_key, tmp_val, n, out);
}

__device__ __forceinline__ float coord_of(float4 p, int a) { return a == 0 ? p.x : (a == 1 ? p.y : p.z); }

// Per segment: longest axis, mid, and what it allocates (one pair if it has a
// child; one next-level segment per non-empty side): pairs | segments << 32.
// lr: the points it sends left | right << 32.
__device__ __forceinline__ unsigned long long seg_decide(const BuildLevel& L, int s, unsigned long long& lr) {
    const int4 sg = L.seg[s];
    const int l = sg.x, r = sg.y;
    float ext[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float lo = coord_of(L.pts[L.perm[a][l]], a);
        const float hi = coord_of(L.pts[L.perm[a][r]], a);
        ext[a] = hi - lo;
    }
    int axis = 0;
    if (ext[1] > ext[axis]) axis = 1;
    if (ext[2] > ext[axis]) axis = 2;
    const int mid = (l + r) >> 1;
    const int has_l = mid > l, has_r = mid < r;
    L.seg_axis[s] = axis;
    L.seg_mid[s] = mid;
    lr = (unsigned long long)(uint32_t)(mid - l) | ((unsigned long long)(uint32_t)(r - mid) << 32);
    return ((has_l || has_r) ? 1ull : 0ull) | ((unsigned long long)(has_l + has_r) << 32);
}

__device__ __forceinline__ void write_child_box(NodeHot* hot, int parent, int side, const float* b) {
    float* f = hot[parent].f;
    if (side == 0) {
        *reinterpret_cast<float4*>(f + 4) = make_float4(b[0], b[1], b[2], b[3]);
        *reinterpret_cast<float2*>(f + 8) = make_float2(b[4], b[5]);
    } else {
        *reinterpret_cast<float2*>(f + 10) = make_float2(b[0], b[1]);
        *reinterpret_cast<float4*>(f + 12) = make_float4(b[2], b[3], b[4], b[5]);
    }
}

// Per segment: write the node and emit the child segments.  before: the pairs and
// segments of the segments before it; first_pair: the level's first pair.
__device__ __forceinline__ void seg_emit(const BuildLevel& L, int s, unsigned long long before, int first_pair,
                                         const Pool& pool, DevHdr* hdr) {
    const int4 sg = L.seg[s];
    const int l = sg.x, r = sg.y, node = sg.z, parent = sg.w;
    const int depth = L.seg_depth[s];
    const int axis = L.seg_axis[s];
    const int mid = L.seg_mid[s];
    const int has_l = mid > l, has_r = mid < r;
    const int pair = (has_l || has_r) ? first_pair + (int)(uint32_t)before : 0;

    const float4 P = L.pts[L.perm[axis][mid]];
    const uint32_t link = ((uint32_t)pair << LK_PAIR_SHIFT) | (has_l ? LK_HASL : 0u) | (has_r ? LK_HASR : 0u);
    *reinterpret_cast<float4*>(pool.hot[node].f) = make_float4(P.x, P.y, P.z, bitsf(link));
    pool.ids[node] = fbits(P.w);
    pool.par[node] = parent;
    pool.cnt[node] = make_int4(r - l + 1, 0, 0, depth);
    pool.meta[node] = (uint32_t)axis;
    atomicMax(&hdr->max_depth, depth);

    float box[6];
    box[0] = L.pts[L.perm[0][l]].x;
    box[1] = L.pts[L.perm[1][l]].y;
    box[2] = L.pts[L.perm[2][l]].z;
    box[3] = L.pts[L.perm[0][r]].x;
    box[4] = L.pts[L.perm[1][r]].y;
    box[5] = L.pts[L.perm[2][r]].z;
    write_child_box(pool.hot, parent, node & 1, box);

    int c = (int)(before >> 32);
    int2 ch = make_int2(-1, -1);
    if (has_l) {
        L.seg_next[c] = make_int4(l, mid - 1, 2 * pair, node);
        L.seg_depth_next[c] = depth + 1;
        ch.x = c++;
    }
    if (has_r) {
        L.seg_next[c] = make_int4(mid + 1, r, 2 * pair + 1, node);
        L.seg_depth_next[c] = depth + 1;
        ch.y = c++;
    }
    L.seg_child[s] = ch;
}

// A level's segments by one workgroup (up to SEG_ONE_MAX of them: decide, scan
// and emit in one launch; each was one of the 8 launches of a level).
__device__ __forceinline__ unsigned long long wave_inclusive_u64(unsigned long long x, int lane) {
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int src = (lane - d) & 63;  // lanes below d ignore what they read
        const unsigned lo = (unsigned)__shfl((int)(unsigned)x, src);
        const unsigned hi = (unsigned)__shfl((int)(unsigned)(x >> 32), src);
        if (lane >= d) x += ((unsigned long long)hi << 32) | lo;
    }
    return x;
}
constexpr int SEG_ONE_MAX = 8192;
__global__ __launch_bounds__(1024) void k_build_seg_one(BuildLevel L, Pool pool, DevHdr* hdr) {
    __shared__ unsigned long long tot_f[16], tot_lr[16];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int count = hdr->seg_count[L.cur], first_pair = hdr->pair_used;
    const int chunk = (count + 1023) >> 10;
    const int b = min(t * chunk, count), e = min(b + chunk, count);
    unsigned long long f = 0, lr = 0;
    for (int s = b; s < e; ++s) {
        unsigned long long x;
        f += seg_decide(L, s, x);
        lr += x;
    }
    const unsigned long long inc_f = wave_inclusive_u64(f, lane), inc_lr = wave_inclusive_u64(lr, lane);
    if (lane == 63) {
        tot_f[w] = inc_f;
        tot_lr[w] = inc_lr;
    }
    __syncthreads();
    unsigned long long run_f = inc_f - f, run_lr = inc_lr - lr;
    for (int i = 0; i < w; ++i) {
        run_f += tot_f[i];
        run_lr += tot_lr[i];
    }
    for (int s = b; s < e; ++s) {
        const int4 sg = L.seg[s];
        const int mid = L.seg_mid[s];
        const int has_l = mid > sg.x, has_r = mid < sg.y;
        L.seg_lr[s] = run_lr;
        seg_emit(L, s, run_f, first_pair, pool, hdr);
        run_f += ((has_l || has_r) ? 1ull : 0ull) | ((unsigned long long)(has_l + has_r) << 32);
        run_lr += (unsigned long long)(uint32_t)(mid - sg.x) | ((unsigned long long)(uint32_t)(sg.y - mid) << 32);
    }
    if (t == 1023) {
        hdr->seg_count[L.cur ^ 1] = (int)(run_f >> 32);
        hdr->pair_used = first_pair + (int)(uint32_t)run_f;
    }
}

// More segments: decide, two scans, emit.
__global__ void k_build_seg_a(BuildLevel L, int bound, DevHdr* hdr) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s == 0) hdr->seg_count[L.cur ^ 1] = 0;
    if (s >= bound) return;
    unsigned long long f = 0, lr = 0;
    if (s < hdr->seg_count[L.cur]) f = seg_decide(L, s, lr);
    L.seg_flags[s] = f;
    L.seg_lr_in[s] = lr;
}
__global__ void k_build_seg_b(BuildLevel L, int bound, Pool pool, DevHdr* hdr) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    const int count = hdr->seg_count[L.cur];
    if (s >= bound || s >= count) return;
    seg_emit(L, s, L.seg_scan[s], hdr->pair_used, pool, hdr);
    if (s == count - 1) {
        const unsigned long long all = L.seg_scan[s] + L.seg_flags[s];
        hdr->seg_count[L.cur ^ 1] = (int)(all >> 32);
        hdr->pair_pending = (int)(uint32_t)all;
    }
}

__global__ void k_build_side(BuildLevel L, DevHdr* hdr) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j == 0) {
        hdr->pair_used += hdr->pair_pending;
        hdr->pair_pending = 0;
    }
    if (j >= L.m) return;
    int s = L.sid[j];
    if (s < 0) return;
    int a = L.seg_axis[s];
    int mid = L.seg_mid[s];
    uint32_t p = L.perm[a][j];
    L.side[p] = (uint8_t)(j < mid ? 0 : (j == mid ? 2 : 1));
}

// The stable partition of the three lists, PART_TILE positions to a workgroup.
// k_build_bits: which positions go left and right, as one bit each, and the
// tile's counts of both.  k_build_scatter: a position's rank among the lefts (or
// rights) of its segment is the tile's prefix (the counts of the tiles before
// it), the bits before it in the tile, less the lefts of the segments before
// its own, which the segments' sizes give (seg_lr).  The bits are 1/4 byte a
// position where a flag and its scan moved 24: a level of 2M points took 25 us
// of flags, 45 of scan and 37 of scatter (now 24 of bits and 31 of scatter).
//
// Up to TILES_SUMMED_MAX tiles each workgroup adds up the tiles before its own;
// that grows with the square of the length, so for longer lists a scan between
// the two launches does (a Build of uniform points, the sums against the scan:
// 1M 1.73 and 1.76 ms, 3M 4.41 and 4.40, 8M 13.4 and 13.1, 64M 195 and 149).
constexpr int PART_TILE = 1024, PART_SB = 256, PART_WORDS = PART_TILE / 64;
constexpr long long TILES_SUMMED_MAX = 3072;

__global__ __launch_bounds__(PART_SB) void k_build_bits(BuildLevel L) {
    __shared__ int cl[PART_SB / 64], cr[PART_SB / 64];
    const int t = threadIdx.x, b = blockIdx.y, lane = t & 63, w = t >> 6;
    const int words = (L.m + 63) >> 6, tiles = gridDim.x;
    int nl = 0, nr = 0;
#pragma unroll
    for (int it = 0; it < PART_TILE / PART_SB; ++it) {
        const int j = blockIdx.x * PART_TILE + it * PART_SB + t;
        int sd = 2;
        if (j < L.m && L.sid[j] >= 0) sd = L.side[L.perm[b][j]];
        const unsigned long long ml = __ballot(sd == 0), mr = __ballot(sd == 1);
        if (lane == 0 && j < L.m) {
            L.bits_l[(size_t)b * words + (j >> 6)] = ml;
            L.bits_r[(size_t)b * words + (j >> 6)] = mr;
        }
        nl += __popcll(ml);
        nr += __popcll(mr);
    }
    if (lane == 0) {
        cl[w] = nl;
        cr[w] = nr;
    }
    __syncthreads();
    if (t == 0) {
        unsigned long long c = 0;
        for (int i = 0; i < PART_SB / 64; ++i) c += (unsigned long long)(uint32_t)cl[i] | ((unsigned long long)(uint32_t)cr[i] << 32);
        L.tile_lr[(size_t)b * tiles + blockIdx.x] = c;
    }
}

__global__ __launch_bounds__(PART_SB) void k_build_scatter(BuildLevel L) {
    __shared__ unsigned long long part[PART_SB / 64];
    __shared__ unsigned long long wl[PART_WORDS], wr[PART_WORDS];
    __shared__ unsigned long long pre[PART_WORDS];  // lefts | rights << 32 before each word, in the list
    const int t = threadIdx.x, b = blockIdx.y, lane = t & 63, w = t >> 6;
    const int words = (L.m + 63) >> 6, tiles = gridDim.x;
    const unsigned long long* __restrict__ counts = L.tile_lr + (size_t)b * tiles;
    unsigned long long sum = 0;
    if (L.tile_pre) {
        // the three lists' tiles scanned behind one another: less the lists before this one
        if (t == 0) sum = L.tile_pre[(size_t)b * tiles + blockIdx.x] - L.tile_pre[(size_t)b * tiles];
    } else {
        for (int i = t; i < (int)blockIdx.x; i += PART_SB) sum += counts[i];
    }
    sum = wave_inclusive_u64(sum, lane);
    if (lane == 63) part[w] = sum;
    if (t < PART_WORDS) {
        const int q = blockIdx.x * PART_WORDS + t;
        wl[t] = q < words ? L.bits_l[(size_t)b * words + q] : 0ull;
        wr[t] = q < words ? L.bits_r[(size_t)b * words + q] : 0ull;
    }
    __syncthreads();
    if (t == 0) {
        unsigned long long run = 0;
        for (int i = 0; i < PART_SB / 64; ++i) run += part[i];
        for (int i = 0; i < PART_WORDS; ++i) {
            pre[i] = run;
            run += (unsigned long long)(uint32_t)__popcll(wl[i]) | ((unsigned long long)(uint32_t)__popcll(wr[i]) << 32);
        }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < PART_TILE / PART_SB; ++it) {
        const int k = it * PART_SB + t, j = blockIdx.x * PART_TILE + k;
        if (j >= L.m) continue;
        const int s = L.sid[j];
        if (s < 0) {
            if (b == 0) L.sid_next[j] = -1;
            continue;
        }
        const int q = k >> 6;
        const unsigned long long below = (1ull << (k & 63)) - 1ull, bit = 1ull << (k & 63);
        const unsigned long long p = pre[q], base = L.seg_lr[s];
        const int mid = L.seg_mid[s];
        int np;
        bool left = (wl[q] & bit) != 0;
        if (left) {
            np = L.seg[s].x + (int)((uint32_t)p - (uint32_t)base) + __popcll(wl[q] & below);
        } else if (wr[q] & bit) {
            np = mid + 1 + (int)((uint32_t)(p >> 32) - (uint32_t)(base >> 32)) + __popcll(wr[q] & below);
        } else {
            if (b == 0) L.sid_next[mid] = -1;  // the segment's node
            continue;
        }
        L.perm_next[b][np] = L.perm[b][j];
        if (b == 0) {
            const int2 ch = L.seg_child[s];
            L.sid_next[np] = left ? ch.x : ch.y;
        }
    }
}

static inline int blocks_for(long long n, int bs) { return (int)((n + bs - 1) / bs); }

// out[j] = pts[perm[j]]: a level's points in list order, so every segment's
// points are contiguous for the one-workgroup build of the levels below.
// Positions whose point is already a node of an upper level (sid < 0) are
// never written by the partitions and hold no valid index: skip them.
// out[j] = the point at list position j; inv[point] = j (positions already
// placed as nodes are skipped: no kernel wrote their list entries).
__global__ void k_gather_list(const float4* __restrict__ pts, const uint32_t* __restrict__ perm,
                              const int* __restrict__ sid, int m, float4* __restrict__ out, int* __restrict__ inv) {
    int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= m) return;
    if (sid[j] < 0) {
        out[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        return;
    }
    const uint32_t p = perm[j];
    out[j] = pts[p];
    if (inv) inv[p] = j;
}
void launch_gather_list(const float4* pts, const uint32_t* perm, const int* sid, int m, float4* out, int* inv,
                        hipStream_t s) {
    if (m <= 0) return;
    hipLaunchKernelGGL(k_gather_list, dim3(blocks_for(m, 256)), dim3(256), 0, s, pts, perm, sid, m, out, inv);
}

void launch_build_keys(const float4* pts, const int* seg_of, int m, int axis, unsigned long long* keys,
                       uint32_t* vals, hipStream_t s) {
    if (m <= 0) return;
    hipLaunchKernelGGL(k_build_keys, dim3(blocks_for(m, 256)), dim3(256), 0, s, pts, seg_of, m, axis, keys, vals);
}
void launch_build_keys32(const float4* pts, int m, int axis, uint32_t* keys, uint32_t* vals, hipStream_t s) {
    if (m <= 0) return;
    hipLaunchKernelGGL(k_build_keys32, dim3(blocks_for(m, 256)), dim3(256), 0, s, pts, m, axis, keys, vals);
}
void launch_build_init_sid(const unsigned long long* k0, int m, int* sid, hipStream_t s) {
    if (m <= 0) return;
    hipLaunchKernelGGL(k_build_init_sid, dim3(blocks_for(m, 256)), dim3(256), 0, s, k0, m, sid);
}
bool build_seg_one_fits(int bound) { return bound <= SEG_ONE_MAX; }
void launch_build_seg_one(const BuildLevel& L, Pool pool, DevHdr* hdr, hipStream_t s) {
    hipLaunchKernelGGL(k_build_seg_one, dim3(1), dim3(1024), 0, s, L, pool, hdr);
}
void launch_build_seg_a(const BuildLevel& L, int bound, DevHdr* hdr, hipStream_t s) {
    hipLaunchKernelGGL(k_build_seg_a, dim3(blocks_for(bound > 0 ? bound : 1, 256)), dim3(256), 0, s, L, bound, hdr);
}
void launch_build_seg_b(const BuildLevel& L, int bound, Pool pool, DevHdr* hdr, hipStream_t s) {
    if (bound <= 0) return;
    hipLaunchKernelGGL(k_build_seg_b, dim3(blocks_for(bound, 256)), dim3(256), 0, s, L, bound, pool, hdr);
}
void launch_build_side(const BuildLevel& L, DevHdr* hdr, hipStream_t s) {
    hipLaunchKernelGGL(k_build_side, dim3(blocks_for(L.m > 0 ? L.m : 1, 256)), dim3(256), 0, s, L, hdr);
}
long long build_tiles(long long m) { return (m + PART_TILE - 1) / PART_TILE; }
bool build_tiles_scanned(long long m) { return build_tiles(m) > TILES_SUMMED_MAX; }
void launch_build_bits(const BuildLevel& L, hipStream_t s) {
    if (L.m <= 0) return;
    hipLaunchKernelGGL(k_build_bits, dim3((unsigned)build_tiles(L.m), 3), dim3(PART_SB), 0, s, L);
}
void launch_build_scatter(const BuildLevel& L, hipStream_t s) {
    if (L.m <= 0) return;
    hipLaunchKernelGGL(k_build_scatter, dim3((unsigned)build_tiles(L.m), 3), dim3(PART_SB), 0, s, L);
}

}  // namespace ikd
