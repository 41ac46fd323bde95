// ikd_build_small.hip — one-launch build of many small subtrees.
//
// The same construction as ikd_build.hip (BuildTree, ikd_Tree.cpp:573-622:
// longest axis with ties to the lower axis, the element of rank mid-l with
// mid = (l+r)>>1 as the node, stable presorted partitions so that equal keys
// keep their input order), but one 256-thread workgroup builds one whole
// segment of at most SMALL_MAX points in LDS: a bitonic sort per axis, then
// one level per block-synchronous step.  Segments, pairs and children are
// numbered in the same order as the global build, so a subtree built here is
// the one the level-synchronous global build makes for the same input.
//
// Node allocation is deterministic: segment g takes the pair range that
// starts at pair_used + exclusive_scan(pairs)[g], where pairs(m) is the number
// of nodes with children in the median tree of m points.
#include <algorithm>

#include "ikd_internal.h"

namespace ikd {

// Three shapes: one lane per segment of at most MICRO_MAX points (most insert
// groups hold one to a few points), one wavefront per segment of at most
// TINY_MAX points, one workgroup for the rest up to SMALL_MAX.  The plan lists
// the segments of the two larger shapes, and one launch builds all three side
// by side: each is a chain of LDS and gather latencies that leaves the device
// almost idle, and one behind the other they took 25 + 38 + 47 us twice per
// mapped scan (now 69 together, at 20 scans 18.2 -> 16.5 ms).
constexpr int MICRO_MAX = 8;
constexpr int TINY_MAX = 128;
constexpr int SMALL_SB = 256;  // threads of a workgroup
constexpr int TINY_WAVES = SMALL_SB / 64;

// Nodes with at least one child in the median-split tree of m points.  A node
// of size x >= 2 leaves children of sizes (x-1)>>1 and x-1-((x-1)>>1), so a
// level holds at most two distinct sizes.
__device__ int median_tree_pairs(int m) {
    int sz[2] = {m, -1};
    long long cnt[2] = {1, 0};
    long long internal = 0;
    while (cnt[0] > 0 || cnt[1] > 0) {
        int nsz[2] = {-1, -1};
        long long ncnt[2] = {0, 0};
        for (int i = 0; i < 2; ++i) {
            if (cnt[i] == 0 || sz[i] < 2) continue;
            internal += cnt[i];
            int parts[2] = {(sz[i] - 1) >> 1, sz[i] - 1 - ((sz[i] - 1) >> 1)};
            for (int p = 0; p < 2; ++p) {
                int x = parts[p];
                if (x < 2) continue;
                int slot = (nsz[0] == x || nsz[0] < 0) ? 0 : 1;
                nsz[slot] = x;
                ncnt[slot] += cnt[i];
            }
        }
        sz[0] = nsz[0];
        sz[1] = nsz[1];
        cnt[0] = ncnt[0];
        cnt[1] = ncnt[1];
    }
    return (int)internal;
}

// Pairs of segment g, and its entry in the list of its shape.
__device__ __forceinline__ int plan_segment(const int4* __restrict__ seg, int g, int S, int micro,
                                            int* __restrict__ lists, DevHdr* hdr) {
    const int m = seg[g].y - seg[g].x + 1;
    if (m <= 0) return 0;
    if (!micro || m > MICRO_MAX) {
        if (m <= TINY_MAX) lists[atomicAdd(&hdr->small_lists[0], 1)] = g;
        else lists[S + atomicAdd(&hdr->small_lists[1], 1)] = g;
    }
    return median_tree_pairs(m);
}

// count_dev (optional) holds the number of live segments among the S slots;
// slots past it take no pairs.  k_small_plan: one workgroup, for up to PLAN_MAX
// segments; pair_scan gets every segment's first pair relative to the pairs this
// build takes, which begin at hdr->pair_base.
constexpr int PLAN_MAX = 8192;
__global__ __launch_bounds__(1024) void k_small_plan(const int4* __restrict__ seg, int S,
                                                     const int* __restrict__ count_dev, int micro,
                                                     int* __restrict__ pair_scan, int* __restrict__ lists,
                                                     DevHdr* hdr) {
    __shared__ int wave_tot[16];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int count = min(count_dev ? *count_dev : S, S);
    const int chunk = (S + 1023) >> 10;
    const int b = min(t * chunk, S), e = min(b + chunk, S);
    if (t < 2) hdr->small_lists[t] = 0;
    __syncthreads();
    int sum = 0;
    for (int g = b; g < e; ++g) {
        const int p = g < count ? plan_segment(seg, g, S, micro, lists, hdr) : 0;
        pair_scan[g] = sum;  // within the thread's run for now
        sum += p;
    }
    int inc = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl(inc, (lane - d) & 63);  // lanes below d ignore what they read
        if (lane >= d) inc += o;
    }
    if (lane == 63) wave_tot[w] = inc;
    __syncthreads();
    int run = inc - sum;
    for (int i = 0; i < w; ++i) run += wave_tot[i];
    for (int g = b; g < e; ++g) pair_scan[g] += run;
    if (t == 1023) {
        hdr->pair_base = hdr->pair_used;
        hdr->pair_used += run + sum;
    }
}

__global__ void k_small_pairs(const int4* __restrict__ seg, int S, const int* __restrict__ count_dev, int micro,
                              int* __restrict__ pairs, int* __restrict__ lists, DevHdr* hdr) {
    int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= S) return;
    const int count = count_dev ? *count_dev : S;
    pairs[g] = g < count ? plan_segment(seg, g, S, micro, lists, hdr) : 0;
}
__global__ void k_small_commit(const int* __restrict__ pairs, const int* __restrict__ scan, int S, DevHdr* hdr) {
    hdr->pair_base = hdr->pair_used;
    hdr->pair_used += scan[S - 1] + pairs[S - 1];
}
__device__ __forceinline__ void write_child_box_s(NodeHot* hot, int parent, int side, const float* b) {
    float* f = hot[parent].f;
    if (side == 0) {
        *reinterpret_cast<float4*>(f + 4) = make_float4(b[0], b[1], b[2], b[3]);
        *reinterpret_cast<float2*>(f + 8) = make_float2(b[4], b[5]);
    } else {
        *reinterpret_cast<float2*>(f + 10) = make_float2(b[0], b[1]);
        *reinterpret_cast<float4*>(f + 12) = make_float4(b[2], b[3], b[4], b[5]);
    }
}

// A build by SB threads: a wavefront of its own (SB = 64; the workgroup's other
// wavefronts build other segments) or a whole workgroup.
template <int SB>
__device__ __forceinline__ int build_thread() {
    return SB == 64 ? (int)(threadIdx.x & 63u) : (int)threadIdx.x;
}
template <int SB>
__device__ __forceinline__ void build_sync() {
    if (SB == 64) {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    } else {
        __syncthreads();
    }
}

// Exclusive scan of one 64-bit value per thread across the building threads
// (*total gets the sum): an inclusive scan inside each wavefront by
// shuffles, then the wavefront totals through LDS (two barriers).  Several
// small counters can ride in one value as bit fields that never overflow.
template <int SB>
__device__ unsigned long long block_exscan_u64(unsigned long long v, unsigned long long* wtot,
                                               unsigned long long* total) {
    const int t = build_thread<SB>(), lane = t & 63, w = t >> 6;
    unsigned long long x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int src = (lane - off) & 63;  // lanes below off ignore what they read
        const unsigned lo = (unsigned)__shfl((int)(unsigned)x, src);
        const unsigned hi = (unsigned)__shfl((int)(unsigned)(x >> 32), src);
        const unsigned long long y = ((unsigned long long)hi << 32) | lo;
        if (lane >= off) x += y;
    }
    if (lane == 63) wtot[w] = x;
    build_sync<SB>();
    unsigned long long base = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < SB / 64; ++i) {
        if (i < w) base += wtot[i];
        tot += wtot[i];
    }
    *total = tot;
    build_sync<SB>();
    return base + x - v;
}

// Ascending bitonic sort of P keys (P a power of two, at most E * SB) held in
// registers: key i lives in x[i / SB] of thread i % SB.  Stages whose partner
// is in the same wavefront exchange by shuffles, stages across the thread's
// own registers by swaps, and only the stages across wavefronts go through
// LDS (xch, SB * E entries).  Keys must be distinct.
template <int SB, int E>
__device__ void reg_bitonic(unsigned long long (&x)[E], int P, unsigned long long* xch) {
    const int t = build_thread<SB>();
    for (int k = 2; k <= P; k <<= 1) {
        for (int j = k >> 1; j > 0; j >>= 1) {
            if (j >= SB) {
                const int ej = j / SB;
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const int e2 = e ^ ej;
                    if (e2 <= e || e2 >= E) continue;
                    const bool up = ((e * SB + t) & k) == 0;
                    const unsigned long long a = x[e], b = x[e2];
                    if ((a > b) == up) {
                        x[e] = b;
                        x[e2] = a;
                    }
                }
            } else if (j >= 64) {
                build_sync<SB>();
#pragma unroll
                for (int e = 0; e < E; ++e) xch[e * SB + t] = x[e];
                build_sync<SB>();
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const int i = e * SB + t;
                    const unsigned long long y = xch[i ^ j];
                    const bool keep_min = ((i & j) == 0) == ((i & k) == 0);
                    x[e] = keep_min ? (x[e] < y ? x[e] : y) : (x[e] > y ? x[e] : y);
                }
            } else {
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const int i = e * SB + t;
                    const unsigned lo = (unsigned)__shfl_xor((int)(unsigned)x[e], j);
                    const unsigned hi = (unsigned)__shfl_xor((int)(unsigned)(x[e] >> 32), j);
                    const unsigned long long y = ((unsigned long long)hi << 32) | lo;
                    const bool keep_min = ((i & j) == 0) == ((i & k) == 0);
                    x[e] = keep_min ? (x[e] < y ? x[e] : y) : (x[e] > y ? x[e] : y);
                }
            }
        }
    }
    build_sync<SB>();  // xch may be reused at once
}

// orig (optional) gives each point's index in the caller's original input:
// equal coordinates are then ordered by it, as the global build's stable
// presorted lists order them; without it, by position in the segment.
template <int SB, int SMAX>
struct BuildLds {
    static constexpr int SEGS = SMAX / 2 + 1;
    unsigned long long skey[SMAX];  // sort keys, then running counts
    unsigned long long wtot[SB / 64];
    float px[SMAX], py[SMAX], pz[SMAX];
    int seg_node[2][SEGS], seg_par[2][SEGS];
    unsigned short lst[2][3][SMAX];
    unsigned short rnk[SMAX];
    short sid[2][SMAX];
    short seg_l[2][SEGS], seg_r[2][SEGS];
    short seg_mid[SEGS], seg_cl[SEGS], seg_cr[SEGS];
    unsigned char side[SMAX];
    unsigned char seg_axis[SEGS];
};

// Segment g by SB threads.
template <int SB, int SMAX>
__device__ void build_segment(BuildLds<SB, SMAX>& L, int g, const float4* __restrict__ pts,
                              const int4* __restrict__ seg, const int* __restrict__ seg_depth,
                              const int* __restrict__ pair_scan, const uint32_t* __restrict__ orig,
                              const SmallLists& pre, const Pool& pool, DevHdr* hdr) {
    const int t = build_thread<SB>();
    const int4 sg = seg[g];
    const int l0 = sg.x;
    const int m = sg.y - sg.x + 1;
    // the list holds this shape's size class; the host guarantees m <= SMALL_MAX
    if (m <= 0 || m > SMAX) return;
    const int depth0 = seg_depth[g];
    int next_pair = hdr->pair_base + pair_scan[g];

    for (int i = t; i < m; i += SB) {
        float4 p = pts[l0 + i];
        L.px[i] = p.x;
        L.py[i] = p.y;
        L.pz[i] = p.z;
    }
    int P = 1;
    while (P < m) P <<= 1;
    if (pre.inv0) {
        // the caller's lists are already sorted (coordinate, original index)
        // per segment, and the points were gathered in x order
        for (int i = t; i < m; i += SB) {
            L.lst[0][0][i] = (unsigned short)i;
            L.lst[0][1][i] = (unsigned short)(pre.inv0[pre.list1[l0 + i]] - l0);
            L.lst[0][2][i] = (unsigned short)(pre.inv0[pre.list2[l0 + i]] - l0);
        }
    } else {
    // tie-break rank of every point: its order by original index, or its position
    constexpr int E = SMAX / SB;
    unsigned long long x[E];
    if (orig) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = e * SB + t;
            x[e] = i < m ? (((unsigned long long)orig[l0 + i] << 16) | (unsigned)i) : ~0ull;
        }
        reg_bitonic<SB, E>(x, P, L.skey);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = e * SB + t;
            if (i < m) L.rnk[x[e] & 0xffffu] = (unsigned short)i;
        }
    } else {
        for (int i = t; i < m; i += SB) L.rnk[i] = (unsigned short)i;
    }
    build_sync<SB>();
    // three stable sorted index lists: key (coordinate, rank, position)
    for (int a = 0; a < 3; ++a) {
        const float* c = a == 0 ? L.px : (a == 1 ? L.py : L.pz);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = e * SB + t;
            x[e] = i < m ? (((unsigned long long)float_key(c[i]) << 32) | ((unsigned)L.rnk[i] << 16) | (unsigned)i)
                         : ~0ull;
        }
        reg_bitonic<SB, E>(x, P, L.skey);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = e * SB + t;
            if (i < m) L.lst[0][a][i] = (unsigned short)(x[e] & 0xffffu);
        }
    }
    build_sync<SB>();
    }
    for (int i = t; i < m; i += SB) L.sid[0][i] = 0;
    if (t == 0) {
        L.seg_l[0][0] = 0;
        L.seg_r[0][0] = (short)(m - 1);
        L.seg_node[0][0] = sg.z;
        L.seg_par[0][0] = sg.w;
    }
    build_sync<SB>();
    unsigned long long* run = L.skey;  // the sort keys' space, reused for running counts
    const int chunk = (m + SB - 1) / SB;
    int ns = 1;
    int cur = 0;
    for (int level = 0; ns > 0; ++level) {
        const int depth = depth0 + level;
        const int per = (ns + SB - 1) / SB;  // contiguous segments per thread keep the order
        int my_pairs = 0, my_children = 0;
        for (int q = 0; q < per; ++q) {
            const int s = t * per + q;
            if (s >= ns) break;
            const int l = L.seg_l[cur][s], r = L.seg_r[cur][s];
            float ext[3];
            ext[0] = L.px[L.lst[cur][0][r]] - L.px[L.lst[cur][0][l]];
            ext[1] = L.py[L.lst[cur][1][r]] - L.py[L.lst[cur][1][l]];
            ext[2] = L.pz[L.lst[cur][2][r]] - L.pz[L.lst[cur][2][l]];
            int axis = 0;
            if (ext[1] > ext[axis]) axis = 1;
            if (ext[2] > ext[axis]) axis = 2;
            const int mid = (l + r) >> 1;
            L.seg_axis[s] = (unsigned char)axis;
            L.seg_mid[s] = (short)mid;
            const int hl = mid > l, hr = mid < r;
            my_pairs += (hl || hr) ? 1 : 0;
            my_children += hl + hr;
        }
        unsigned long long tot2;
        const unsigned long long off2 =
            block_exscan_u64<SB>((unsigned long long)my_pairs | ((unsigned long long)my_children << 32), L.wtot, &tot2);
        int pair_off = (int)(unsigned)off2, child_off = (int)(off2 >> 32);
        const int tot_pairs = (int)(unsigned)tot2, tot_children = (int)(tot2 >> 32);
        for (int q = 0; q < per; ++q) {
            const int s = t * per + q;
            if (s >= ns) break;
            const int l = L.seg_l[cur][s], r = L.seg_r[cur][s], mid = L.seg_mid[s], axis = L.seg_axis[s];
            const int node = L.seg_node[cur][s], parent = L.seg_par[cur][s];
            const int hl = mid > l, hr = mid < r;
            const int pair = (hl || hr) ? next_pair + pair_off++ : 0;
            const int piv = L.lst[cur][axis][mid];
            const uint32_t link = ((uint32_t)pair << LK_PAIR_SHIFT) | (hl ? LK_HASL : 0u) | (hr ? LK_HASR : 0u);
            const float4 P4 = pts[l0 + piv];
            *reinterpret_cast<float4*>(pool.hot[node].f) = make_float4(P4.x, P4.y, P4.z, bitsf(link));
            pool.ids[node] = fbits(P4.w);
            pool.par[node] = parent;
            pool.cnt[node] = make_int4(r - l + 1, 0, 0, depth);
            pool.meta[node] = (uint32_t)axis;
            float box[6] = {L.px[L.lst[cur][0][l]], L.py[L.lst[cur][1][l]], L.pz[L.lst[cur][2][l]],
                            L.px[L.lst[cur][0][r]], L.py[L.lst[cur][1][r]], L.pz[L.lst[cur][2][r]]};
            write_child_box_s(pool.hot, parent, node & 1, box);
            int cl = -1, cr = -1;
            if (hl) {
                cl = child_off++;
                L.seg_l[cur ^ 1][cl] = (short)l;
                L.seg_r[cur ^ 1][cl] = (short)(mid - 1);
                L.seg_node[cur ^ 1][cl] = 2 * pair;
                L.seg_par[cur ^ 1][cl] = node;
            }
            if (hr) {
                cr = child_off++;
                L.seg_l[cur ^ 1][cr] = (short)(mid + 1);
                L.seg_r[cur ^ 1][cr] = (short)r;
                L.seg_node[cur ^ 1][cr] = 2 * pair + 1;
                L.seg_par[cur ^ 1][cr] = node;
            }
            L.seg_cl[s] = (short)cl;
            L.seg_cr[s] = (short)cr;
        }
        if (t == 0) atomicMax(&hdr->max_depth, depth);
        next_pair += tot_pairs;
        build_sync<SB>();
        if (tot_children == 0) break;
        // side of every live position, read off its segment's axis list
        for (int j = t; j < m; j += SB) {
            const int s = L.sid[cur][j];
            if (s < 0) continue;
            const int mid = L.seg_mid[s];
            L.side[L.lst[cur][L.seg_axis[s]][j]] = (unsigned char)(j < mid ? 0 : (j == mid ? 2 : 1));
        }
        build_sync<SB>();
        // stable partition of the three lists at once: for every position, the
        // numbers of left and right entries of each list before it, as six
        // 10-bit fields of one value (no field reaches 1024: at most m - 1
        // entries move), so one scan serves all three lists
        unsigned long long cnt6 = 0;
        for (int q = 0; q < chunk; ++q) {
            const int j = t * chunk + q;
            if (j >= m) break;
            if (L.sid[cur][j] < 0) continue;
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                const unsigned char sd = L.side[L.lst[cur][b][j]];
                if (sd < 2) cnt6 += 1ull << (20 * b + 10 * sd);
            }
        }
        unsigned long long tot6;
        unsigned long long acc = block_exscan_u64<SB>(cnt6, L.wtot, &tot6);
        for (int q = 0; q < chunk; ++q) {
            const int j = t * chunk + q;
            if (j >= m) break;
            run[j] = acc;
            if (L.sid[cur][j] < 0) continue;
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                const unsigned char sd = L.side[L.lst[cur][b][j]];
                if (sd < 2) acc += 1ull << (20 * b + 10 * sd);
            }
        }
        build_sync<SB>();
        for (int b = 0; b < 3; ++b) {
            for (int q = 0; q < chunk; ++q) {
                const int j = t * chunk + q;
                if (j >= m) break;
                const int s = L.sid[cur][j];
                if (s < 0) {
                    if (b == 0) L.sid[cur ^ 1][j] = -1;
                    continue;
                }
                const int p = L.lst[cur][b][j];
                const unsigned char sd = L.side[p];
                if (sd == 2) {
                    if (b == 0) L.sid[cur ^ 1][L.seg_mid[s]] = -1;
                    continue;
                }
                const int l = L.seg_l[cur][s], mid = L.seg_mid[s];
                // fields only grow along the list, so the packed difference
                // subtracts field by field without borrows
                const int before = (int)(((run[j] - run[l]) >> (20 * b + 10 * sd)) & 1023ull);
                const int np = sd == 0 ? l + before : mid + 1 + before;
                L.lst[cur ^ 1][b][np] = (unsigned short)p;
                if (b == 0) L.sid[cur ^ 1][np] = sd == 0 ? L.seg_cl[s] : L.seg_cr[s];
            }
        }
        build_sync<SB>();
        ns = tot_children;
        cur ^= 1;
    }
    build_sync<SB>();  // the next segment of the list reuses the LDS arrays
}

// One lane builds one segment of at most MICRO_MAX points: the median tree of
// k_build_small (axis of the longest extent, ties to the lower axis; node =
// the element of rank (n-1)>>1 in (coordinate, position) order; both sides
// keep the segment's order).  The lane keeps the work order as 4-bit
// positions packed in one register and its pending ranges in LDS (nothing
// indexed at run time lives in private memory); pairs are taken from the
// segment's range one internal node at a time.  Larger segments (or every
// segment when micro is off) go to the size-class lists.
constexpr int MICRO_BS = SMALL_SB;
constexpr int MICRO_STACK = 6;  // pending ranges: at most one per level below the current one
struct MicroLds {
    // per lane: (lo | hi << 4 | level << 8), slot node, slot parent
    int stk_r[MICRO_STACK][MICRO_BS], stk_node[MICRO_STACK][MICRO_BS], stk_par[MICRO_STACK][MICRO_BS];
};
__device__ __forceinline__ float micro_coord(const float4& q, int axis) {
    return axis == 0 ? q.x : (axis == 1 ? q.y : q.z);
}
__device__ void build_micro(MicroLds& L, int g, const float4* __restrict__ pts, const int4* __restrict__ seg,
                            const int* __restrict__ seg_depth, const int* __restrict__ pair_scan, int S,
                            const int* __restrict__ count_dev, const Pool& pool, DevHdr* hdr) {
    const int tid = threadIdx.x;
    if (g >= S || (count_dev && g >= *count_dev)) return;
    const int4 sg = seg[g];
    const int m = sg.y - sg.x + 1;
    if (m <= 0 || m > MICRO_MAX) return;
    const float4* P = pts + sg.x;
    uint64_t perm = 0x76543210ull;  // nibble i: the position at work-order slot i
    int next_pair = hdr->pair_base + pair_scan[g];
    const int depth0 = seg_depth[g];
    int nw = 1;
    L.stk_r[0][tid] = m << 4;
    L.stk_node[0][tid] = sg.z;
    L.stk_par[0][tid] = sg.w;
    int deepest = depth0;
    while (nw > 0) {
        --nw;
        const int rr = L.stk_r[nw][tid];
        const int lo = rr & 15, hi = (rr >> 4) & 15, depth = depth0 + (rr >> 8);
        const int node = L.stk_node[nw][tid], parent = L.stk_par[nw][tid];
        const int cnt = hi - lo;
        // bounds in key order, as the sorted lists give them (-0 below +0)
        const float4 q0 = P[(perm >> (4 * lo)) & 15];
        float mn[3] = {q0.x, q0.y, q0.z}, mx[3] = {q0.x, q0.y, q0.z};
        for (int i = lo + 1; i < hi; ++i) {
            const float4 q = P[(perm >> (4 * i)) & 15];
            const float c[3] = {q.x, q.y, q.z};
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                if (float_key(c[a]) < float_key(mn[a])) mn[a] = c[a];
                if (float_key(c[a]) > float_key(mx[a])) mx[a] = c[a];
            }
        }
        const float ext[3] = {mx[0] - mn[0], mx[1] - mn[1], mx[2] - mn[2]};
        int axis = 0;
        if (ext[1] > ext[axis]) axis = 1;
        if (ext[2] > ext[axis]) axis = 2;
        // the element of rank (cnt-1)>>1 in (coordinate, position) order
        const int want = (cnt - 1) >> 1;
        int pos = -1;
        uint32_t kp = 0;
        for (int i = lo; i < hi; ++i) {
            const int pi = (int)((perm >> (4 * i)) & 15);
            const uint32_t ka = float_key(micro_coord(P[pi], axis));
            int rank = 0;
            for (int j = lo; j < hi; ++j) {
                const int pj = (int)((perm >> (4 * j)) & 15);
                const uint32_t kb = float_key(micro_coord(P[pj], axis));
                rank += (kb < ka || (kb == ka && pj < pi)) ? 1 : 0;
            }
            if (rank == want) {
                pos = pi;
                kp = ka;
            }
        }
        // stable split: ranks below the pivot's first, then the pivot, then the ones above
        uint64_t left = 0, right = 0;
        int nl = 0, nr = 0;
        for (int i = lo; i < hi; ++i) {
            const int pi = (int)((perm >> (4 * i)) & 15);
            if (pi == pos) continue;
            const uint32_t kb = float_key(micro_coord(P[pi], axis));
            if (kb < kp || (kb == kp && pi < pos)) left |= (uint64_t)pi << (4 * nl++);
            else right |= (uint64_t)pi << (4 * nr++);
        }
        const uint64_t run = left | ((uint64_t)pos << (4 * nl)) | (right << (4 * (nl + 1)));
        const uint64_t mask = ((1ull << (4 * cnt)) - 1) << (4 * lo);
        perm = (perm & ~mask) | (run << (4 * lo));
        const int hl = nl > 0, hr = nr > 0;
        const int pair = (hl || hr) ? next_pair++ : 0;
        const uint32_t link = ((uint32_t)pair << LK_PAIR_SHIFT) | (hl ? LK_HASL : 0u) | (hr ? LK_HASR : 0u);
        const float4 P4 = P[pos];
        *reinterpret_cast<float4*>(pool.hot[node].f) = make_float4(P4.x, P4.y, P4.z, bitsf(link));
        pool.ids[node] = fbits(P4.w);
        pool.par[node] = parent;
        pool.cnt[node] = make_int4(cnt, 0, 0, depth);
        pool.meta[node] = (uint32_t)axis;
        const float box[6] = {mn[0], mn[1], mn[2], mx[0], mx[1], mx[2]};
        write_child_box_s(pool.hot, parent, node & 1, box);
        deepest = depth > deepest ? depth : deepest;
        const int lv = (rr >> 8) + 1;
        if (hr) {
            L.stk_r[nw][tid] = (lo + nl + 1) | (hi << 4) | (lv << 8);
            L.stk_node[nw][tid] = 2 * pair + 1;
            L.stk_par[nw][tid] = node;
            ++nw;
        }
        if (hl) {
            L.stk_r[nw][tid] = lo | ((lo + nl) << 4) | (lv << 8);
            L.stk_node[nw][tid] = 2 * pair;
            L.stk_par[nw][tid] = node;
            ++nw;
        }
    }
    atomicMax(&hdr->max_depth, deepest);
}

// The three shapes in one launch: the workgroups [0, nb_small) share the list
// of segments above TINY_MAX points, the wavefronts of the next nb_tiny the list
// of those above MICRO_MAX, and the lanes of the rest take one segment each.
__global__ __launch_bounds__(SMALL_SB) void k_build_segments(const float4* __restrict__ pts,
                                                             const int4* __restrict__ seg,
                                                             const int* __restrict__ seg_depth,
                                                             const int* __restrict__ pair_scan, int S,
                                                             const int* __restrict__ count_dev,
                                                             const int* __restrict__ lists,
                                                             const uint32_t* __restrict__ orig, SmallLists pre,
                                                             Pool pool, DevHdr* hdr, int nb_small, int nb_tiny) {
    __shared__ union {
        BuildLds<SMALL_SB, SMALL_MAX> small;
        BuildLds<64, TINY_MAX> tiny[TINY_WAVES];
        MicroLds micro;
    } lds;
    const int b = blockIdx.x;
    if (b < nb_small) {
        const int n = hdr->small_lists[1];
        for (int i = b; i < n; i += nb_small)
            build_segment<SMALL_SB, SMALL_MAX>(lds.small, lists[S + i], pts, seg, seg_depth, pair_scan, orig, pre, pool,
                                               hdr);
    } else if (b < nb_small + nb_tiny) {
        const int n = hdr->small_lists[0], w = threadIdx.x >> 6;
        for (int i = (b - nb_small) * TINY_WAVES + w; i < n; i += nb_tiny * TINY_WAVES)
            build_segment<64, TINY_MAX>(lds.tiny[w], lists[i], pts, seg, seg_depth, pair_scan, orig, pre, pool, hdr);
    } else {
        build_micro(lds.micro, (b - nb_small - nb_tiny) * MICRO_BS + (int)threadIdx.x, pts, seg, seg_depth, pair_scan,
                    S, count_dev, pool, hdr);
    }
}

static inline int blocks_for(long long n, int bs) { return (int)((n + bs - 1) / bs); }

bool small_plan_fits(int S) { return S <= PLAN_MAX; }
// the lane build follows the position tie rule only: presorted or
// original-order inputs go to the larger shapes
static int micro_ok(const uint32_t* orig, const SmallLists& pre) { return (!orig && !pre.inv0) ? 1 : 0; }

void launch_small_plan(const int4* seg, int S, const int* count_dev, const uint32_t* orig, const SmallLists& pre,
                       int* pair_scan, int* lists, DevHdr* hdr, hipStream_t s) {
    if (S <= 0) return;
    hipLaunchKernelGGL(k_small_plan, dim3(1), dim3(1024), 0, s, seg, S, count_dev, micro_ok(orig, pre), pair_scan,
                       lists, hdr);
}
void launch_small_pairs(const int4* seg, int S, const int* count_dev, const uint32_t* orig, const SmallLists& pre,
                        int* pairs, int* lists, DevHdr* hdr, hipStream_t s) {
    if (S <= 0) return;
    launch_fill_i32(hdr->small_lists, 0, 2, s);
    hipLaunchKernelGGL(k_small_pairs, dim3(blocks_for(S, 256)), dim3(256), 0, s, seg, S, count_dev, micro_ok(orig, pre),
                       pairs, lists, hdr);
}
void launch_small_commit(const int* pairs, const int* pair_scan, int S, DevHdr* hdr, hipStream_t s) {
    if (S <= 0) return;
    hipLaunchKernelGGL(k_small_commit, dim3(1), dim3(1), 0, s, pairs, pair_scan, S, hdr);
}
void launch_build_small(const float4* pts, const int4* seg, const int* seg_depth, const int* pair_scan, int S,
                        const int* count_dev, const uint32_t* orig, SmallLists pre, const int* lists, Pool pool,
                        DevHdr* hdr, hipStream_t s) {
    if (S <= 0) return;
    // wide enough to fill the device when a list is long
    const int nb_small = std::min(S, 512), nb_tiny = std::min(blocks_for(S, TINY_WAVES), 512);
    const int nb_micro = micro_ok(orig, pre) ? blocks_for(S, MICRO_BS) : 0;
    hipLaunchKernelGGL(k_build_segments, dim3(nb_small + nb_tiny + nb_micro), dim3(SMALL_SB), 0, s, pts, seg, seg_depth,
                       pair_scan, S, count_dev, lists, orig, pre, pool, hdr, nb_small, nb_tiny);
}

}  // namespace ikd
