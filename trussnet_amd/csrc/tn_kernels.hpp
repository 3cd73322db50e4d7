// tn_kernels.hpp -- the relaxation's gfx950 kernels.
//
// Rebuild (src/v2m_particles.cpp:771-820): k_keys (cell key + count per cell),
// k_scan_* (exclusive scan: cell starts), k_place and k_permute (the nodes renumbered in
// cell order), k_brick_count and k_brick_order (the order of the searches), k_truss (each
// node's candidates, one wave per 64 nodes), k_lists (the K nearest of them in order).
// Iteration (src/v2m_particles.cpp:828-947): k_force, k_move_easy + k_move,
// k_stats (histogram, max, Verlet count, refresh flags, FIRE power partial sums),
// k_truss_node (own-list refresh of the nodes past a full skin, which k_stats lists),
// k_control (one block: FIRE's update, p99, the stop and rebuild decisions).
//
// Node slots: at every rebuild the nodes are renumbered in cell order (slot t holds
// the node at old slot sorted[t]), so a wave's nodes, their list entries and their
// neighbours lie close in memory. id[t] is the node's index in the caller's arrays:
// it orders equal distances in the K-lists, as the reference's node index does, and
// places the results; slot_of is its inverse. The lists hold slots.
#pragma once

#include "tn_device.hpp"

namespace tnk {

using namespace tnd;

constexpr int kWave = 64;
constexpr int kBlock = 256;

// The device control block: per-iteration accumulators, FIRE's state and the
// loop decisions. The host reads its head after each iteration.
struct Ctl {
    // decisions and stats (read back by the host)
    int32_t it;            // iterations done
    int32_t done;          // converged: the loop stops
    int32_t rebuild;       // a rebuild is due before the next iteration
    int32_t rebuilds;
    float last_move, last_p99;
    int32_t fire_resets;
    float fire_dt;
    int32_t zero_v;        // FIRE reset: the next move reads every velocity as zero
    int32_t power_fallbacks;   // iterations whose power sign needed the serial sum
    int32_t nrefresh;      // nodes queued for an own-list refresh this iteration
    int32_t nhalf;         // nodes past skin/2 (this iteration)
    int32_t nmove;         // interface nodes queued for the trapped step (this iteration)
    int32_t nmove_int;     // interior nodes queued for the trapped step (crossing or in snap range)
    int32_t nmove_rest;    // other nodes queued for the general trapped step (this iteration)
    int32_t nmove_def;     // nodes a lean pass handed to the general step (this iteration)
    int32_t moved_rest;    // nmove_rest as of the end of the moves (the count itself is then cleared)
    // FIRE (FireCtl, src/v2m_particles.h:47-76)
    float dt0, dt, dtmax, alpha;
    int32_t npos;
    // accumulators, cleared by k_control
    uint32_t hist[32];
    uint32_t mmax_bits;
    int32_t order_cnt[4];  // node counts by type rank (interface, junction, interior, corner)
    double power;
};

// ---- small utilities ------------------------------------------------------------

__global__ void k_fill_i32(int32_t* __restrict__ a, int64_t m, int32_t v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m) {
        a[i] = v;
    }
}

__device__ __forceinline__ uint64_t lanemask_lt() {
    const int lane = threadIdx.x & (kWave - 1);
    return lane ? (~0ull >> (kWave - lane)) : 0ull;
}

// exclusive scan of one int per thread over a 256-thread block; *total = block sum
__device__ __forceinline__ int block_excl_scan(int v, int* lds4, int* total) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int y = __shfl_up(x, d, kWave);
        if (lane >= d) {
            x += y;
        }
    }
    if (lane == kWave - 1) {
        lds4[w] = x;
    }
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int k = 0; k < kBlock / kWave; ++k) {
        const int s = lds4[k];
        base += k < w ? s : 0;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return base + x - v;
}

// ---- smallest and largest of an array ---------------------------------------------

// mm[0]: the smallest of a, mm[1]: the largest of a and 0 (kPositive: of its positive
// values), as float bits in signed-integer order; start from { +inf's bits, 0 }. NaNs are
// passed over. Each block reduces its share in registers and adds one pair of atomics: an
// atomic a value, all to two words, took 5.9 ms for 16.8 M values where this streams them
// in 0.03 ms.
__device__ __forceinline__ int32_t ordered_bits(float v) {
    const int32_t b = (int32_t)__float_as_uint(v);
    return b ^ ((b >> 31) & 0x7FFFFFFF);
}

template <bool kPositive>
__global__ __launch_bounds__(kBlock) void k_minmax(const float* __restrict__ a, int64_t n, int32_t* __restrict__ mm) {
    __shared__ float lds[2][kBlock / kWave];
    float lo = __builtin_huge_valf(), hi = 0.0f;
    const int64_t step = (int64_t)gridDim.x * kBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += step) {
        const float v = a[i];
        if (!kPositive || v > 0.0f) {
            lo = fminf(lo, v);
            hi = fmaxf(hi, v);
        }
    }
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, d, kWave));
        hi = fmaxf(hi, __shfl_xor(hi, d, kWave));
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & (kWave - 1)) == 0) {
        lds[0][w] = lo;
        lds[1][w] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < kBlock / kWave; ++k) {
            lo = fminf(lo, lds[0][k]);
            hi = fmaxf(hi, lds[1][k]);
        }
        atomicMin(&mm[0], ordered_bits(lo));
        atomicMax(&mm[1], ordered_bits(hi));
    }
}

constexpr int kMinmaxGrid = 1024;   // blocks at most (4 a CU)

// ---- exclusive scan (int32), tiles of 4096 ----------------------------------------

constexpr int kScanItems = 16;
constexpr int kScanTile = kBlock * kScanItems;
constexpr int kScanTiles = 1024;   // tiles whose sums every block may add up itself (4 a thread)

__global__ __launch_bounds__(kBlock) void k_scan_reduce(const int32_t* __restrict__ in, int64_t m,
                                                        int32_t* __restrict__ bsum) {
    __shared__ int lds4[4];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        s += base + k < m ? in[base + k] : 0;
    }
    int tot;
    block_excl_scan(s, lds4, &tot);
    if (threadIdx.x == 0) {
        bsum[blockIdx.x] = tot;
    }
}

// one block: exclusive scan of the tile sums in place, chunk by chunk
__global__ __launch_bounds__(kBlock) void k_scan_top(int32_t* __restrict__ bsum, int64_t nb) {
    __shared__ int lds4[4];
    int carry = 0;
    for (int64_t c0 = 0; c0 < nb; c0 += kScanTile) {
        const int64_t base = c0 + (int64_t)threadIdx.x * kScanItems;
        int v[kScanItems];
        int s = 0;
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            v[k] = base + k < nb ? bsum[base + k] : 0;
            s += v[k];
        }
        int tot;
        int run = carry + block_excl_scan(s, lds4, &tot);
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            if (base + k < nb) {
                bsum[base + k] = run;
            }
            run += v[k];
        }
        carry += tot;
    }
}

// kTop: bsum holds the tiles' sums, not their scan, and each block adds up the ones
// before its own (at most kScanTiles of them: a launch fewer, and cheaper than the one
// block that would scan them)
template <bool kTop>
__global__ __launch_bounds__(kBlock) void k_scan_down(const int32_t* in, int32_t* out, int64_t m,
                                                      const int32_t* __restrict__ bsum) {
    __shared__ int lds4[4];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    int v[kScanItems];
    int s = 0, before = 0;
    if (kTop) {
        int part = 0;
        for (unsigned k = threadIdx.x; k < blockIdx.x; k += kBlock) {
            part += bsum[k];
        }
        block_excl_scan(part, lds4, &before);
    } else {
        before = bsum[blockIdx.x];
    }
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = base + k < m ? in[base + k] : 0;
        s += v[k];
    }
    int tot;
    int run = before + block_excl_scan(s, lds4, &tot);
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        if (base + k < m) {
            out[base + k] = run;
        }
        run += v[k];
    }
}

// ---- keys (v2m_h_at + v2m_level_of + v2m_bin_key; count per cell) ---------------

// X.w is v2m_h_at at the node (set with every move), the size the rebuild takes.
// The nodes sit in cell order from the previous rebuild, so neighbouring lanes
// mostly share a key: each run of equal keys in a wave adds its length at once, and its
// nodes take the places in their cell that the count stood at (in arrival order: k_permute
// puts a cell's nodes in slot order).
__global__ __launch_bounds__(kBlock) void k_keys(Hash H, const float4* __restrict__ X, int n, float tskin,
                                                 int32_t* __restrict__ key, int32_t* __restrict__ cnt,
                                                 int32_t* __restrict__ place) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const int lane = threadIdx.x & (kWave - 1);
    const bool valid = i < n;
    int k = -1;
    if (valid) {
        const float4 x = X[i];
        k = cell_key(H, level_for(H, tskin * x.w), x.x, x.y, x.z);
        key[i] = k;
    }
    const int prev = __shfl_up(k, 1, kWave);
    const bool head = valid && (lane == 0 || prev != k);
    const uint64_t heads = __ballot(head);
    const int nvalid = __popcll(__ballot(valid));   // the valid lanes are a prefix
    int at = 0;
    if (head) {
        const uint64_t later = lane == kWave - 1 ? 0ull : heads & (~0ull << (lane + 1));
        const int end = later ? __ffsll((long long)later) - 1 : nvalid;
        at = atomicAdd(&cnt[k], end - lane);
    }
    if (valid) {   // (lane 0 is a head: every lane has one at or below it)
        const int first = 63 - __clzll((long long)(heads & (~0ull >> (kWave - 1 - lane))));
        place[i] = __shfl(at, first, kWave) + lane - first;
    }
}

// The slots gathered by cell: slot i to its cell's start plus its place there.
__global__ __launch_bounds__(kBlock) void k_place(const int32_t* __restrict__ key, const int32_t* __restrict__ place,
                                                  const int32_t* __restrict__ cstart, int n,
                                                  int32_t* __restrict__ bycell) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) {
        bycell[cstart[key[i]] + place[i]] = i;
    }
}

// ---- the K-nearest search's query order ------------------------------------------
//
// k_truss serves the nodes a wave at a time. In slot order (cells in x-fastest row
// order) a wave's 64 nodes lie along a row of cells, and the union of their scan
// boxes is long; taken brick by brick instead (4 x 4 x 4 cells of a level, cells
// z, y, x within a brick, bricks in x-fastest order) they are compact, and the union,
// which a wave loads and tests as a whole, is about a quarter smaller. The order is a
// counting sort of the slots by brick position: a cell's slots stay contiguous.

constexpr int kBrickEdge = 4;
static_assert(kBrickEdge == 4, "k_brick_count takes a position apart in 2-bit fields");

struct BrickMap {
    int nb[TN_MAXLEV][3];   // bricks per axis at each level
    int off[TN_MAXLEV];     // each level's first position (64 a brick)
    int size;               // positions in all
};

// the brick-order position of cell key k
__device__ __forceinline__ int brick_pos(const Hash& H, const BrickMap& B, int k) {
    int L = 0;
    while (L + 1 < H.nlev && k >= H.off[L + 1]) {
        ++L;
    }
    const int local = k - H.off[L], nx = H.dim[L][0], ny = H.dim[L][1];
    const int cx = local % nx, cy = (local / nx) % ny, cz = local / (nx * ny);
    const int brick = (cx / kBrickEdge) + B.nb[L][0] * ((cy / kBrickEdge) + B.nb[L][1] * (cz / kBrickEdge));
    const int within = (cx % kBrickEdge) + kBrickEdge * ((cy % kBrickEdge) + kBrickEdge * (cz % kBrickEdge));
    return B.off[L] + brick * (kBrickEdge * kBrickEdge * kBrickEdge) + within;
}

// the node count of each brick-order position's cell (0 at a position of no cell and at
// the end), every position written
__global__ __launch_bounds__(kBlock) void k_brick_count(Hash H, BrickMap B, const int32_t* __restrict__ cstart,
                                                        int32_t* __restrict__ cnt) {
    const int pos = blockIdx.x * kBlock + threadIdx.x;
    if (pos > B.size) {
        return;
    }
    int c = 0;
    if (pos < B.size) {
        int L = 0;
        while (L + 1 < H.nlev && pos >= B.off[L + 1]) {
            ++L;
        }
        const int within = (pos - B.off[L]) & 63, brick = (pos - B.off[L]) >> 6;
        const int bx = brick % B.nb[L][0], by = (brick / B.nb[L][0]) % B.nb[L][1], bz = brick / (B.nb[L][0] * B.nb[L][1]);
        const int cx = bx * kBrickEdge + (within & 3), cy = by * kBrickEdge + ((within >> 2) & 3),
                  cz = bz * kBrickEdge + (within >> 4);
        if (cx < H.dim[L][0] && cy < H.dim[L][1] && cz < H.dim[L][2]) {
            const int k = H.off[L] + cx + H.dim[L][0] * (cy + H.dim[L][1] * cz);
            c = cstart[k + 1] - cstart[k];
        }
    }
    cnt[pos] = c;
}

// the slots in brick order: slot s goes to its cell's start in that order plus its rank
// in the cell (start: the exclusive scan of k_brick_count's counts)
__global__ __launch_bounds__(kBlock) void k_brick_order(Hash H, BrickMap B, const int32_t* __restrict__ key, int n,
                                                        const int32_t* __restrict__ cstart,
                                                        const int32_t* __restrict__ start,
                                                        int32_t* __restrict__ order) {
    const int s = blockIdx.x * kBlock + threadIdx.x;
    if (s < n) {
        const int k = key[s];
        order[start[brick_pos(H, B, k)] + (s - cstart[k])] = s;
    }
}

// ---- stable LSD radix sort of (key, id) by key, 8-bit digits --------------------------

constexpr int kRadixItems = 8;
constexpr int kRadixTile = kBlock * kRadixItems;

__global__ __launch_bounds__(kBlock) void k_radix_hist(const int32_t* __restrict__ keys, int n, int shift, int nblk,
                                                       int32_t* __restrict__ bhist) {
    __shared__ int lh[256];
    lh[threadIdx.x] = 0;
    __syncthreads();
    const int base = blockIdx.x * kRadixTile;
#pragma unroll
    for (int it = 0; it < kRadixItems; ++it) {
        const int e = base + it * kBlock + threadIdx.x;
        if (e < n) {
            atomicAdd(&lh[(keys[e] >> shift) & 255], 1);
        }
    }
    __syncthreads();
    bhist[(size_t)threadIdx.x * nblk + blockIdx.x] = lh[threadIdx.x];
}

// Scatter one tile: element order within the tile is (round, thread), and each
// element's rank among equal digits counts the earlier ones -- a stable pass.
// vals_in == nullptr: the values are the element indices (the node ids).
__global__ __launch_bounds__(kBlock) void k_radix_scatter(const int32_t* __restrict__ keys_in,
                                                          const int32_t* __restrict__ vals_in, int n, int shift,
                                                          int nblk, const int32_t* __restrict__ offs,
                                                          int32_t* __restrict__ keys_out,
                                                          int32_t* __restrict__ vals_out) {
    __shared__ int goff[256];
    __shared__ int run[256];
    __shared__ int wcnt[kBlock / kWave][256];
    const int tid = threadIdx.x, w = tid >> 6;
    goff[tid] = offs[(size_t)tid * nblk + blockIdx.x];
    run[tid] = 0;
    const int base = blockIdx.x * kRadixTile;
    const uint64_t below = lanemask_lt();
    for (int it = 0; it < kRadixItems; ++it) {
        const int e = base + it * kBlock + tid;
        const bool valid = e < n;
        const int key = valid ? keys_in[e] : 0;
        const int val = valid ? (vals_in ? vals_in[e] : e) : 0;
        const int d = valid ? ((key >> shift) & 255) : 256;
        // lanes of this wave holding the same digit (9 bits: 256 = no element)
        uint64_t peers = ~0ull;
#pragma unroll
        for (int b = 0; b < 9; ++b) {
            const uint64_t bal = __ballot((d >> b) & 1);
            peers &= ((d >> b) & 1) ? bal : ~bal;
        }
        const int rank_w = __popcll(peers & below);
#pragma unroll
        for (int k = 0; k < kBlock / kWave; ++k) {
            wcnt[k][tid] = 0;
        }
        __syncthreads();
        if (valid && rank_w == 0) {
            wcnt[w][d] = __popcll(peers);
        }
        __syncthreads();
        {
            int acc = run[tid];
#pragma unroll
            for (int k = 0; k < kBlock / kWave; ++k) {
                const int c = wcnt[k][tid];
                wcnt[k][tid] = acc;
                acc += c;
            }
            run[tid] = acc;
        }
        __syncthreads();
        if (valid) {
            const int pos = goff[d] + wcnt[w][d] + rank_w;
            keys_out[pos] = key;
            vals_out[pos] = val;
        }
        __syncthreads();
    }
}

// ---- renumbering in cell order ---------------------------------------------------------

// The nodes renumbered in cell order, a cell's nodes by their old slots: the stable sort
// by key. bycell holds each cell's old slots in arrival order (k_place), and a node's rank
// among them (read from LDS) is its place: two launches where the radix sort this
// replaces took three passes of five (2.5 M nodes: 126 us of sorting and 66 of renumbering
// a rebuild before, 11 and 80 now; 3 k nodes: 37 and 6, now 6 and 7). The rank costs a
// comparison for every node of the cell, so it grows with the square of a cell's nodes as
// their search does. A cell longer than the window is read by the block together, tile by
// tile, which keeps it a tenth of the search's time or less: 495 k nodes that the voxel
// trap stacks up (hundreds in a cell) 103 -> 29 us, each node reading the cell's places by
// itself -> tiles; 100 k nodes of a few cells 4.24 -> 0.66 ms, their search 7.0.
// Ps and P0 (the positions as of this rebuild) and Ms (id, typ | lab << 8) are written in
// the new order, and keyS the nodes' keys.
struct NodeArrays {
    float4* X;
    float4* V;
    uint8_t* typ;
    uint32_t* part;
    uint16_t* lab;
    int32_t* id;
    uint8_t* sticky;   // handed back to the general move pass before (may be null)
};

__global__ __launch_bounds__(kBlock) void k_permute(const int32_t* __restrict__ bycell,
                                                    const int32_t* __restrict__ key,
                                                    const int32_t* __restrict__ cstart, int n, NodeArrays in,
                                                    NodeArrays out, float4* __restrict__ Ps,
                                                    float4* __restrict__ P0, int2* __restrict__ Ms,
                                                    int32_t* __restrict__ slot_of, int32_t* __restrict__ keyS) {
    constexpr int kSide = kBlock / 2, kTile = 2 * kBlock;
    __shared__ __align__(16) int near[kTile];   // bycell around the block: most cells' slots; then tiles
    __shared__ int reach[2];                    // where the first node's cell begins, where the last one's ends
    const int tid = threadIdx.x, p0 = blockIdx.x * kBlock, p = p0 + tid, n0 = p0 - kSide, n1 = n0 + kTile;
    for (int j = tid; j < kTile; j += kBlock) {
        near[j] = n0 + j >= 0 && n0 + j < n ? bycell[n0 + j] : 0;
    }
    __syncthreads();
    int s = 0, k = 0, b = 0, e = 0, t = 0;
    if (p < n) {
        s = near[kSide + tid];
        k = key[s];
        b = cstart[k];
        e = cstart[k + 1];
        const int b1 = max(b, n0), e1 = min(e, n1);
        t = b;
#pragma unroll 4
        for (int q = b1; q < e1; ++q) {
            t += near[q - n0] < s ? 1 : 0;
        }
    }
    if (tid == 0) {
        reach[0] = b;
    }
    if (p == min(n, p0 + kBlock) - 1) {
        reach[1] = e;
    }
    __syncthreads();
    // the slots of a long cell at places q0 .. q1 - 1, outside the window (all threads of the
    // block; mine: of this node's cell, the one that reaches out of the window on that side)
    auto beyond = [&](int q0, int q1, bool mine) {
        for (int at = q0; at < q1; at += kTile) {
            for (int j = tid; j < kTile; j += kBlock) {
                near[j] = at + j < q1 ? bycell[at + j] : INT_MAX;
            }
            __syncthreads();
            if (mine) {
                const int4* tile = reinterpret_cast<const int4*>(near);
                const int m = (min(kTile, q1 - at) + 3) / 4;
#pragma unroll 4
                for (int j = 0; j < m; ++j) {
                    const int4 v = tile[j];
                    t += (v.x < s ? 1 : 0) + (v.y < s ? 1 : 0) + (v.z < s ? 1 : 0) + (v.w < s ? 1 : 0);
                }
            }
            __syncthreads();
        }
    };
    beyond(reach[0], n0, b < n0);
    beyond(n1, reach[1], e > n1);
    if (p < n) {
        keyS[t] = k;
        const float4 x = in.X[s];
        out.X[t] = x;
        Ps[t] = x;
        P0[t] = x;
        out.V[t] = in.V[s];
        const int ty = in.typ[s];
        out.typ[t] = (uint8_t)ty;
        out.part[t] = in.part[s];
        const int l = in.lab[s];
        out.lab[t] = (uint16_t)l;
        const int o = in.id[s];
        out.id[t] = o;
        if (in.sticky) {
            out.sticky[t] = in.sticky[s];
        }
        Ms[t] = make_int2(o, ty | (l << 8));
        slot_of[o] = t;
    }
}

// ---- K-nearest lists, one wave per 64 nodes in cell order ----------------------------
//
// v2m_neighbors (src/opencl/v2m_particle_body.cl:73-151) for 64 query nodes at once.
// The queries are consecutive in cell order, so their scan boxes overlap. Per group
// of lanes (one cell row, a bounded span along it) the wave lists the rows of the
// union of its lanes' boxes over their levels (rows no lane reaches are skipped),
// reads all their cell starts at once, and tests the concatenation of the rows'
// candidates in full chunks of 64 staged in LDS: a distance prefilter on the
// matrix cores, then for every possible hit of a lane that scans the candidate's
// row the reference's exact test and its other checks (not the node itself, no
// interior bar across labels): in k_lists, or here once a buffer fills, which is then cut
// back to its 24 best. k_lists keeps the first 24 in (distance, id) order. The list equals
// the reference's:
// its K smallest valid candidates in (distance, id) order, of those in the cells of the
// lane's own box, the reference's scan region. Where every node's reach fits its level's
// cell (H.prune) a bar ends inside the box but for the rounding of the two reaches, so
// only a bar that could be past it by that (kDoubtful) is asked for its cells; otherwise
// every one is.

constexpr int kTrussWave = 64;   // one wave per block
constexpr int kCollect = 32;   // per-lane candidate buffer (entries): half a wave's lanes hold one when it is cut back
// waves a SIMD: 160 registers and no spill (at 4, 128 registers, 2.5 M nodes took longer)
constexpr int kTrussOcc = 3;
constexpr int kMinRoom = 4;    // a lane with less room than this (and more possible hits) settles first

// ---- wave-wide reductions and scans on DPP (64 lanes, all active) ----------------
//
// Each step combines a lane with a lane of its row (16 lanes) through the data-
// parallel-primitives operand modifier, then rows with row broadcasts (lane 15 of a
// row into the next, lane 31 into the upper two), so the reduction never touches LDS.
// dpp_ctrl: quad_perm [1,0,3,2] 0xB1, [2,3,0,1] 0x4E; row_shr:k 0x110 + k;
// row_mirror 0x140, row_half_mirror 0x141; row_bcast:15 0x142, row_bcast:31 0x143.

template <int kCtrl, int kRowMask = 0xF>
__device__ __forceinline__ int dpp(int old, int v) {
    return __builtin_amdgcn_update_dpp(old, v, kCtrl, kRowMask, 0xF, false);
}

// the reduction of v over the wave under op (commutative, idempotent), as a uniform value
template <typename Op>
__device__ __forceinline__ int wave_reduce(int v, Op op) {
    v = op(v, dpp<0xB1>(v, v));
    v = op(v, dpp<0x4E>(v, v));
    v = op(v, dpp<0x141>(v, v));
    v = op(v, dpp<0x140>(v, v));
    v = op(v, dpp<0x142, 0xA>(v, v));
    v = op(v, dpp<0x143, 0xC>(v, v));
    return __builtin_amdgcn_readlane(v, kWave - 1);
}

__device__ __forceinline__ int wave_min(int v) {
    return wave_reduce(v, [](int a, int b) { return min(a, b); });
}

__device__ __forceinline__ int wave_max(int v) {
    return wave_reduce(v, [](int a, int b) { return max(a, b); });
}

// the largest of non-negative floats (their bits order as unsigned integers do)
__device__ __forceinline__ float wave_max_nonneg(float v) {
    return __uint_as_float((uint32_t)wave_reduce((int)__float_as_uint(v), [](int a, int b) {
        return (int)max((uint32_t)a, (uint32_t)b);
    }));
}

// exclusive prefix sum over the wave; *total: the sum of all lanes
__device__ __forceinline__ int wave_excl_scan(int v, int lane, int* total) {
    (void)lane;
    int x = v;
    x += dpp<0x111>(0, x);   // row_shr: a lane with no source adds 0
    x += dpp<0x112>(0, x);
    x += dpp<0x114>(0, x);
    x += dpp<0x118>(0, x);
    x += dpp<0x142, 0xA>(0, x);
    x += dpp<0x143, 0xC>(0, x);
    *total = __builtin_amdgcn_readlane(x, kWave - 1);
    return x - v;
}

// (distance, id) order of the K-list (src/opencl/v2m_particle_body.cl:128-141)
__device__ __forceinline__ bool before(float da, int ja, float db, int jb) {
    return da < db || (da == db && ja < jb);
}

// A list entry as one 64-bit key: the distance's bits above the id. Distances are
// >= +0, whose bits order as the floats do, so the keys order as (distance, id), the
// K-list's order (src/opencl/v2m_particle_body.cl:128-141).
__device__ __forceinline__ uint64_t list_key(float d, int id) {
    return ((uint64_t)__float_as_uint(d) << 32) | (uint32_t)id;
}

// Sort N <= 32 keys in registers: Batcher's odd-even merge network for 32, less the
// comparators that reach past N (K. E. Batcher, Sorting networks and their applications,
// AFIPS 1968), every index known at compile time (24: 132 comparators, 32: 191).
template <int N>
__device__ __forceinline__ void merge_sort(uint64_t (&k)[32]) {
    static_assert(N <= 32, "the network is for 32 keys");
#pragma unroll
    for (int p = 1; p < 32; p <<= 1) {
#pragma unroll
        for (int d = p; d > 0; d >>= 1) {
#pragma unroll
            for (int i = 0; i + d < N; ++i) {
                // (i, i + d) is a comparator: i in the first half of its pair of runs of d
                // (offset by d % p), both in one block of 2 p
                if (i >= d % p && ((i - d % p) / d) % 2 == 0 && i / (2 * p) == (i + d) / (2 * p)) {
                    const uint64_t x = k[i], y = k[i + d];
                    const bool swap = x > y;
                    k[i] = swap ? y : x;
                    k[i + d] = swap ? x : y;
                }
            }
        }
    }
}

// ---- settling a few lanes' buffers with the whole wave -----------------------------------
//
// When only some lanes' buffers are full, the wave cuts them back two at a time, one per
// half-wave: lane i of a half holds entry i of its buffer, and its key's rank among the 32
// (they differ) is counted against all of them, broadcast from LDS. The 32 comparisons do
// not wait for each other, as the 15 steps of a sorting network do: waves of stacked nodes,
// the last of a launch to end, spend most of their time here (495 k nodes in the voxel
// field: 2.31 -> 2.23 ms a rebuild).

__device__ __forceinline__ uint64_t readlane64(uint64_t v, int l) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), l);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ float readlane_f(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// The reference looks for the other ends at level L in the cells from that of p - r to that
// of p + r along each axis, r = ((t + skin) h_i + b_L) / 2. An end at most r from p has its
// cell among them (rounding keeps order, so p + r does not round below it); past r, the
// 32-bit difference is at least r and d^2 at least r^2 as rounded. A bar has d^2 < rj^2, rj =
// (t + skin) / 2 (h_i + h_j), and b_L >= (t + skin) h_j as rounded: r >= rj (1 - 4 u), u =
// 2^-24, so a bar past the cells has d^2 >= rj^2 (1 - 11 u), the squares' and the product's
// own roundings counted. The bars from kDoubtful rj^2 on (32 u) are asked for their cells.
constexpr float kDoubtful = 1.0f - 0x1p-19f;

// whether the candidate c at level L lies in the reference's scan region of the node at
// (x, y, z) of reach R (v2m_neighbors, src/opencl/v2m_particle_body.cl:73-151)
__device__ __forceinline__ bool in_region(const Hash& H, int L, float x, float y, float z, float R, float4 c) {
    const float r = 0.5f * (R + H.b0 * (float)(1 << L));
    const int cx = cell_coord(H, L, c.x, H.ox, 0), cy = cell_coord(H, L, c.y, H.oy, 1), cz = cell_coord(H, L, c.z, H.oz, 2);
    return cx >= cell_coord(H, L, x - r, H.ox, 0) && cx <= cell_coord(H, L, x + r, H.ox, 0) &&
           cy >= cell_coord(H, L, y - r, H.oy, 1) && cy <= cell_coord(H, L, y + r, H.oy, 1) &&
           cz >= cell_coord(H, L, z - r, H.oz, 2) && cz <= cell_coord(H, L, z + r, H.oz, 2);
}

// A wave's queries, lane by lane (the search's view of its 64 nodes).
struct WaveQueries {
    float px, py, pz, h;   // position and size
    int slot;
};

// Cut the slot buffers of the lanes in sm (wave-uniform) back to their best 24 bars (in
// order); their cnt becomes the bars left and kth the 24th key when there are 24. All
// lanes take part: the exact test and the keys are formed from the slots, relative to the
// owner's query.
__device__ __forceinline__ void settle_slot_lanes(uint32_t* cb, uint64_t* keys, int lane, uint64_t sm, int& cnt, uint64_t& kth,
                                                  const float4* __restrict__ Ps, const int2* __restrict__ Ms,
                                                  const WaveQueries& Q, const Hash& H, float half) {
    // the pair of lanes settled next, with its entries already on their way while the pair
    // before it is sorted (a wave of stacked nodes settles a hundred times in a row)
    const bool lo = lane < 32;
    const int i = lane & 31;
    int a = 0, b = 0, sl = 0, id = 0;
    bool in = false;
    float4 c = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    auto next = [&]() {
        a = __builtin_ctzll(sm);
        sm &= sm - 1;
        b = sm ? __builtin_ctzll(sm) : a;
        sm &= sm ? sm - 1 : 0ull;
        const int ca = __builtin_amdgcn_readlane(cnt, a), cb_n = __builtin_amdgcn_readlane(cnt, b);
        in = i < (lo ? ca : cb_n);
        sl = in ? (int)cb[i * kTrussWave + (lo ? a : b)] : 0;
        c = Ps[sl];
        id = Ms[sl].x;
    };
    next();
    for (;;) {
        const int a0 = a, b0 = b;
        const float xa = readlane_f(Q.px, a), ya = readlane_f(Q.py, a), za = readlane_f(Q.pz, a), ha = readlane_f(Q.h, a);
        const float xb = readlane_f(Q.px, b), yb = readlane_f(Q.py, b), zb = readlane_f(Q.pz, b), hb = readlane_f(Q.h, b);
        const int qa = __builtin_amdgcn_readlane(Q.slot, a), qb = __builtin_amdgcn_readlane(Q.slot, b);
        const float ex = c.x - (lo ? xa : xb), ey = c.y - (lo ? ya : yb), ez = c.z - (lo ? za : zb);
        const float d2 = ex * ex + ey * ey + ez * ez;
        const float rj = half * ((lo ? ha : hb) + c.w), rj2 = rj * rj;
        bool bar = in && d2 < rj2 && sl != (lo ? qa : qb);
        if (bar && d2 >= kDoubtful * rj2) {
            const float T = 2.0f * half;
            bar = in_region(H, level_for(H, T * c.w), lo ? xa : xb, lo ? ya : yb, lo ? za : zb, T * (lo ? ha : hb), c);
        }
        uint64_t v = bar ? list_key(sqrtf(d2), id) : ~0ull;
        int slot = sl;
        const bool more = sm != 0;
        if (more) {   // (of other lanes than a0 and b0: their columns are not written below)
            next();
        }
        keys[lane] = v;
        __syncthreads();
        const ulonglong2* mine = reinterpret_cast<const ulonglong2*>(keys + (lane & 32));
        int rank = 0;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const ulonglong2 k = mine[e];
            rank += (k.x < v ? 1 : 0) + (k.y < v ? 1 : 0);
        }
        const bool bars1 = v != ~0ull;
        if (bars1 && rank < kK) {
            cb[rank * kTrussWave + (lo ? a0 : b0)] = (uint32_t)slot;
        }
        const uint64_t bars = __ballot(bars1), last = __ballot(bars1 && rank == kK - 1);
        const int na = __popcll(bars & 0xFFFFFFFFull), nb = __popcll(bars >> 32);
        const uint32_t la = (uint32_t)last, lb = (uint32_t)(last >> 32);
        const uint64_t ka = la ? readlane64(v, __ffs((int)la) - 1) : ~0ull;
        const uint64_t kb = lb ? readlane64(v, 32 + __ffs((int)lb) - 1) : ~0ull;
        if (lane == a0) {
            cnt = min(na, kK);
            kth = ka;
        }
        if (lane == b0) {
            cnt = min(nb, kK);
            kth = kb;
        }
        __syncthreads();   // the keys are read
        if (!more) {
            break;
        }
    }
}

// ---- the distance prefilter on the matrix cores ------------------------------------------
//
// For query p (this lane's node) and candidate c, with both taken relative to a
// wave-uniform origin and k = (t + skin) / 2, the exact test is d^2 < (k (h_p + h_c))^2.
// Its difference d^2 - k^2 (h_p + h_c)^2 is a dot product of two 6-vectors,
//   b_c = (-2c, -2 k^2 h_c, 1, |c|^2 - k^2 h_c^2),  a_p = (p, h_p, |p|^2 - k^2 h_p^2, 1),
// so the 64 x 64 differences of a chunk of candidates and a wave's queries come from
// four 32 x 32 tiles of v_mfma_f32_32x32x2f32 (three K-steps each), candidates along
// the rows and queries along the columns. A candidate whose difference is below a
// rounding margin is a possible hit; every possible hit is then tested exactly as
// before, so the prefilter only has to keep every true hit.
// (v_mfma_f32_32x32x2f32: lane l supplies A[l % 32][l / 32] and B[l / 32][l % 32];
// its output register e holds D[8 (e / 4) + 4 (l / 32) + e % 4][l % 32]. So in the
// tile of its own query's columns a lane holds half of the tile's candidate rows
// for its query, and lane l ^ 32 holds the other half.)
//
// Around the twelve matrix operations a chunk costs few others. The accumulators start at
// minus the margin, so that a possible hit is a sign bit, taken into the mask with one
// funnel shift each. Lane l holds candidate chunk_index(l), the one whose row makes the 16
// mask bits of either half of the wave 16 consecutive candidates. Operands and masks change
// halves with v_permlane32_swap. (With compares and selects a bit, the operands formed
// twice from LDS and the masks spread nibble by nibble, a chunk took about 450 vector
// instructions instead of 190.)

typedef float f32x16 __attribute__((ext_vector_type(16)));

// the candidate of the chunk that lane l holds, the lane that holds candidate k, and a
// mask of lanes as one of candidates (bits 2, 3 and 4 of the index change places)
__device__ __forceinline__ int chunk_index(int lane) {
    return (lane & 0x23) | ((lane & 4) << 2) | ((lane & 0x18) >> 1);
}
__device__ __forceinline__ int chunk_lane(int k) {
    return (k & 0x23) | ((k & 0x0C) << 1) | ((k & 0x10) >> 2);
}
__device__ __forceinline__ uint64_t by_index(uint64_t lanes) {
    // nibbles 8 a + 4 hh of each half to 4 a + 16 hh: even ones below, odd ones above
    const uint64_t lo = lanes & 0x0F0F0F0F0F0F0F0Full, hi = (lanes >> 4) & 0x0F0F0F0F0F0F0F0Full;
    auto pack = [](uint64_t x) {   // the low nibble of each byte, packed within each half
        x = (x | (x >> 4)) & 0x00FF00FF00FF00FFull;
        return (x | (x >> 8)) & 0x0000FFFF0000FFFFull;
    };
    return pack(lo) | (pack(hi) << 16);
}

// lanes 32..63 of a and lanes 0..31 of b exchanged
__device__ __forceinline__ void swap_halves(float& a, float& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(r[0]);
    b = __uint_as_float(r[1]);
}

// this lane's B operands: queries 32 c + l % 32 (c = the column tile), three K-steps
struct QueryOps {
    float b[2][3];
};

// the six components of a lane's query, K-index 2 t + l / 32: (k0, k1), (k2, k3), (k4, k5)
__device__ __forceinline__ QueryOps query_ops(float k0, float k1, float k2, float k3, float k4, float k5) {
    QueryOps o;
    swap_halves(k0, k1);
    swap_halves(k2, k3);
    swap_halves(k4, k5);
    o.b[0][0] = k0;
    o.b[1][0] = k1;
    o.b[0][1] = k2;
    o.b[1][1] = k3;
    o.b[0][2] = k4;
    o.b[1][2] = k5;
    return o;
}

// the signs of one output tile: bit e for register e
__device__ __forceinline__ uint32_t tile_signs(const f32x16& acc) {
    uint32_t m = 0;
#pragma unroll
    for (int e = 15; e >= 0; --e) {   // (m << 1) | sign
        m = __builtin_amdgcn_alignbit(m, __float_as_uint(acc[e]), 31);
    }
    return m;
}

// The 64-bit mask of this lane's query over the chunk's candidates whose dot product is
// below the margin, from lane l's operands of candidate chunk_index(l) (K-index 2 t and
// 2 t + 1 in a_t[0] and a_t[1])
__device__ __forceinline__ uint64_t tiles_below(const QueryOps& qo, float (&a0)[2], float (&a1)[2], float (&a2)[2],
                                                float margin) {
    swap_halves(a0[0], a0[1]);   // [r]: candidates of lanes 32 r .. 32 r + 31
    swap_halves(a1[0], a1[1]);
    swap_halves(a2[0], a2[1]);
    f32x16 start;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        start[e] = -margin;
    }
    uint32_t out[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {   // the row tile
        uint32_t bits[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {   // queries 32 c .. 32 c + 31 (the column tile)
            f32x16 acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a0[r], qo.b[c][0], start, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a1[r], qo.b[c][1], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a2[r], qo.b[c][2], acc, 0, 0, 0);
            bits[c] = tile_signs(acc);
        }
        // a lane's own column tile is l / 32: candidates 0..15 of the row tile from the lower
        // half's registers, 16..31 from the upper half's
        const auto x = __builtin_amdgcn_permlane32_swap(bits[0], bits[1], false, false);
        out[r] = x[0] | (x[1] << 16);
    }
    return ((uint64_t)out[1] << 32) | out[0];
}

// the 64-bit mask of this lane's query over the chunk's candidates (lane l's own:
// candidate chunk_index(l), at v) whose difference, relative to the origin o, is below
// the margin
__device__ __forceinline__ uint64_t chunk_hits(const QueryOps& qo, float4 v, float ox, float oy, float oz, float k2,
                                               float margin) {
    const bool some = v.x < __builtin_huge_valf();
    const float cx = v.x - ox, cy = v.y - oy, cz = v.z - oz;
    const float C = cx * cx + cy * cy + cz * cz - k2 * v.w * v.w;
    // K-index 2 t + l / 32: (-2 cx, -2 cy), (-2 cz, -2 k^2 h), (1, |c|^2 - k^2 h^2); past the
    // chunk's end an infinite difference, above the margin in any unit of length
    float a0[2] = { some ? -2.0f * cx : 0.0f, some ? -2.0f * cy : 0.0f };
    float a1[2] = { some ? -2.0f * cz : 0.0f, some ? -2.0f * k2 * v.w : 0.0f };
    float a2[2] = { some ? 1.0f : 0.0f, some ? C : __builtin_huge_valf() };
    return tiles_below(qo, a0, a1, a2, margin);
}

// The same for d^2 < near^2, near: this lane's 24th best distance so far. The terms of d^2 -
// near^2 are (-2c, 1, |c|^2) . (p, |p|^2 - near^2, 1), so it takes the same three steps. A
// wave of stacked nodes meets hundreds of possible bars a node of which a tenth comes
// before the node's 24th: only those are then tested one by one (495 k nodes moved in the
// voxel field, 48 rebuilds: k_truss and k_lists 3.02 -> 2.40 ms a rebuild).
__device__ __forceinline__ uint64_t chunk_near(float qx, float qy, float qz, float near2, float4 v, float ox, float oy,
                                               float oz, float margin) {
    const bool some = v.x < __builtin_huge_valf();
    const float cx = v.x - ox, cy = v.y - oy, cz = v.z - oz;
    const QueryOps qo = query_ops(qx, qy, qz, qx * qx + qy * qy + qz * qz - near2, 1.0f, 0.0f);
    float a0[2] = { some ? -2.0f * cx : 0.0f, some ? -2.0f * cy : 0.0f };
    float a1[2] = { some ? -2.0f * cz : 0.0f, some ? 1.0f : 0.0f };
    float a2[2] = { some ? cx * cx + cy * cy + cz * cz : __builtin_huge_valf(), 0.0f };
    return tiles_below(qo, a0, a1, a2, margin);
}

// The rows of one group, collected before any of their candidates is loaded: the
// cell-start reads of all rows are then issued together, and the candidates of all
// rows (and levels) are concatenated into full chunks.
constexpr int kMaxRanges = 64;


// The lists of all nodes at a rebuild: query q is the node in slot q. The buffers hold
// the candidates' slots (4 bytes): 12 KB of LDS a wave, so that 13 waves fit a CU. While
// no buffer of the wave has filled, every possible hit is appended as it is (93 of 100
// are bars) and the exact test is left to k_lists, which forms the distances anyway: a few
// instructions a hit, each lane its own. From the first full buffer on (nodes that stack
// up on the voxel faces, and the grids with no reach bound) a wave tests its possible hits
// as (query, candidate) pairs, one a lane, and takes in only what beats its query's 24th
// best so far. Rows of up to 32 slots leave the kernel: 24 in the list's own row, the rest
// in tail0 and tail1.
__global__ __launch_bounds__(kTrussWave, kTrussOcc) void k_truss(Hash H, TrussIn in, int n, int32_t* __restrict__ nbr,
                                                                      int4* __restrict__ tail0, int4* __restrict__ tail1,
                                                                      int32_t* __restrict__ nnb) {
    __shared__ float4 cpos[kTrussWave];   // the chunk's candidates: position, h
    __shared__ int cid[kTrussWave];       // their ids
    __shared__ int crow[kTrussWave];      // their row (index into the row table)
    // the row table of the current group: cell-start indices of the row's first cell and
    // one past its last, the lanes that scan the row, its level; after the cell starts
    // are read: the row's first slot and its position in the concatenation
    __shared__ int r_lev[kMaxRanges], r_sa[kMaxRanges], r_beg[kMaxRanges], r_len[kMaxRanges];
    // the rows' keys are read before any round: a settling's sort keys take their place, and a
    // round's (query lane, candidate) pairs
    __shared__ __align__(16) uint64_t r_keys[kMaxRanges];
    static_assert(kMaxRanges >= kTrussWave, "the pairs and sort keys share the row keys' array");
    int* const r_key0 = reinterpret_cast<int*>(r_keys);
    int* const r_key1 = r_key0 + kMaxRanges;
    int* const pairs = r_key0;
    __shared__ uint64_t r_mask[kMaxRanges];
    __shared__ uint32_t cb[kCollect * kTrussWave];   // the lanes' lists (candidate slots)
    __shared__ int cslot[kTrussWave];                // the chunk's candidates' slots
    const int lane = threadIdx.x;
    const float tskin = in.t + in.skin;
    const float half = tskin * 0.5f;   // (t + skin) * 0.5f * (hi + hj), left to right
    const float k2 = half * half;
    const float inf = __builtin_huge_valf();
    const int cidx = chunk_index(lane);
    for (int qb = blockIdx.x * kTrussWave; qb < n; qb += gridDim.x * kTrussWave) {
        const bool active = qb + lane < n;
        const int q = active ? in.order[qb + lane] : 0;   // the node in slot q
        float px = 0.0f, py = 0.0f, pz = 0.0f, hi = 0.0f, Ri = 0.0f;
        int Li = 0, ti_int = 0, li = 0;
        if (active) {   // the node in slot q (nodes are in cell order)
            const float4 xi = in.X[q];
            px = xi.x;
            py = xi.y;
            pz = xi.z;
            hi = xi.w;
            Ri = tskin * hi;
            Li = level_for(H, Ri);
            const int2 mi = in.Ms[q];
            ti_int = (mi.y & 0xFF) == TN_INTERIOR;
            li = mi.y >> 8;
        }
        // The lanes are served in groups that share their level and a row of bricks and lie
        // within one brick of the group's first lane along it, so that a group's union of
        // scan boxes stays tight (a wave of queries can straddle bricks).
        int grow = -1, gx = 0;
        if (active) {
            const int cy = cell_coord(H, Li, py, H.oy, 1), cz = cell_coord(H, Li, pz, H.oz, 2);
            grow = (Li << 26) | ((cz / kBrickEdge) << 13) | (cy / kBrickEdge);
            gx = cell_coord(H, Li, px, H.ox, 0) / kBrickEdge;
        }
        // the label of the wave's interior queries, if they have one in common
        const uint64_t qint = __ballot(ti_int != 0);
        const int wl = qint ? __builtin_amdgcn_readlane(li, __builtin_ctzll(qint)) : 0;
        const bool one_label = __ballot(ti_int && li != wl) == 0ull;
        bool pending = active;
        // The lane's buffer holds cnt keys; once it has been cut back to the 24 best, kth is
        // the 24th of them, and a candidate must come before it to enter.
        int cnt = 0;
        uint64_t kth = ~0ull;
        bool near = false;   // (wave-uniform: some lane has 24 bars, and kth bounds what it still takes)
        bool cut = !H.prune;   // (wave-uniform: some lane's buffer has been, or the pairs are needed anyway)
        const WaveQueries Q{ px, py, pz, hi, q };
        for (;;) {
            const uint64_t pm = __ballot(pending);
            if (!pm) {
                break;
            }
            const int lead = __ffsll((long long)pm) - 1;
            const int lrow = __shfl(grow, lead, kWave), lx = __shfl(gx, lead, kWave);
            const bool ingroup = pending && grow == lrow && abs(gx - lx) <= 1;
            pending = pending && !ingroup;
            // the prefilter's origin: the group's first query; its query operands
            const float gox = __shfl(px, lead, kWave), goy = __shfl(py, lead, kWave), goz = __shfl(pz, lead, kWave);
            const float qx = px - gox, qy = py - goy, qz = pz - goz;
            const float q2 = qx * qx + qy * qy + qz * qz;
            const QueryOps qops = query_ops(qx, qy, qz, hi, q2 - k2 * hi * hi, 1.0f);
            const float P2 = wave_max_nonneg(ingroup ? q2 : 0.0f), HP = wave_max_nonneg(ingroup ? hi : 0.0f);
            // The prefilter's margin, 2^-16 of a bound S on the terms of a true hit's difference:
            // its candidate lies within the bar's reach of the query, so |c| <= |p| + k (h_p +
            // h_c), and h_c is at most the grid's largest h. (A candidate farther off may be
            // misjudged either way: it is no hit, and the exact test says so.)
            const float hs = HP + H.hbig, Cmax = sqrtf(P2) + half * hs;
            const float margin = (2.0f * (P2 + Cmax * Cmax) + 2.0f * k2 * hs * hs) * (1.0f / 65536.0f);
            int nr = 0;   // rows in the table (wave-uniform)
            // Read the cell starts of the table's rows, then test the concatenation of their
            // candidates chunk by chunk: the distance prefilter on the matrix cores, then the
            // exact test and the reference's other checks for each possible hit of a lane
            // that scans the candidate's row; the valid ones are appended as (distance, id).
            auto flush = [&]() {
                __syncthreads();   // the table's rows are written
                int sa = 0, len = 0;
                if (lane < nr) {
                    sa = in.cstart[r_key0[lane]];
                    len = in.cstart[r_key1[lane]] - sa;
                }
                int total = 0;
                const int beg = wave_excl_scan(len, lane, &total);
                if (lane < nr) {
                    r_sa[lane] = sa;
                    r_beg[lane] = beg;
                    r_len[lane] = len;
                }
                const int rows = nr;
                nr = 0;
                __syncthreads();
                // The candidates of chunk base + 64 are loaded while chunk base is tested: always,
                // past the end slot 0's. (With the loads under a branch, the wait for the chunk's
                // own candidates has to hold on the path without them too, and waits for the loads
                // just issued: 2.5 M nodes 1.35 instead of 1.31 ms a rebuild.)
                int rfirst = 0;   // the row holding the loaded chunk's first candidate
                float4 npos;
                int2 nms;
                int nrow, nslot;
                bool nin;
                // Once a buffer has filled, the chunks left take their candidates evenly spread
                // over what is left of the concatenation, from sfirst on, sstep of them: in the
                // rows' order the distances fall as the scan comes up to a node, so that almost
                // every candidate beats the 24th so far and the buffers fill again and again (495 k
                // nodes in the voxel field: 2.25 -> 1.65 ms a rebuild).
                int sfirst = -1, sstep = 1;
                auto fetch = [&](int base) {
                    if (sfirst < 0 && near && H.prune) {
                        sfirst = base;
                        sstep = (total - base + kTrussWave - 1) / kTrussWave;
                    }
                    int p, lo;   // the candidate and its row: the last that starts at or before it
                    if (sfirst < 0) {
                        while (rfirst + 1 < rows && r_beg[rfirst + 1] <= base) {
                            ++rfirst;
                        }
                        p = base + cidx;
                        lo = rfirst;
                        while (lo + 1 < rows && r_beg[lo + 1] <= p) {
                            ++lo;
                        }
                    } else {
                        p = sfirst + cidx * sstep + (base - sfirst) / kTrussWave;
                        lo = 0;
                        for (int d = kMaxRanges / 2; d > 0; d >>= 1) {
                            lo = lo + d < rows && r_beg[lo + d] <= p ? lo + d : lo;
                        }
                    }
                    nin = p < total;
                    const int s = nin ? r_sa[lo] + (p - r_beg[lo]) : 0;
                    npos = in.Ps[s];
                    nms = in.Ms[s];
                    nslot = s;
                    nrow = lo;
                };
                fetch(0);
                for (int base = 0; base < total; base += kTrussWave) {
                    __syncthreads();   // the previous chunk is consumed
                    cslot[cidx] = nslot;
                    // past the end: far away, it fails every test
                    const bool some = nin;
                    const float4 mine_c = some ? npos : make_float4(inf, inf, inf, 0.0f);
                    const int2 mine_m = some ? nms : make_int2(-1, 0);
                    if (cut) {
                        cpos[cidx] = mine_c;
                        cid[cidx] = mine_m.x;
                        crow[cidx] = nrow;
                    }
                    const int mine_row = nrow;
                    __syncthreads();
                    fetch(base + kTrussWave);
                    uint64_t hit = chunk_hits(qops, mine_c, gox, goy, goz, k2, margin);
                    if (!H.prune) {
                        // the candidates of the rows this lane scans (its level range, its own
                        // box); where every reach fits its level's cell, only the bars that could
                        // be past the box by rounding are asked, where their lengths are formed
                        const int cn = min(kTrussWave, total - base);
                        uint64_t elig = 0;
                        const int r0 = crow[0], r1 = crow[cn - 1];
                        for (int r = r0; r <= r1; ++r) {
                            const int a = max(r_beg[r] - base, 0), b = min(r_beg[r] + r_len[r] - base, cn);
                            if (b > a && ((r_mask[r] >> lane) & 1ull)) {
                                elig |= (b - a == kTrussWave ? ~0ull : ((1ull << (b - a)) - 1)) << a;
                            }
                        }
                        hit &= elig;
                    }
                    hit = ingroup ? hit : 0ull;
                    // no bar between interior nodes of two labels
                    if (one_label) {   // (one mask then: 1.42 -> 1.35 ms for 2.5 M nodes)
                        const uint64_t foreign = __ballot((mine_m.y & 0xFF) == TN_INTERIOR && (mine_m.y >> 8) != wl && mine_m.x >= 0);
                        if (foreign) {
                            hit = ti_int ? hit & ~by_index(foreign) : hit;
                        }
                    } else {
                        const bool inside = (mine_m.y & 0xFF) == TN_INTERIOR;
                        const int cl = mine_m.y >> 8;
                        uint64_t left = by_index(__ballot(inside && mine_m.x >= 0));
                        while (left) {   // the labels of the chunk's interior candidates (mostly one)
                            const int l = __builtin_amdgcn_readlane(cl, chunk_lane(__builtin_ctzll(left)));
                            const uint64_t of = by_index(__ballot(inside && cl == l));
                            hit = ti_int && li != l ? hit & ~of : hit;
                            left &= ~of;
                        }
                    }
                    if (near) {
                        const bool full = kth != ~0ull;   // (a lane with fewer bars takes any)
                        const float dk = full ? __uint_as_float((uint32_t)(kth >> 32)) : 0.0f;
                        const uint64_t nearer = chunk_near(qx, qy, qz, dk * dk, mine_c, gox, goy, goz, margin);
                        hit = full ? hit & nearer : hit;
                    }
                    if (!cut && __ballot(cnt + __popcll(hit) > kCollect)) {   // a buffer fills
                        cut = true;
                        cpos[cidx] = mine_c;
                        cid[cidx] = mine_m.x;
                        crow[cidx] = mine_row;
                        __syncthreads();
                    }
                    if (!cut) {
                        while (hit) {   // (each lane its own)
                            const int k = __builtin_ctzll(hit);
                            hit &= hit - 1;
                            cb[cnt * kTrussWave + lane] = (uint32_t)cslot[k];
                            ++cnt;
                        }
                        continue;
                    }
                    // The possible hits as (query lane, candidate) pairs, up to 64 a round, one
                    // a lane: the exact test and the reference's other checks, and the valid
                    // ones appended to their query's buffer, packed in pair order.
                    while (__ballot(hit != 0ull)) {
                        const int pc = __popcll(hit);
                        // little room for them: keep the 24 best so far
                        const uint64_t sm = __ballot(pc > kCollect - cnt && kCollect - cnt < kMinRoom);
                        if (sm) {
                            settle_slot_lanes(cb, r_keys, lane, sm, cnt, kth, in.Ps, in.Ms, Q, H, half);
                            near = true;
                        }
                        const int want = min(pc, kCollect - cnt);
                        int npair = 0;
                        const int s0 = wave_excl_scan(want, lane, &npair);
                        const int take = max(0, min(want, kTrussWave - s0));
                        npair = min(npair, kTrussWave);
                        for (int e = 0; e < take; ++e) {
                            const int k = __builtin_ctzll(hit);
                            hit &= hit - 1;
                            pairs[s0 + e] = (lane << 6) | k;
                        }
                        __syncthreads();   // the pairs are written
                        const int pr = lane < npair ? pairs[lane] : 0;
                        const int o = pr >> 6, k = pr & 63;
                        // the owner's query, from its lane (every lane takes part in the shuffles)
                        const float ox_ = __shfl(px, o, kWave), oy_ = __shfl(py, o, kWave);
                        const float oz_ = __shfl(pz, o, kWave), oh = __shfl(hi, o, kWave);
                        const int oslot = __shfl(q, o, kWave);
                        const int os0 = __shfl(s0, o, kWave), ocnt = __shfl(cnt, o, kWave);
                        const uint64_t okth = __shfl(kth, o, kWave);
                        int cs = 0;
                        bool valid = false;
                        if (lane < npair) {
                            const float4 c = cpos[k];
                            cs = cslot[k];
                            const float ex = c.x - ox_, ey = c.y - oy_, ez = c.z - oz_;
                            const float d2 = ex * ex + ey * ey + ez * ez;
                            const float rj = half * (oh + c.w), rj2 = rj * rj;
                            valid = d2 < rj2 && cs != oslot;   // a bar, and not the node itself
                            if (valid && (!H.prune || d2 >= kDoubtful * rj2)) {   // the reference's own scan region only
                                valid = in_region(H, r_lev[crow[k]], ox_, oy_, oz_, tskin * oh, c);
                            }
                            valid = valid && list_key(sqrtf(d2), cid[k]) < okth;
                        }
                        const uint64_t vm = __ballot(valid);
                        // the owner's pairs are [s0, s0 + take) of its round: a valid pair's place is
                        // the owner's count plus the valid pairs of the owner before it
                        if (valid) {
                            const int at = ocnt + __popcll(vm & lanemask_lt() & ~((1ull << (os0 & 63)) - 1));
                            cb[at * kTrussWave + o] = (uint32_t)cs;
                        }
                        if (take > 0) {
                            const uint64_t span = take == kTrussWave ? ~0ull : ((1ull << take) - 1);
                            cnt += __popcll((vm >> s0) & span);
                        }
                        __syncthreads();   // the pairs are consumed
                    }
                }
            };
            const int lmin = wave_min(ingroup ? max(Li - 1, 0) : INT_MAX);
            const int lmax = wave_max(ingroup ? min(Li + 1, H.nlev - 1) : -1);
            for (int L = lmin; L <= lmax; ++L) {
                const bool mine = ingroup && L >= Li - 1 && L <= Li + 1;
                const float bL = H.b0 * (float)(1 << L);
                const float r = 0.5f * (Ri + bL);
                int x0 = INT_MAX, x1 = -1, y0 = INT_MAX, y1 = -1, z0 = INT_MAX, z1 = -1;
                if (mine) {
                    x0 = cell_coord(H, L, px - r, H.ox, 0);
                    x1 = cell_coord(H, L, px + r, H.ox, 0);
                    y0 = cell_coord(H, L, py - r, H.oy, 1);
                    y1 = cell_coord(H, L, py + r, H.oy, 1);
                    z0 = cell_coord(H, L, pz - r, H.oz, 2);
                    z1 = cell_coord(H, L, pz + r, H.oz, 2);
                }
                const int Y0 = wave_min(y0), Y1 = wave_max(y1), Z0 = wave_min(z0), Z1 = wave_max(z1);
                // rows beyond reach are skipped (a valid bar is shorter than r; margin for rounding)
                const float rw = r * 1.0001f + 1e-3f * bL + 2e-6f * (fabsf(px) + fabsf(py) + fabsf(pz));
                const float rr = rw * rw;
                // the level's grid (uniform: kept in scalar registers through the rows)
                const int nx = __builtin_amdgcn_readfirstlane(H.dim[L][0]);
                const int ny = __builtin_amdgcn_readfirstlane(H.dim[L][1]);
                const int nz1 = __builtin_amdgcn_readfirstlane(H.dim[L][2]) - 1, ny1 = ny - 1;
                const int koff = __builtin_amdgcn_readfirstlane(H.off[L]);
                const float inv_bL = 1.0f / bL;
                for (int cz = Z0; cz <= Z1; ++cz) {
                    const float zlo = cz == 0 ? -inf : H.oz + (float)cz * bL;
                    const float zhi = cz == nz1 ? inf : H.oz + (float)(cz + 1) * bL;
                    const float dz = fmaxf(0.0f, fmaxf(zlo - pz, pz - zhi));
                    for (int cy = Y0; cy <= Y1; ++cy) {
                        const float ylo = cy == 0 ? -inf : H.oy + (float)cy * bL;
                        const float yhi = cy == ny1 ? inf : H.oy + (float)(cy + 1) * bL;
                        const float dy = fmaxf(0.0f, fmaxf(ylo - py, py - yhi));
                        const bool row_own = mine && cz >= z0 && cz <= z1 && cy >= y0 && cy <= y1;
                        int xa = INT_MAX, xb = -1;
                        if (row_own) {
                            if (!H.prune) {
                                xa = x0;
                                xb = x1;
                            } else {
                                // The x-extent of the ball of radius rw in this row. A valid
                                // candidate lies at least (rw - rj) / 2 >= 5e-4 bL inside it (rj <= r,
                                // the bar's reach), far more than the error of the hardware square
                                // root and of the multiplication by 1 / bL (below 1e-4 cells), so
                                // these approximate cells never drop a candidate.
                                const float rem = rr - dz * dz - dy * dy;
                                if (rem >= 0.0f) {
                                    const float w = __builtin_amdgcn_sqrtf(rem);
                                    const int ca = (int)floorf((px - w - H.ox) * inv_bL);
                                    const int cb_ = (int)floorf((px + w - H.ox) * inv_bL);
                                    xa = max(x0, min(max(ca, 0), nx - 1));
                                    xb = min(x1, min(max(cb_, 0), nx - 1));
                                }
                            }
                        }
                        const int XA = wave_min(xa), XB = wave_max(xb);
                        if (XA > XB) {
                            continue;
                        }
                        const uint64_t scan = __ballot(xa <= xb);   // the lanes with cells in the row
                        if (lane == 0) {
                            const int krow = koff + nx * (cy + ny * cz);
                            r_key0[nr] = krow + XA;
                            r_key1[nr] = krow + XB + 1;
                            r_mask[nr] = scan;
                            r_lev[nr] = L;
                        }
                        if (++nr == kMaxRanges) {
                            flush();
                        }
                    }
                }
            }
            if (nr > 0) {
                flush();
            }
        }   // the groups
        if (active) {   // in any order, the entries past the count read by nobody
            nnb[q] = cnt;
            int4* row = reinterpret_cast<int4*>(nbr + (size_t)q * kK);
#pragma unroll
            for (int e = 0; e < kCollect; e += 4) {
                if (e < cnt) {
                    const int4 v = make_int4((int)cb[e * kTrussWave + lane], (int)cb[(e + 1) * kTrussWave + lane],
                                             (int)cb[(e + 2) * kTrussWave + lane], (int)cb[(e + 3) * kTrussWave + lane]);
                    if (e < kK) {
                        row[e / 4] = v;
                    } else if (e == kK) {
                        tail0[q] = v;
                    } else {
                        tail1[q] = v;
                    }
                }
            }
        }
        __syncthreads();   // the buffers are reused by the next block of queries
    }
}

// The rows k_truss left (up to 32 slots, in any order) tested exactly and put in
// (distance, id) order, the first 24 kept. In a launch of its own, a lane a node in slot
// order, its rows and the neighbours' positions are read and written whole lines at a time;
// at the end of k_truss, whose lanes hold nodes in brick order, the same work was a gather
// of the ids, one of their slots and 24 scattered stores a node, its 64 key registers
// bounding the search (2.5 M nodes: 2.25 ms in one kernel, 1.31 + 0.22 ms in two). The
// keys are (distance, slot): the ids are read only in a wave where two distances tie, whose
// lanes then sort by (distance, id) and look the slots up (neighbours exchanged until all
// ids are in order took up to a pass a tied entry: 152 us instead of 80 for 495 k nodes in
// the voxel field). Bound by the gathers of the positions.
template <int N>
__device__ __forceinline__ int sort_row(const Hash& H, const float4* __restrict__ Ps, const int2* __restrict__ Ms, int t,
                                        int m, float4 xi, float half, const int4* __restrict__ row, const int4* __restrict__ tail0,
                                        const int4* __restrict__ tail1, const int32_t* __restrict__ slot_of,
                                        uint64_t (&k)[32]) {
    constexpr int kB = 8;
    int s[N];
    uint32_t doubt = 0;   // the bars that could be past the scan region by rounding
#pragma unroll
    for (int e = 0; e < N; e += 4) {
        const int4 j4 = e < kK ? row[e / 4] : (e == kK ? tail0[t] : tail1[t]);
        s[e] = e < m ? j4.x : t;
        s[e + 1] = e + 1 < m ? j4.y : t;
        s[e + 2] = e + 2 < m ? j4.z : t;
        s[e + 3] = e + 3 < m ? j4.w : t;
    }
#pragma unroll
    for (int e0 = 0; e0 < N; e0 += kB) {
        float4 x[kB];
#pragma unroll
        for (int e = 0; e < kB; ++e) {
            x[e] = Ps[s[e0 + e]];
        }
#pragma unroll
        for (int e = 0; e < kB; ++e) {   // the reference's test (an entry past the row's end is the node itself)
            const float ex = x[e].x - xi.x, ey = x[e].y - xi.y, ez = x[e].z - xi.z;
            const float d2 = ex * ex + ey * ey + ez * ez;
            const float rj = half * (xi.w + x[e].w), rj2 = rj * rj;
            const bool bar = d2 < rj2 && s[e0 + e] != t;
            k[e0 + e] = bar ? list_key(sqrtf(d2), s[e0 + e]) : ~0ull;
            doubt |= bar && d2 >= kDoubtful * rj2 ? 1u << (e0 + e) : 0u;
        }
    }
#pragma clang loop unroll(disable)
    while (doubt) {   // (rare)
        const int at = __builtin_ctz(doubt);
        doubt &= doubt - 1;
        int j = t;
#pragma unroll
        for (int e = 0; e < N; ++e) {
            j = e == at ? (int)(uint32_t)k[e] : j;
        }
        const float4 c = Ps[j];
        const float T = 2.0f * half;
        if (!in_region(H, level_for(H, T * c.w), xi.x, xi.y, xi.z, T * xi.w, c)) {
#pragma unroll
            for (int e = 0; e < N; ++e) {
                k[e] = e == at ? ~0ull : k[e];
            }
        }
    }
    merge_sort<N>(k);
    int bars = 0;
    bool tie = false;
#pragma unroll
    for (int e = 0; e < N; ++e) {
        bars += k[e] != ~0ull ? 1 : 0;
        if (e > 0) {
            tie = tie || (k[e] != ~0ull && (k[e - 1] >> 32) == (k[e] >> 32));
        }
    }
    if (__ballot(tie)) {   // by (distance, id) then, and the slots looked up
#pragma unroll
        for (int e = 0; e < N; ++e) {
            k[e] = k[e] != ~0ull ? (k[e] >> 32) << 32 | (uint32_t)Ms[(int)(uint32_t)k[e]].x : ~0ull;
        }
        merge_sort<N>(k);
#pragma unroll
        for (int e = 0; e < kK; ++e) {
            k[e] = k[e] != ~0ull ? (uint32_t)slot_of[(int)(uint32_t)k[e]] : 0ull;
        }
    }
    return bars < kK ? bars : kK;
}

__global__ __launch_bounds__(kBlock) void k_lists(Hash H, const float4* __restrict__ Ps, const int2* __restrict__ Ms, int n,
                                                  float half, int32_t* __restrict__ nbr, const int4* __restrict__ tail0,
                                                  const int4* __restrict__ tail1, const int32_t* __restrict__ slot_of,
                                                  int32_t* __restrict__ nnb) {
    const int g = blockIdx.x * kBlock + threadIdx.x;
    const bool valid = g < n;
    const int t = valid ? g : 0;
    const int m = valid ? nnb[t] : 0;
    int4* row = reinterpret_cast<int4*>(nbr + (size_t)t * kK);
    const float4 xi = Ps[t];
    uint64_t k[32];
    const int bars = __ballot(m > kK) ? sort_row<32>(H, Ps, Ms, t, m, xi, half, row, tail0, tail1, slot_of, k)
                                      : sort_row<kK>(H, Ps, Ms, t, m, xi, half, row, tail0, tail1, slot_of, k);
    if (valid) {
        nnb[t] = bars;
#pragma unroll
        for (int e = 0; e < kK; e += 4) {
            row[e / 4] = make_int4((int)(uint32_t)k[e], (int)(uint32_t)k[e + 1], (int)(uint32_t)k[e + 2],
                                   (int)(uint32_t)k[e + 3]);
        }
    }
}

// ---- own-list refresh: one wave per node --------------------------------------------
//
// The nodes past a full skin refresh their own list every iteration
// (src/v2m_particles.cpp:925-931: the current position and size against the cells
// and candidate positions of the last rebuild; then P0 = P). They are few (about
// 0.1% of the nodes) and scattered, so each gets a whole wave: the lanes test the
// node's candidates 64 at a time with coalesced loads, valid ones are appended to
// the wave's list in LDS, and the K best in (distance, id) order are picked by rank
// (the order is total, so ranks are distinct). The scan region and the row pruning
// are k_truss's for a single lane.

constexpr int kRefreshCap = 256;   // LDS list entries (cut back to the best K when full)

// Keep the K best of the cnt entries of (cd, cj), in order, at [0, min(cnt, K)).
__device__ __forceinline__ int keep_best(float* cd, int* cj, int cnt, int lane) {
    constexpr int kPer = kRefreshCap / kWave;
    float d[kPer];
    int j[kPer], rank[kPer];
#pragma unroll
    for (int t = 0; t < kPer; ++t) {
        const int e = lane + t * kWave;
        d[t] = e < cnt ? cd[e] : 0.0f;
        j[t] = e < cnt ? cj[e] : 0;
        rank[t] = 0;
    }
    for (int e = 0; e < cnt; ++e) {
        const float de = cd[e];
        const int je = cj[e];
#pragma unroll
        for (int t = 0; t < kPer; ++t) {
            rank[t] += before(de, je, d[t], j[t]) ? 1 : 0;
        }
    }
    __syncthreads();   // every entry is read before any is moved
#pragma unroll
    for (int t = 0; t < kPer; ++t) {
        if (lane + t * kWave < cnt && rank[t] < kK) {
            cd[rank[t]] = d[t];
            cj[rank[t]] = j[t];
        }
    }
    __syncthreads();
    return cnt < kK ? cnt : kK;
}

__device__ __forceinline__ void k_truss_node_body(Hash H, TrussIn in, int n, const int32_t* __restrict__ list, const Ctl* __restrict__ ctl, int32_t* __restrict__ nbr, int32_t* __restrict__ nnb, float4* __restrict__ P0, int bid, int nblk) {
    __shared__ float cd[kRefreshCap];
    __shared__ int cj[kRefreshCap];
    const int lane = threadIdx.x;
    // after k_control: a rebuild (which rebuilds every list and sets P0 = P) or the end of
    // the loop follows, so no refreshed list would ever be read
    const int m = ctl->rebuild || ctl->done ? 0 : ctl->nrefresh;
    const float tskin = in.t + in.skin;
    for (int q = bid; q < m; q += nblk) {
        const int i = list[q];   // the node's slot
        const float4 xi = in.X[i];
        const float px = xi.x, py = xi.y, pz = xi.z, hi = xi.w;
        const float Ri = tskin * hi;
        const int Li = level_for(H, Ri);
        const int ti_int = in.typ[i] == TN_INTERIOR;
        const int li = in.lab[i];
        int cnt = 0;   // the wave's list length (the same in every lane)
        const int l0 = Li - 1 > 0 ? Li - 1 : 0, l1 = Li + 1 < H.nlev - 1 ? Li + 1 : H.nlev - 1;
        for (int L = l0; L <= l1; ++L) {
            const float bL = H.b0 * (float)(1 << L);
            const float r = 0.5f * (Ri + bL);
            const int x0 = cell_coord(H, L, px - r, H.ox, 0), x1 = cell_coord(H, L, px + r, H.ox, 0);
            const int y0 = cell_coord(H, L, py - r, H.oy, 1), y1 = cell_coord(H, L, py + r, H.oy, 1);
            const int z0 = cell_coord(H, L, pz - r, H.oz, 2), z1 = cell_coord(H, L, pz + r, H.oz, 2);
            const float rw = r * 1.0001f + 1e-3f * bL + 2e-6f * (fabsf(px) + fabsf(py) + fabsf(pz));
            const float rr = rw * rw;
            const int ny1 = H.dim[L][1] - 1, nz1 = H.dim[L][2] - 1;
            for (int cz = z0; cz <= z1; ++cz) {
                const float zlo = cz == 0 ? -__builtin_huge_valf() : H.oz + (float)cz * bL;
                const float zhi = cz == nz1 ? __builtin_huge_valf() : H.oz + (float)(cz + 1) * bL;
                const float dz = fmaxf(0.0f, fmaxf(zlo - pz, pz - zhi));
                for (int cy = y0; cy <= y1; ++cy) {
                    const float ylo = cy == 0 ? -__builtin_huge_valf() : H.oy + (float)cy * bL;
                    const float yhi = cy == ny1 ? __builtin_huge_valf() : H.oy + (float)(cy + 1) * bL;
                    const float dy = fmaxf(0.0f, fmaxf(ylo - py, py - yhi));
                    int xa = x0, xb = x1;
                    if (H.prune) {
                        const float rem = rr - dz * dz - dy * dy;
                        if (rem < 0.0f) {
                            continue;
                        }
                        const float wx = sqrtf(rem);
                        xa = max(x0, cell_coord(H, L, px - wx, H.ox, 0));
                        xb = min(x1, cell_coord(H, L, px + wx, H.ox, 0));
                        if (xa > xb) {
                            continue;
                        }
                    }
                    const int krow = H.off[L] + H.dim[L][0] * (cy + H.dim[L][1] * cz);
                    const int sa = in.cstart[krow + xa], sb = in.cstart[krow + xb + 1];
                    for (int base = sa; base < sb; base += kWave) {
                        const int s = base + lane;
                        bool ok = false;
                        float dist = 0.0f;
                        int j = 0;
                        if (s < sb) {
                            const float4 c = in.Ps[s];
                            const float ex = c.x - px, ey = c.y - py, ez = c.z - pz;
                            const float d2 = ex * ex + ey * ey + ez * ez;
                            const float rj = tskin * 0.5f * (hi + c.w);
                            if (d2 < rj * rj) {   // slot s: the candidate's current type, its id
                                ok = s != i && !(ti_int && in.typ[s] == TN_INTERIOR && in.lab[s] != li);
                                j = in.Ms[s].x;
                                dist = sqrtf(d2);
                            }
                        }
                        const uint64_t vm = __ballot(ok);
                        if (vm) {
                            const int add = __popcll(vm);
                            if (cnt + add > kRefreshCap) {
                                cnt = keep_best(cd, cj, cnt, lane);
                            }
                            if (ok) {
                                const int pos = cnt + __popcll(vm & lanemask_lt());
                                cd[pos] = dist;
                                cj[pos] = j;
                            }
                            cnt += add;
                        }
                    }
                }
            }
        }
        __syncthreads();   // the appends are visible to every lane
        const int kk = keep_best(cd, cj, cnt, lane);
        if (lane < kk) {
            nbr[(size_t)i * kK + lane] = in.slot_of[cj[lane]];
        }
        if (lane == 0) {
            nnb[i] = kk;
            P0[i] = xi;
        }
        __syncthreads();   // the list is read before the next node reuses it
    }
}

__global__ __launch_bounds__(kWave) void k_truss_node(Hash H, TrussIn in, int n, const int32_t* __restrict__ list, const Ctl* __restrict__ ctl, int32_t* __restrict__ nbr, int32_t* __restrict__ nnb, float4* __restrict__ P0) {
    k_truss_node_body(H, in, n, list, ctl, nbr, nnb, P0, blockIdx.x, gridDim.x);
}

// ---- node counts by type: interface, junction, interior, corner ------------------------

__device__ __forceinline__ int type_rank(int t) {
    return t == TN_INTERFACE ? 0 : (t == TN_JUNCTION ? 1 : (t == TN_INTERIOR ? 2 : 3));
}

// lanes of this wave whose node has type rank r (4 ballots)
__device__ __forceinline__ void rank_masks(bool valid, int r, uint64_t* m) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        m[k] = __ballot(valid && r == k);
    }
}

__global__ __launch_bounds__(kBlock) void k_order_count(const uint8_t* __restrict__ typ, int n, Ctl* __restrict__ ctl) {
    __shared__ int c[4];
    if (threadIdx.x < 4) {
        c[threadIdx.x] = 0;
    }
    __syncthreads();
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const bool valid = i < n;
    uint64_t m[4];
    rank_masks(valid, valid ? type_rank(typ[i] & 3) : 0, m);
    if ((threadIdx.x & (kWave - 1)) == 0) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (m[k]) {
                atomicAdd(&c[k], __popcll(m[k]));
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < 4 && c[threadIdx.x]) {
        atomicAdd(&ctl->order_cnt[threadIdx.x], c[threadIdx.x]);
    }
}

// ---- force --------------------------------------------------------------------------

// append i to queue for the lanes with flag set (one atomic on *count per wave)
__device__ __forceinline__ void wave_append(bool flag, int i, int32_t* count, int32_t* __restrict__ queue) {
    const uint64_t m = __ballot(flag);
    if (m) {
        const int lead = __ffsll((long long)m) - 1;
        int base = 0;
        if ((int)(threadIdx.x & (kWave - 1)) == lead) {
            base = atomicAdd(count, __popcll(m));
        }
        base = __shfl(base, lead, kWave);
        if (flag) {
            queue[base + __popcll(m & lanemask_lt())] = i;
        }
    }
}


// The forces; with queue_rest, also the junction nodes queued for the general move
// pass (their moves need no result of k_move_easy, so that pass can start as soon as
// the forces are done) and flagged in skip for k_move_easy, which leaves them alone
// without reading their type (the general pass may be rewriting it).
// The forces, and the queue of the general move pass that starts beside k_move_easy:
// the junction nodes and, when `sticky` is given, the nodes a lean pass has handed back
// before (their move is the same whichever pass computes it; queued here, it leaves the
// iteration's critical path).
__device__ __forceinline__ void k_force_body(const float4* __restrict__ X, const uint8_t* __restrict__ typ, const int32_t* __restrict__ nbr, const int32_t* __restrict__ nnb, float fscale, float fsurf, int n, float4* __restrict__ F, Ctl* __restrict__ ctl, int32_t* __restrict__ queue_rest, uint8_t* __restrict__ skip, const uint8_t* __restrict__ sticky, int bid, int nblk) {
    const int i = bid * kBlock + threadIdx.x;
    bool junction = false;
    if (i == 0) {   // the counts that the iteration's later kernels fill
        ctl->nhalf = 0;
        ctl->nrefresh = 0;
        ctl->nmove = 0;
        ctl->nmove_int = 0;
        ctl->nmove_def = 0;
    }
    if (i < n) {
        F[i] = bar_force(X, typ, nbr, nnb, fscale, fsurf, i);
        if (queue_rest) {
            junction = typ[i] == TN_JUNCTION || (sticky && sticky[i]);
            skip[i] = junction ? 1 : 0;
        }
    }
    if (queue_rest) {
        wave_append(junction, i, &ctl->nmove_rest, queue_rest);
    }
}

__global__ __launch_bounds__(kBlock) void k_force(const float4* __restrict__ X, const uint8_t* __restrict__ typ, const int32_t* __restrict__ nbr, const int32_t* __restrict__ nnb, float fscale, float fsurf, int n, float4* __restrict__ F, Ctl* __restrict__ ctl, int32_t* __restrict__ queue_rest, uint8_t* __restrict__ skip, const uint8_t* __restrict__ sticky) {
    k_force_body(X, typ, nbr, nnb, fscale, fsurf, n, F, ctl, queue_rest, skip, sticky, blockIdx.x, gridDim.x);
}

// ---- move (v2m_move, src/opencl/v2m_particle_body.cl:844-935) ----------------------

struct MoveArgs {
    float dt, maxstep, snap;
    int fire;
    int lanes;   // nodes per wave of the general pass at least (a launch shape; results do not depend on it)
};

__device__ __forceinline__ uint32_t pack_part(int b, int c) {
    return (uint32_t)(b & 0xFFFF) | ((uint32_t)(c & 0xFFFF) << 16);
}

// The FIRE / Jacobi part of v2m_move (src/opencl/v2m_particle_body.cl:853-912) for a
// node that is not a corner: the step s, capped at maxstep h, the power a . v, and
// whether the node moves at all (a settled node, |s| < 5e-4 h, stays put).
struct NodeStep {
    float s[3];
    float pw;
    bool moves;
};

// (v_at(): the node's velocity, read only when FIRE uses it)
template <class VAt>
__device__ __forceinline__ NodeStep node_step_with(const MoveArgs& ma, const Ctl* __restrict__ ctl, float4 Fi,
                                                   VAt v_at, float h) {
    NodeStep r;
    r.pw = 0.0f;
    const float stiff = Fi.w > 1.0f ? Fi.w : 1.0f;
    const float ac[3] = { Fi.x / stiff, Fi.y / stiff, Fi.z / stiff };
    if (ma.fire) {
        const float fdt = ctl->dt, falpha = ctl->alpha;
        float v[3] = { 0.0f, 0.0f, 0.0f };
        if (!ctl->zero_v) {
            const float4 v4 = v_at();
            v[0] = v4.x;
            v[1] = v4.y;
            v[2] = v4.z;
        }
        const float pv = ac[0] * v[0] + ac[1] * v[1] + ac[2] * v[2];
        r.pw = pv;
        if (pv < 0.0f) {
            v[0] = v[1] = v[2] = 0.0f;
        } else {
            const float vn = sqrtf(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
            const float an = sqrtf(ac[0] * ac[0] + ac[1] * ac[1] + ac[2] * ac[2]);
            if (an > 0.0f) {
                for (int k = 0; k < 3; ++k) {
                    v[k] = (1.0f - falpha) * v[k] + falpha * vn * ac[k] / an;
                }
            }
        }
        for (int k = 0; k < 3; ++k) {
            v[k] += fdt * ac[k];
            r.s[k] = fdt * v[k];
        }
    } else {
        for (int k = 0; k < 3; ++k) {
            r.s[k] = ma.dt * ac[k];
        }
    }
    const float sl = sqrtf(r.s[0] * r.s[0] + r.s[1] * r.s[1] + r.s[2] * r.s[2]);
    r.moves = !(sl < 5e-4f * h);
    if (r.moves && sl > ma.maxstep * h) {
        for (int k = 0; k < 3; ++k) {
            r.s[k] *= ma.maxstep * h / sl;
        }
    }
    return r;
}

__device__ __forceinline__ NodeStep node_step(const MoveArgs& ma, const Ctl* __restrict__ ctl, float4 Fi,
                                              const float4* __restrict__ V, int i, float h) {
    return node_step_with(ma, ctl, Fi, [&] { return V[i]; }, h);
}

// the writes that end v2m_move for node i (src/opencl/v2m_particle_body.cl:921-934)
__device__ __forceinline__ void move_store(const MoveArgs& ma, const Ctl* __restrict__ ctl, int i, float4 x, int ty0,
                                           uint32_t pp, const NodeState& ns, float m, float p_w,
                                           float4* __restrict__ X, float4* __restrict__ V,
                                           uint8_t* __restrict__ typ, uint32_t* __restrict__ part,
                                           float* __restrict__ mv, float* __restrict__ pw) {
    if (m > 0.0f) {
        X[i] = make_float4(ns.p.x, ns.p.y, ns.p.z, ns.hn);
    }
    if (ns.ty != ty0) {
        typ[i] = (uint8_t)ns.ty;
    }
    const uint32_t np = pack_part(ns.b, ns.c);
    if (np != pp) {
        part[i] = np;
    }
    if (ma.fire) {
        const float fdt = ctl->dt;
        float4 vout = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (m > 0.0f && ns.ty == ty0) {
            vout = make_float4((ns.p.x - x.x) / fdt, (ns.p.y - x.y) / fdt, (ns.p.z - x.z) / fdt, 0.0f);
        }
        V[i] = vout;
        pw[i] = p_w;
    }
    mv[i] = m;
}

// Pass 1 of the move, over every node in slot order but the junction nodes (queued
// by k_force for the general pass): corners, settled nodes and interior nodes whose
// step stays in their own region with no interface within snap range are finished
// here, exactly as v2m_move finishes them. The interface nodes and the interior
// nodes that cross or may snap are queued, untouched, for the lean k_move passes.
// Most nodes are interior, and this pass needs a fraction of the registers of the
// full trapped step.
// Append i to queue a (lanes with fa set) and to queue b (fb), one atomic per block
// and queue: the 2 M-node pass would otherwise send tens of thousands of atomics to
// the same two counters. Every thread of the block must arrive here.
__device__ __forceinline__ void block_append2(bool fa, bool fb, int i, int32_t* ca, int32_t* __restrict__ qa,
                                              int32_t* cb, int32_t* __restrict__ qb) {
    constexpr int kW = kBlock / kWave;
    __shared__ int cnt[2][kW + 1];
    const uint64_t ma = __ballot(fa), mb = __ballot(fb);
    const int w = threadIdx.x >> 6, lane = threadIdx.x & (kWave - 1);
    if (lane == 0) {
        cnt[0][w] = __popcll(ma);
        cnt[1][w] = __popcll(mb);
    }
    __syncthreads();
    if (threadIdx.x < 2) {   // the block's offsets of its waves, then one atomic per queue
        int tot = 0;
        for (int k = 0; k < kW; ++k) {
            const int c = cnt[threadIdx.x][k];
            cnt[threadIdx.x][k] = tot;
            tot += c;
        }
        cnt[threadIdx.x][kW] = tot ? atomicAdd(threadIdx.x == 0 ? ca : cb, tot) : 0;
    }
    __syncthreads();
    const uint64_t below = lanemask_lt();
    if (fa) {
        qa[cnt[0][kW] + cnt[0][w] + __popcll(ma & below)] = i;
    }
    if (fb) {
        qb[cnt[1][kW] + cnt[1][w] + __popcll(mb & below)] = i;
    }
}

// F: PlainField when every grid of the launch is a label volume with its apron slots
// (tn_apron.hpp): the kernel then holds no other field mode; Field for the others.
template <class F>
__device__ __forceinline__ void k_move_easy_body(F f, MoveArgs ma, Ctl* __restrict__ ctl, int n, const float4* __restrict__ Fo, float4* __restrict__ X, float4* __restrict__ V, uint8_t* __restrict__ typ, uint32_t* __restrict__ part, const uint16_t* __restrict__ lab, float* __restrict__ mv, float* __restrict__ pw, int32_t* __restrict__ queue, int32_t* __restrict__ queue_int, const uint8_t* __restrict__ skip, int bid, int nblk) {
    const int g = bid * kBlock + threadIdx.x;
    int i = 0;
    bool surf = false, inner = false;   // the two lean queues
    // The node's own values, read at once rather than each behind the test that needs
    // it (a node another pass moves reads values it then leaves unused).
    const bool in = g < n;
    const int sk = in ? skip[g] : 1;
    const int ty0 = in ? typ[g] : 0;
    const float4 x = in ? X[g] : make_float4(0.0f, 0.0f, 0.0f, 1.0f);
    const float4 Fi = in ? Fo[g] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float4 Vi = in && ma.fire ? V[g] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const int a = in ? lab[g] : 0;
    const uint32_t pp = in ? part[g] : 0u;
    if (in && !sk) {   // (junction nodes: queued by k_force for the general pass)
        i = g;
        if (ty0 == TN_INTERFACE) {
            surf = true;
        } else if (ty0 == TN_CORNER) {
            if (ma.fire) {
                V[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                pw[i] = 0.0f;
            }
            mv[i] = 0.0f;
        } else {
            const float h = x.w;
            const NodeStep st = node_step_with(ma, ctl, Fi, [&] { return Vi; }, h);
            if (!st.moves) {
                if (ma.fire) {
                    V[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    pw[i] = st.pw;
                }
                mv[i] = 0.0f;
            } else {
                // trapped_step's interior branch up to its first decision
                const P3 p = p3(x.x, x.y, x.z);
                const P3 q = p3(p.x + st.s[0], p.y + st.s[1], p.z + st.s[2]);
                // h at the target, loaded before the owner query's chain of loads (it is
                // needed unless the node turns out to cross or to snap)
                const float hq = size_at(f, q.x, q.y, q.z);
                const OwnerPsi own = owner_psi_at(f, a, q);
                if (own.best != a) {
                    inner = true;
                } else if (own.sec != kNoLab && ma.snap > 0.0f) {
                    const float4 gq = own.g;
                    const float gn = sqrtf(gq.x * gq.x + gq.y * gq.y + gq.z * gq.z);
                    inner = gn > 1e-9f && gq.w / gn < ma.snap * h;
                }
                if (!inner) {   // the rest of trapped_step for an interior node that stays interior
                    NodeState ns;
                    ns.p = p;
                    ns.hn = h;
                    ns.ty = TN_INTERIOR;
                    ns.b = (int)(pp & 0xFFFF);
                    ns.c = (int)(pp >> 16);
                    float m = 0.0f;
                    const float lim = (ma.maxstep + fmaxf(ma.snap, 0.5f)) * h;
                    const float m2 = dist2(q, p);
                    if (!(m2 <= lim * lim)) {
                        ns.b = kNoLab;
                    } else {
                        ns.p = q;
                        ns.hn = hq;
                        m = sqrtf(m2) / h;
                    }
                    move_store(ma, ctl, i, x, TN_INTERIOR, pp, ns, m, st.pw, X, V, typ, part, mv, pw);
                }
            }
        }
    }
    // queue the rest, one atomic per block and queue
    block_append2(surf, inner, i, &ctl->nmove, queue, &ctl->nmove_int, queue_int);
}

template <class F>
__global__ __launch_bounds__(kBlock) void k_move_easy(F f, MoveArgs ma, Ctl* __restrict__ ctl, int n, const float4* __restrict__ Fo, float4* __restrict__ X, float4* __restrict__ V, uint8_t* __restrict__ typ, uint32_t* __restrict__ part, const uint16_t* __restrict__ lab, float* __restrict__ mv, float* __restrict__ pw, int32_t* __restrict__ queue, int32_t* __restrict__ queue_int, const uint8_t* __restrict__ skip) {
    k_move_easy_body(f, ma, ctl, n, Fo, X, V, typ, part, lab, mv, pw, queue, queue_int, skip, blockIdx.x,
                             gridDim.x);
}

#ifndef TN_REST_LANES
#define TN_REST_LANES 4
#endif
constexpr int kRestLanes = TN_REST_LANES;   // nodes per wave in k_move<kGeneral>
// a lean pass spreads up to this many nodes per wave before it fills whole waves
#ifndef TN_LEAN_SPREAD
#define TN_LEAN_SPREAD 4
#endif
constexpr int kLeanSpread = TN_LEAN_SPREAD;

// waves per SIMD the full move kernel is compiled for (its register budget: 512 / waves)
#ifndef TN_MOVE_WAVES
#define TN_MOVE_WAVES 1
#endif

// v2m_move for queued node i; true: handed back (a lean mode, a third label near)
template <int kMode, class F>
__device__ __forceinline__ bool move_node(const F& f, const MoveArgs& ma, const Ctl* __restrict__ ctl, int i,
                                          const float4* __restrict__ Fo, float4* __restrict__ X,
                                          float4* __restrict__ V, uint8_t* __restrict__ typ,
                                          uint32_t* __restrict__ part, const uint16_t* __restrict__ lab,
                                          float* __restrict__ mv, float* __restrict__ pw) {
    const float4 x = X[i];
    const float h = x.w;   // h at the node: v2m_h_at(P_i), kept current by every move
    const int ty0 = kMode == kLeanInterface ? TN_INTERFACE : (kMode == kLeanInterior ? TN_INTERIOR : typ[i]);
    const uint32_t pp = part[i];
    NodeState ns;
    ns.p = p3(x.x, x.y, x.z);
    ns.hn = h;
    ns.ty = ty0;
    ns.b = (int)(pp & 0xFFFF);
    ns.c = (int)(pp >> 16);
    float m = 0.0f;
    const NodeStep st = node_step(ma, ctl, Fo[i], V, i, h);   // queued nodes are never corners
    if (st.moves) {
        m = trapped_step<kMode>(f, h, p3(st.s[0], st.s[1], st.s[2]), ma.maxstep, ma.snap, lab[i], ns);
        if (kMode != kGeneral && m == kDeferred) {
            return true;
        }
    }
    move_store(ma, ctl, i, x, ty0, pp, ns, m, st.pw, X, V, typ, part, mv, pw);
    return false;
}

// The whole move in voxel-trap mode (v2m_move with voxmode, src/opencl/v2m_particle_body.cl:
// 844-935 and 549-650): every node in one pass; corners and settled nodes stay.
// The voxel-trap move, pass 1, a lane per node: corners, settled nodes and interior
// nodes whose step meets no wall and no wall within snap range are finished here; the
// rest (face and edge scans) are queued, untouched, for pass 2.
__device__ __forceinline__ void k_move_voxel_body(const Field& f, const MoveArgs& ma, const Ctl* __restrict__ ctl,
                                                  int n, const float4* __restrict__ F, float4* __restrict__ X,
                                                  float4* __restrict__ V, uint8_t* __restrict__ typ,
                                                  uint32_t* __restrict__ part, const uint16_t* __restrict__ lab,
                                                  float* __restrict__ mv, float* __restrict__ pw,
                                                  int32_t* __restrict__ queue, int32_t* __restrict__ qcount, int bid) {
    const int i = bid * kBlock + threadIdx.x;
    bool defer = false;
    if (i < n) {
        const float4 x = X[i];
        const float h = x.w;
        const int ty0 = typ[i];
        const uint32_t pp = part[i];
        NodeState ns;
        ns.p = p3(x.x, x.y, x.z);
        ns.hn = h;
        ns.ty = ty0;
        ns.b = (int)(pp & 0xFFFF);
        ns.c = (int)(pp >> 16);
        float m = 0.0f, p_w = 0.0f;
        if (ty0 != TN_CORNER) {
            const NodeStep st = node_step(ma, ctl, F[i], V, i, h);
            p_w = st.pw;
            if (st.moves) {
                m = voxel_step<false>(f, h, ma.snap, lab[i], st.s, ns);
                defer = m == kDeferred;
            }
        }
        if (!defer) {
            move_store(ma, ctl, i, x, ty0, pp, ns, m, p_w, X, V, typ, part, mv, pw);
        }
    }
    wave_append(defer, i, qcount, queue);
}

__global__ __launch_bounds__(kBlock) void k_move_voxel(Field f, MoveArgs ma, const Ctl* __restrict__ ctl, int n,
                                                       const float4* __restrict__ F, float4* __restrict__ X,
                                                       float4* __restrict__ V, uint8_t* __restrict__ typ,
                                                       uint32_t* __restrict__ part, const uint16_t* __restrict__ lab,
                                                       float* __restrict__ mv, float* __restrict__ pw,
                                                       int32_t* __restrict__ queue, int32_t* __restrict__ qcount) {
    k_move_voxel_body(f, ma, ctl, n, F, X, V, typ, part, lab, mv, pw, queue, qcount, blockIdx.x);
}

// Pass 2: a wave per queued node, every lane on the same node (the same values in
// every lane), the face and edge scans split over the wave; lane 0 stores.
__device__ __forceinline__ void k_move_voxel_wave_body(const Field& f, const MoveArgs& ma, const Ctl* __restrict__ ctl,
                                                       const int32_t* __restrict__ queue,
                                                       const int32_t* __restrict__ qcount,
                                                       const float4* __restrict__ F, float4* __restrict__ X,
                                                       float4* __restrict__ V, uint8_t* __restrict__ typ,
                                                       uint32_t* __restrict__ part, const uint16_t* __restrict__ lab,
                                                       float* __restrict__ mv, float* __restrict__ pw, int bid,
                                                       int nblk) {
    constexpr int kWaves = kBlock / kWave;
    const int count = *qcount;
    for (int g = bid * kWaves + (int)(threadIdx.x >> 6); g < count; g += nblk * kWaves) {
        const int i = queue[g];
        const float4 x = X[i];
        const float h = x.w;
        const int ty0 = typ[i];
        const uint32_t pp = part[i];
        NodeState ns;
        ns.p = p3(x.x, x.y, x.z);
        ns.hn = h;
        ns.ty = ty0;
        ns.b = (int)(pp & 0xFFFF);
        ns.c = (int)(pp >> 16);
        const NodeStep st = node_step(ma, ctl, F[i], V, i, h);   // queued nodes move
        const float m = voxel_step<true>(f, h, ma.snap, lab[i], st.s, ns);
        if ((threadIdx.x & (kWave - 1)) == 0) {
            move_store(ma, ctl, i, x, ty0, pp, ns, m, st.pw, X, V, typ, part, mv, pw);
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_move_voxel_wave(Field f, MoveArgs ma, const Ctl* __restrict__ ctl,
                                                            const int32_t* __restrict__ queue,
                                                            const int32_t* __restrict__ qcount,
                                                            const float4* __restrict__ F, float4* __restrict__ X,
                                                            float4* __restrict__ V, uint8_t* __restrict__ typ,
                                                            uint32_t* __restrict__ part,
                                                            const uint16_t* __restrict__ lab, float* __restrict__ mv,
                                                            float* __restrict__ pw) {
    k_move_voxel_wave_body(f, ma, ctl, queue, qcount, F, X, V, typ, part, lab, mv, pw, blockIdx.x, gridDim.x);
}

// Pass 2: v2m_move (src/opencl/v2m_particle_body.cl:844-935) for the queued nodes,
// *count of them. kLeanInterface / kLeanInterior: interface or interior nodes, with
// their branch of the trapped step only and no out-of-line calls (whose register
// budgets would bound the kernel's occupancy); a node with a third label near is
// appended to (defer_count, defer_queue) for a later kGeneral pass. kGeneral: the
// whole trapped step (junction nodes and the handed-back ones). Each node's move
// reads and writes only that node's state, so the passes over disjoint queues may
// run concurrently.
template <int kMode, class F>
__device__ __forceinline__ void k_move_body(F f, MoveArgs ma, Ctl* __restrict__ ctl, const int32_t* __restrict__ queue, const float4* __restrict__ Fo, float4* __restrict__ X, float4* __restrict__ V, uint8_t* __restrict__ typ, uint32_t* __restrict__ part, const uint16_t* __restrict__ lab, float* __restrict__ mv, float* __restrict__ pw, const int32_t* __restrict__ qcount, int32_t* __restrict__ defer_count, int32_t* __restrict__ defer_queue, uint8_t* __restrict__ sticky, int bid, int nblk) {
    // A fixed grid strides over the queue, whose length only the device knows. A
    // short queue's nodes follow long, divergent paths (projections onto interfaces
    // and junction curves), and a wave executes every path its lanes take, so they
    // are spread thinly over the grid's waves (lean passes: one to kLeanSpread nodes per
    // wave; the general pass: from kRestLanes, measured best); a long queue fills whole
    // waves, whose lanes then share the issue slots.
    constexpr bool kLean = kMode != kGeneral;
    constexpr int kWaves = kBlock / kWave;
    const int count = *qcount;
    const int waves = (int)nblk * kWaves;
    const int spread = (count + waves - 1) / waves;
    int lpw;
    if (kLean) {
        lpw = spread < 1 ? 1 : (spread > kLeanSpread ? kWave : spread);
    } else {
        const int rl = ma.lanes > 0 ? ma.lanes : kRestLanes;
        lpw = spread < rl ? rl : (spread > kWave ? kWave : spread);
    }
    const int per_block = lpw * kWaves;
    const int lane = threadIdx.x & (kWave - 1);
    const int slot = lane < lpw ? (threadIdx.x >> 6) * lpw + lane : -1;
    for (int base = bid * per_block; base < count; base += nblk * per_block) {
        const int g = base + slot;
        bool defer = false;
        int i = 0;
        if (slot >= 0 && g < count) {
            i = queue[g];
            defer = move_node<kMode>(f, ma, ctl, i, Fo, X, V, typ, part, lab, mv, pw);
        }
        if (kLean) {   // every lane of the wave is here
            wave_append(defer, i, defer_count, defer_queue);
            if (defer && sticky) {   // from the next iteration on, queued by k_force
                sticky[i] = 1;
            }
        }
    }
}

template <int kMode, class F>
__global__ __launch_bounds__(kBlock, TN_MOVE_WAVES) void k_move(F f, MoveArgs ma, Ctl* __restrict__ ctl, const int32_t* __restrict__ queue, const float4* __restrict__ Fo, float4* __restrict__ X, float4* __restrict__ V, uint8_t* __restrict__ typ, uint32_t* __restrict__ part, const uint16_t* __restrict__ lab, float* __restrict__ mv, float* __restrict__ pw, const int32_t* __restrict__ qcount, int32_t* __restrict__ defer_count, int32_t* __restrict__ defer_queue, uint8_t* __restrict__ sticky) {
    k_move_body<kMode>(f, ma, ctl, queue, Fo, X, V, typ, part, lab, mv, pw, qcount, defer_count, defer_queue,
                               sticky, blockIdx.x, gridDim.x);
}

constexpr int kMoveGrid = 2048;       // blocks of a lean k_move at most
constexpr int kMoveRestGrid = 512;    // blocks of k_move<kGeneral>: the waves resident at its register budget


// ---- per-iteration reductions + Verlet bookkeeping ----------------------------------

// The histogram bin of src/v2m_particles.cpp:881: clamp(20 + floor(log2f(m)), 0, 31).
// floor(log2f(m)) is the binary exponent of m, except just below a power of two,
// where the rounded log2f reaches the next integer; thr[e + 21] is the smallest
// float below 2^e whose log2f rounds up to e (from the host's log2f).
__device__ __forceinline__ int hist_bin(float m, const float* __restrict__ thr) {
    if (!(m > 0.0f)) {
        return 0;
    }
    int e;
    frexpf(m, &e);   // m in [2^(e-1), 2^e)
    int fl = e - 1;
    if (e >= -21 && e <= 13 && m >= thr[e + 21]) {
        fl = e;
    }
    const int b = 20 + fl;
    return b < 0 ? 0 : (b > 31 ? 31 : b);
}

constexpr int kHistThr = 35;   // exponents -21..13
constexpr int kStatsBlocks = 2048;   // k_stats' grid at most (8 blocks per CU)
constexpr int kHeldChunks = 8;       // chunks of nodes after which a block writes out what it lists

// Per iteration: the histogram, the largest move, the count past skin/2, the
// nodes past a full skin (listed: their own lists are refreshed), and FIRE's
// power partial sums (src/v2m_particles.cpp:849-937). Counts are reduced per
// wave with ballots before any atomic, and the listed nodes gathered in LDS, so that a
// block takes its place in the list once (a pass of its own over a flag a node, as
// before, cost 8 us an iteration at 2.5 M nodes and a launch at any size; 57 us there). LDS holds
// every node of kHeldChunks chunks, and the block writes the list out after that many
// whatever it holds: the chunk's number is the same in every wave, while the count held
// may already be another wave's next, and the writing has barriers that all must reach.
__device__ __forceinline__ void k_stats_body(const float4* __restrict__ X, const float4* __restrict__ P0, const float* __restrict__ mv, const float* __restrict__ pw, int n, float skin, int fire, const float* __restrict__ thr, Ctl* __restrict__ ctl, int32_t* __restrict__ refresh, double2* __restrict__ partials, int bid, int nblk) {
    __shared__ int held[kHeldChunks * kBlock];   // nodes to list
    __shared__ int nheld, held_at;
    __shared__ uint32_t lh[32];
    __shared__ uint32_t lmax;
    __shared__ int lhalf;
    __shared__ double lps[kBlock / kWave][2];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    if (tid < 32) {
        lh[tid] = 0;
    }
    if (tid == 0) {
        lmax = 0;
        lhalf = 0;
        nheld = 0;
        if (bid == 0) {   // (the moves are done: the queue is free for the next k_force)
            ctl->moved_rest = ctl->nmove_rest;
            ctl->nmove_rest = 0;
        }
    }
    // every thread of the block: the held nodes into the list
    auto list_held = [&]() {
        const int m = nheld;
        if (tid == 0 && m) {
            held_at = atomicAdd(&ctl->nrefresh, m);
        }
        __syncthreads();
        for (int e = tid; e < m; e += kBlock) {
            refresh[held_at + e] = held[e];
        }
        __syncthreads();
        if (tid == 0) {
            nheld = 0;
        }
        __syncthreads();
    };
    double bs = 0.0, ba = 0.0;   // this block's power partial sums (thread 0), chunk by chunk
    int chunks = 0;              // chunks since the block last wrote its list out
    // chunks of kBlock nodes, grid-strided: each block adds its counts to the control
    // block once, and its partial sums have a fixed shape
    for (int c = bid; (int64_t)c * kBlock < n; c += nblk) {
        __syncthreads();   // lps of the previous chunk has been read, its nodes are held
        if (chunks == kHeldChunks) {
            list_held();
            chunks = 0;
        }
        ++chunks;
        const int i = c * kBlock + tid;
        double ps = 0.0, pa = 0.0;
        int bin = -1;
        uint32_t mbits = 0;
        bool half = false, far = false;
        if (i < n) {
            const float m = mv[i];
            bin = hist_bin(m, thr);
            mbits = __float_as_uint(m);
            const float4 x = X[i], x0 = P0[i];
            const float ex = x.x - x0.x, ey = x.y - x0.y, ez = x.z - x0.z;
            const float h = x.w;
            const float m2 = ex * ex + ey * ey + ez * ez, s2 = skin * skin * h * h;
            far = m2 > s2;
            half = !far && m2 > 0.25f * s2;
            if (fire) {
                ps = (double)pw[i];
                pa = fabs(ps);
            }
        }
        const uint64_t fm = __ballot(far);
        if (fm) {
            const int lead = __ffsll((long long)fm) - 1;
            int at = 0;
            if (lane == lead) {
                at = atomicAdd(&nheld, __popcll(fm));
            }
            at = __shfl(at, lead, kWave);
            if (far) {
                held[at + __popcll(fm & lanemask_lt())] = i;
            }
        }
        // histogram: one LDS add per (wave, occupied bin)
        uint64_t left = __ballot(bin >= 0);
        while (left) {
            const int b = __shfl(bin, __ffsll((long long)left) - 1, kWave);
            const uint64_t same = __ballot(bin == b);
            if (lane == 0) {
                atomicAdd(&lh[b], (uint32_t)__popcll(same));
            }
            left &= ~same;
        }
#pragma unroll
        for (int d = kWave / 2; d > 0; d >>= 1) {
            mbits = max(mbits, (uint32_t)__shfl_xor((int)mbits, d, kWave));
        }
        const int nh = __popcll(__ballot(half));
        if (lane == 0) {
            atomicMax(&lmax, mbits);
            if (nh) {
                atomicAdd(&lhalf, nh);
            }
        }
        if (fire) {   // fixed-shape tree: the partial sums are reproducible
#pragma unroll
            for (int d = kWave / 2; d > 0; d >>= 1) {
                ps += __shfl_xor(ps, d, kWave);
                pa += __shfl_xor(pa, d, kWave);
            }
            if (lane == 0) {
                lps[tid >> 6][0] = ps;
                lps[tid >> 6][1] = pa;
            }
            __syncthreads();
            if (tid == 0) {
                bs += (lps[0][0] + lps[1][0]) + (lps[2][0] + lps[3][0]);
                ba += (lps[0][1] + lps[1][1]) + (lps[2][1] + lps[3][1]);
            }
        }
    }
    __syncthreads();
    if (nheld) {
        list_held();
    }
    if (tid < 32 && lh[tid]) {
        atomicAdd(&ctl->hist[tid], lh[tid]);
    }
    if (tid == 0) {
        atomicMax(&ctl->mmax_bits, lmax);
        if (lhalf) {
            atomicAdd(&ctl->nhalf, lhalf);
        }
        if (fire) {
            partials[bid] = make_double2(bs, ba);
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_stats(const float4* __restrict__ X, const float4* __restrict__ P0, const float* __restrict__ mv, const float* __restrict__ pw, int n, float skin, int fire, const float* __restrict__ thr, Ctl* __restrict__ ctl, int32_t* __restrict__ refresh, double2* __restrict__ partials) {
    k_stats_body(X, P0, mv, pw, n, skin, fire, thr, ctl, refresh, partials, blockIdx.x, gridDim.x);
}

// ---- field queries at given points (the queries the move makes, for checking) ---------

// phi_a (v2m_phi_f), psi_ab and its gradient (v2m_psi_grad), the owner and the
// runner-up (v2m_label_of) at X[3k..3k+2]; any output may be null.
template <class F>
__global__ __launch_bounds__(kBlock) void k_field_points(F f, int a, int b, int m, const float* __restrict__ X,
                                                         float* __restrict__ phi, float* __restrict__ psi,
                                                         float* __restrict__ grad, int32_t* __restrict__ label,
                                                         int32_t* __restrict__ second) {
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= m) {
        return;
    }
    const P3 p = p3(X[3 * k], X[3 * k + 1], X[3 * k + 2]);
    if (phi) {
        phi[k] = phi_point(f, a, p);
    }
    if (psi || grad) {
        const float4 g = psi_grad_once(f, a, b, p);
        if (psi) {
            psi[k] = g.w;
        }
        if (grad) {
            grad[3 * k] = g.x;
            grad[3 * k + 1] = g.y;
            grad[3 * k + 2] = g.z;
        }
    }
    if (label || second) {
        const int2 o = owner_at(f, p);
        if (label) {
            label[k] = o.x;
        }
        if (second) {
            second[k] = o.y;
        }
    }
}

// ---- control (one block) ---------------------------------------------------------------

struct CtlArgs {
    int n, max_iters, fire, rebuild_div;
    float dptol;
    int nparts;
    int force_serial;   // take the serial power sum every FIRE iteration (the exact path, for its tests)
};

// FIRE's power P = sum pw, whose sign (P >= 0) drives FireCtl::update
// (src/v2m_particles.h:58-73). The CPU path sums pw serially in double
// (src/v2m_particles.cpp:849-855). Here the partial sums are combined in a fixed
// tree; with A = sum |pw|, both that sum and the serial one are within
// (n + 64) * 2^-53 * A of the exact sum, so when |S| exceeds twice that bound both
// have the exact sum's sign. Otherwise the serial sum is recomputed here, in index
// order, exactly as the CPU does.
//
// The control block goes to the host from here, by stores to pinned memory (host, if it is
// not null), and the own-list refreshes are launched after the event that the host waits
// for: a copy between the refreshes and the event cost each iteration its own latency, and
// the host enqueued the next iteration only after both (435 k nodes, 100 iterations: 42.1 ->
// 41.2 ms; at 75 k nodes to convergence the runs of one side differ by more than the gain).
__device__ __forceinline__ void k_control_step(CtlArgs ca, Ctl* __restrict__ ctl, const double2* __restrict__ partials, const float* __restrict__ pw, const int32_t* __restrict__ slot_of, int bid, int nblk) {
    __shared__ double red[kBlock][2];
    __shared__ float chunk[kScanTile];
    __shared__ int use_serial;
    const int tid = threadIdx.x;
    double s = 0.0, a = 0.0;
    if (ca.fire) {
        for (int k = tid; k < ca.nparts; k += kBlock) {
            const double2 p = partials[k];
            s += p.x;
            a += p.y;
        }
    }
    red[tid][0] = s;
    red[tid][1] = a;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if (tid < w) {
            red[tid][0] += red[tid + w][0];
            red[tid][1] += red[tid + w][1];
        }
        __syncthreads();
    }
    double P = red[0][0];
    if (tid == 0) {
        const double A = red[0][1];
        const double bound = 2.0 * ((double)ca.n + 64.0) * 0x1p-53 * A;
        use_serial = ca.fire && (ca.force_serial || (A > 0.0 && !(fabs(P) > bound)));
    }
    __syncthreads();
    if (use_serial) {   // the CPU's own summation, in node index (id) order
        double pt = 0.0;
        for (int c0 = 0; c0 < ca.n; c0 += kScanTile) {
            for (int k = tid; k < kScanTile; k += kBlock) {
                chunk[k] = c0 + k < ca.n ? pw[slot_of[c0 + k]] : 0.0f;
            }
            __syncthreads();
            if (tid == 0) {
                const int m = ca.n - c0 < kScanTile ? ca.n - c0 : kScanTile;
                for (int k = 0; k < m; ++k) {
                    pt += chunk[k];
                }
            }
            __syncthreads();
        }
        P = pt;
    }
    if (tid != 0) {
        return;
    }
    const int it = ctl->it;
    if (use_serial) {
        ctl->power_fallbacks += 1;
    }
    ctl->power = P;
    if (ca.fire) {   // FireCtl::update
        if (P >= 0.0) {
            ctl->zero_v = 0;
            if (++ctl->npos > 5) {
                const float up = ctl->dt * 1.1f;
                ctl->dt = up < ctl->dtmax ? up : ctl->dtmax;
                ctl->alpha *= 0.99f;
            }
        } else {
            ctl->zero_v = 1;
            ctl->npos = 0;
            const float down = ctl->dt * 0.5f, lo = 0.05f * ctl->dt0;
            ctl->dt = down < lo ? lo : down;
            ctl->alpha = 0.1f;
            ctl->fire_resets += 1;
        }
    }
    ctl->it = it + 1;
    ctl->last_move = __uint_as_float(ctl->mmax_bits);
    ctl->fire_dt = ca.fire ? ctl->dt : 0.0f;
    int acc = 0, b99 = 31;
    for (int b = 0; b < 32; ++b) {
        acc += (int)ctl->hist[b];
        if ((double)acc >= 0.99 * (double)ca.n) {
            b99 = b;
            break;
        }
    }
    const float p99 = ldexpf(1.0f, b99 - 20 + 1);
    ctl->last_p99 = p99;
    const int done = p99 < ca.dptol && (!ca.fire || ctl->dt >= 0.25f * ctl->dt0);
    ctl->done = done;
    ctl->rebuild = 0;
    if (!done) {
        const int endgame = it >= ca.max_iters * 4 / 5 || p99 < 4.0f * ca.dptol;
        const int div = endgame ? (ca.rebuild_div > 1000 ? ca.rebuild_div : 1000) : ca.rebuild_div;
        ctl->rebuild = ctl->nhalf > ca.n / div;
    }
    for (int b = 0; b < 32; ++b) {
        ctl->hist[b] = 0;
    }
    ctl->mmax_bits = 0;
}

// the control, then the block to the host (host may be null)
__device__ __forceinline__ void k_control_body(CtlArgs ca, Ctl* __restrict__ ctl, const double2* __restrict__ partials, const float* __restrict__ pw, const int32_t* __restrict__ slot_of, Ctl* host, int bid, int nblk) {
    k_control_step(ca, ctl, partials, pw, slot_of, bid, nblk);
    if (!host) {
        return;
    }
    __syncthreads();   // the first thread's stores are done
    static_assert(sizeof(Ctl) % 4 == 0, "Ctl is copied in words");
    const volatile uint32_t* src = reinterpret_cast<const volatile uint32_t*>(ctl);
    volatile uint32_t* dst = reinterpret_cast<volatile uint32_t*>(host);
    for (int k = threadIdx.x; k < (int)(sizeof(Ctl) / 4); k += kBlock) {
        dst[k] = src[k];
    }
    __threadfence_system();
}

__global__ __launch_bounds__(kBlock) void k_control(CtlArgs ca, Ctl* __restrict__ ctl, const double2* __restrict__ partials, const float* __restrict__ pw, const int32_t* __restrict__ slot_of, Ctl* host) {
    k_control_body(ca, ctl, partials, pw, slot_of, host, blockIdx.x, gridDim.x);
}

// ---- grouped launches: one launch runs an iteration's kernel for many plans -------
//
// Each plan's arguments sit in a device table; a block finds its plan and its block
// index within that plan's grid (bplan / bfirst, per grid shape) and runs the same
// body a single-plan launch of that grid runs, so every plan computes exactly what
// its own launches would.

enum GridShape { kShNodes, kShLean, kShGen, kShParts, kShRefresh, kShOne, kShapes };

struct PlanIter {
    Field f;
    Hash H;
    TrussIn tin;
    MoveArgs ma;
    CtlArgs ca;
    int n, fire, nparts, voxel;   // voxel: the voxel-trap move (no queues)
    float fscale, fsurf, skin;
    Ctl* ctl;
    int32_t* nbr;
    int32_t* nnb;
    float4 *X, *V, *F, *P0;
    uint8_t* typ;
    uint32_t* part;
    const uint16_t* lab;
    float *mv, *pw;
    const float* thr;
    uint8_t* flag;
    double2* partials;
    int32_t *rqueue, *mq, *mqi, *mq2, *mqd;
    const int32_t* slot_of;
    uint8_t* sticky;   // handed back to the general pass before (k_force queues them there)
    int nblk[kShapes];
};

#define TN_PLAN_BLOCK(shape)                              \
    const int v_ = bplan[blockIdx.x];                     \
    const PlanIter& P = tab[v_];                          \
    const int bid_ = (int)blockIdx.x - bfirst[v_];        \
    const int nb_ = P.nblk[shape]

__global__ __launch_bounds__(kBlock) void kg_force(const PlanIter* __restrict__ tab, const int32_t* __restrict__ bplan,
                                                   const int32_t* __restrict__ bfirst) {
    TN_PLAN_BLOCK(kShNodes);
    k_force_body(P.X, P.typ, P.nbr, P.nnb, P.fscale, P.fsurf, P.n, P.F, P.ctl, P.voxel ? nullptr : P.mq2, P.flag,
                 P.sticky, bid_, nb_);
}

template <class F>
__global__ __launch_bounds__(kBlock) void kg_move_easy(const PlanIter* __restrict__ tab,
                                                       const int32_t* __restrict__ bplan,
                                                       const int32_t* __restrict__ bfirst) {
    TN_PLAN_BLOCK(kShNodes);
    if (P.voxel) {   // the voxel-trap move's pass 1; pass 2 takes the interface queue's place
        k_move_voxel_body(P.f, P.ma, P.ctl, P.n, P.F, P.X, P.V, P.typ, P.part, P.lab, P.mv, P.pw, P.mq, &P.ctl->nmove,
                          bid_);
        return;
    }
    k_move_easy_body(as_field<F>(P.f), P.ma, P.ctl, P.n, P.F, P.X, P.V, P.typ, P.part, P.lab, P.mv, P.pw, P.mq, P.mqi, P.flag,
                             bid_, nb_);
}

// the four move passes: kQueue 0 = the general queue, 1 = interior (lean), 2 =
// interface (lean), 3 = the handed-back nodes (general)
template <int kQueue, class F>
__global__ __launch_bounds__(kBlock, TN_MOVE_WAVES) void kg_move(const PlanIter* __restrict__ tab,
                                                                 const int32_t* __restrict__ bplan,
                                                                 const int32_t* __restrict__ bfirst) {
    constexpr int kMode = kQueue == 1 ? kLeanInterior : (kQueue == 2 ? kLeanInterface : kGeneral);
    TN_PLAN_BLOCK(kMode == kGeneral ? kShGen : kShLean);
    if (P.voxel) {   // the voxel-trap move's pass 2 (its only queue)
        if (kQueue == 2) {
            k_move_voxel_wave_body(P.f, P.ma, P.ctl, P.mq, &P.ctl->nmove, P.F, P.X, P.V, P.typ, P.part, P.lab, P.mv,
                                   P.pw, bid_, nb_);
        }
        return;
    }
    const int32_t* queue = kQueue == 0 ? P.mq2 : (kQueue == 1 ? P.mqi : (kQueue == 2 ? P.mq : P.mqd));
    const int32_t* count = kQueue == 0 ? &P.ctl->nmove_rest
                                       : (kQueue == 1 ? &P.ctl->nmove_int
                                                      : (kQueue == 2 ? &P.ctl->nmove : &P.ctl->nmove_def));
    const bool lean = kMode != kGeneral;
    k_move_body<kMode>(as_field<F>(P.f), P.ma, P.ctl, queue, P.F, P.X, P.V, P.typ, P.part, P.lab, P.mv, P.pw, count,
                       lean ? &P.ctl->nmove_def : nullptr, lean ? P.mqd : nullptr, lean ? P.sticky : nullptr, bid_,
                       nb_);
}

__global__ __launch_bounds__(kBlock) void kg_stats(const PlanIter* __restrict__ tab, const int32_t* __restrict__ bplan,
                                                   const int32_t* __restrict__ bfirst) {
    TN_PLAN_BLOCK(kShParts);
    k_stats_body(P.X, P.P0, P.mv, P.pw, P.n, P.skin, P.fire, P.thr, P.ctl, P.rqueue, P.partials, bid_, nb_);
}

__global__ __launch_bounds__(kWave) void kg_truss_node(const PlanIter* __restrict__ tab,
                                                       const int32_t* __restrict__ bplan,
                                                       const int32_t* __restrict__ bfirst) {
    TN_PLAN_BLOCK(kShRefresh);
    k_truss_node_body(P.H, P.tin, P.n, P.rqueue, P.ctl, P.nbr, P.nnb, P.P0, bid_, nb_);
}

__global__ __launch_bounds__(kBlock) void kg_control(const PlanIter* __restrict__ tab,
                                                     const int32_t* __restrict__ bplan,
                                                     const int32_t* __restrict__ bfirst, Ctl* host) {
    TN_PLAN_BLOCK(kShOne);
    k_control_body(P.ca, P.ctl, P.partials, P.pw, P.slot_of, host + v_, bid_, nb_);
}

#undef TN_PLAN_BLOCK

__global__ void k_order_begin(Ctl* __restrict__ ctl) {
    if (threadIdx.x < 4) {
        ctl->order_cnt[threadIdx.x] = 0;
    }
}

}  // namespace tnk
