// nb_keys.hip -- stage 2, the octree build (buildtree.cl:12-200), from sorted
// octant-path keys instead of insertion.
//
// A body's place in the reference's octree is fixed by its octant path: the
// octant at each level, taken against cell centres that the reference derives
// from the root with one FP32 recurrence (buildtree.cl:124-136), and a body
// sits in the first level where no other body shares its path. So every body
// works out its own path with that same recurrence, 3 bits per level, and the
// bodies are sorted by it. The cells are the path prefixes that at
// least two bodies share; from the sorted keys they follow without any
// pointer chasing:
//   * a binary radix tree over the sorted keys (Karras, "Maximizing
//     parallelism in the construction of BVHs, octrees, and k-d trees", HPG
//     2012): internal node i finds its key range and split by binary searches
//     on delta(i, j), the common prefix length of keys i and j in bits;
//   * an octree cell of level k is the prefix of 3k bits: binary node X holds
//     the cells of the levels k with 3k in (delta(parent(X)), delta(X)] -- a
//     chain of them when the bodies of X share several more octants, exactly
//     as the reference's split loop creates them (buildtree.cl:106-165);
//   * the parent of X's top cell is the deepest cell of the nearest binary
//     ancestor that holds any, and it sits in the slot of its octant at the
//     parent's level; a body sits in the deepest cell of its nearest
//     ancestor that holds one.
// The result is written in the layout the rest of the pipeline reads:
// epoch-tagged child slots (a slot of an older epoch reads as empty, so the
// last step's tree needs no clearing) and per-cell records, cells numbered in
// key order with the root as cell 0. The sorted body order is the
// octant-path (Morton) order that the sort stage produces (sort.cl:12-76).
//
// Keys hold 21 levels in 63 bits (level 0 in the top bits). Bodies that share
// all 21 (rare: 2 of 4M in the clustered benchmark universe) form runs of
// equal keys, which are ordered by their paths extended to 84 levels: in a bucket
// that fits LDS every body counts the smaller ones of its run; in a larger bucket
// and after the radix passes one thread orders a run (after the passes in
// registers up to kMaxRun bodies, else through global memory). Limit: cells on levels below kBuildLevelLimit (bodies at
// most that deep); beyond it the build stops with a depth error, and a tree
// of more cells than the pool holds stops it with a pool error.
#include "nb_device.h"

namespace nb {

constexpr int kKeyLevels = 21; // levels per 64-bit key word (63 bits)
constexpr int kDeepWords = 3;  // key words past the first: levels 21 .. 83
constexpr int kMaxRun = 16;    // bodies sharing the first 21 levels, per run

// a child slot of the current tree: (epoch << 32) | child (nb_tree.hip reads them)
__device__ __forceinline__ unsigned long long slot_tag(uint32_t ep, int v)
{
    return ((unsigned long long)ep << 32) | (uint32_t)v;
}

__device__ __forceinline__ int key_octant(float cx, float cy, float cz, float4 p)
{
    return (cx < p.x ? 1 : 0) | (cy < p.y ? 2 : 0) | (cz < p.z ? 4 : 0);
}

// the child centre of octant `o` (buildtree.cl:124-136: x = parent - r/2 +
// (bit ? r : 0), r the parent's half size)
__device__ __forceinline__ void key_descend(float &cx, float &cy, float &cz, float &r, int o)
{
    const float rh = r * 0.5f;
    cx = (cx - rh) + ((o & 1) ? r : 0.0f);
    cy = (cy - rh) + ((o & 2) ? r : 0.0f);
    cz = (cz - rh) + ((o & 4) ? r : 0.0f);
    r = rh;
}

// the key of a body at p: 21 levels of its octant path from the root cell
__device__ __forceinline__ unsigned long long path_key(float cx, float cy, float cz, float r, float4 p)
{
    unsigned long long k = 0;
#pragma unroll
    for (int L = 0; L < kKeyLevels; ++L) {
        const int o = key_octant(cx, cy, cz, p);
        k = (k << 3) | (unsigned long long)o;
        key_descend(cx, cy, cz, r, o);
    }
    return k;
}

// The level counters of the tree to be built, and no levels until it is there
// (one block of at least kMaxDepth threads): a build that an error stops leaves
// none to summarize.
__device__ __forceinline__ void clear_levels(const Dev &d)
{
    const int t = threadIdx.x;
    if (t < kMaxDepth) d.lvl_count[t * kLevelLine] = d.lvl_count[(kMaxDepth + t) * kLevelLine] = 0;
    if (t == 0) {
        d.ctl->levels = 0;
        d.ctl->live_cells = 0;
    }
}

// ---------------------------------------------------------------------------
// Keys: 21 levels of each body's octant path, level 0 in bits 62..60, for the
// bodies in the order `order` (the identity when null).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_keys(Dev d, const int *__restrict__ order, unsigned long long *key, int *val)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const Ctl *ctl = d.ctl;
    if (blockIdx.x == 0) clear_levels(d);
    if (i >= d.n || ctl->error) return;
    const int b = order ? order[i] : i;
    key[i] = path_key(ctl->root[0], ctl->root[1], ctl->root[2], ctl->radius, d.pm4[b]);
    val[i] = b;
}

// ---------------------------------------------------------------------------
// LSD radix sort of (key, body) by 8-bit digits, 8 passes. A tile of
// kRsTile keys per block: per-tile digit counts (k_rs_count), their
// digit-major exclusive offsets over the tiles (k_rs_offsets), then each tile
// ranks its keys stably, sorts itself by digit in LDS and writes each digit's
// run out contiguously (k_rs_scatter).
// ---------------------------------------------------------------------------
constexpr int kRsThreads = 256;
constexpr int kRsPer = 8;
constexpr int kRsTile = kRsThreads * kRsPer; // 2048 keys
constexpr int kRsBins = 256;
static_assert(kRsTile == kKeyTile, "the engine sizes the per-tile arrays with kKeyTile");

__global__ __launch_bounds__(kRsThreads) void k_rs_count(const unsigned long long *__restrict__ key, int n, int shift,
                                                         unsigned *__restrict__ hist, int ntiles)
{
    __shared__ unsigned h[kRsBins];
    const int t = threadIdx.x;
    h[t] = 0;
    __syncthreads();
    const int base = blockIdx.x * kRsTile;
#pragma unroll
    for (int j = 0; j < kRsPer; ++j) {
        const int idx = base + j * kRsThreads + t;
        if (idx < n) atomicAdd(&h[(unsigned)(key[idx] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[(size_t)t * ntiles + blockIdx.x] = h[t];
}

// Block b: the exclusive prefix of digit b's counts over the tiles (into
// offs) and the digit's total. 1024 threads, each a contiguous run of tiles.
__global__ __launch_bounds__(1024) void k_rs_offsets(const unsigned *__restrict__ hist, int ntiles,
                                                     unsigned *__restrict__ offs, unsigned *__restrict__ total)
{
    __shared__ unsigned s[1024];
    const int t = threadIdx.x, b = blockIdx.x;
    const int per = (ntiles + 1023) / 1024;
    const unsigned *h = hist + (size_t)b * ntiles;
    unsigned *o = offs + (size_t)b * ntiles;
    unsigned sum = 0;
    for (int k = 0; k < per; ++k) {
        const int tile = t * per + k;
        if (tile < ntiles) sum += h[tile];
    }
    s[t] = sum;
    __syncthreads();
    for (int st = 1; st < 1024; st <<= 1) {
        const unsigned u = t >= st ? s[t - st] : 0u;
        __syncthreads();
        s[t] += u;
        __syncthreads();
    }
    unsigned run = s[t] - sum; // exclusive
    for (int k = 0; k < per; ++k) {
        const int tile = t * per + k;
        if (tile < ntiles) {
            o[tile] = run;
            run += h[tile];
        }
    }
    if (t == 1023) total[b] = s[1023];
}

__device__ __forceinline__ unsigned long long lanemask_lt()
{
    const int lane = threadIdx.x & 63;
    return lane ? (~0ull >> (64 - lane)) : 0ull;
}

// exclusive scan of one value per thread over a 256-thread block (v[t] in,
// the result returned); `s` is 256 words of LDS
__device__ __forceinline__ unsigned block_excl_scan256(unsigned v, unsigned *s)
{
    const int t = threadIdx.x;
    s[t] = v;
    __syncthreads();
    for (int st = 1; st < 256; st <<= 1) {
        const unsigned u = t >= st ? s[t - st] : 0u;
        __syncthreads();
        s[t] += u;
        __syncthreads();
    }
    const unsigned r = s[t] - v;
    __syncthreads();
    return r;
}

// One tile. A key's place in the tile sorted by digit = the tile's keys of
// smaller digits + its rank among the keys of its digit, counted in input
// order: keys of its digit in earlier rounds of 256, in earlier waves of this
// round, and in lower lanes of its wave (from eight ballots of the digit's
// bits). The tile is sorted in LDS, then written out in tile order, so that
// consecutive threads write consecutive places of each digit's run.
__global__ __launch_bounds__(kRsThreads) void k_rs_scatter(const unsigned long long *__restrict__ kin,
                                                           const int *__restrict__ vin,
                                                           unsigned long long *__restrict__ kout,
                                                           int *__restrict__ vout, int n, int shift,
                                                           const unsigned *__restrict__ hist,
                                                           const unsigned *__restrict__ offs,
                                                           const unsigned *__restrict__ total, int ntiles)
{
    __shared__ unsigned long long sk[kRsTile];
    __shared__ int sv[kRsTile];
    __shared__ unsigned gstart[kRsBins]; // global place of this tile's first key of each digit
    __shared__ unsigned lstart[kRsBins]; // its place in the tile
    __shared__ unsigned run[kRsBins];    // keys of each digit placed so far
    __shared__ unsigned cnt[4][kRsBins]; // per wave and digit, this round
    __shared__ unsigned scratch[kRsBins];
    const int t = threadIdx.x, w = t >> 6;
    const int tile = blockIdx.x, base = tile * kRsTile;
    const int tcount = min(kRsTile, n - base);
    const unsigned tot = total[t];
    const unsigned digit_base = block_excl_scan256(tot, scratch);
    gstart[t] = digit_base + offs[(size_t)t * ntiles + tile];
    lstart[t] = block_excl_scan256(hist[(size_t)t * ntiles + tile], scratch);
    run[t] = 0;
    cnt[0][t] = cnt[1][t] = cnt[2][t] = cnt[3][t] = 0;
    __syncthreads();
    const unsigned long long below = lanemask_lt();
    for (int j = 0; j < kRsPer; ++j) {
        const int li = j * kRsThreads + t;
        const bool valid = li < tcount;
        const unsigned long long k = valid ? kin[base + li] : 0ull;
        const int v = valid ? vin[base + li] : 0;
        const unsigned dg = (unsigned)(k >> shift) & 255u;
        unsigned long long peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const unsigned long long bal = __ballot((dg >> b) & 1u);
            peers &= ((dg >> b) & 1u) ? bal : ~bal;
        }
        const int rank = __popcll(peers & below);
        if (valid && rank == 0) cnt[w][dg] = (unsigned)__popcll(peers);
        __syncthreads();
        if (valid) {
            unsigned at = lstart[dg] + run[dg] + (unsigned)rank;
            for (int ww = 0; ww < w; ++ww) at += cnt[ww][dg];
            sk[at] = k;
            sv[at] = v;
        }
        __syncthreads();
        {
            run[t] += cnt[0][t] + cnt[1][t] + cnt[2][t] + cnt[3][t];
            cnt[0][t] = cnt[1][t] = cnt[2][t] = cnt[3][t] = 0;
        }
        __syncthreads();
    }
    for (int li = t; li < tcount; li += kRsThreads) {
        const unsigned long long k = sk[li];
        const unsigned dg = (unsigned)(k >> shift) & 255u;
        const unsigned dest = gstart[dg] + ((unsigned)li - lstart[dg]);
        kout[dest] = k;
        vout[dest] = sv[li];
    }
}

// ---------------------------------------------------------------------------
// Warm sort. After the first step the bodies come in the last tree's order
// (sorted[]), which the new keys nearly keep, and the last tree's sorted keys
// are still in kb_key[0]. Bucketing by splitters taken from those keys then
// moves most bodies a short way and every bucket is small:
//   * splitters: every kBucketT-th of the last tree's sorted keys (with the
//     bounding box, make_splitter);
//   * a body's bucket: the number of splitters <= its key. A block's bodies
//     are consecutive in the last order, so their buckets are nearly all in
//     a window of kWin around the one their places suggest: searched in an
//     LDS copy of the window's splitters, counted in LDS, one atomic per
//     bucket and block (k_keys_warm, with the keys); the counts' exclusive
//     scan (k_bucket_scan); then each body takes the next place of its
//     bucket the same way (k_bucket_scatter);
//   * each bucket is sorted by one block (k_bucket_sort): up to kBucketCap
//     bodies in LDS, a larger bucket (stale order) by radix passes through
//     device memory.
// The order inside a bucket before its sort depends on the atomics; the keys
// are distinct after the run ordering below (equal keys are ordered by their
// deeper levels), so the result does not.
// ---------------------------------------------------------------------------
constexpr int kBsThreads = 256; // blocks of the bucket sort
constexpr int kBsWaves = kBsThreads / 64;
static_assert(kBsThreads == kRsBins, "a thread per digit");

// the splitters of the next warm build alone (launch_bbox does it otherwise)
__global__ __launch_bounds__(256) void k_splitters(Dev d, int S)
{
    if (d.ctl->error) return;
    make_splitter(d, blockIdx.x * blockDim.x + threadIdx.x, S);
}

// the first j with spl[j] > k (S if none): spl is non-decreasing; searched
// outward from g, then by bisection (global memory). Invariant: (lo < 0 or spl[lo] <= k) and
// (hi >= S or spl[hi] > k).
__device__ __forceinline__ int bucket_of(const unsigned long long *__restrict__ spl, int S, unsigned long long k, int g)
{
    g = min(max(g, 0), S);
    int lo, hi;
    if (g < S && spl[g] <= k) {
        lo = g;
        hi = g + 1;
        for (int step = 1; hi < S && spl[hi] <= k; hi = lo + step) {
            lo = hi;
            step <<= 1;
        }
        hi = min(hi, S);
    } else {
        hi = g;
        lo = g - 1;
        for (int step = 1; lo >= 0 && spl[lo] > k; lo = hi - step) {
            hi = lo;
            step <<= 1;
        }
        lo = max(lo, -1);
    }
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (spl[mid] <= k) lo = mid;
        else hi = mid;
    }
    return hi;
}

// Bucket windows: a block's bodies (consecutive in the last tree's order)
// expect buckets near first / kBucketT + 1; buckets w0 .. w0 + kWin - 1 (w0
// = that - kWin / 4) are searched in an LDS copy of their splitters and
// counted in LDS bins, one LDS atomic per body; a body outside the window is
// searched in global memory and goes to its bucket's counter directly. Lanes
// that elect one atomic per bin and wave take a round per bin: build stage, us,
// with election and 64 buckets / one atomic a body and 64 / and 128: 32,768 bodies
// (disk, dt 0.025) 65 / 62 / 58, 1M (Plummer, dt 0.025) 150 / 144 / 141, 4M
// clusters (dt 1e-3) 368 / 364 / 361.
constexpr int kWinPer = 8;
constexpr int kWinBodies = 256 * kWinPer;
constexpr int kWin = 128;

// ws[0 .. kWin]: spl[w0 - 1 .. w0 + kWin - 1], 0 below the first splitter
// and ~0 past the last (keys use 63 bits); block-wide, before a barrier
__device__ __forceinline__ void load_window(const unsigned long long *__restrict__ spl, int S, int w0,
                                            unsigned long long *ws)
{
    const int t = threadIdx.x;
    if (t <= kWin) {
        const int j = w0 - 1 + t;
        ws[t] = j < 0 ? 0ull : (j >= S ? ~0ull : spl[j]);
    }
}

// bucket of k if it is one of w0 .. w0 + kWin - 1, else -1
__device__ __forceinline__ int bucket_in_window(const unsigned long long *ws, int w0, unsigned long long k)
{
    if (k < ws[0] || k >= ws[kWin]) return -1;
    int lo = 0, hi = kWin; // ws[lo] <= k < ws[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (ws[mid] <= k) lo = mid;
        else hi = mid;
    }
    return w0 - 1 + hi;
}

// Warm keys: body order[i] (the last tree's order) at place i: its key and
// value, its bucket (bid) and the bucket counts. Its record comes from
// `staged` (the records in that order, as the last fused update wrote them)
// when given, else from pm4. A block takes kWarmPer * 256 places, whose
// buckets are expected near first / kBucketT + 1; the window starts kWin / 4
// below. Every load is issued before the arithmetic.
constexpr int kWarmPer = 4;
constexpr int kWarmBodies = 256 * kWarmPer;

__global__ __launch_bounds__(256) void k_keys_warm(Dev d, const int *__restrict__ order,
                                                   const float4 *__restrict__ staged,
                                                   const unsigned long long *__restrict__ spl, int S,
                                                   unsigned long long *__restrict__ key, int *__restrict__ val,
                                                   int *__restrict__ bid, unsigned *__restrict__ bcnt)
{
    __shared__ unsigned h[kWin];
    __shared__ unsigned long long ws[kWin + 1];
    const int t = threadIdx.x, first = blockIdx.x * kWarmBodies;
    const int n = d.n;
    const Ctl *ctl = d.ctl;
    const int err = ctl->error;
    if (blockIdx.x == 0) clear_levels(d);
    const int w0 = first / kBucketT + 1 - kWin / 4;
    if (t < kWin) h[t] = 0;
    int b[kWarmPer];
    float4 p[kWarmPer];
#pragma unroll
    for (int j = 0; j < kWarmPer; ++j) {
        const int ic = min(first + j * 256 + t, n - 1);
        b[j] = order[ic];
        p[j] = staged ? staged[ic] : d.pm4[b[j]];
    }
    load_window(spl, S, w0, ws);
    if (block_stops(err)) return;
    const float rx = ctl->root[0], ry = ctl->root[1], rz = ctl->root[2], rr = ctl->radius;
#pragma unroll
    for (int j = 0; j < kWarmPer; ++j) {
        const int i = first + j * 256 + t;
        const bool valid = i < n;
        const unsigned long long k = path_key(rx, ry, rz, rr, p[j]);
        int bk = valid ? bucket_in_window(ws, w0, k) : -1;
        if (bk >= 0) {
            atomicAdd(&h[bk - w0], 1u);
        } else if (valid) {
            bk = bucket_of(spl, S, k, i / kBucketT + 1);
            atomicAdd(&bcnt[bk], 1u);
        }
        if (valid) {
            key[i] = k;
            val[i] = b[j];
            bid[i] = bk;
        }
    }
    __syncthreads();
    if (t < kWin && h[t]) atomicAdd(&bcnt[w0 + t], h[t]);
}

// exclusive scan of the S + 1 bucket counts: bstart[0 .. S+1] (one block).
// Chunks of kBsChunk counts go through LDS (coalesced loads and stores; the
// 8 of a thread padded to 9 words, so its reads hit distinct banks), each
// thread scans 8 consecutive counts, and the chunk's carry moves on.
constexpr int kBsPer = 8;
constexpr int kBsChunk = 1024 * kBsPer;

__device__ __forceinline__ int bs_pad(int i) { return i + i / kBsPer; }

__global__ __launch_bounds__(1024) void k_bucket_scan(const Ctl *ctl, const unsigned *__restrict__ bcnt, int S,
                                                      unsigned *__restrict__ bstart)
{
    __shared__ unsigned c[kBsChunk + kBsChunk / kBsPer];
    __shared__ unsigned wsum[16];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    if (block_stops(ctl->error)) return;
    const int nb = S + 1;
    unsigned carry = 0;
    for (int c0 = 0; c0 < nb; c0 += kBsChunk) {
#pragma unroll
        for (int k = 0; k < kBsPer; ++k) {
            const int i = k * 1024 + t;
            c[bs_pad(i)] = c0 + i < nb ? bcnt[c0 + i] : 0u;
        }
        __syncthreads();
        unsigned v[kBsPer], sum = 0;
#pragma unroll
        for (int k = 0; k < kBsPer; ++k) {
            v[k] = c[bs_pad(t * kBsPer + k)];
            sum += v[k];
        }
        unsigned x = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        if (lane == 63) wsum[w] = x;
        __syncthreads();
        unsigned below = 0, total = 0;
#pragma unroll
        for (int ww = 0; ww < 16; ++ww) {
            const unsigned ws = wsum[ww];
            below += ww < w ? ws : 0u;
            total += ws;
        }
        unsigned run = carry + below + x - sum;
#pragma unroll
        for (int k = 0; k < kBsPer; ++k) {
            c[bs_pad(t * kBsPer + k)] = run;
            run += v[k];
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kBsPer; ++k) {
            const int i = k * 1024 + t;
            if (c0 + i < nb) bstart[c0 + i] = c[bs_pad(i)];
        }
        carry += total;
        __syncthreads();
    }
    if (t == 0) bstart[nb] = carry;
}

// Each body takes the next place of its bucket: LDS counters for the buckets
// of the block's window (one global atomic per bucket and block), a global
// atomic for a bucket outside it. SCAN (S < kScatterScan): every block works out
// the buckets' starts from their counts by itself, and the first block keeps
// them for the sort; a launch less (4.5 us) for about 1 us of it.
constexpr int kScatterScan = 1024;

// exclusive scan of v over 256 threads, wave by wave; wsum: 4 words of LDS.
// Ends with wsum[3] = the total.
__device__ __forceinline__ unsigned scan256_total(unsigned v, unsigned *wsum)
{
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    unsigned x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    const unsigned w0 = wsum[0], w1 = wsum[1], w2 = wsum[2], w3 = wsum[3];
    __syncthreads();
    if (t == 0) wsum[3] = w0 + w1 + w2 + w3;
    return x - v + (w > 0 ? w0 : 0u) + (w > 1 ? w1 : 0u) + (w > 2 ? w2 : 0u);
}

template <bool SCAN>
__global__ __launch_bounds__(256) void k_bucket_scatter(const Ctl *ctl, const unsigned long long *__restrict__ kin,
                                                        const int *__restrict__ vin, const int *__restrict__ bid,
                                                        unsigned long long *__restrict__ kout, int *__restrict__ vout,
                                                        int n, const unsigned *__restrict__ bcnt, int S,
                                                        unsigned *__restrict__ bstart, unsigned *__restrict__ bfill)
{
    __shared__ unsigned h[kWin], hb[kWin];
    __shared__ unsigned starts[SCAN ? kScatterScan : 1], wsum[4];
    const int err = ctl->error;
    const int t = threadIdx.x, first = blockIdx.x * kWinBodies;
    const int w0 = first / kBucketT + 1 - kWin / 4;
    if (t < kWin) h[t] = 0;
    unsigned long long k[kWinPer];
    int v[kWinPer], b[kWinPer];
#pragma unroll
    for (int j = 0; j < kWinPer; ++j) {
        const int i = min(first + j * 256 + t, n - 1);
        k[j] = kin[i];
        v[j] = vin[i];
        b[j] = bid[i];
    }
    if (SCAN) {
        unsigned c[4], sum = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = 4 * t + q;
            c[q] = i <= S ? bcnt[i] : 0u;
            sum += c[q];
        }
        unsigned run = scan256_total(sum, wsum);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int i = 4 * t + q;
            starts[i] = run;
            if (blockIdx.x == 0 && i <= S) bstart[i] = run;
            run += c[q];
        }
        if (blockIdx.x == 0 && t == 0) bstart[S + 1] = (unsigned)n;
    }
    if (__syncthreads_or(err)) return;
    const auto start = [&](int bk) { return SCAN ? starts[bk] : bstart[bk]; };
    unsigned at[kWinPer];
#pragma unroll
    for (int j = 0; j < kWinPer; ++j) {
        const bool valid = first + j * 256 + t < n;
        const unsigned o = (unsigned)(b[j] - w0);
        if (!valid) continue;
        at[j] = o < (unsigned)kWin ? atomicAdd(&h[o], 1u) : start(b[j]) + atomicAdd(&bfill[b[j]], 1u);
    }
    __syncthreads();
    if (t < kWin) hb[t] = h[t] ? start(w0 + t) + atomicAdd(&bfill[w0 + t], h[t]) : 0u;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kWinPer; ++j) {
        if (first + j * 256 + t >= n) continue;
        const unsigned o = (unsigned)(b[j] - w0);
        const unsigned pos = o < (unsigned)kWin ? hb[o] + at[j] : at[j];
        kout[pos] = k[j];
        vout[pos] = v[j];
    }
}

// ---------------------------------------------------------------------------
// First builds of up to kColdBodies bodies. There is no last order, so the
// splitters come from a sample: one block sorts the keys of 1024 or 2048 bodies
// spread over the indices and takes every (samples / (S + 1))-th (k_sample).
// Blocks of kColdPer bodies then find each body's bucket among all S <= 1024
// splitters in LDS, count the buckets in LDS and take their places in each
// bucket with one atomic per bucket and block (k_keys_cold); the scan of the
// counts gives the buckets' starts (k_cold_scatter), and the buckets are sorted
// as in a warm build. Four launches where the radix sort takes 26: the first
// build of 16,384 bodies takes 58 us instead of 187, of 100,003 87 instead of
// 200.
// A bucket has at least 2 samples to its name on average, so that one above
// kColdCap = 8 times its size (Gamma(2) > 16: 2e-6) is rare.
// ---------------------------------------------------------------------------
constexpr int kColdCap = 1024; // bodies of a bucket sorted in LDS
constexpr int kColdPer = 512;
constexpr int kColdMax = kColdBodies / kColdT; // splitters
constexpr int kSampleThreads = 1024;

// The value of lane ^ STEP: DPP moves (quad_perm, row_half_mirror then the
// reversed quads, row_ror) and the row swaps of permlane, which leave the LDS
// unit alone.
template <int CTRL> __device__ __forceinline__ unsigned dpp_u(unsigned v)
{
    return (unsigned)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, false);
}

template <int STEP> __device__ __forceinline__ unsigned lane_xor(unsigned v)
{
    if constexpr (STEP == 1) return dpp_u<0xB1>(v);
    if constexpr (STEP == 2) return dpp_u<0x4E>(v);
    if constexpr (STEP == 4) return dpp_u<0x1B>(dpp_u<0x141>(v));
    if constexpr (STEP == 8) return dpp_u<0x128>(v);
    const bool high = (threadIdx.x & STEP) != 0;
    if constexpr (STEP == 16) {
        const auto s = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        return high ? s[0] : s[1];
    } else {
        const auto s = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return high ? s[0] : s[1];
    }
}

template <int STEP> __device__ __forceinline__ unsigned long long lane_xor64(unsigned long long v)
{
    return (unsigned long long)lane_xor<STEP>((unsigned)(v >> 32)) << 32 | lane_xor<STEP>((unsigned)v);
}

template <int R, class Other>
__device__ __forceinline__ void keep(unsigned long long (&k)[R], bool smaller, const Other &other)
{
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const unsigned long long o = other(r);
        if ((o < k[r]) == smaller) k[r] = o;
    }
}

// The index of sample i: multiples of the golden ratio modulo 1 spread evenly, and
// unlike equal strides they keep no step with an order that has a period (a
// lattice, row by row, of which equal strides may see one face).
__device__ __forceinline__ int sample_index(int i, int n)
{
    return (int)(((unsigned long long)((unsigned)i * 0x9E3779B1u) * (unsigned)n) >> 32);
}

// R samples per thread, places R t .. R t + R - 1 of the bitonic sort: partners
// `step` places apart are in the thread's registers, in its wave, or in LDS.
template <int R> __global__ __launch_bounds__(kSampleThreads) void k_sample(Dev d, int S)
{
    constexpr int T = kSampleThreads, M = R * T;
    static_assert(R == 1 || R == 2, "partners in a thread: places 0 and 1");
    __shared__ unsigned long long sk[R][T];
    const Ctl *ctl = d.ctl;
    if (block_stops(ctl->error)) return;
    const int t = threadIdx.x, n = d.n;
    const float rx = ctl->root[0], ry = ctl->root[1], rz = ctl->root[2], rr = ctl->radius;
    unsigned long long k[R];
#pragma unroll
    for (int r = 0; r < R; ++r) k[r] = path_key(rx, ry, rz, rr, d.pm4[sample_index(R * t + r, n)]);
    for (int j = t; j <= S; j += T) d.kb_bcnt[j] = 0;
    for (int size = 2; size <= M; size <<= 1) {
        const bool up = (R * t & size) == 0;
        for (int step = size >> 1; step >= R; step >>= 1) {
            const bool smaller = ((R * t & step) == 0) == up;
            const int lanes = step / R; // the same in every thread
            switch (lanes) {
            case 1: keep(k, smaller, [&](int r) { return lane_xor64<1>(k[r]); }); break;
            case 2: keep(k, smaller, [&](int r) { return lane_xor64<2>(k[r]); }); break;
            case 4: keep(k, smaller, [&](int r) { return lane_xor64<4>(k[r]); }); break;
            case 8: keep(k, smaller, [&](int r) { return lane_xor64<8>(k[r]); }); break;
            case 16: keep(k, smaller, [&](int r) { return lane_xor64<16>(k[r]); }); break;
            case 32: keep(k, smaller, [&](int r) { return lane_xor64<32>(k[r]); }); break;
            default:
                __syncthreads();
#pragma unroll
                for (int r = 0; r < R; ++r) sk[r][t] = k[r];
                __syncthreads();
                keep(k, smaller, [&](int r) { return sk[r][t ^ lanes]; });
            }
        }
        if constexpr (R == 2) {
            const unsigned long long lo = min(k[0], k[1]), hi = max(k[0], k[1]);
            k[0] = up ? lo : hi;
            k[1] = up ? hi : lo;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) sk[r][t] = k[r];
    __syncthreads();
    for (int j = t; j < S; j += T) {
        const int at = (int)((long long)(j + 1) * M / (S + 1));
        d.kb_spl[j] = sk[at % R][at / R];
    }
}

// (key, body) in the bodies' order, and where[i] = place in the bucket << 11 |
// bucket (a place is below 2^17, a bucket at most 2^10)
__global__ __launch_bounds__(256) void k_keys_cold(Dev d, int S, unsigned long long *__restrict__ key,
                                                   int *__restrict__ where)
{
    __shared__ unsigned long long spl[kColdMax];
    __shared__ unsigned h[kColdMax + 1];
    const Ctl *ctl = d.ctl;
    const int t = threadIdx.x, n = d.n, first = blockIdx.x * kColdPer;
    if (blockIdx.x == 0) clear_levels(d);
    if (__syncthreads_or(ctl->error)) return;
    for (int j = t; j < S; j += 256) spl[j] = d.kb_spl[j];
    for (int j = t; j <= S; j += 256) h[j] = 0;
    __syncthreads();
    const float rx = ctl->root[0], ry = ctl->root[1], rz = ctl->root[2], rr = ctl->radius;
    constexpr int per = kColdPer / 256;
    unsigned long long k[per];
    int b[per];
    unsigned at[per];
#pragma unroll
    for (int u = 0; u < per; ++u) {
        const int i = first + u * 256 + t;
        k[u] = path_key(rx, ry, rz, rr, d.pm4[min(i, n - 1)]);
        if (i < n) key[i] = k[u];
        b[u] = 0;
    }
    // b = the splitters <= k, all bodies of the thread at once
#pragma unroll
    for (int step = kColdMax; step > 0; step >>= 1) {
#pragma unroll
        for (int u = 0; u < per; ++u)
            if (b[u] + step <= S && spl[b[u] + step - 1] <= k[u]) b[u] += step;
    }
#pragma unroll
    for (int u = 0; u < per; ++u) {
        if (first + u * 256 + t >= n) b[u] = -1;
        else at[u] = atomicAdd(&h[b[u]], 1u);
    }
    __syncthreads();
    for (int j = t; j <= S; j += 256)
        if (h[j]) h[j] = atomicAdd(&d.kb_bcnt[j], h[j]);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < per; ++u)
        if (b[u] >= 0) where[first + u * 256 + t] = (int)((h[b[u]] + at[u]) << 11 | (unsigned)b[u]);
}

__global__ __launch_bounds__(256) void k_cold_scatter(const Ctl *ctl, int n, int S, const unsigned *__restrict__ bcnt,
                                                      const unsigned long long *__restrict__ kin,
                                                      const int *__restrict__ where,
                                                      unsigned long long *__restrict__ kout, int *__restrict__ vout,
                                                      unsigned *__restrict__ bstart)
{
    constexpr int per = (kColdMax + 1 + 255) / 256;
    __shared__ unsigned starts[per * 256], wsum[4];
    const int err = ctl->error;
    const int t = threadIdx.x, i = blockIdx.x * 256 + t;
    const unsigned long long k = i < n ? kin[i] : 0ull;
    const int w = i < n ? where[i] : 0;
    unsigned c[per], sum = 0;
#pragma unroll
    for (int q = 0; q < per; ++q) {
        const int j = per * t + q;
        c[q] = j <= S ? bcnt[j] : 0u;
        sum += c[q];
    }
    unsigned run = scan256_total(sum, wsum);
#pragma unroll
    for (int q = 0; q < per; ++q) {
        const int j = per * t + q;
        starts[j] = run;
        if (blockIdx.x == 0 && j <= S) bstart[j] = run;
        run += c[q];
    }
    if (blockIdx.x == 0 && t == 0) bstart[S + 1] = (unsigned)n;
    if (__syncthreads_or(err) || i >= n) return;
    const unsigned pos = starts[w & 2047] + ((unsigned)w >> 11);
    kout[pos] = k;
    vout[pos] = i;
}

struct RankLds {
    unsigned cnt[kBsWaves][kRsBins]; // per wave and digit in a round; then their exclusive prefix over the waves
    unsigned lstart[kRsBins];        // first place of each digit
    unsigned run[kRsBins];           // places of each digit taken by earlier rounds
    unsigned tot[kRsBins];           // digit counts; then each round's per-digit total
    unsigned wsum[kBsWaves];
};

// exclusive scan over the first 256 threads of the block (each passes v; the
// others pass anything and ignore the result); every thread must call it
__device__ __forceinline__ unsigned scan256_excl(unsigned v, unsigned *wsum)
{
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    unsigned x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    unsigned add = 0;
    for (int ww = 0; ww < w && ww < 4; ++ww) add += wsum[ww];
    __syncthreads();
    return add + x - v;
}

// One stable pass over m keys by the 8 bits at `shift`: (sk, sv) -> (dk, dv),
// all m places of dk/dv written. Rounds of kBsThreads keys in input order: a
// key's place = its digit's first place + the places earlier rounds took + the
// keys of its digit in lower waves of this round + its rank in its wave (eight
// ballots of the digit's bits). The pointers are LDS or global.
template <class SK, class SV, class DK, class DV>
__device__ void rank_pass(SK sk, SV sv, DK dk, DV dv, int m, int shift, RankLds &R)
{
    const int t = threadIdx.x, w = t >> 6;
    if (t < kRsBins) R.tot[t] = 0;
    for (int x = t; x < kBsWaves * kRsBins; x += kBsThreads) (&R.cnt[0][0])[x] = 0;
    __syncthreads();
    for (int j = t; j < m; j += kBsThreads) atomicAdd(&R.tot[(unsigned)(sk[j] >> shift) & 255u], 1u);
    __syncthreads();
    const unsigned ls = scan256_excl(t < kRsBins ? R.tot[t] : 0u, R.wsum);
    if (t < kRsBins) {
        R.lstart[t] = ls;
        R.run[t] = 0;
    }
    __syncthreads();
    const int lane = t & 63;
    const unsigned long long below = lane ? (~0ull >> (64 - lane)) : 0ull;
    for (int r0 = 0; r0 < m; r0 += kBsThreads) {
        const int j = r0 + t;
        const bool valid = j < m;
        const unsigned long long k = valid ? sk[j] : 0ull;
        const int v = valid ? sv[j] : 0;
        const unsigned dg = (unsigned)(k >> shift) & 255u;
        unsigned long long peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const unsigned long long bal = __ballot((dg >> b) & 1u);
            peers &= ((dg >> b) & 1u) ? bal : ~bal;
        }
        const int rank = __popcll(peers & below);
        if (valid && rank == 0) R.cnt[w][dg] = (unsigned)__popcll(peers);
        __syncthreads();
        if (t < kRsBins) {
            unsigned acc = 0;
#pragma unroll
            for (int ww = 0; ww < kBsWaves; ++ww) {
                const unsigned c = R.cnt[ww][t];
                R.cnt[ww][t] = acc;
                acc += c;
            }
            R.tot[t] = acc;
        }
        __syncthreads();
        if (valid) {
            const unsigned at = R.lstart[dg] + R.run[dg] + R.cnt[w][dg] + (unsigned)rank;
            dk[at] = k;
            dv[at] = v;
        }
        __syncthreads();
        if (t < kRsBins) {
            R.run[t] += R.tot[t];
#pragma unroll
            for (int ww = 0; ww < kBsWaves; ++ww) R.cnt[ww][t] = 0;
        }
        __syncthreads();
    }
}

// the highest key bit that differs inside key[0 .. m-1] (-1: all equal)
template <class SK>
__device__ int varying_top_bit(SK key, int m, unsigned long long *red)
{
    const int t = threadIdx.x;
    if (t == 0) *red = 0ull;
    __syncthreads();
    const unsigned long long k0 = key[0];
    unsigned long long x = 0;
    for (int j = t; j < m; j += kBsThreads) x |= key[j] ^ k0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x |= __shfl_xor(x, o);
    if ((t & 63) == 0 && x) atomicOr(red, x);
    __syncthreads();
    const unsigned long long all = *red;
    __syncthreads();
    return all ? 63 - __clzll((long long)all) : -1;
}

// ---------------------------------------------------------------------------
// Runs of equal 21-level keys: their bodies' paths extended to 84 levels
// (deep[0..2][pos], levels 21 .. 83), each run ordered by them: by the bucket
// sort in a warm build, by one thread per run (k_deep_runs) after the radix
// sort.
// ---------------------------------------------------------------------------
// levels 21 .. 83 of body p's path, three words of 21 levels
__device__ __forceinline__ void deep_words(float rx, float ry, float rz, float rr, float4 p,
                                           unsigned long long *out)
{
    float cx = rx, cy = ry, cz = rz, r = rr;
    for (int L = 0; L < kKeyLevels; ++L) key_descend(cx, cy, cz, r, key_octant(cx, cy, cz, p));
    for (int w = 0; w < kDeepWords; ++w) {
        unsigned long long x = 0;
        for (int L = 0; L < kKeyLevels; ++L) {
            const int o = key_octant(cx, cy, cz, p);
            x = (x << 3) | (unsigned long long)o;
            key_descend(cx, cy, cz, r, o);
        }
        out[w] = x;
    }
}

// deep path of run element x before that of y (words at base[w * n + .])
__device__ __forceinline__ bool deep_less(const unsigned long long *base, size_t n, int x, int y)
{
    for (int w = 0; w < kDeepWords; ++w) {
        const unsigned long long a = base[w * n + x], b = base[w * n + y];
        if (a != b) return a < b;
    }
    return false;
}

// A run longer than kMaxRun (bodies i .. i+m-1): ordered through global
// memory by one thread. The deep words go to `deep` in the run's current
// order, a permutation of the run is merge-sorted (stable, in perm with tmp
// as the merge buffer), then the bodies and their deep words are gathered
// through staging copies. perm, tmp, stage_k and stage_v are n-element
// buffers that nothing else uses at this point; each run works in its own
// range [i, i+m) of them.
__device__ void order_long_run(const Dev &d, int i, int m, int *val, unsigned long long *deep, int *perm, int *tmp,
                               unsigned long long *stage_k, int *stage_v)
{
    const size_t n = (size_t)d.n;
    const Ctl *ctl = d.ctl;
    const float rx = ctl->root[0], ry = ctl->root[1], rz = ctl->root[2], rr = ctl->radius;
    for (int a = 0; a < m; ++a) {
        unsigned long long w3[kDeepWords];
        deep_words(rx, ry, rz, rr, d.pm4[val[i + a]], w3);
        for (int w = 0; w < kDeepWords; ++w) deep[w * n + i + a] = w3[w];
        perm[i + a] = a;
    }
    const unsigned long long *base = deep + i;
    int *src = perm + i, *dst = tmp + i;
    for (int width = 1; width < m; width <<= 1) {
        for (int lo = 0; lo < m; lo += 2 * width) {
            const int mid = min(lo + width, m), hi = min(lo + 2 * width, m);
            int a = lo, b = mid, o = lo;
            while (a < mid && b < hi) dst[o++] = deep_less(base, n, src[b], src[a]) ? src[b++] : src[a++];
            while (a < mid) dst[o++] = src[a++];
            while (b < hi) dst[o++] = src[b++];
        }
        int *t = src;
        src = dst;
        dst = t;
    }
    for (int a = 0; a < m; ++a) stage_v[i + a] = val[i + src[a]];
    for (int a = 0; a < m; ++a) val[i + a] = stage_v[i + a];
    for (int w = 0; w < kDeepWords; ++w) {
        for (int a = 0; a < m; ++a) stage_k[i + a] = deep[w * n + i + src[a]];
        for (int a = 0; a < m; ++a) deep[w * n + i + a] = stage_k[i + a];
    }
    for (int a = 1; a < m; ++a)
        if (!deep_less(base, n, a - 1, a)) flag_error(d.ctl, kErrDepth); // one 84-level path
}

// Bucket blockIdx.x of the S + 1, in place in (key, val), and the runs of equal
// keys in it (a run is never split: its keys fall into one bucket).
//
// A bucket of up to kBucketCap bodies stays in LDS: one distribution by the 8
// highest key bits that vary inside it, whose order inside a digit is free,
// then every key counts the smaller keys of its digit, which gives its place.
// A digit holds a few keys (a bucket covers about a cell of 256 bodies, 8 bits
// are two to three levels below it), so the counts are short; a digit that
// holds them all costs kBucketCap reads, no more. Five barriers and about 40
// dependent LDS accesses in all, where radix passes over every varying digit
// took some 30 of each per pass (one wave per bucket, 5 or 6 passes):
// bound by that latency, not by bandwidth or the adds. One launch instead of
// three (buckets, large buckets, runs): 16,384 bodies 29 -> 6.0 us, 1M 42 ->
// 22 us, 4M 85 -> 58 us.
// Keys that meet an equal key get their levels 21 .. 83 here too, and their
// place among the equals by counting the smaller of those.
//
// A larger bucket goes through device memory by stable radix passes ((tkey,
// tval) are free n-element buffers), and one thread orders each of its runs.
constexpr int kCountStep = 4; // keys a count reads at once
template <int CAP> struct BucketLds {
    unsigned long long sk[CAP + kCountStep]; // past the bucket: ~0 (keys use 63 bits)
    unsigned long long dw[kDeepWords][CAP]; // deep words of the keys that have equals
    int sv[CAP];
    unsigned start[kRsBins + 1];
    unsigned cnt[kRsBins];
    unsigned wsum[kBsWaves];
    unsigned long long diff[kBsWaves];
};

__device__ void sort_large_bucket(const Dev &d, unsigned long long *key, int *val, unsigned long long *deep,
                                  unsigned long long *tkey, int *tval, int *perm, int *tmp, int base, int m,
                                  bool warm, RankLds &R, unsigned long long *red)
{
    const int t = threadIdx.x;
    if (warm && t == 0) atomicAdd(&d.ctl->large_buckets, 1);
    unsigned long long *k0 = key + base, *k1 = tkey + base;
    int *v0 = val + base, *v1 = tval + base;
    const int top = varying_top_bit(k0, m, red);
    bool in_tmp = false;
    for (int shift = 0; shift <= top; shift += 8) {
        if (in_tmp) rank_pass(k1, v1, k0, v0, m, shift, R);
        else rank_pass(k0, v0, k1, v1, m, shift, R);
        in_tmp = !in_tmp;
    }
    if (in_tmp) {
        for (int j = t; j < m; j += kBsThreads) {
            k0[j] = k1[j];
            v0[j] = v1[j];
        }
    }
    __syncthreads();
    for (int j = t; j + 1 < m; j += kBsThreads) {
        const unsigned long long k = k0[j];
        if (k0[j + 1] != k || (j > 0 && k0[j - 1] == k)) continue; // not the start of a run
        int run = 2;
        while (j + run < m && k0[j + run] == k) ++run;
        order_long_run(d, base + j, run, val, deep, perm, tmp, tkey, tval);
    }
}

template <int CAP>
__global__ __launch_bounds__(kBsThreads) void k_bucket_sort(Dev d, unsigned long long *__restrict__ key,
                                                            int *__restrict__ val,
                                                            unsigned long long *__restrict__ deep,
                                                            unsigned long long *__restrict__ tkey,
                                                            int *__restrict__ tval, int *__restrict__ perm,
                                                            int *__restrict__ tmp,
                                                            const unsigned *__restrict__ bstart, bool warm)
{
    __shared__ union {
        BucketLds<CAP> b;
        struct {
            RankLds rank;
            unsigned long long red;
        } large;
    } lds;
    constexpr int kPer = CAP / kBsThreads;
    static_assert(CAP % kBsThreads == 0, "whole rows of the block");
    const Ctl *ctl = d.ctl;
    const int t = threadIdx.x, w = t >> 6;
    const int base = (int)bstart[blockIdx.x], m = (int)bstart[blockIdx.x + 1] - base;
    // the same decision in every wave: a bucket sorted at the same time may flag
    // an error, and a wave that left then would leave its keys out of the counts
    if (__syncthreads_or(ctl->error) || m <= 1) return;
    if (m > CAP) {
        sort_large_bucket(d, key, val, deep, tkey, tval, perm, tmp, base, m, warm, lds.large.rank, &lds.large.red);
        return;
    }
    BucketLds<CAP> &s = lds.b;
    const size_t n = (size_t)d.n;
    unsigned long long k[kPer], diff = 0;
    int v[kPer];
    const unsigned long long k0 = key[base];
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
        const int i = r * kBsThreads + t;
        k[r] = i < m ? key[base + i] : k0;
        v[r] = i < m ? val[base + i] : 0;
        diff |= k[r] ^ k0;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) diff |= __shfl_xor(diff, o);
    if ((t & 63) == 0) s.diff[w] = diff;
    s.cnt[t] = 0;
    __syncthreads();
    diff = s.diff[0] | s.diff[1] | s.diff[2] | s.diff[3];
    const int top = diff ? 63 - __clzll((long long)diff) : 0;
    const int shift = max(0, top - 7);
    unsigned at[kPer];
#pragma unroll
    for (int r = 0; r < kPer; ++r)
        if (r * kBsThreads + t < m) at[r] = atomicAdd(&s.cnt[(unsigned)(k[r] >> shift) & 255u], 1u);
    __syncthreads();
    const unsigned mine = s.cnt[t];
    s.start[t] = scan256_excl(mine, s.wsum);
    if (t == 0) s.start[kRsBins] = (unsigned)m;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
        if (r * kBsThreads + t >= m) continue;
        const unsigned p = s.start[(unsigned)(k[r] >> shift) & 255u] + at[r];
        s.sk[p] = k[r];
        s.sv[p] = v[r];
    }
    if (t < kCountStep) s.sk[m + t] = ~0ull;
    __syncthreads();
    // from here a thread's elements are the places i of the distributed order
    bool run = false;
    int place[kPer];
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
        const int i = r * kBsThreads + t;
        place[r] = -1;
        if (i >= m) continue;
        const unsigned long long kk = s.sk[i];
        const unsigned dg = (unsigned)(kk >> shift) & 255u;
        const int lo = (int)s.start[dg], hi = (int)s.start[dg + 1];
        int less = 0, same = 0;
        for (int j = lo; j < hi; j += kCountStep) { // the keys past hi are larger
#pragma unroll
            for (int q = 0; q < kCountStep; ++q) {
                const unsigned long long kj = s.sk[j + q];
                less += kj < kk ? 1 : 0;
                same += kj == kk ? 1 : 0;
            }
        }
        k[r] = kk;
        v[r] = s.sv[i];
        place[r] = lo + less;
        at[r] = (unsigned)same;
        run |= same > 1;
    }
    if (__syncthreads_or(run)) {
        const float rx = ctl->root[0], ry = ctl->root[1], rz = ctl->root[2], rr = ctl->radius;
#pragma unroll
        for (int r = 0; r < kPer; ++r) {
            if (place[r] < 0 || at[r] < 2) continue;
            unsigned long long w3[kDeepWords];
            deep_words(rx, ry, rz, rr, d.pm4[v[r]], w3);
#pragma unroll
            for (int q = 0; q < kDeepWords; ++q) s.dw[q][r * kBsThreads + t] = w3[q];
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kPer; ++r) {
            if (place[r] < 0 || at[r] < 2) continue;
            const int i = r * kBsThreads + t;
            const unsigned dg = (unsigned)(k[r] >> shift) & 255u;
            const int lo = (int)s.start[dg], hi = (int)s.start[dg + 1];
            const unsigned long long a0 = s.dw[0][i], a1 = s.dw[1][i], a2 = s.dw[2][i];
            int before = 0;
            for (int j = lo; j < hi; ++j) {
                if (s.sk[j] != k[r] || j == i) continue;
                const unsigned long long b0 = s.dw[0][j], b1 = s.dw[1][j], b2 = s.dw[2][j];
                if (b0 == a0 && b1 == a1 && b2 == a2) {
                    // two bodies on one 84-level path are closer than the tree can separate
                    flag_error(d.ctl, kErrDepth);
                    before += j < i ? 1 : 0;
                } else {
                    before += b0 < a0 || (b0 == a0 && (b1 < a1 || (b1 == a1 && b2 < a2))) ? 1 : 0;
                }
            }
            place[r] += before;
            const size_t o = (size_t)(base + place[r]);
            deep[o] = a0;
            deep[n + o] = a1;
            deep[2 * n + o] = a2;
        }
    }
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
        if (place[r] < 0) continue;
        key[base + place[r]] = k[r];
        val[base + place[r]] = v[r];
    }
}

__global__ __launch_bounds__(256) void k_deep_runs(Dev d, const unsigned long long *__restrict__ key, int *val,
                                                   unsigned long long *__restrict__ deep, int *perm, int *tmp,
                                                   unsigned long long *stage_k, int *stage_v)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int n = d.n;
    Ctl *ctl = d.ctl;
    if (i + 1 >= n || ctl->error) return;
    const unsigned long long k = key[i];
    if (key[i + 1] != k || (i > 0 && key[i - 1] == k)) return; // not the start of a run
    int m = 2;
    while (i + m < n && key[i + m] == k) ++m;
    if (m > kMaxRun) {
        order_long_run(d, i, m, val, deep, perm, tmp, stage_k, stage_v);
        return;
    }
    unsigned long long dk[kMaxRun][kDeepWords];
    int vv[kMaxRun];
    const float rx = ctl->root[0], ry = ctl->root[1], rz = ctl->root[2], rr = ctl->radius;
    for (int a = 0; a < m; ++a) {
        vv[a] = val[i + a];
        deep_words(rx, ry, rz, rr, d.pm4[vv[a]], dk[a]);
    }
    // stable insertion sort by the deep words
    for (int a = 1; a < m; ++a) {
        unsigned long long c0 = dk[a][0], c1 = dk[a][1], c2 = dk[a][2];
        const int cv = vv[a];
        int b = a - 1;
        while (b >= 0 && (dk[b][0] > c0 || (dk[b][0] == c0 && (dk[b][1] > c1 || (dk[b][1] == c1 && dk[b][2] > c2))))) {
            dk[b + 1][0] = dk[b][0];
            dk[b + 1][1] = dk[b][1];
            dk[b + 1][2] = dk[b][2];
            vv[b + 1] = vv[b];
            --b;
        }
        dk[b + 1][0] = c0;
        dk[b + 1][1] = c1;
        dk[b + 1][2] = c2;
        vv[b + 1] = cv;
    }
    for (int a = 0; a < m; ++a) {
        // two bodies on one 84-level path are closer than the tree can separate
        if (a > 0 && dk[a][0] == dk[a - 1][0] && dk[a][1] == dk[a - 1][1] && dk[a][2] == dk[a - 1][2])
            flag_error(ctl, kErrDepth);
        val[i + a] = vv[a];
        for (int w = 0; w < kDeepWords; ++w) deep[(size_t)w * n + i + a] = dk[a][w];
    }
}

// Common prefix in bits (3 per level) of sorted bodies i and j, whose keys are
// ki and kj.
__device__ __forceinline__ int delta_of(unsigned long long ki, unsigned long long kj,
                                        const unsigned long long *__restrict__ deep, int n, int i, int j)
{
    const unsigned long long x = ki ^ kj;
    if (x) return __clzll((long long)x) - 1;
    // equal 21-level keys: i and j are in one run, whose deep words are set
#pragma unroll
    for (int w = 0; w < kDeepWords; ++w) {
        const unsigned long long y = deep[(size_t)w * n + i] ^ deep[(size_t)w * n + j];
        if (y) return 63 * (w + 1) + __clzll((long long)y) - 1;
    }
    return 63 * (kDeepWords + 1);
}

// Common prefix of sorted keys i and j in bits (3 per level); -1 outside.
__device__ __forceinline__ int key_delta(const unsigned long long *__restrict__ key,
                                         const unsigned long long *__restrict__ deep, int n, int i, int j)
{
    if (j < 0 || j >= n) return -1;
    return delta_of(key[i], key[j], deep, n, i, j);
}

// octant of sorted body `pos` at `level`
__device__ __forceinline__ int key_digit(const unsigned long long *__restrict__ key,
                                         const unsigned long long *__restrict__ deep, int n, int pos, int level)
{
    const int w = level / kKeyLevels, L = level % kKeyLevels;
    const unsigned long long x = w == 0 ? key[pos] : deep[(size_t)(w - 1) * n + pos];
    return (int)((x >> (3 * (kKeyLevels - 1 - L))) & 7ull);
}

// ---------------------------------------------------------------------------
// Binary radix tree over the sorted keys (Karras 2012, fig. 4), internal node
// i of n - 1 (node 0 is the root): its range [lo, hi] and split, the parent
// links of its two children (internal or body), and the octree levels it
// holds: ktop .. ktop + own - 1, the levels k with 3k in (delta(parent),
// delta(i)]. delta(parent) is the larger of the prefixes the range shares with
// its two outside neighbours (the parent extends the range towards the
// neighbour that shares more; -1 for the root).
//
// The searches of a block's nodes read the keys from a window in LDS (the
// block's own keys and kBtHalo on each side, loaded once, coalesced); only a
// probe past the window (a node whose range reaches further) reads the key
// from device memory. Most ranges are short, so the searches' dependent loads
// become LDS reads.
// ---------------------------------------------------------------------------
constexpr int kBtThreads = 512;
constexpr int kBtHalo = 512;
constexpr int kBtSpan = kBtThreads + 2 * kBtHalo;

// keys through the block's LDS window where it has them, else from device memory
struct KeysAny {
    const unsigned long long *ks;
    const unsigned long long *__restrict__ key;
    int base;
    __device__ __forceinline__ unsigned long long operator()(int j) const
    {
        const unsigned t = (unsigned)(j - base);
        return t < (unsigned)kBtSpan ? ks[t] : key[j];
    }
};

// delta(i, j) > dd for i's key ki, with lim = limit(dd). Keys use 63 bits, so
// delta = clz(ki ^ kj) - 1 below 63, and delta > dd (dd < 63) holds exactly
// when ki ^ kj < 2^(62 - dd) (equal keys included: their delta is >= 63); one
// 64-bit compare instead of the count of leading zeros. A dd of 63 or more (i
// inside a run of equal keys) compares the deep words.
__device__ __forceinline__ unsigned long long delta_limit(int dd) { return dd < 63 ? 1ull << (62 - dd) : 0ull; }

template <class K>
__device__ __forceinline__ bool delta_above(const K &ka, const unsigned long long *__restrict__ deep, int n, int i,
                                            unsigned long long ki, int j, int dd, unsigned long long lim)
{
    if (j < 0 || j >= n) return false;
    if (lim) return (ki ^ ka(j)) < lim;
    return delta_of(ki, ka(j), deep, n, i, j) > dd;
}

template <class K>
__device__ __forceinline__ int delta_at(const K &ka, const unsigned long long *__restrict__ deep, int n, int i,
                                        unsigned long long ki, int j)
{
    return j < 0 || j >= n ? -1 : delta_of(ki, ka(j), deep, n, i, j);
}

struct BinOut {
    int *__restrict__ iparent, *__restrict__ lparent, *__restrict__ lo, *__restrict__ own, *__restrict__ ktop;
    int *__restrict__ obase, *__restrict__ tsum, *__restrict__ tdep;
};

// Internal node i: its searches, then its outputs (own and top also returned).
// dir and dmin come from the neighbours i - 1 and i + 1. n <= 2^26 (the pool
// limit), so every probe fits an int.
template <class K>
__device__ __forceinline__ int2 bintree_node(const Dev &d, const K &ka, const unsigned long long *__restrict__ deep,
                                             int n, int i, const BinOut &o)
{
    const unsigned long long ki = ka(i);
    const int dir = delta_at(ka, deep, n, i, ki, i + 1) - delta_at(ka, deep, n, i, ki, i - 1) > 0 ? 1 : -1;
    const int dmin = delta_at(ka, deep, n, i, ki, i - dir);
    const unsigned long long lmin = delta_limit(dmin);
    int lmax = 2;
    while (delta_above(ka, deep, n, i, ki, i + lmax * dir, dmin, lmin)) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (delta_above(ka, deep, n, i, ki, i + (l + t) * dir, dmin, lmin)) l += t;
    const int j = i + l * dir;
    const int dn = delta_at(ka, deep, n, i, ki, j);
    const unsigned long long ln = delta_limit(dn);
    int s = 0, t = l;
    do {
        t = (t + 1) >> 1;
        if (delta_above(ka, deep, n, i, ki, i + (s + t) * dir, dn, ln)) s += t;
    } while (t > 1);
    const int lo = min(i, j), hi = max(i, j);
    // of keys in order the split lies inside the range; the bounds keep the
    // links below inside their arrays whatever the keys are
    const int g = max(lo, min(i + s * dir + min(dir, 0), hi - 1));
    if (lo == g) o.lparent[g] = i;
    else o.iparent[g] = i;
    if (hi == g + 1) o.lparent[g + 1] = i;
    else o.iparent[g + 1] = i;
    o.lo[i] = lo;
    if (i == 0) o.iparent[0] = -1;
    const int dp = max(delta_at(ka, deep, n, lo, ka(lo), lo - 1), delta_at(ka, deep, n, hi, ka(hi), hi + 1));
    const int kt = dp < 0 ? 0 : dp / 3 + 1;
    int kb = dn / 3;
    if (kb >= kBuildLevelLimit) {
        flag_error(d.ctl, kErrDepth);
        kb = kBuildLevelLimit - 1;
    }
    const int own = max(0, kb - kt + 1);
    o.own[i] = own;
    o.ktop[i] = kt;
    return make_int2(own, kt);
}

// SCAN: a block's nodes are also a tile of the scan of the cells that the nodes
// hold (-> their first cells): obase = the cells of the tile's earlier nodes,
// tsum = the tile's cells, tdep = the tile's depth (the deepest cell's level +
// 1: its children are bodies); and the cells of each level are counted.
template <bool SCAN>
__global__ __launch_bounds__(kBtThreads) void k_bintree(Dev d, const unsigned long long *__restrict__ key,
                                                        const unsigned long long *__restrict__ deep, BinOut o)
{
    __shared__ unsigned long long ks[kBtSpan];
    __shared__ int wsum[SCAN ? kBtThreads / 64 : 1], wdep[SCAN ? kBtThreads / 64 : 1];
    __shared__ int h[SCAN ? kMaxDepth : 1];
    const int n = d.n, t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int err = d.ctl->error;
    const int base = (int)blockIdx.x * kBtThreads - kBtHalo;
    if (SCAN && t < kMaxDepth) h[t] = 0;
    for (int u = t; u < kBtSpan; u += kBtThreads) {
        const int g = base + u;
        ks[u] = g >= 0 && g < n ? key[g] : 0ull;
    }
    // one decision for the block: bintree_node of another block may flag a depth
    // error meanwhile, and a window without the keys of waves that left would be
    // searched as if it were in order
    if (block_stops(err)) return;
    const int i = (int)blockIdx.x * kBtThreads + t;
    int2 node = make_int2(0, 0); // cells held, level of the first
    if (i < n - 1) node = bintree_node(d, KeysAny{ks, key, base}, deep, n, i, o);
    if (!SCAN) return;
    for (int k = 0; k < node.x; ++k) atomicAdd(&h[node.y + k], 1);
    int dep = node.x > 0 ? node.y + node.x : 0;
#pragma unroll
    for (int q = 32; q > 0; q >>= 1) dep = max(dep, __shfl_xor(dep, q));
    int x = node.x; // inclusive scan over the wave
#pragma unroll
    for (int q = 1; q < 64; q <<= 1) {
        const int y = __shfl_up(x, q);
        if (lane >= q) x += y;
    }
    if (lane == 63) {
        wsum[w] = x;
        wdep[w] = dep;
    }
    __syncthreads();
    int before = 0, all = 0, deepest = 0;
#pragma unroll
    for (int q = 0; q < kBtThreads / 64; ++q) {
        before += q < w ? wsum[q] : 0;
        all += wsum[q];
        deepest = max(deepest, wdep[q]);
    }
    if (i < n - 1) o.obase[i] = before + x - node.x;
    if (t == 0) {
        o.tsum[blockIdx.x] = all;
        o.tdep[blockIdx.x] = deepest;
    }
    if (t < kMaxDepth && h[t]) atomicAdd(&d.lvl_count[t * kLevelLine], h[t]);
}

// the running maximum of the depths (buildtree.cl:199)
__device__ __forceinline__ void raise_depth(Ctl *ctl, int dep)
{
    if (dep > 0) __hip_atomic_fetch_max(&ctl->max_depth, dep, __ATOMIC_RELAXED, AGENT);
}

// The cell count C (the total of the scan), the pool check and the root's
// record: by one thread.
__device__ __forceinline__ void finish_count(const Dev &d, int C)
{
    Ctl *ctl = d.ctl;
    if (C > d.cap) {
        flag_error(ctl, kErrPool);
    } else {
        ctl->n_cells = C;
        d.cinfo[0] = make_int4(-1, 0, (int)ctl->epoch, 0);
    }
}

// ---------------------------------------------------------------------------
// Exclusive scan of the cells each internal node holds (-> its first cell):
// tiles of kScanTile scanned with their sums kept (k_scan_tiles), the sums
// scanned by one block (k_scan_sums); readers add the two.
// The same passes find the tree's depth: the deepest cell's level + 1, per tile
// and then over the tiles, into the running maximum with one atomic.
// This is the way of large trees (build_levels): the binary tree's blocks would
// wait for their slowest node to scan, which costs more than these launches.
// ---------------------------------------------------------------------------
constexpr int kScanPer = 4; // one int4 per thread: coalesced
constexpr int kScanTile = 256 * kScanPer;
static_assert(kScanTile >= kKeyScanTile && kBtThreads >= kKeyScanTile,
              "the engine sizes the tile sums with kKeyScanTile");

__device__ __forceinline__ int4 load4(const int *__restrict__ a, int i0, int m)
{
    if (i0 + 3 < m) return *reinterpret_cast<const int4 *>(a + i0);
    return make_int4(i0 < m ? a[i0] : 0, i0 + 1 < m ? a[i0 + 1] : 0, i0 + 2 < m ? a[i0 + 2] : 0, 0);
}

__global__ __launch_bounds__(256) void k_scan_tiles(const Ctl *ctl, const int *__restrict__ in,
                                                    const int *__restrict__ ktop, int *__restrict__ out, int m,
                                                    int *__restrict__ sums, int *__restrict__ tdepth)
{
    __shared__ int wsum[4], wdep[4];
    const int err = ctl->error;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int i0 = blockIdx.x * kScanTile + t * kScanPer;
    const int4 v = load4(in, i0, m), kt = load4(ktop, i0, m);
    const int acc = v.x + v.y + v.z + v.w;
    int dep = 0;
    if (v.x > 0) dep = max(dep, kt.x + v.x);
    if (v.y > 0) dep = max(dep, kt.y + v.y);
    if (v.z > 0) dep = max(dep, kt.z + v.z);
    if (v.w > 0) dep = max(dep, kt.w + v.w);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) dep = max(dep, __shfl_xor(dep, o));
    if (lane == 0) wdep[w] = dep;
    int x = acc; // inclusive scan of the per-thread totals over the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[w] = x;
    if (block_stops(err)) return;
    int run = x - acc;
    for (int ww = 0; ww < w; ++ww) run += wsum[ww];
    const int4 e = make_int4(run, run + v.x, run + v.x + v.y, run + v.x + v.y + v.z);
    if (i0 + 3 < m) {
        *reinterpret_cast<int4 *>(out + i0) = e;
    } else {
        if (i0 < m) out[i0] = e.x;
        if (i0 + 1 < m) out[i0 + 1] = e.y;
        if (i0 + 2 < m) out[i0 + 2] = e.z;
    }
    if (t == 0) {
        sums[blockIdx.x] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
        tdepth[blockIdx.x] = max(max(wdep[0], wdep[1]), max(wdep[2], wdep[3]));
    }
}

// one block: exclusive scan of the tile sums in place (each thread a run of
// them)
__global__ __launch_bounds__(1024) void k_scan_sums(Dev d, int *__restrict__ sums, int ntiles,
                                                   const int *__restrict__ tdepth)
{
    __shared__ int s[1024];
    __shared__ int wdep[16];
    Ctl *ctl = d.ctl;
    const int err = ctl->error;
    const int t = threadIdx.x;
    const int per = (ntiles + 1023) / 1024;
    int acc = 0, dep = 0;
    for (int k = 0; k < per; ++k) {
        const int j = t * per + k;
        if (j < ntiles) {
            acc += sums[j];
            dep = max(dep, tdepth[j]);
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) dep = max(dep, __shfl_xor(dep, o));
    if ((t & 63) == 0) wdep[t >> 6] = dep;
    s[t] = acc;
    if (block_stops(err)) return;
    for (int st = 1; st < 1024; st <<= 1) {
        const int u = t >= st ? s[t - st] : 0;
        __syncthreads();
        s[t] += u;
        __syncthreads();
    }
    int run = s[t] - acc;
    for (int k = 0; k < per; ++k) {
        const int j = t * per + k;
        if (j < ntiles) {
            const int c = sums[j];
            sums[j] = run;
            run += c;
        }
    }
    if (t == 0) {
        for (int k = 0; k < 16; ++k) dep = max(dep, wdep[k]);
        raise_depth(ctl, dep);
        finish_count(d, s[1023]);
    }
}

// ---------------------------------------------------------------------------
// Cells and slots. Cell first_cell(i) + (k - ktop[i]) is internal node i's cell
// of level k; the root (level 0, held by binary node 0) is cell 0.
// ---------------------------------------------------------------------------
struct KeyTree {
    const unsigned long long *key, *deep;
    const int *val, *iparent, *lparent, *lo, *own, *ktop, *obase, *tsum;
};

// The deepest cell of the nearest binary ancestor (p itself included) that
// holds a cell, or -1 (an inconsistent tree; the caller flags it). A node that
// holds none shares its level with its parent, so the walk is at most a few
// steps; it is bounded anyway.
template <class T> __device__ __forceinline__ int holding_cell(const KeyTree &kt, const T &tile, int p)
{
    for (int steps = 0; steps < 4 * kBuildLevelLimit * 3 && p >= 0; ++steps) {
        const int o = kt.own[p];
        if (o != 0) return kt.obase[p] + tile(p) + o - 1;
        p = kt.iparent[p];
    }
    return -1;
}

// one body: the root is the one cell
__global__ void k_one_cell(Dev d)
{
    Ctl *ctl = d.ctl;
    if (ctl->error) return;
    ctl->n_cells = 1;
    d.cinfo[0] = make_int4(-1, 0, (int)ctl->epoch, 0);
    d.lvl_list[0] = 0;
    for (int k = 0; k <= kMaxDepth; ++k) ctl->lvl_start[k] = k > 0 ? 1 : 0;
    ctl->levels = 1;
    ctl->live_cells = 1;
}

// Position g: the cells of internal node g (g < n - 1) -- each in the slot of
// its octant in its parent, and its record -- and sorted body g, in the
// deepest cell of its nearest holding ancestor, at the level one below the
// larger prefix it shares with a neighbour. The kernel is bound by the
// latency of its dependent reads, not by its arithmetic: a thread takes
// kLinkPer positions (kLinkPer * 256 apart in a block's span), and their
// loads are issued together, in two rounds of independent reads (clamped
// indices, no branch in between).
constexpr int kLinkPer = 2;
constexpr int kLinkSpan = 256 * kLinkPer;

template <class T>
__device__ __forceinline__ int deepest_of(const KeyTree &kt, const T &tile, int own, int ob, int p)
{
    // the holding cell of binary node p, given the cells it holds and the
    // first of them: p itself when it holds any, else the walk up from its parent
    return own != 0 ? ob + own - 1 : (p >= 0 ? holding_cell(kt, tile, kt.iparent[p]) : -1);
}

// SCAN (after k_bintree<true>, at most kLinkSums tiles): every block scans the
// tile sums by itself, and the first block does what k_scan_sums does with
// their total; a block also puts its cells into the lists of their levels
// (lvl_list): it counts them by level, takes that many places of each level
// with one atomic, and places them as it writes the cells.
constexpr int kLinkSums = 1024;
static_assert(kBuildLevels <= kLinkSums * kBtThreads, "k_link scans the tiles of every tree it groups by level");

template <bool SCAN>
__global__ __launch_bounds__(256) void k_link(Dev d, KeyTree kt, int ntiles, const int *__restrict__ tdep)
{
    constexpr int kTile = SCAN ? kBtThreads : kScanTile;
    __shared__ int sums[SCAN ? kLinkSums : 1];
    __shared__ unsigned wsum[4];
    __shared__ int h[SCAN ? kMaxDepth : 1], at[SCAN ? kMaxDepth : 1];
    const int n = d.n, t = threadIdx.x;
    Ctl *ctl = d.ctl;
    const int err = ctl->error;
    const uint32_t ep = ctl->epoch;
    const int g0 = blockIdx.x * kLinkSpan + t;
    if (n < 2) { // the root holds the one body
        if (g0 == 0 && !err) d.slot[key_digit(kt.key, kt.deep, n, 0, 0)] = slot_tag(ep, kt.val[0]);
        return;
    }
    if (SCAN && t < kMaxDepth) h[t] = 0;
    // round 1: each position's node and leaf records and the keys around it
    int own[kLinkPer], top[kLinkPer], lo[kLinkPer], ip[kLinkPer], ob[kLinkPer], lp[kLinkPer];
    int body[kLinkPer];
    unsigned long long kg[kLinkPer], km[kLinkPer], kq[kLinkPer];
#pragma unroll
    for (int u = 0; u < kLinkPer; ++u) {
        const int g = min(g0 + u * 256, n - 1);
        const int gi = min(g, n - 2);
        own[u] = kt.own[gi];
        top[u] = kt.ktop[gi];
        lo[u] = kt.lo[gi];
        ip[u] = kt.iparent[gi];
        ob[u] = kt.obase[gi];
        lp[u] = kt.lparent[g];
        body[u] = kt.val[g];
        kg[u] = kt.key[g];
        km[u] = kt.key[max(g - 1, 0)];
        kq[u] = kt.key[min(g + 1, n - 1)];
    }
    if (SCAN) {
        constexpr int per = kLinkSums / 256;
        unsigned c[per], sum = 0;
#pragma unroll
        for (int q = 0; q < per; ++q) {
            const int j = per * t + q;
            c[q] = j < ntiles ? (unsigned)kt.tsum[j] : 0u;
            sum += c[q];
        }
        unsigned run = scan256_total(sum, wsum);
#pragma unroll
        for (int q = 0; q < per; ++q) {
            sums[per * t + q] = (int)run;
            run += c[q];
        }
    }
    // the same decision in every wave: another block may flag an error meanwhile
    if (__syncthreads_or(err)) return;
    if (SCAN) {
        const int C = (int)wsum[3];
        if (blockIdx.x == 0) {
            int dep = 0;
            for (int j = t; j < ntiles; j += 256) dep = max(dep, tdep[j]);
#pragma unroll
            for (int q = 32; q > 0; q >>= 1) dep = max(dep, __shfl_xor(dep, q));
            if ((t & 63) == 0) raise_depth(ctl, dep);
            if (t == 0) finish_count(d, C);
        }
        if (C > d.cap) return; // every block sees it: no cell is written
    }
    const auto tile = [&](int i) { return SCAN ? sums[i / kTile] : kt.tsum[i / kTile]; };
    // round 2: the parents' records, and the key of each node's first body
    int own_ip[kLinkPer], ob_ip[kLinkPer], own_lp[kLinkPer], ob_lp[kLinkPer];
    unsigned long long klo[kLinkPer];
#pragma unroll
    for (int u = 0; u < kLinkPer; ++u) {
        const int ipc = max(ip[u], 0);
        own_ip[u] = kt.own[ipc];
        ob_ip[u] = kt.obase[ipc] + tile(ipc);
        own_lp[u] = kt.own[lp[u]];
        ob_lp[u] = kt.obase[lp[u]] + tile(lp[u]);
        klo[u] = kt.key[lo[u]];
    }
    if (SCAN) {
#pragma unroll
        for (int u = 0; u < kLinkPer; ++u)
            if (g0 + u * 256 < n - 1)
                for (int k = 0; k < own[u]; ++k) atomicAdd(&h[top[u] + k], 1);
        __syncthreads();
        if (t < kMaxDepth) { // the first wave
            const int cells = d.lvl_count[t * kLevelLine];
            int x = cells;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(x, o);
                if (t >= o) x += y;
            }
            at[t] = x - cells + (h[t] ? atomicAdd(&d.lvl_count[(kMaxDepth + t) * kLevelLine], h[t]) : 0);
            if (blockIdx.x == 0) {
                const unsigned long long some = __ballot(cells > 0);
                ctl->lvl_start[t] = x - cells;
                if (t == kMaxDepth - 1) {
                    ctl->lvl_start[kMaxDepth] = x;
                    ctl->live_cells = x;
                    ctl->levels = 64 - __clzll((long long)some);
                }
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < kLinkPer; ++u) {
        const int g = g0 + u * 256;
        if (g >= n) break;
        if (g < n - 1 && own[u] > 0) {
            int par = -1;
            if (top[u] > 0) {
                par = deepest_of(kt, tile, own_ip[u], ob_ip[u], ip[u]);
                if (par < 0) {
                    flag_error(ctl, kErrSync);
                    return;
                }
            }
            const int base = ob[u] + tile(g);
            for (int k = top[u]; k < top[u] + own[u]; ++k) {
                const int cid = base + (k - top[u]);
                if (k > 0) {
                    const int L = k - 1;
                    const int dg = L < kKeyLevels ? (int)((klo[u] >> (3 * (kKeyLevels - 1 - L))) & 7ull)
                                                  : key_digit(kt.key, kt.deep, n, lo[u], L);
                    d.slot[(size_t)par * 8 + dg] = slot_tag(ep, n + cid);
                    d.cinfo[cid] = make_int4(par, k | (dg << 8), (int)ep, 0);
                }
                if (SCAN) d.lvl_list[atomicAdd(&at[k], 1)] = cid;
                par = cid;
            }
        }
        const int par = deepest_of(kt, tile, own_lp[u], ob_lp[u], lp[u]);
        if (par < 0) {
            flag_error(ctl, kErrSync);
            return;
        }
        // common prefixes with the neighbours from the keys in hand (the deep
        // words only when a key is repeated)
        const int dm = g == 0 ? -1
                              : (kg[u] != km[u] ? __clzll((long long)(kg[u] ^ km[u])) - 1
                                                : key_delta(kt.key, kt.deep, n, g, g - 1));
        const int dq = g == n - 1 ? -1
                                  : (kg[u] != kq[u] ? __clzll((long long)(kg[u] ^ kq[u])) - 1
                                                    : key_delta(kt.key, kt.deep, n, g, g + 1));
        const int lv = max(dm, dq) / 3;
        const int dg = lv < kKeyLevels ? (int)((kg[u] >> (3 * (kKeyLevels - 1 - lv))) & 7ull)
                                       : key_digit(kt.key, kt.deep, n, g, lv);
        d.slot[(size_t)par * 8 + dg] = slot_tag(ep, body[u]);
    }
}

// ---------------------------------------------------------------------------
// launcher
// ---------------------------------------------------------------------------
hipError_t launch_build_keys(const Dev &d, bool warm, bool staged, bool splitters, hipStream_t st)
{
    const int n = d.n;
    const dim3 b256(256), g256((n + 255) / 256);
    unsigned long long *ka = d.kb_key[0], *kb = d.kb_key[1];
    int *va = d.kb_val[0], *vb = d.kb_val[1];
    if (warm) {
        // keys in the last tree's order into [1], splitters from the last
        // tree's sorted keys in [0], bucketed into [0], each bucket sorted in
        // place ([1] is the spill space of large buckets)
        // (the buckets of the bodies go to kb_lo, which the binary tree fills later)
        const int S = bucket_samples(n);
        const dim3 gw((n + kWinBodies - 1) / kWinBodies);
        if (!splitters) hipLaunchKernelGGL(k_splitters, dim3((S + 1 + 255) / 256), b256, 0, st, d, S);
        hipLaunchKernelGGL(k_keys_warm, dim3((n + kWarmBodies - 1) / kWarmBodies), b256, 0, st, d, d.sorted,
                           staged ? d.bnode : nullptr, d.kb_spl, S, kb, vb, d.kb_lo, d.kb_bcnt);
        if (S < kScatterScan) {
            hipLaunchKernelGGL(k_bucket_scatter<true>, gw, b256, 0, st, d.ctl, kb, vb, d.kb_lo, ka, va, n, d.kb_bcnt, S,
                               d.kb_bstart, d.kb_bfill);
        } else {
            hipLaunchKernelGGL(k_bucket_scan, dim3(1), dim3(1024), 0, st, d.ctl, d.kb_bcnt, S, d.kb_bstart);
            hipLaunchKernelGGL(k_bucket_scatter<false>, gw, b256, 0, st, d.ctl, kb, vb, d.kb_lo, ka, va, n, d.kb_bcnt,
                               S, d.kb_bstart, d.kb_bfill);
        }
        // (the binary tree's arrays, written later, serve the runs of large buckets)
        hipLaunchKernelGGL(k_bucket_sort<kBucketCap>, dim3(S + 1), dim3(kBsThreads), 0, st, d, ka, va, d.kb_deep, kb,
                           vb, d.kb_ipar, d.kb_lpar, d.kb_bstart, true);
    } else if (n <= kColdBodies) {
        const int S = cold_samples(n);
        const dim3 gc((n + kColdPer - 1) / kColdPer);
        const dim3 one(1), ts(kSampleThreads);
        if (n <= kColdBodies / 2) hipLaunchKernelGGL(k_sample<1>, one, ts, 0, st, d, S);
        else hipLaunchKernelGGL(k_sample<2>, one, ts, 0, st, d, S);
        hipLaunchKernelGGL(k_keys_cold, gc, b256, 0, st, d, S, kb, d.kb_lo);
        hipLaunchKernelGGL(k_cold_scatter, g256, b256, 0, st, d.ctl, n, S, d.kb_bcnt, kb, d.kb_lo, ka, va, d.kb_bstart);
        hipLaunchKernelGGL(k_bucket_sort<kColdCap>, dim3(S + 1), dim3(kBsThreads), 0, st, d, ka, va, d.kb_deep, kb, vb,
                           d.kb_ipar, d.kb_lpar, d.kb_bstart, false);
    } else {
        const int ntiles = (n + kRsTile - 1) / kRsTile;
        hipLaunchKernelGGL(k_keys, g256, b256, 0, st, d, nullptr, ka, va);
        for (int pass = 0; pass < 8; ++pass) {
            const int shift = 8 * pass;
            hipLaunchKernelGGL(k_rs_count, dim3(ntiles), dim3(kRsThreads), 0, st, ka, n, shift, d.kb_hist, ntiles);
            hipLaunchKernelGGL(k_rs_offsets, dim3(kRsBins), dim3(1024), 0, st, d.kb_hist, ntiles, d.kb_offs, d.kb_tot);
            hipLaunchKernelGGL(k_rs_scatter, dim3(ntiles), dim3(kRsThreads), 0, st, ka, va, kb, vb, n, shift, d.kb_hist,
                               d.kb_offs, d.kb_tot, ntiles);
            unsigned long long *tk = ka;
            ka = kb;
            kb = tk;
            int *tv = va;
            va = vb;
            vb = tv;
        }
        // eight passes: the sorted keys are back in kb_key[0] / kb_val[0]; the
        // other pair and the binary tree's arrays (written later) serve long runs
        hipLaunchKernelGGL(k_deep_runs, g256, b256, 0, st, d, ka, va, d.kb_deep, d.kb_ipar, d.kb_lpar, kb, vb);
    }
    KeyTree kt{ka, d.kb_deep, va, d.kb_ipar, d.kb_lpar, d.kb_lo, d.kb_own, d.kb_ktop, d.kb_obase, d.kb_scan};
    const dim3 gl((n + kLinkSpan - 1) / kLinkSpan), gi((n + kBtThreads - 2) / kBtThreads);
    const BinOut bo{d.kb_ipar, d.kb_lpar, d.kb_lo, d.kb_own, d.kb_ktop, d.kb_obase, d.kb_scan, d.kb_tdep};
    if (n < 2) {
        hipLaunchKernelGGL(k_one_cell, dim3(1), dim3(1), 0, st, d);
        hipLaunchKernelGGL(k_link<false>, gl, b256, 0, st, d, kt, 0, d.kb_tdep);
    } else if (build_levels(n)) {
        hipLaunchKernelGGL(k_bintree<true>, gi, dim3(kBtThreads), 0, st, d, ka, d.kb_deep, bo);
        hipLaunchKernelGGL(k_link<true>, gl, b256, 0, st, d, kt, (int)gi.x, d.kb_tdep);
    } else {
        const int m = n - 1, nt = (m + kScanTile - 1) / kScanTile;
        hipLaunchKernelGGL(k_bintree<false>, gi, dim3(kBtThreads), 0, st, d, ka, d.kb_deep, bo);
        hipLaunchKernelGGL(k_scan_tiles, dim3(nt), dim3(256), 0, st, d.ctl, d.kb_own, d.kb_ktop, d.kb_obase, m,
                           d.kb_scan, d.kb_tdep);
        hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(1024), 0, st, d, d.kb_scan, nt, d.kb_tdep);
        hipLaunchKernelGGL(k_link<false>, gl, b256, 0, st, d, kt, nt, d.kb_tdep);
    }
    return hipGetLastError();
}

} // namespace nb
