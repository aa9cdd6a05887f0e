// nb_device.h -- device helpers shared by the force traversals.
#pragma once

#include "nb_internal.h"

namespace nb {

#define AGENT __HIP_MEMORY_SCOPE_AGENT

constexpr float kFar = __builtin_huge_valf();
constexpr int kStack = 512; // >= 7 * 64 + 8 entries: the deepest possible push pattern
constexpr uint64_t kAllLanes = ~0ull;

// Entries of the stack of K waves that share a vote group. One wave (K = 1)
// walks depth first: at most 7 siblings wait per level. K waves take the K
// top entries together; the limit kSplitTop above which they take one entry at
// a time (depth first from there, again at most 7 per level) bounds the stack
// for every tree of kMaxDepth levels: kSplitTop + the children of one round +
// 7 per level.
constexpr int kSplitTop = 512;
template <int K> constexpr int split_stack() { return K == 1 ? kStack : kSplitTop + 8 * K + kStack; }
constexpr unsigned kSplitBad = 1u << 16; // a wave's report of a corrupt tree, above its push count

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// v_writelane_b32: `old` with lane `lane` (wave-uniform) set to the
// wave-uniform value v; one instruction (LLVM's amdgcn.writelane intrinsic,
// which this compiler exposes under no builtin name)
__device__ int amdgcn_writelane_i32(int v, int lane, int old) __asm("llvm.amdgcn.writelane.i32");

__device__ __forceinline__ unsigned lane_write(unsigned old, unsigned v, int lane)
{
    return (unsigned)amdgcn_writelane_i32((int)v, lane, (int)old);
}

// After a round of K waves in which this one opened npush cells: a barrier, by
// which the round's entries are read, then the cells that the lower waves and
// that all opened. False when some wave says the tree is corrupt. Every wave of
// the block calls it; `pushed` holds K words.
template <int K>
__device__ __forceinline__ bool count_round(unsigned *pushed, int wv, int lane, int npush, bool bad, unsigned &before,
                                            unsigned &total)
{
    if (lane == 0) pushed[wv] = (unsigned)npush | (bad ? kSplitBad : 0u);
    __syncthreads();
    before = total = 0;
#pragma unroll
    for (int w = 0; w < K; ++w) {
        const unsigned c = pushed[w];
        before += w < wv ? c : 0u;
        total += c;
    }
    total = __builtin_amdgcn_readfirstlane(total);
    return total < kSplitBad;
}

// End of a round of K waves that took `take` entries off the top of the shared
// stack of sp entries, this wave having opened npush cells (entry j in lane j
// of `push`): the new entries go behind those of the lower waves, and sp
// becomes the new count. False when the tree is corrupt (some wave says so, or
// the stack would overflow).
template <int K, class Entry>
__device__ __forceinline__ bool end_round(Entry *stk, unsigned *pushed, int wv, int lane, int take, int npush, Entry push,
                                          bool bad, int &sp)
{
    unsigned before, total;
    // the same in every wave
    if (!count_round<K>(pushed, wv, lane, npush, bad, before, total) || sp - take + (int)total > split_stack<K>())
        return false;
    if (lane < npush) stk[sp - take + (int)before + lane] = push;
    sp += (int)total - take;
    if (sp) __syncthreads();
    return true;
}

// K waves that share a group and part: breadth first, a cell each per round,
// until the queue holds FRONT cells; then each wave takes every K-th of them
// and walks their subtrees by itself, depth first. After STRETCH visits, or
// with nothing left, a wave waits for the others, and what all of them have
// left is dealt out again, every K-th entry to one wave: the subtrees differ in
// size, and without that the waves end far apart. The queue is a ring of kQueue
// entries; a wave's own stack holds what it is dealt (at most kDealt entries:
// with more left in all, the waves go on with what they have) and 7 entries for
// each level below. The order depends on the tree alone. stk: parted_stack
// words, the root in the first (before a barrier); visit(entry, opened) calls
// opened(entry) for what it opens and may set bad. Returns bad.
constexpr int kQueue = 512, kOwnStack = 576, kDealt = 120;
template <int K> constexpr int parted_stack() { return kQueue + K * kOwnStack; }

template <int K, int FRONT, int STRETCH, class Visit>
__device__ __forceinline__ bool walk_parted(unsigned *stk, unsigned *pushed, int wv, int lane, unsigned cap, bool &bad,
                                            Visit &&visit)
{
    static_assert(FRONT - 1 + 8 * K <= kQueue && (FRONT - 1 + 8 * K + K - 1) / K <= kDealt && kDealt <= 128 &&
                      kDealt + 7 * kMaxDepth + 8 <= kOwnStack && K * kOwnStack < (int)kSplitBad,
                  "the queue and the stacks hold every tree of kMaxDepth levels");
    int head = 0, tail = 1; // the same in every wave
    while (tail > head && tail - head < FRONT) {
        const int take = min(tail - head, K);
        int npush = 0;
        unsigned push = 0; // entry j of this wave's children in lane j
        if (wv < take) {
            const unsigned cur = __builtin_amdgcn_readfirstlane(stk[(head + wv) % kQueue]);
            if ((cur >> 6) >= cap) { // the pool holds `cap` cells: corrupt
                bad = true;
            } else {
                visit(cur, [&](unsigned e) {
                    push = lane_write(push, e, npush);
                    ++npush;
                });
            }
        }
        unsigned before, total;
        if (!count_round<K>(pushed, wv, lane, npush, bad, before, total)) return true;
        if (lane < npush) stk[(tail + (int)before + lane) % kQueue] = push;
        head += take;
        tail += (int)total;
        __syncthreads();
    }
    unsigned *own = stk + kQueue + wv * kOwnStack;
    int sp = (tail - head + K - 1 - wv) / K;
    for (int i = lane; i < sp; i += 64) own[i] = stk[(head + wv + K * (sp - 1 - i)) % kQueue];
    __builtin_amdgcn_wave_barrier();
    for (;;) {
        for (int v = 0; v < STRETCH && sp > 0; ++v) {
            --sp;
            const unsigned cur = __builtin_amdgcn_readfirstlane(own[sp]);
            if ((cur >> 6) >= cap) {
                bad = true;
                break;
            }
            visit(cur, [&](unsigned e) {
                own[sp] = e; // every lane, one address
                ++sp;
            });
        }
        unsigned before, total;
        if (!count_round<K>(pushed, wv, lane, sp, bad, before, total)) return true;
        if (total == 0) return false;
        const bool deal = total <= (unsigned)(K * kDealt); // the same in every wave
        unsigned e[2];
        if (deal) {
            sp = ((int)total + K - 1 - wv) / K;
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int j = lane + 64 * r;
                if (j >= sp) continue;
                const unsigned at = wv + K * j; // place in the stacks one after the other
                unsigned start = 0, from = 0, next = 0;
#pragma unroll
                for (int w = 0; w < K - 1; ++w) {
                    next += pushed[w];
                    if (at >= next) {
                        start = next;
                        from = w + 1;
                    }
                }
                e[r] = stk[kQueue + from * kOwnStack + (at - start)];
            }
        }
        __syncthreads(); // read by every wave: the stacks and the counts
        if (deal) {
#pragma unroll
            for (int r = 0; r < 2; ++r)
                if (lane + 64 * r < sp) own[lane + 64 * r] = e[r];
            __builtin_amdgcn_wave_barrier();
        }
    }
}

__device__ __forceinline__ void kahan_add(float &sum, float &comp, float x)
{
    const float y = x - comp;
    const float t = sum + y;
    comp = (t - sum) - y;
    sum = t;
}

__device__ __forceinline__ void flag_error(Ctl *ctl, int code)
{
    int expected = 0;
    __hip_atomic_compare_exchange_strong(&ctl->error, &expected, code, __ATOMIC_RELAXED,
                                         __ATOMIC_RELAXED, AGENT);
}

// One decision for all waves of a block on the device error word: `err` as
// thread 0 read it, behind a barrier. Another block, or a kernel on another
// stream, may set the word between two waves' reads, and a wave that left by
// itself would owe the others what it should have put into LDS. Called once per
// kernel, by every thread.
__device__ __forceinline__ bool block_stops(int err)
{
    __shared__ int stop;
    if (threadIdx.x == 0) stop = err;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(stop) != 0;
}

// Splitter j of a warm build (j < S = bucket_samples(n)): the key at position
// j * kBucketT of the last tree's sorted keys, so non-decreasing (a decrease
// means the buffer does not hold them and stops the build with an error), and
// the counters of bucket j (j <= S) cleared.
__device__ __forceinline__ void make_splitter(const Dev &d, int j, int S)
{
    if (j > S) return;
    if (j < S) {
        const unsigned long long *key = d.kb_key[0];
        const unsigned long long k = key[(size_t)j * kBucketT];
        d.kb_spl[j] = k;
        if (j > 0 && key[(size_t)(j - 1) * kBucketT] > k) flag_error(d.ctl, kErrSync);
    }
    d.kb_bcnt[j] = 0;
    d.kb_bfill[j] = 0;
}

// Epilogue for one body: velocity correction and store (calculateforce.cl:
// 174-185), optionally the kick-drift-kick of integrate.cl:29-43 (mode 1), or
// only the acceleration into the probe buffer (mode 2).
__device__ __forceinline__ void finish_body(const Dev &d, int pos, float4 me, float fx, float fy,
                                            float fz, int mode, int step)
{
    const int b = d.sorted[pos];
    if (mode == 2) {
        d.probe[b] = make_float4(fx, fy, fz, 0.0f);
        return;
    }
    const float dt = d.dt;
    const float4 v0 = d.vel4[b];
    float vx = v0.x, vy = v0.y, vz = v0.z;
    if (step > 0) {
        const float4 a0 = d.acc4[b];
        vx = vx + ((fx - a0.x) * dt) * 0.5f;
        vy = vy + ((fy - a0.y) * dt) * 0.5f;
        vz = vz + ((fz - a0.z) * dt) * 0.5f;
    }
    d.acc4[b] = make_float4(fx, fy, fz, 0.0f);
    if (mode == 1) {
        const float dvx = (fx * dt) * 0.5f, dvy = (fy * dt) * 0.5f, dvz = (fz * dt) * 0.5f;
        const float vhx = vx + dvx, vhy = vy + dvy, vhz = vz + dvz;
        float4 p = me; // this body's (x, y, z, m)
        if (d.fp64) {
            const double4 q = d.pos64[b];
            const double x = fma((double)vhx, (double)dt, q.x);
            const double y = fma((double)vhy, (double)dt, q.y);
            const double z = fma((double)vhz, (double)dt, q.z);
            d.pos64[b] = make_double4(x, y, z, 0.0);
            p.x = (float)x; p.y = (float)y; p.z = (float)z;
        } else {
            p.x = fmaf(vhx, dt, p.x);
            p.y = fmaf(vhy, dt, p.y);
            p.z = fmaf(vhz, dt, p.z);
        }
        d.pm4[b] = p;
        d.bnode[pos] = p; // the new record in sorted order, read by the next build
        vx = vhx + dvx;
        vy = vhy + dvy;
        vz = vhz + dvz;
    }
    d.vel4[b] = make_float4(vx, vy, vz, 0.0f);
}

} // namespace nb
