// nb_force.hip -- force traversal (calculateforce.cl:25-188) for gfx950, and
// the FP64 direct sum used to measure force errors.
//
// A wave takes 64 consecutive sorted positions. A vote group is G consecutive
// lanes (G = 16, 32 or 64; 16 is the reference's work-group vote of
// calculateforce.cl:145 and 64 is one wave). Visiting a cell tests all of its
// (at most 8, compacted) children: bodies always interact, a child cell is
// accepted by a group only if every lane of the group has d^2 + eps^2 >=
// dq[depth], and a child that a group does not accept is opened by that group.
// Which nodes interact therefore matches the reference exactly; only the order
// of the terms differs.
//
// The wave walks the union of its groups' traversals: a stack entry is a cell
// (cell << 6 | depth) and the groups that opened it, and a cell is visited once
// for all of them. The cell is wave-uniform, so its children's indices and
// their (x, y, z, m) (contiguous in cchild and cdata: 32 + 128 bytes) arrive
// through scalar loads whatever G is, and the vector ALU only does the per-body
// arithmetic. Lanes whose group did not open the cell take an infinite
// softening: their 1 / sqrt(d^2) is 0, so they add nothing and accept every
// child. The groups of a wave are neighbours in the tree's order and open
// nearly the same cells, and never more than one 64-lane group would: a cell
// is opened when some lane of some group that reached it rejects it. With a
// stack per 16-lane group the four groups of a wave were at different cells,
// each child came through vector loads, and three quarters of the lanes idled
// in most of the branches: 25.5 -> 10.0 ms at 4M clustered bodies (theta 0.4,
// vote 16), 6.03 -> 2.76 ms at 1M Plummer bodies (theta 0.5, vote 16).
//
// Bound: vector issue. Of the 14 issue slots of a term (3 sub, 3 fma, rsq =
// 2, 3 mul, 3 fma), 3,690 terms per body at 1M Plummer bodies (theta 0.5,
// vote 64) are 52k of the 69k slots that a wave takes; 1.89 ms (2.37 ms before
// the scalar side was cut and the FP64 sums), 98 % of vector issue.
//
// Accumulation: the terms of one visited cell (<= 8) are summed in FP32 and
// added into FP64 sums. An FP64 add issues at the rate of an FP32 add here, so
// convert and add (6 instructions per cell) cost half of a compensated FP32
// sum (12) and keep more bits. A wave that walks narrow groups alone keeps the
// compensated sums (see waves_per_group).
#include "nb_device.h"

#include <type_traits>

namespace nb {

// Groups as bits: bit f stands for the 16 lanes of field f, and a vote group of
// 32 or 64 lanes is two or four fields. group_bits: the groups in which a lane
// of r is set; field_lanes: the lanes of the fields f. (s_quadmask ors each
// four bits into one, s_bitreplicate doubles each bit; neither has a builtin.)
template <int G> __device__ __forceinline__ unsigned group_bits(uint64_t r)
{
    static_assert(G == 16 || G == 32 || G == 64, "vote width");
    if constexpr (G == 64) return r ? 15u : 0u;
    uint64_t quads;
    asm("s_quadmask_b64 %0, %1" : "=s"(quads) : "s"(r) : "scc");
    unsigned f;
    asm("s_quadmask_b32 %0, %1" : "=s"(f) : "s"((unsigned)quads) : "scc");
    if constexpr (G == 32) f |= ((f >> 1) & 5u) | ((f << 1) & 10u);
    return f;
}

__device__ __forceinline__ uint64_t field_lanes(unsigned f)
{
    uint64_t x = f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const unsigned lo = (unsigned)x;
        asm("s_bitreplicate_b64_b32 %0, %1" : "=s"(x) : "s"(lo));
    }
    return x;
}

// the softened monopole term of mass m at (dx, dy, dz), d2 = |d|^2 + eps^2
__device__ __forceinline__ void add_term(float dx, float dy, float dz, float d2, float m, float &px, float &py,
                                         float &pz)
{
    const float ri = __builtin_amdgcn_rsqf(d2);
    const float f = m * (ri * ri * ri);
    px = fmaf(dx, f, px);
    py = fmaf(dy, f, py);
    pz = fmaf(dz, f, pz);
}

// One visit at vote width 64: the children of cell `e >> 6` (on level e & 63)
// against the wave's bodies. The terms' sum goes to (px, py, pz), the number of
// children is returned; opened(entry) is called for every child that is
// opened. Every branch is wave-uniform. Child cells sit at the front of the
// cell's record and bodies at its back, and their counts in the first two index
// words (nb_internal.h): a body costs a compare and a branch on the scalar
// side, a cell two more for its vote. The scalar unit issues one instruction
// per SIMD and four cycles like the vector one, and with a test of each child's
// kind it is the busier of the two: 1.92 against 2.65 ms at 1M Plummer bodies,
// theta 0.5.
template <bool SPLIT, class Opened>
__device__ __forceinline__ int visit_wide(unsigned e, float thr, float4 me, float eps2, const int *__restrict__ cchild,
                                          const float4 *__restrict__ cdata, float &px, float &py, float &pz,
                                          bool &bad, Opened &&opened)
{
    const size_t c = e >> 6;
    const i32x8 ch = *reinterpret_cast<const i32x8 *>(cchild + c * 8);
    const f32x16 q0 = *reinterpret_cast<const f32x16 *>(cdata + c * 8);
    const f32x16 q1 = *reinterpret_cast<const f32x16 *>(cdata + c * 8 + 4);
    // all loads issued together (the compiler would put the second half
    // behind the first children's work, one more round trip per visit)
    if constexpr (SPLIT) asm volatile("" ::"s"(ch), "s"(q0), "s"(q1));
    const int nbody = (int)((unsigned)ch[0] >> kCountShift);
    int ncell = (int)((unsigned)ch[1] >> kCountShift);
    // cells live on kMaxDepth levels: child cells below the last are corrupt
    // (and not followed, so a visit never descends past it)
    if ((e & 63u) == kMaxDepth - 1 && ncell > 0) {
        bad = true;
        ncell = 0;
    }
    px = py = pz = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if (k >= ncell) break;
        const f32x16 &q = k < 4 ? q0 : q1;
        const float dx = q[4 * (k & 3)] - me.x, dy = q[4 * (k & 3) + 1] - me.y, dz = q[4 * (k & 3) + 2] - me.z;
        const float d2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
        // 3 = ordered >=
        if (__builtin_amdgcn_fcmpf(d2, thr, 3) != kAllLanes)
            opened(((unsigned)ch[k] << 6) | ((e & 63u) + 1u));
        else
            add_term(dx, dy, dz, d2, q[4 * (k & 3) + 3], px, py, pz);
    }
#pragma unroll
    for (int k = 7; k >= 0; --k) {
        if (7 - k >= nbody) break;
        const f32x16 &q = k < 4 ? q0 : q1;
        const float dx = q[4 * (k & 3)] - me.x, dy = q[4 * (k & 3) + 1] - me.y, dz = q[4 * (k & 3) + 2] - me.z;
        const float d2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
        add_term(dx, dy, dz, d2, q[4 * (k & 3) + 3], px, py, pz);
    }
    return nbody + ncell;
}

// The same for narrower votes. fields: the groups that opened the cell; act:
// their lanes; opened(entry, groups) for every child that some group opens.
// The children come in octant order, each with its kind: with the order of the
// cells' walk and the compensated sums of the kernel below, a wave alone then
// adds every body's terms exactly as its group by itself would.
template <int G, bool SPLIT, class Opened>
__device__ __forceinline__ int visit_narrow(unsigned e, unsigned fields, uint64_t act, float thr, float4 me,
                                          float eps2, const int *__restrict__ cchild,
                                          const float4 *__restrict__ cdata, float &px, float &py, float &pz,
                                          bool &bad, Opened &&opened)
{
    const size_t c = e >> 6;
    const i32x8 ch = *reinterpret_cast<const i32x8 *>(cchild + c * 8);
    const f32x16 q0 = *reinterpret_cast<const f32x16 *>(cdata + c * 8);
    const f32x16 q1 = *reinterpret_cast<const f32x16 *>(cdata + c * 8 + 4);
    // all loads issued together (the compiler would put the second half
    // behind the first children's work, one more round trip per visit)
    if constexpr (SPLIT) asm volatile("" ::"s"(ch), "s"(q0), "s"(q1));
    const int nchild = (int)((unsigned)ch[0] >> kCountShift) & 15;
    const unsigned below = (e & 63u) + 1u;
    const float e2 = __builtin_amdgcn_inverse_ballot_w64(act) ? eps2 : kFar;
    px = py = pz = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if (k >= nchild) break;
        const f32x16 &q = k < 4 ? q0 : q1;
        const float dx = q[4 * (k & 3)] - me.x, dy = q[4 * (k & 3) + 1] - me.y, dz = q[4 * (k & 3) + 2] - me.z;
        const float d2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, e2)));
        const float m = q[4 * (k & 3) + 3];
        // the lanes that reject the child, a cell (the asm keeps the vote in
        // a branch of its own: 2.94 -> 2.76 ms at 1M Plummer bodies, theta
        // 0.5, vote 16, against an arm of its own for bodies)
        uint64_t r = 0;
        if (ch[k] >= 0) {
            r = act & ~__builtin_amdgcn_fcmpf(d2, thr, 3); // 3 = ordered >=
            asm volatile("");
        }
        if (r) {
            const unsigned rej = group_bits<G>(r); // the groups that open this child
            // cells live on kMaxDepth levels: one below the last is corrupt
            // (and not followed)
            if (below < (unsigned)kMaxDepth) opened(((unsigned)ch[k] << 6) | below, rej);
            else bad = true;
            // some groups accept, some open: the latter add nothing (the asm
            // keeps the compiler from joining this arm's sums with the
            // other's behind a flag: 4 % of the kernel)
            if (rej != fields) {
                add_term(dx, dy, dz, d2, __builtin_amdgcn_inverse_ballot_w64(field_lanes(rej)) ? 0.f : m, px, py, pz);
                asm volatile("" : "+v"(px), "+v"(py), "+v"(pz));
            }
        } else {
            add_term(dx, dy, dz, d2, m, px, py, pz);
        }
    }
    return nchild;
}

template <int G> struct StackEntry {
    using type = uint2;
};
template <> struct StackEntry<64> {
    using type = unsigned;
};

// The epilogue's per-wave sums overlay the stacks.
template <int G, int K> constexpr int force_lds()
{
    const int entries = K == 1 ? kStack : G < 64 ? split_stack<K>() : parted_stack<K>();
    const int stack = entries * (int)sizeof(typename StackEntry<G>::type), red = K == 1 ? 0 : K * 3 * 64 * 8;
    return ((stack > red ? stack : red) + 15) & ~15;
}

// K waves share the group of 64 positions (K > 1: few groups, so that one
// wave per group would leave the chip idle). With narrow votes they take the
// stack's top K entries in rounds: wave w visits the w-th from the top, and
// after a barrier pushes what it opened behind the lower waves' entries. At
// width 64 they part after a first stretch of rounds (walk_parted): a round
// lasts as long as its slowest visit (taking turns to the end: 442 us at
// 100,003 bodies, two spheres, 980 at 262,144). Parted waves stay even because
// what they have left is dealt out anew every 8 visits, with four waves 16: 372
// -> 331 us at 100,003 bodies and 873 -> 766 at 262,144 (two spheres), 128 -> 112
// at 65,536 (ball), against parting at 256 cells, the best of 64 to 512, with no
// dealing. Every 8 / 16 / 24 visits 331 / 345 / 368 us at 100,003 bodies, 777 / 766 /
// 792 at 262,144 (a series on another card than that of waves_per_group). With dealing the first stretch can be short: parting at 256 /
// 128 / 64 cells 355 / 352 / 345 us (8 waves, every 16). The order depends on nothing but the tree, and so
// do the sums. (Eight waves per SIMD by the
// attribute: the scalar registers would otherwise allow seven, 1.90 against
// 2.19 ms at 1M Plummer bodies, theta 0.5, vote 64.)
template <int G, int K>
__global__ __launch_bounds__(64 * K) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_force(
    Dev d, const int *__restrict__ cchild, const float4 *__restrict__ cdata, int mode)
{
    __shared__ __attribute__((aligned(16))) unsigned char lds[force_lds<G, K>()];
    __shared__ float dq_s[kMaxDepth];
    __shared__ unsigned pushed[K];
    __shared__ unsigned long long wint[K];
    // (cell << 6 | depth), with narrow votes beside the groups that opened it
    using Entry = typename StackEntry<G>::type;
    Entry *stk = reinterpret_cast<Entry *>(lds);
    auto entry = [](unsigned e, unsigned f) {
        if constexpr (G < 64) return make_uint2(e, f);
        else return e;
    };
    auto take_entry = [](Entry v, unsigned &e, unsigned &f) {
        if constexpr (G < 64) {
            e = __builtin_amdgcn_readfirstlane(v.x);
            f = __builtin_amdgcn_readfirstlane(v.y);
        } else {
            e = __builtin_amdgcn_readfirstlane(v);
        }
    };
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = K == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = d.n;
    Ctl *ctl = d.ctl;
    // several waves decide together, at the barrier before their walk: one that
    // left by itself would leave its count of a round unwritten, which the
    // others add up, and they stop when the sum is zero
    const int err = ctl->error;
    if (K == 1 && err) return;
    if (ctl->max_depth > kMaxDepth) { // calculateforce.cl:69-73
        if (tid == 0) flag_error(ctl, kErrDepth);
        return;
    }
    for (int i = tid; i < kMaxDepth; i += 64 * K) dq_s[i] = ctl->dq[i];
    const int step = ctl->step;

    const int pos = blockIdx.x * 64 + lane;
    const bool valid = pos < n;
    // a lane past the last body sits at infinity: its d^2 is infinite, so it
    // accepts every cell and never holds up the vote (its sums are discarded)
    const float4 me = valid ? d.pm4[d.sorted[pos]] : make_float4(kFar, kFar, kFar, 0.f);
    const uint64_t vmask = __ballot(valid);
    const float eps2 = d.eps2;
    const unsigned cap = (unsigned)d.cap;
    double sx = 0.0, sy = 0.0, sz = 0.0;
    float fx = 0.f, fy = 0.f, fz = 0.f, kx = 0.f, ky = 0.f, kz = 0.f; // narrow votes, K = 1
    // Interactions: every child of a visited cell meets the lanes that opened
    // it, except where it is opened in turn, which is a visit of its own: the
    // sum over the visits of (children - 1) x lanes, plus the root's lanes.
    unsigned long long inter = 0;
    bool bad = false;

    if constexpr (K == 1) {
        __syncthreads();
        unsigned cur = 0, fields = 15u; // root cell 0 at depth 0, opened by every group
        int sp = 0;
        for (;;) {
            const uint64_t act = G < 64 ? field_lanes(fields) : kAllLanes;
            float px, py, pz;
            auto opened = [&](unsigned e, unsigned f = 15u) {
                stk[sp] = entry(e, f); // every lane, one address
                ++sp;
            };
            const float thr = dq_s[cur & 63u];
            int children;
            if constexpr (G < 64)
                children = visit_narrow<G, false>(cur, fields, act, thr, me, eps2, cchild, cdata, px, py, pz, bad, opened);
            else
                children = visit_wide<false>(cur, thr, me, eps2, cchild, cdata, px, py, pz, bad, opened);
            if constexpr (G < 64) {
                // only the lanes that opened the cell, as each group alone
                // would sum
                if (__builtin_amdgcn_inverse_ballot_w64(act)) {
                    kahan_add(fx, kx, px);
                    kahan_add(fy, ky, py);
                    kahan_add(fz, kz, pz);
                }
            } else {
                sx += (double)px;
                sy += (double)py;
                sz += (double)pz;
            }
            inter += (G < 64 ? (unsigned long long)(unsigned)__popcll(act & vmask) : 1ull) * (unsigned)(children - 1);
            if (sp == 0) break;
            --sp;
            take_entry(stk[sp], cur, fields);
            if ((cur >> 6) >= cap) { // the pool holds `cap` cells: corrupt
                bad = true;
                break;
            }
        }
    } else {
        if (tid == 0) stk[0] = entry(0, 15u); // root cell 0 at depth 0
        if (block_stops(err)) return;
        if constexpr (G < 64) {
            int sp = 1; // the same in every wave
            for (;;) {
                const int take = sp > kSplitTop ? 1 : min(sp, K);
                int npush = 0;
                unsigned push = 0, pushf = 0; // entry j of this wave's children in lane j
                if (wv < take) {
                    unsigned cur, fields;
                    take_entry(stk[sp - 1 - wv], cur, fields);
                    if ((cur >> 6) >= cap) { // the pool holds `cap` cells: corrupt
                        bad = true;
                    } else {
                        const uint64_t act = field_lanes(fields);
                        float px, py, pz;
                        const int children = visit_narrow<G, true>(
                            cur, fields, act, dq_s[cur & 63u], me, eps2, cchild, cdata, px, py, pz, bad,
                            [&](unsigned e, unsigned f) {
                                push = lane_write(push, e, npush);
                                pushf = lane_write(pushf, f, npush);
                                ++npush;
                            });
                        sx += (double)px;
                        sy += (double)py;
                        sz += (double)pz;
                        inter += (unsigned long long)(unsigned)__popcll(act & vmask) * (unsigned)(children - 1);
                    }
                }
                if (!end_round<K>(stk, pushed, wv, lane, take, npush, entry(push, pushf), bad, sp)) {
                    bad = true;
                    break;
                }
                if (sp == 0) break;
            }
        } else {
            bad = walk_parted<K, 8 * K, K == 4 ? 16 : 8>(stk, pushed, wv, lane, cap, bad, [&](unsigned cur, auto &&opened) {
                float px, py, pz;
                const int children =
                    visit_wide<false>(cur, dq_s[cur & 63u], me, eps2, cchild, cdata, px, py, pz, bad, opened);
                sx += (double)px;
                sy += (double)py;
                sz += (double)pz;
                inter += (unsigned)(children - 1);
            });
        }
        // the waves' sums in wave order
        __syncthreads();
        double *red = reinterpret_cast<double *>(lds);
        red[(wv * 3 + 0) * 64 + lane] = sx;
        red[(wv * 3 + 1) * 64 + lane] = sy;
        red[(wv * 3 + 2) * 64 + lane] = sz;
        if (lane == 0) wint[wv] = inter;
        __syncthreads();
        if (wv > 0) return;
#pragma unroll 1
        for (int w = 1; w < K; ++w) {
            sx += red[(w * 3 + 0) * 64 + lane];
            sy += red[(w * 3 + 1) * 64 + lane];
            sz += red[(w * 3 + 2) * 64 + lane];
            inter += wint[w];
        }
    }
    if (bad && lane == 0) flag_error(ctl, kErrStack);
    if constexpr (G < 64 && K == 1) {
        if (valid) finish_body(d, pos, me, fx - kx, fy - ky, fz - kz, mode, step);
    } else {
        if (valid) finish_body(d, pos, me, (float)sx, (float)sy, (float)sz, mode, step);
    }
    // device interaction counters: one atomic per block
    if (lane == 0) {
        const unsigned nv = (unsigned)__popcll(vmask);
        __hip_atomic_fetch_add(&ctl->tally[blockIdx.x % kTallies].all, G < 64 ? inter + nv : (inter + 1) * nv,
                               __ATOMIC_RELAXED, AGENT);
    }
}

// Waves per group, by the number of groups. One wave per group leaves the
// 1,024 SIMDs (8 waves each) short of waves below about 8,192 groups, and a
// visit is a chain of a stack read and scalar loads; more waves shorten the
// chain of visits but wait for each other. us of the force stage, 1 / 4 / 8 / 16
// waves (one series on one card):
//   vote 64
//   16,384 bodies (256 groups), ball, theta 0.5      282 / 97 / 63 / 46
//   32,768 (512), two spheres, theta 0.4             654 / 228 / 144 / 118
//   40,960 (640), two spheres                        710 / 244 / 157 / 171
//   40,960 (640), disk, theta 1.22                   99 / 43 / 38 / 47
//   100,003 (1,563), two spheres                     862 / 345 / 323 / 360
//   131,072 (2,048), two spheres                     930 / 439 / 404 / 476
//   131,072 (2,048), disk                            111 / 63 / 76 / 101
//   262,144 (4,096), two spheres                     1125 / 750 / 762 / 944
//   400,000 (6,250), two spheres                     1319 / 1121 / 1154 / 1454
//   400,000 (6,250), disk                            150 / 146 / 191 / 285
//   524,288 (8,192), two spheres                     1600 / 1437 / 1499 / 1909
//   524,288 (8,192), disk                            170 / 182 / 245 / 374
//   vote 16 (32 alike)
//   16,384 (256), ball, theta 0.5                    391 / 194 / 102 / 74
//   32,768 (512), disk, theta 1.22                   136 / 61 / 43 / 40
//   40,960 (640), ball                               514 / 255 / 144 / 146
//   65,536 (1,024), ball                             537 / 300 / 175 / 190
//   65,536 (1,024), disk                             140 / 73 / 55 / 72
//   100,003 (1,563), ball                            599 / 390 / 264 / 289
//   262,144 (4,096), ball                            764 / 832 / 591 / 700
//   400,000 (6,250), ball                            928 / 1215 / 897 / 1072
// The narrow line is no crossing: 8 waves would be the faster up to 4,096 groups.
// From 641 groups on a wave alone keeps, at that price, the order of its group's own
// depth-first walk, and so every body's sum bit for bit as a walk per group gives
// it; below, where a step gains three times and more, the order is given up. The
// sums of both orders are equally far from 64 bits (16,384 bodies, ball: rms 4.9e-8
// and 4.8e-8 of the acceleration; 32,768, disk: 8.7e-8 and 8.4e-8), but a run may
// grow their difference: a rotating disk at the reference's vote and time step (0.025)
// to 2e-5 of the velocities in 20 steps at 1,000 and 16,384 bodies, 6e-5 at 32,768
// and 65,536, 3e-4 at 262,144 (the body that differs most).
static int waves_per_group(int groups, bool narrow)
{
    if (narrow) return groups <= 640 ? 16 : 1;
    return groups <= 576 ? 16 : groups <= 1792 ? 8 : groups <= 6400 ? 4 : 1;
}

template <int G> static void launch_force_g(const Dev &d, int mode, hipStream_t st)
{
    const int groups = (d.n + 63) / 64;
    const dim3 grid(groups);
    const int *cc = d.cchild;
    const float4 *cd = d.cdata;
    const int k = waves_per_group(groups, G < 64);
    if (k == 16) hipLaunchKernelGGL((k_force<G, 16>), grid, dim3(1024), 0, st, d, cc, cd, mode);
    else if (k == 1) hipLaunchKernelGGL((k_force<G, 1>), grid, dim3(64), 0, st, d, cc, cd, mode);
    else if constexpr (G == 64) {
        if (k == 8) hipLaunchKernelGGL((k_force<G, 8>), grid, dim3(512), 0, st, d, cc, cd, mode);
        else hipLaunchKernelGGL((k_force<G, 4>), grid, dim3(256), 0, st, d, cc, cd, mode);
    }
}

hipError_t launch_force(const Dev &d, int vote, int mode, hipStream_t st)
{
    switch (vote) {
    case 16: launch_force_g<16>(d, mode, st); break;
    case 32: launch_force_g<32>(d, mode, st); break;
    case 64: launch_force_g<64>(d, mode, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// FP64 direct sum on sampled bodies (the error yardstick; G = 1): block (t, s)
// sums the bodies [s * chunk, (s + 1) * chunk) for 64 targets: 4 threads per
// target stride through the chunk, whose bodies are staged through LDS
// (converted to FP64) once for all 64 targets. 1 / sqrt(r^2) starts from the
// FP64 hardware estimate (v_rsq_f64) and takes one FP64 Newton step,
// y (3/2 - r^2 y^2 / 2), which squares its relative error (the parity test
// holds it to 1e-12). Partial sums per (target, chunk) are combined by a second
// kernel in a fixed order, so the result is deterministic.
//
// Three sums: the accelerations; the softened potentials
// sum_{j != i} m_j / sqrt(r^2 + eps^2) alone (in the w component); and, for the
// total energy of all bodies, each target's potential from the bodies after it
// only, so that every pair is worked out once (a block whose chunk ends before
// its targets has nothing to do). Bound: FP64 issue, 20 slots a pair for the
// accelerations (the estimate takes four), 15 for a potential: the exact
// potential of 131,072 bodies 11.8 -> 3.8 ms against all pairs with
// accelerations beside it.
// ---------------------------------------------------------------------------
constexpr int kDirChunks = 64;  // source chunks
constexpr int kDirTargets = 64; // targets per block
constexpr int kDirTile = 256;   // bodies staged per LDS tile

template <DirectSum SUM>
__global__ __launch_bounds__(256) void k_direct64(Dev d, const int *__restrict__ idx, int ns, double4 *part)
{
    __shared__ double4 tile[kDirTile];
    __shared__ double4 red[256];
    const int n = d.n;
    const int t0 = blockIdx.x * kDirTargets;
    const int chunk = (n + kDirChunks - 1) / kDirChunks;
    int lo = min(n, (int)blockIdx.y * chunk);
    const int hi = min(n, lo + chunk);
    const int tl = threadIdx.x & (kDirTargets - 1); // target of this thread
    // 0..3: which quarter of each tile (the wave's index: uniform, so the
    // source loop below is counted in scalar registers)
    const int sub = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kDirTargets);
    const int tgt = t0 + tl;
    double tx = 0.0, ty = 0.0, tz = 0.0;
    int self = -1;
    if (tgt < ns) {
        const int b = idx[tgt];
        if (b >= 0 && b < n) {
            const float4 p = d.pm4[b];
            tx = p.x; ty = p.y; tz = p.z;
            self = b;
        }
    }
    // kDirectPhiAfter: the targets are consecutive bodies; sources from the
    // first one's successor on
    int first = 0, last = 0; // the block's first and last target
    if (SUM == kDirectPhiAfter) {
        first = __builtin_amdgcn_readfirstlane(idx[t0]);
        last = first + min(kDirTargets, ns - t0) - 1;
        lo = max(lo, first + 1);
    }
    const double eps2 = (double)d.eps2;
    double ax = 0.0, ay = 0.0, az = 0.0, phi = 0.0;
    for (int base = lo; base < hi; base += kDirTile) {
        __syncthreads();
        const int j = base + threadIdx.x;
        const float4 pj = j < hi ? d.pm4[j] : make_float4(0.f, 0.f, 0.f, 0.f);
        tile[threadIdx.x] = make_double4(pj.x, pj.y, pj.z, pj.w);
        __syncthreads();
        const int cnt = min(kDirTile, hi - base);
        // one source's terms, added in source order; TEST: the tile may hold
        // sources that this target leaves out
        auto pair = [&](int k, auto test) {
            const double4 s = tile[k];
            const double dx = s.x - tx, dy = s.y - ty, dz = s.z - tz;
            const double r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, eps2)));
            double ri = __builtin_amdgcn_rsq(r2);
            ri = ri * fma(-0.5 * r2, ri * ri, 1.5);
            if (SUM == kDirectAcc) {
                const double f = s.w * ri * ri * ri;
                ax = fma(dx, f, ax);
                ay = fma(dy, f, ay);
                az = fma(dz, f, az);
            } else if (test) {
                const bool in = SUM == kDirectPhi ? base + k != self : base + k > self;
                phi = fma(s.w, in ? ri : 0.0, phi);
            } else {
                phi = fma(s.w, ri, phi);
            }
        };
        // four sources per round: their loads and arithmetic overlap, only the
        // final adds are chained (the same order as one at a time)
        auto sweep = [&](auto test) {
            int k = sub;
            for (; k + 12 < cnt; k += 16) {
                pair(k, test);
                pair(k + 4, test);
                pair(k + 8, test);
                pair(k + 12, test);
            }
            for (; k < cnt; k += 4) pair(k, test);
        };
        if (SUM == kDirectPhi || (SUM == kDirectPhiAfter && base <= last))
            sweep(std::true_type{});
        else
            sweep(std::false_type{});
    }
    red[threadIdx.x] = make_double4(ax, ay, az, phi);
    __syncthreads();
    if (sub == 0 && tgt < ns) {
        double4 r = red[tl];
        for (int k = 1; k < 4; ++k) {
            const double4 o = red[tl + k * kDirTargets];
            r.x += o.x; r.y += o.y; r.z += o.z; r.w += o.w;
        }
        part[(size_t)tgt * kDirChunks + blockIdx.y] = r;
    }
}

__global__ __launch_bounds__(256) void k_direct64_reduce(const double4 *part, int ns, double4 *out)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ns) return;
    double4 r = make_double4(0.0, 0.0, 0.0, 0.0);
    for (int k = 0; k < kDirChunks; ++k) {
        const double4 o = part[(size_t)t * kDirChunks + k];
        r.x += o.x; r.y += o.y; r.z += o.z; r.w += o.w;
    }
    out[t] = r;
}

// part must hold ns * 64 entries, out ns entries
hipError_t launch_direct64(const Dev &d, const int *idx, int ns, double4 *part, double4 *out, DirectSum sum,
                           hipStream_t st)
{
    if (ns <= 0) return hipSuccess;
    const dim3 grid((ns + kDirTargets - 1) / kDirTargets, kDirChunks);
    switch (sum) {
    case kDirectAcc: hipLaunchKernelGGL(k_direct64<kDirectAcc>, grid, dim3(256), 0, st, d, idx, ns, part); break;
    case kDirectPhi: hipLaunchKernelGGL(k_direct64<kDirectPhi>, grid, dim3(256), 0, st, d, idx, ns, part); break;
    case kDirectPhiAfter:
        hipLaunchKernelGGL(k_direct64<kDirectPhiAfter>, grid, dim3(256), 0, st, d, idx, ns, part);
        break;
    }
    hipLaunchKernelGGL(k_direct64_reduce, dim3((ns + 255) / 256), dim3(256), 0, st, (const double4 *)part, ns,
                       out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// FP64 sums over all bodies for the diagnostics: per block (grid-stride over
// bodies, fixed grid) the mass, momentum, kinetic energy, angular momentum
// about the origin and first moment of mass; the host adds the blocks in order.
// ---------------------------------------------------------------------------
constexpr int kMomTerms = 11; // m, p(3), ke, L(3), m x(3)

__global__ __launch_bounds__(256) void k_moments(Dev d, double *part)
{
    __shared__ double red[kMomTerms][256];
    double acc[kMomTerms];
#pragma unroll
    for (int k = 0; k < kMomTerms; ++k) acc[k] = 0.0;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < d.n; i += kMomentBlocks * 256) {
        const float4 p = d.pm4[i];
        const float4 v = d.vel4[i];
        double x = p.x, y = p.y, z = p.z;
        if (d.fp64) {
            const double4 q = d.pos64[i];
            x = q.x; y = q.y; z = q.z;
        }
        const double m = p.w, vx = v.x, vy = v.y, vz = v.z;
        acc[0] += m;
        acc[1] += m * vx;
        acc[2] += m * vy;
        acc[3] += m * vz;
        acc[4] += 0.5 * m * (vx * vx + vy * vy + vz * vz);
        acc[5] += m * (y * vz - z * vy);
        acc[6] += m * (z * vx - x * vz);
        acc[7] += m * (x * vy - y * vx);
        acc[8] += m * x;
        acc[9] += m * y;
        acc[10] += m * z;
    }
#pragma unroll
    for (int k = 0; k < kMomTerms; ++k) red[k][threadIdx.x] = acc[k];
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o)
#pragma unroll
            for (int k = 0; k < kMomTerms; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x < kMomTerms) part[(size_t)blockIdx.x * kMomTerms + threadIdx.x] = red[threadIdx.x][0];
}

hipError_t launch_moments(const Dev &d, double *part, hipStream_t st)
{
    hipLaunchKernelGGL(k_moments, dim3(kMomentBlocks), dim3(256), 0, st, d, part);
    return hipGetLastError();
}

} // namespace nb
