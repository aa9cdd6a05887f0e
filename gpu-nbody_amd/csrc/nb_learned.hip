// nb_learned.hip -- the learned coarse-theta correction for gfx950.
//
// Coarse traversal. The wave-uniform traversal of the force stage (one wave
// = one vote group of 64 sorted bodies, a cell is taken when all 64 lanes
// accept it) with a coarser test. A lane accepts a cell of extent b (the
// largest distance of its bodies from its centre of mass, bounded in
// summarize) and mass m at s^2 = |d|^2 + eps^2 when
//     s^2 >= b^2 / theta_c^2 + eps^2           (extent test: |d| >= b / theta_c)
//     s^2 >= (m b^3)^(2/5) (alpha^2 |a_old|^2)^(-1/5)
//                                              (relative test: m b^3 / s^5, the
//                                               size of the first term left
//                                               out, within alpha |a_old|; its
//                                               two factors are rounded to FP32
//                                               once, per cell and per body)
// with a_old the body's acceleration of the previous step (the relative test
// is off for a lane while there is none). Every accepted cell contributes its
// monopole and its quadrupole under the softened kernel: with d = centre of
// mass - body and the cell's traceless second moment Q and trace T about its
// centre of mass,
//     a = m d / s^3 - Q d / s^5 + 5/2 (d.Q.d - T eps^2) d / s^7 .
// (The T eps^2 term is the part of the second-order expansion of the
// softened kernel that the traceless Q does not carry; it matters once cells
// sit within a few softening lengths.) Bodies interact as point masses. The
// training targets use the same kernel with the force stage's opening table
// (kOutAccel).
// A visited cell's bodies come first (its quadrupole records are on their way
// from memory meanwhile), then each child cell is tested and, when taken,
// added at once: with all tests before all terms the squared distance of a taken
// cell was worked out twice (3.27 -> 2.97 ms at 4M clustered bodies, alpha
// 0.0175; the bodies' and cells' places in the record make each loop a run of
// one kind, so no branch has three ways). Bound: vector issue.
//
// Features. Per body, 24 numbers in a frame built from the body's own coarse
// acceleration a: e1 = a / |a|, e2 = the part of the quadrupole acceleration
// a_q perpendicular to e1, normalized, e3 = e1 x e2. Vectors are projected on
// the frame and divided by |a|, so the features do not change under rotations
// and under a common scaling of the masses. Per accepted cell the traversal
// only keeps the quadrupole part and the cell mass apart; the rest comes once
// per body from wave reductions.
//    0-2  acceleration from bodies (a_b)
//    3-4  a_q along e1, e2 (its e3 component is 0 by construction)
//    5-7  a minus the mean coarse acceleration of the group
//    8-10 offset of the body from its group's centroid, over the group radius
//   11-13 the group's mean a_b
//   14-16 the group's mean a_q
//   17-18 log(1 + accepted cells), log(1 + bodies met)
//   19-20 log(|a_q| / |a|), log(|a_b| / |a|)
//   21    accepted-cell mass / (accepted-cell mass + body mass met)
//   22    log(group radius / root radius)
//   23    cosine between the cell monopole part and a_b
//
// Network. 24 -> 64 -> 64 -> 3 with tanh-GELU. Inference runs in the epilogue
// of the coarse traversal itself: the wave's 64 bodies go through
// v_mfma_f32_16x16x32_bf16 (BF16 operands, FP32 accumulation) in the
// transposed form Z^T = W^T X^T, 16 bodies (one B-operand column block) at a
// time: 4 + 8 + 2 matrix instructions per block. The features reach the
// operand layout through LDS once; between layers, each lane's D registers
// already hold what it needs as the next B operand (the weights are stored
// with the matching order of k), and the three outputs return to their own
// lanes by shuffles. The corrected acceleration then goes straight into the
// body update, so the update overlaps with other waves' traversal. Training:
// forward, backward and weight gradients in one kernel on the FP32 matrix
// instruction, the gradient's sum and Adam in a second, all sums in a fixed
// order.
#include "nb_device.h"

namespace nb {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// numerics shared by inference and training
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint16_t to_bf16(float f)
{
    // round to nearest even (inputs are finite)
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

// tanh(y) = 1 - 2 / (exp(2y) + 1) with the hardware reciprocal (1 ulp): the
// network is BF16 at inference, so an IEEE division buys nothing here;
// saturates correctly at both ends (rcp(inf) = 0, rcp(1) = 1)
__device__ __forceinline__ float tanh_fast(float y)
{
    return 1.0f - 2.0f * __builtin_amdgcn_rcpf(__expf(2.0f * y) + 1.0f);
}

constexpr float kGeluC = 0.7978845608028654f; // sqrt(2 / pi)
constexpr float kGeluA = 0.044715f;

__device__ __forceinline__ float clipz(float z) { return fminf(fmaxf(z, -kClipZ), kClipZ); }

// Inference GELU in the logistic form of the same function,
// 0.5 x (1 + tanh(u)) = x / (1 + exp(-2 u)), u = sqrt(2/pi) (x + 0.044715 x^3),
// with the hardware 2^x and reciprocal: 7 instructions. Limits: x -> +inf
// gives x, x -> -inf gives -0 (2^+inf = inf, 1 / inf = 0).
constexpr float kGeluK1 = -2.0f * kGeluC * 1.4426950408889634f;          // -2 c log2(e)
constexpr float kGeluK2 = -2.0f * kGeluC * kGeluA * 1.4426950408889634f; // -2 c a log2(e)

__device__ __forceinline__ float gelu_infer(float x)
{
    const float s = fmaf(kGeluK2, x * x, kGeluK1);
    return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(s * x));
}

// two floats to packed BF16, round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi)
{
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 h = {(__bf16)lo, (__bf16)hi};
    return __builtin_bit_cast(uint32_t, h);
}

__device__ __forceinline__ bf16x8 load_bf16x8(const uint16_t *p)
{
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const u16x8 *>(p));
}

// ---------------------------------------------------------------------------
// BF16 matrix-core network (shared by the learned step and the test path)
//
// v_mfma_f32_16x16x32_bf16 operand layout (lane l, i16 = l % 16, g = l / 16):
//   A: row i16 of the 16-row block, k = 8 g .. 8 g + 7
//   B: column i16 of the 16-column block, k = 8 g .. 8 g + 7
//   D: column i16, rows 4 g .. 4 g + 3
// ---------------------------------------------------------------------------
// GELU of two accumulator blocks (their biases came in as the accumulators'
// initial values), packed to BF16
__device__ __forceinline__ bf16x8 pack_gelu(f32x4 lo, f32x4 hi)
{
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 h = {pack_bf16(gelu_infer(lo[0]), gelu_infer(lo[1])), pack_bf16(gelu_infer(lo[2]), gelu_infer(lo[3])),
                     pack_bf16(gelu_infer(hi[0]), gelu_infer(hi[1])), pack_bf16(gelu_infer(hi[2]), gelu_infer(hi[3]))};
    return __builtin_bit_cast(bf16x8, h);
}

__device__ __forceinline__ f32x4 as_f32x4(float4 v) { return f32x4{v.x, v.y, v.z, v.w}; }

// Runs the wave's 64 rows of normalized BF16 features (fs: LDS, row r at
// fs + 24 r) through the network; lane r receives the residual of row r.
__device__ __forceinline__ void mlp_wave(const uint16_t *fs, const Mlp &m, int lane, float &y0, float &y1,
                                         float &y2)
{
    const int i16 = lane & 15, g = lane >> 4;
    const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
    y0 = y1 = y2 = 0.f;
    // one 16-body column block at a time, not unrolled: the epilogue must not
    // raise the register count of the traversal it ends
#pragma unroll 1
    for (int cb = 0; cb < 4; ++cb) {
        const bf16x8 xb = g < 3 ? load_bf16x8(fs + (cb * 16 + i16) * kFeat + 8 * g)
                                : __builtin_bit_cast(bf16x8, u16x8{0, 0, 0, 0, 0, 0, 0, 0});
        // each layer in two halves of 32 hidden rows (two 16-row blocks),
        // each half's activations packed before the next half starts: fewer
        // accumulators live at once
        const float4 *b1 = reinterpret_cast<const float4 *>(m.b1 + 4 * g);
        const float4 *b2 = reinterpret_cast<const float4 *>(m.b2 + 4 * g);
        bf16x8 h1[2];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            const f32x4 p0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load_bf16x8(m.w1f + ((2 * hf) * 64 + lane) * 8), xb,
                                                                     as_f32x4(b1[8 * hf]), 0, 0, 0);
            const f32x4 p1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                load_bf16x8(m.w1f + ((2 * hf + 1) * 64 + lane) * 8), xb, as_f32x4(b1[8 * hf + 4]), 0, 0, 0);
            h1[hf] = pack_gelu(p0, p1);
            __builtin_amdgcn_sched_barrier(0);
        }
        bf16x8 h2[2];
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            f32x4 p[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int rb = 2 * hf + q;
                p[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load_bf16x8(m.w2f + ((rb * 2 + 0) * 64 + lane) * 8),
                                                               h1[0], as_f32x4(b2[4 * rb]), 0, 0, 0);
                p[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load_bf16x8(m.w2f + ((rb * 2 + 1) * 64 + lane) * 8),
                                                               h1[1], p[q], 0, 0, 0);
            }
            h2[hf] = pack_gelu(p[0], p[1]);
            __builtin_amdgcn_sched_barrier(0);
        }
        const bf16x8 h2a = h2[0], h2b = h2[1];
        f32x4 d3 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load_bf16x8(m.w3f + lane * 8), h2a, z4, 0, 0, 0);
        d3 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load_bf16x8(m.w3f + (64 + lane) * 8), h2b, d3, 0, 0, 0);
        // outputs 0..2 of the column block's bodies sit in lanes 0..15 (g = 0)
        const float t0 = __shfl(d3[0], i16), t1 = __shfl(d3[1], i16), t2 = __shfl(d3[2], i16);
        if (g == cb) {
            y0 = t0 + m.b3[0];
            y1 = t1 + m.b3[1];
            y2 = t2 + m.b3[2];
        }
    }
}

// ---------------------------------------------------------------------------
// Coarse traversal
// ---------------------------------------------------------------------------
#define NB_COARSE_PARAMS                                                                                     \
    Dev d, Learn L, const int *__restrict__ cchild, const float4 *__restrict__ cdata,                        \
        const float4 *__restrict__ cqa, const float4 *__restrict__ cqb, const float2 *__restrict__ cmac,     \
        const int *__restrict__ groups, int ngroups,                                                         \
        const float4 *__restrict__ rec, float *__restrict__ xraw, float4 *__restrict__ frame_out,            \
        float4 *__restrict__ acc_out, int fmode
#define NB_COARSE_PASS \
    d, L, cchild, cdata, cqa, cqb, cmac, groups, ngroups, rec, xraw, frame_out, acc_out, fmode

// K waves share a vote group, as in k_force (nb_force.hip): one wave walks depth
// first; K start breadth first and part, and their sums are added in wave order.
template <int OUT, int K, bool REC> __device__ __forceinline__ void coarse_traverse(int gslot, NB_COARSE_PARAMS)
{
    constexpr bool kFeatOn = OUT == kOutLearned || OUT == kOutRaw;
    constexpr bool kGeo = OUT == kOutAccel; // the fine traversal: the force stage's opening table
    // the stack; after the traversal the waves' sums overlay it, and the
    // learned step's 64 rows of BF16 features (64 x 24 x 2 bytes)
    constexpr int kRedBytes = K == 1 ? 0 : K * 64 * (kFeatOn ? 9 * 4 : 3 * 8);
    constexpr int kFeatBytes = OUT == kOutLearned ? 64 * kFeat * 2 : 0;
    constexpr int kStackBytes = (K == 1 ? kStack : parted_stack<K>()) * 4;
    constexpr int kLds = kStackBytes > kRedBytes ? (kStackBytes > kFeatBytes ? kStackBytes : kFeatBytes)
                                                 : (kRedBytes > kFeatBytes ? kRedBytes : kFeatBytes);
    struct WaveTotals {
        float smb;
        int bodies, cells, visits;
    };
    __shared__ __attribute__((aligned(16))) unsigned char lds[kLds];
    // a visited cell's children's quadrupole records, (qa, qb) per child, for
    // the accepted cells' uniform LDS reads
    __shared__ float4 qst[K][16];
    __shared__ float dq_s[kMaxDepth];
    __shared__ unsigned pushed[K];
    __shared__ WaveTotals totals[K];
    unsigned *stk = reinterpret_cast<unsigned *>(lds); // (cell << 6 | depth)
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wv = K == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = d.n;
    Ctl *ctl = d.ctl;
    const int err = ctl->error; // several waves decide together, as in k_force
    if (K == 1 && err) return;
    if (ctl->max_depth > kMaxDepth) {
        if (tid == 0) flag_error(ctl, kErrDepth);
        return;
    }
    // REC: the step's own scalars, as k_pair_records kept them
    const PairCtl *pc = REC ? reinterpret_cast<const PairCtl *>(rec + 2 * 64 * (size_t)ngroups) : nullptr;
    if (kGeo)
        for (int i = tid; i < kMaxDepth; i += 64 * K) dq_s[i] = pc->dq[i];
    const int step = REC ? pc->step : ctl->step;
    const float root_r = REC ? pc->radius : ctl->radius;

    int g = gslot;
    if (groups) {
        if (gslot >= ngroups) return;
        g = groups[gslot];
    }
    const int pos = g * 64 + lane;
    const bool valid = pos >= 0 && pos < n;
    if (__ballot(valid) == 0ull) return; // the same in every wave of the block
    // a lane past the last body sits at infinity: its d^2 is infinite, so it
    // accepts every cell and never holds up the vote (its sums are discarded)
    // REC: the groups' records and accelerations as k_pair_records copied them
    float4 me = make_float4(kFar, kFar, kFar, 0.f);
    if (valid) me = REC ? rec[2 * ((size_t)gslot * 64 + lane)] : d.pm4[d.sorted[pos]];
    const float eps2 = d.eps2;
    const unsigned cap = (unsigned)d.cap;
    // the body's factor (alpha^2 |a_old|^2)^(-1/5) of the relative test's
    // threshold; 0 switches it off (no previous acceleration yet, as in the
    // force stage's kick, or alpha = 0)
    float a5 = 0.f;
    if (!kGeo && valid && step > 0 && d.alpha2_coarse > 0.f) {
        const float4 a0 = REC ? rec[2 * ((size_t)gslot * 64 + lane) + 1] : d.acc4[d.sorted[pos]];
        const float a2 = fmaf(a0.x, a0.x, fmaf(a0.y, a0.y, a0.z * a0.z));
        if (a2 > 0.f) a5 = (float)pow((double)(d.alpha2_coarse * a2), -0.2);
    }

    // The learned step and the features keep three FP32 running sums --
    // bodies (b), cell monopoles (s) and cell quadrupoles (q): the features
    // need them apart, and the step's error bound is 1e-3. The coarse force
    // alone sums a visited cell's terms in FP32 and adds them into FP64 sums
    // (t; convert and add issue like two FP32 adds), the fine pass into
    // compensated FP32 sums (s, k), in the order of its walk.
    double tx = 0.0, ty = 0.0, tz = 0.0;
    float kx = 0.f, ky = 0.f, kz = 0.f;
    float sx = 0.f, sy = 0.f, sz = 0.f;
    float bx = 0.f, by = 0.f, bz = 0.f;
    float qx = 0.f, qy = 0.f, qz = 0.f;
    float smb = 0.f; // mass of the bodies met (the accepted cells hold the rest)
    // children met so far: every child cell of a visited cell is accepted or
    // visited in turn
    int nbod = 0, nchild = 0, nvisit = 0;
    bool bad = false;

    // One visit of cell e >> 6 on level e & 63; opened(entry) for the
    // children to visit. Every branch is wave-uniform.
    auto visit = [&](unsigned e, auto &&opened) {
        const size_t c = e >> 6;
        const i32x8 ch = *reinterpret_cast<const i32x8 *>(cchild + c * 8);
        const f32x16 q0 = *reinterpret_cast<const f32x16 *>(cdata + c * 8);
        const f32x16 q1 = *reinterpret_cast<const f32x16 *>(cdata + c * 8 + 4);
        f32x16 mc;
        if constexpr (!kGeo) mc = *reinterpret_cast<const f32x16 *>(cmac + c * 8);
        float thr = 0.f;
        if constexpr (kGeo) thr = dq_s[e & 63u];
        // the children's quadrupole records, child k in lanes k, k + 8, ...:
        // two vector loads issued now, waited for after the bodies; each from
        // the cell's uniform base plus an unsigned lane offset (no 64-bit
        // address adds per lane)
        const float4 qav = (cqa + c * 8)[(unsigned)lane & 7u];
        const float4 qbv = (cqb + c * 8)[(unsigned)lane & 7u];
        // child cells at the front of the record, bodies at its back
        const int nbody = (int)((unsigned)ch[0] >> kCountShift);
        int ncell = (int)((unsigned)ch[1] >> kCountShift);
        if ((e & 63u) == kMaxDepth - 1 && ncell > 0) { // no level below: corrupt
            bad = true;
            ncell = 0;
        }
        nbod += nbody;
        nchild += ncell;
        ++nvisit;
        float px = 0.f, py = 0.f, pz = 0.f, cx = 0.f, cy = 0.f, cz = 0.f; // this cell's bodies and child cells
        float &bpx = kFeatOn ? bx : px, &bpy = kFeatOn ? by : py, &bpz = kFeatOn ? bz : pz;
        float &mpx = kFeatOn ? sx : kGeo ? cx : px, &mpy = kFeatOn ? sy : kGeo ? cy : py, &mpz = kFeatOn ? sz : kGeo ? cz : pz;
#pragma unroll
        for (int k = 7; k >= 0; --k) {
            if (7 - k >= nbody) break;
            const f32x16 &q = k < 4 ? q0 : q1;
            const int o = 4 * (k & 3);
            const float dx = q[o] - me.x, dy = q[o + 1] - me.y, dz = q[o + 2] - me.z;
            const float d2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
            const float ri = __builtin_amdgcn_rsqf(d2);
            const float f = q[o + 3] * (ri * ri * ri);
            bpx = fmaf(dx, f, bpx);
            bpy = fmaf(dy, f, bpy);
            bpz = fmaf(dz, f, bpz);
            if (kFeatOn) smb += q[o + 3];
        }
        // the records into this wave's LDS rows: an accepted cell reads its two
        // with uniform LDS reads, no VALU
        if (ncell) {
            if (lane < 8) {
                qst[wv][2 * lane] = qav;
                qst[wv][2 * lane + 1] = qbv;
            }
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if (k >= ncell) break;
            const f32x16 &q = k < 4 ? q0 : q1;
            const int o = 4 * (k & 3);
            const float dx = q[o] - me.x, dy = q[o + 1] - me.y, dz = q[o + 2] - me.z;
            const float d2 = fmaf(dx, dx, fmaf(dy, dy, fmaf(dz, dz, eps2)));
            // The coarse test: the extent (threshold b^2 / theta_c^2 + eps^2
            // from summarize), then the relative test (threshold the product
            // of the cell's and the body's factors) only when every lane
            // passed it. Lane masks come straight from the compares (3 =
            // ordered >=, 5 = ordered <=).
            bool take = __builtin_amdgcn_fcmpf(d2, kGeo ? thr : mc[2 * k], 3) == kAllLanes;
            if (!kGeo && take) take = __builtin_amdgcn_fcmpf(mc[2 * k + 1] * a5, d2, 5) == kAllLanes;
            if (!take) {
                opened(((unsigned)ch[k] << 6) | ((e & 63u) + 1u));
                continue;
            }
            const float4 qa = qst[wv][2 * k], qb = qst[wv][2 * k + 1]; // (Qxx, Qyy, Qzz, T eps^2), (Qxy, Qxz, Qyz, 0)
            const float ri = __builtin_amdgcn_rsqf(d2);
            const float r2i = ri * ri;
            const float r3 = r2i * ri;
            const float f = q[o + 3] * r3;
            const float Qx = fmaf(qa.x, dx, fmaf(qb.x, dy, qb.y * dz));
            const float Qy = fmaf(qb.x, dx, fmaf(qa.y, dy, qb.z * dz));
            const float Qz = fmaf(qb.y, dx, fmaf(qb.z, dy, qa.z * dz));
            const float dQd = fmaf(Qx, dx, fmaf(Qy, dy, Qz * dz));
            const float r5 = r3 * r2i;
            if (kFeatOn) {
                // the quadrupole part as r5 (u d - Q d), u = 5/2 (d.Q.d - T eps^2) / s^2
                const float u = (dQd - qa.w) * (2.5f * r2i);
                mpx = fmaf(dx, f, mpx);
                mpy = fmaf(dy, f, mpy);
                mpz = fmaf(dz, f, mpz);
                qx = fmaf(r5, fmaf(u, dx, -Qx), qx);
                qy = fmaf(r5, fmaf(u, dy, -Qy), qy);
                qz = fmaf(r5, fmaf(u, dz, -Qz), qz);
            } else {
                const float c2 = (dQd - qa.w) * ((2.5f * r5) * r2i);
                // monopole and quadrupole radial terms share one factor
                const float h = f + c2;
                mpx = fmaf(dx, h, fmaf(-r5, Qx, mpx));
                mpy = fmaf(dy, h, fmaf(-r5, Qy, mpy));
                mpz = fmaf(dz, h, fmaf(-r5, Qz, mpz));
            }
        }
        if constexpr (!kFeatOn) {
            if constexpr (kGeo) {
                kahan_add(sx, kx, px + cx);
                kahan_add(sy, ky, py + cy);
                kahan_add(sz, kz, pz + cz);
            } else {
                tx += (double)px;
                ty += (double)py;
                tz += (double)pz;
            }
        }
    };

    if constexpr (K == 1) {
        if (kGeo) __syncthreads();
        unsigned cur = 0; // root cell 0 at depth 0
        int sp = 0;
        for (;;) {
            visit(cur, [&](unsigned e) {
                stk[sp] = e; // every lane, one address
                ++sp;
            });
            if (sp == 0) break;
            --sp;
            cur = __builtin_amdgcn_readfirstlane(stk[sp]);
            if ((cur >> 6) >= cap) { // the pool holds `cap` cells: corrupt
                bad = true;
                break;
            }
        }
    } else {
        if (tid == 0) stk[0] = 0; // root cell 0 at depth 0
        if (block_stops(err)) return;
        bad = walk_parted<K, 64, 32>(stk, pushed, wv, lane, cap, bad, visit);
        // the waves' sums in wave order
        __syncthreads();
        if (lane == 0) totals[wv] = WaveTotals{smb, nbod, nchild, nvisit};
        float *rf = reinterpret_cast<float *>(lds);
        double *rd = reinterpret_cast<double *>(lds);
        if constexpr (kFeatOn) {
            const float v[9] = {bx, by, bz, sx, sy, sz, qx, qy, qz};
#pragma unroll
            for (int i = 0; i < 9; ++i) rf[(wv * 9 + i) * 64 + lane] = v[i];
        } else {
            rd[(wv * 3 + 0) * 64 + lane] = tx;
            rd[(wv * 3 + 1) * 64 + lane] = ty;
            rd[(wv * 3 + 2) * 64 + lane] = tz;
        }
        __syncthreads();
        if (wv > 0) return;
#pragma unroll 1
        for (int w = 1; w < K; ++w) {
            if constexpr (kFeatOn) {
                const float *o = rf + w * 9 * 64 + lane;
                bx += o[0 * 64]; by += o[1 * 64]; bz += o[2 * 64];
                sx += o[3 * 64]; sy += o[4 * 64]; sz += o[5 * 64];
                qx += o[6 * 64]; qy += o[7 * 64]; qz += o[8 * 64];
            } else {
                tx += rd[(w * 3 + 0) * 64 + lane];
                ty += rd[(w * 3 + 1) * 64 + lane];
                tz += rd[(w * 3 + 2) * 64 + lane];
            }
            smb += totals[w].smb;
            nbod += totals[w].bodies;
            nchild += totals[w].cells;
            nvisit += totals[w].visits;
        }
    }
    const int nc = nchild - (nvisit - 1); // accepted cells
    if (bad && lane == 0) flag_error(ctl, kErrStack);
    if constexpr (OUT == kOutLearned || OUT == kOutFinish) {
        // the group's cost for the next launch order, in interactions: a
        // visited cell (its loads and up to eight tests) weighs about three
        const long long cost = (long long)nbod + nc + 3ll * nvisit;
        if (lane == 0) d.gcost[g] = cost < 0x7fffffffll ? (int)cost : 0x7fffffff;
    }
    const float ax = kFeatOn ? (bx + sx) + qx : kGeo ? sx - kx : (float)tx;
    const float ay = kFeatOn ? (by + sy) + qy : kGeo ? sy - ky : (float)ty;
    const float az = kFeatOn ? (bz + sz) + qz : kGeo ? sz - kz : (float)tz;
    const int slot = gslot * 64 + lane;
    if constexpr (OUT == kOutAccel) {
        if (valid) acc_out[slot] = make_float4(ax, ay, az, 0.f);
    } else if constexpr (OUT == kOutFinish) {
        if (valid) finish_body(d, pos, me, ax, ay, az, fmode, step);
    } else {
        // group centroid and radius, mean acceleration and mean body part
        // (wave reductions over the valid lanes)
        const float nv = (float)__popcll(__ballot(valid));
        float gx = valid ? me.x : 0.f, gy = valid ? me.y : 0.f, gz = valid ? me.z : 0.f;
        float gax = valid ? ax : 0.f, gay = valid ? ay : 0.f, gaz = valid ? az : 0.f;
        float gbx = valid ? bx : 0.f, gby = valid ? by : 0.f, gbz = valid ? bz : 0.f;
        float gqx = valid ? qx : 0.f, gqy = valid ? qy : 0.f, gqz = valid ? qz : 0.f;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            gqx += __shfl_xor(gqx, o);
            gqy += __shfl_xor(gqy, o);
            gqz += __shfl_xor(gqz, o);
            gx += __shfl_xor(gx, o);
            gy += __shfl_xor(gy, o);
            gz += __shfl_xor(gz, o);
            gax += __shfl_xor(gax, o);
            gay += __shfl_xor(gay, o);
            gaz += __shfl_xor(gaz, o);
            gbx += __shfl_xor(gbx, o);
            gby += __shfl_xor(gby, o);
            gbz += __shfl_xor(gbz, o);
        }
        // the features end as BF16 network inputs: hardware reciprocal,
        // square root and logarithm (about 1 ulp) instead of the IEEE sequences
        const float inv_nv = __builtin_amdgcn_rcpf(nv);
        gx *= inv_nv;
        gy *= inv_nv;
        gz *= inv_nv;
        gax *= inv_nv;
        gay *= inv_nv;
        gaz *= inv_nv;
        gbx *= inv_nv;
        gby *= inv_nv;
        gbz *= inv_nv;
        gqx *= inv_nv;
        gqy *= inv_nv;
        gqz *= inv_nv;
        const float ox = me.x - gx, oy = me.y - gy, oz = me.z - gz;
        float rg = valid ? __builtin_amdgcn_sqrtf(ox * ox + oy * oy + oz * oz) : 0.f;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) rg = fmaxf(rg, __shfl_xor(rg, o));

        float f[kFeat];
#pragma unroll
        for (int i = 0; i < kFeat; ++i) f[i] = 0.f;
        const float A = __builtin_amdgcn_sqrtf(ax * ax + ay * ay + az * az);
        float e2x = 0.f, e2y = 0.f, e2z = 0.f;
        if (A > 0.f) {
            const float inv = __builtin_amdgcn_rcpf(A);
            const float e1x = ax * inv, e1y = ay * inv, e1z = az * inv;
            const float qe1 = qx * e1x + qy * e1y + qz * e1z;
            float wx = qx - qe1 * e1x, wy = qy - qe1 * e1y, wz = qz - qe1 * e1z;
            float W = __builtin_amdgcn_sqrtf(wx * wx + wy * wy + wz * wz);
            if (!(W > 0.f)) {
                // no quadrupole direction: the coordinate axis least aligned with e1
                const float fx = fabsf(e1x), fy = fabsf(e1y), fz = fabsf(e1z);
                const float tx = (fx <= fy && fx <= fz) ? 1.f : 0.f;
                const float ty = (tx == 0.f && fy <= fz) ? 1.f : 0.f;
                const float tz = (tx == 0.f && ty == 0.f) ? 1.f : 0.f;
                const float te1 = tx * e1x + ty * e1y + tz * e1z;
                wx = tx - te1 * e1x;
                wy = ty - te1 * e1y;
                wz = tz - te1 * e1z;
                W = __builtin_amdgcn_sqrtf(wx * wx + wy * wy + wz * wz);
            }
            const float iW = __builtin_amdgcn_rcpf(W);
            e2x = wx * iW;
            e2y = wy * iW;
            e2z = wz * iW;
            const float e3x = e1y * e2z - e1z * e2y;
            const float e3y = e1z * e2x - e1x * e2z;
            const float e3z = e1x * e2y - e1y * e2x;
#define NB_LOC(X, Y, Z, I)                                                                         \
    f[I] = ((X) * e1x + (Y) * e1y + (Z) * e1z) * inv;                                             \
    f[(I) + 1] = ((X) * e2x + (Y) * e2y + (Z) * e2z) * inv;                                       \
    f[(I) + 2] = ((X) * e3x + (Y) * e3y + (Z) * e3z) * inv
            NB_LOC(bx, by, bz, 0);
            f[3] = qe1 * inv;
            f[4] = (qx * e2x + qy * e2y + qz * e2z) * inv;
            NB_LOC(ax - gax, ay - gay, az - gaz, 5);
            if (rg > 0.f) {
                const float ir = __builtin_amdgcn_rcpf(rg);
                f[8] = (ox * e1x + oy * e1y + oz * e1z) * ir;
                f[9] = (ox * e2x + oy * e2y + oz * e2z) * ir;
                f[10] = (ox * e3x + oy * e3y + oz * e3z) * ir;
            }
            NB_LOC(gbx, gby, gbz, 11);
            NB_LOC(gqx, gqy, gqz, 14);
            f[17] = __logf(1.0f + (float)nc); // counts below 2^24: 1 + n is exact
            f[18] = __logf(1.0f + (float)nbod);
            const float qn = __builtin_amdgcn_sqrtf(qx * qx + qy * qy + qz * qz);
            const float bn = __builtin_amdgcn_sqrtf(bx * bx + by * by + bz * bz);
            f[19] = __logf(fmaxf(qn * inv, 1e-30f));
            f[20] = __logf(fmaxf(bn * inv, 1e-30f));
            // accepted-cell mass over the mass met: every body is met once, as a
            // body or inside an accepted cell, so the cells hold the total
            // mass (the root's) minus the bodies' (one sum fewer in the loop)
            const float mtot = (float)d.com64[0].w;
            f[21] = mtot > 0.f ? (mtot - smb) * __builtin_amdgcn_rcpf(mtot) : 0.f;
            f[22] = __logf(fmaxf(rg * __builtin_amdgcn_rcpf(root_r), 1e-30f));
            const float mx = ax - bx - qx, my = ay - by - qy, mz = az - bz - qz;
            const float mn = __builtin_amdgcn_sqrtf(mx * mx + my * my + mz * mz);
            f[23] = (mn > 0.f && bn > 0.f) ? (mx * bx + my * by + mz * bz) * __builtin_amdgcn_rcpf(mn * bn) : 0.f;
#undef NB_LOC
        }
        if constexpr (OUT == kOutRaw) {
            if (valid) {
                float *o = xraw + (size_t)slot * kFeat;
#pragma unroll
                for (int i = 0; i < kFeat; i += 4)
                    *reinterpret_cast<float4 *>(o + i) = make_float4(f[i], f[i + 1], f[i + 2], f[i + 3]);
                frame_out[2 * (size_t)slot] = make_float4(ax, ay, az, A);
                frame_out[2 * (size_t)slot + 1] = make_float4(A * e2x, A * e2y, A * e2z, 0.f);
            }
        } else {
            // the learned step: normalized BF16 features into this wave's LDS
            // rows, the network, the correction, the body update
            uint16_t *fs = reinterpret_cast<uint16_t *>(lds);
            uint32_t w[kFeat / 2];
#pragma unroll
            for (int i = 0; i < kFeat; i += 2) {
                const uint32_t h = pack_bf16(clipz((f[i] - L.mlp.xmu[i]) * L.mlp.xrs[i]),
                                             clipz((f[i + 1] - L.mlp.xmu[i + 1]) * L.mlp.xrs[i + 1]));
                w[i / 2] = valid ? h : 0u;
            }
            uint4 *o = reinterpret_cast<uint4 *>(fs + lane * kFeat);
            o[0] = make_uint4(w[0], w[1], w[2], w[3]);
            o[1] = make_uint4(w[4], w[5], w[6], w[7]);
            o[2] = make_uint4(w[8], w[9], w[10], w[11]);
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            __builtin_amdgcn_wave_barrier();
            float y0, y1, y2;
            mlp_wave(fs, L.mlp, lane, y0, y1, y2);
            // residual = |a| (y0 e1 + y1 e2 + y2 e3)
            float rx = ax, ry = ay, rz = az;
            if (A > 0.f) {
                const float iA = __builtin_amdgcn_rcpf(A);
                const float e1x = ax * iA, e1y = ay * iA, e1z = az * iA;
                const float e3x = e1y * e2z - e1z * e2y, e3y = e1z * e2x - e1x * e2z, e3z = e1x * e2y - e1y * e2x;
                rx += A * (y0 * e1x + y1 * e2x + y2 * e3x);
                ry += A * (y0 * e1y + y1 * e2y + y2 * e3y);
                rz += A * (y0 * e1z + y1 * e2z + y2 * e3z);
            }
            if (valid) finish_body(d, pos, me, rx, ry, rz, fmode, step);
        }
    }
    // device interaction counters: one atomic each per block
    const unsigned long long nvalid = (unsigned long long)__popcll(__ballot(valid));
    if (lane == 0) {
        Tally *t = &ctl->tally[blockIdx.x % kTallies];
        __hip_atomic_fetch_add(&t->all, (unsigned long long)(unsigned)(nbod + nc) * nvalid, __ATOMIC_RELAXED, AGENT);
        __hip_atomic_fetch_add(&t->cells, (unsigned long long)(unsigned)nc * nvalid, __ATOMIC_RELAXED, AGENT);
    }
}

// The kernels. Seven waves per SIMD at least, by the attribute (learned step
// at 4M clustered bodies 2.97 ms at six, 2.87 ms at seven, where 14 registers
// of its epilogue spill; the coarse force at eight would spill scalar
// registers in the loop, 0.85 -> 1.29 ms at 700,001 bodies).
template <int OUT, int K>
__global__ __launch_bounds__(64 * K) __attribute__((amdgpu_waves_per_eu(7, 8))) void k_coarse64(
    NB_COARSE_PARAMS)
{
    coarse_traverse<OUT, K, false>((int)blockIdx.x, NB_COARSE_PASS);
}

// A step's training pairs, both passes over the listed groups in one launch: the
// fine pass (targets) in the blocks 0 .. ngroups - 1, the raw one (features)
// after them. One wave per group, in the order of its walk: some features are
// ill-conditioned (the direction of the part of the quadrupole acceleration
// across a, where that part is small), targets are the small difference of two
// accelerations, and Adam turns rounding into full steps where a parameter's
// gradient nearly cancels. With waves sharing a group (978 + 270 -> 247 us for
// 256 groups of a 262,144-body run) equally exact sums moved trained weights
// by up to 4e-3. The few long chains run beside the step's force pass instead
// (the engine puts them on a stream of their own, on copies of the bodies'
// records). They are the longer of the two, so their waves issue first on the
// SIMDs they share: a step of pairs at 262,144 bodies 1.255 -> 1.193 ms.
__global__ __launch_bounds__(64) void k_pairs(NB_COARSE_PARAMS)
{
    __builtin_amdgcn_s_setprio(3);
    if ((int)blockIdx.x < ngroups)
        coarse_traverse<kOutAccel, 1, true>((int)blockIdx.x, NB_COARSE_PASS);
    else
        coarse_traverse<kOutRaw, 1, true>((int)blockIdx.x - ngroups, NB_COARSE_PASS);
}

// The records and accelerations of the listed groups' bodies, 64 slots a group,
// and behind them the step's scalars: with both, the pairs read nothing that the
// next step's bounding box and build write
__global__ __launch_bounds__(256) void k_pair_records(Dev d, const int *__restrict__ groups, int slots,
                                                      float4 *__restrict__ rec)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (blockIdx.x == 0) {
        PairCtl *pc = reinterpret_cast<PairCtl *>(rec + 2 * (size_t)slots);
        if (threadIdx.x < kMaxDepth) pc->dq[threadIdx.x] = d.ctl->dq[threadIdx.x];
        if (threadIdx.x == 0) {
            pc->radius = d.ctl->radius;
            pc->step = d.ctl->step;
        }
    }
    if (i >= slots) return;
    const int pos = groups[i >> 6] * 64 + (i & 63);
    if (pos < 0 || pos >= d.n) return;
    const int b = d.sorted[pos];
    rec[2 * (size_t)i] = d.pm4[b];
    rec[2 * (size_t)i + 1] = d.acc4[b];
}

// One block: a histogram of the groups' cost classes (1 + floor(log2 cost),
// 0 for no cost yet), then the groups by class, the most expensive first.
// Inside a class the groups keep roughly their sorted (spatial) order, so
// neighbouring waves still share tree cells in the caches; measured at 4M
// clustered bodies, classes of one octave beat four classes per octave
// (139.9 against 139.4 steps/s; 137.3 in sorted order). The order inside a
// class is not fixed, and the forces do not depend on the order in which
// groups run.
__device__ __forceinline__ int cost_key(int c)
{
    return c <= 0 ? 0 : 32 - __clz(c); // 1 + floor(log2 c) <= 31 < kCostKeys
}

// Claims h[key] + (rank of this lane among the wave's active lanes with the
// same key) with one LDS atomic per distinct key in the wave (neighbouring
// groups mostly share a class, so that is one or two atomics, not 64). Every
// lane of the wave calls it; the loop runs once per distinct key.
__device__ __forceinline__ int wave_claim(int *h, int key, bool active)
{
    const int lane = threadIdx.x & 63;
    const unsigned long long below = (1ull << lane) - 1ull;
    unsigned long long rem = __ballot(active);
    int slot = 0;
    while (rem) {
        const int leader = __ffsll((long long)rem) - 1;
        const int k = __shfl(key, leader);
        const bool mine = active && key == k;
        const unsigned long long m = __ballot(mine);
        int base = 0;
        if (lane == leader) base = atomicAdd(&h[k], __popcll(m));
        base = __shfl(base, leader);
        if (mine) slot = base + __popcll(m & below);
        rem &= ~m;
    }
    return slot;
}

// Each pass reads the costs kOrderBatch per thread at a time, all loads in
// flight together (one block cannot hide a load's latency otherwise: the
// first version, one load per round trip, took 103 us at 4M bodies).
constexpr int kOrderBatch = 16;

__global__ __launch_bounds__(1024) void k_group_order(const int *__restrict__ cost, int ng, int *__restrict__ order)
{
    __shared__ int h[kCostKeys];
    const int tid = threadIdx.x;
    if (tid < kCostKeys) h[tid] = 0;
    __syncthreads();
    for (int base = 0; base < ng; base += 1024 * kOrderBatch) { // uniform bound: whole waves call wave_claim
        int key[kOrderBatch];
#pragma unroll
        for (int j = 0; j < kOrderBatch; ++j) {
            const int g = base + j * 1024 + tid;
            key[j] = g < ng ? cost_key(cost[g]) : -1;
        }
#pragma unroll
        for (int j = 0; j < kOrderBatch; ++j) (void)wave_claim(h, key[j], key[j] >= 0);
    }
    __syncthreads();
    if (tid == 0) {
        int acc = 0;
        for (int k = kCostKeys - 1; k >= 0; --k) {
            const int t = h[k];
            h[k] = acc;
            acc += t;
        }
    }
    __syncthreads();
    // the same costs as the histogram read (the engine runs this kernel after
    // the pass that wrote them and holds the next pass until it is done), so
    // every group lands in [0, ng) exactly once
    for (int base = 0; base < ng; base += 1024 * kOrderBatch) {
        int key[kOrderBatch];
#pragma unroll
        for (int j = 0; j < kOrderBatch; ++j) {
            const int g = base + j * 1024 + tid;
            key[j] = g < ng ? cost_key(cost[g]) : -1;
        }
#pragma unroll
        for (int j = 0; j < kOrderBatch; ++j) {
            const int slot = wave_claim(h, key[j], key[j] >= 0);
            if (key[j] >= 0) order[slot] = base + j * 1024 + tid;
        }
    }
}

hipError_t launch_group_order(const Dev &d, hipStream_t st)
{
    const int ng = (d.n + 63) / 64;
    if (ng <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_group_order, dim3(1), dim3(1024), 0, st, (const int *)d.gcost, ng, d.gorder);
    return hipGetLastError();
}

// Waves per group, by the number of groups (see waves_per_group in
// nb_force.hip; the waves part at 64 cells: a group opens a few hundred, and
// breadth first keeps every wave of a round busy, where rounds off the top of a
// stack took 10 to 40 % longer). us of the force stage, 1 / 4 / 8 / 16 waves,
// coarse and learned (theta_c 0.9, alpha 0.02):
//   16,384 bodies (256 groups), Plummer      300 / 118 / 93 / 86      309 / 128 / 85 / 77
//   40,960 (640), Plummer                    365 / 137 / 114 / 171    377 / 146 / 103 / 149
//   65,536 (1,024), halo and disk            384 / 153 / 147 / 245    392 / 153 / 133 / 207
//   100,003 (1,563), clusters                268 / 114 / 154 / 283    280 / 125 / 141 / 265
//   262,144 (4,096), halo and disk           516 / 295 / 453 / 887    543 / 317 / 383 / 719
//   524,288 (8,192), halo and disk           680 / 553 / 910 / 1859   720 / 614 / 764 / 1460
//   700,001 (10,938), halo and disk          697 / 706 / 1202 / -     730 / 786 / 1019 / -
static int coarse_waves_per_group(int groups)
{
    return groups <= 320 ? 16 : groups <= 1280 ? 8 : groups <= 9216 ? 4 : 1;
}

hipError_t launch_coarse(const Dev &d, const Learn &L, int out, const int *groups, int ngroups, float *xraw,
                         float4 *frame_out, int fmode, hipStream_t st)
{
    const int waves = groups ? ngroups : (d.n + 63) / 64;
    if (waves <= 0) return hipSuccess;
    const float4 *rec = nullptr;
    float4 *acc_out = nullptr;
#define NB_COARSE_ARGS                                                                             \
    d, L, (const int *)d.cchild, (const float4 *)d.cdata, (const float4 *)d.cqa, (const float4 *)d.cqb, \
        (const float2 *)d.cmac, groups, ngroups, rec, xraw, frame_out, acc_out, fmode
#define NB_COARSE_LAUNCH(OUT)                                                                                  \
    switch (coarse_waves_per_group(waves)) {                                                                   \
    case 16: hipLaunchKernelGGL((k_coarse64<OUT, 16>), dim3(waves), dim3(1024), 0, st, NB_COARSE_ARGS); break; \
    case 8: hipLaunchKernelGGL((k_coarse64<OUT, 8>), dim3(waves), dim3(512), 0, st, NB_COARSE_ARGS); break;    \
    case 4: hipLaunchKernelGGL((k_coarse64<OUT, 4>), dim3(waves), dim3(256), 0, st, NB_COARSE_ARGS); break;    \
    default: hipLaunchKernelGGL((k_coarse64<OUT, 1>), dim3(waves), dim3(64), 0, st, NB_COARSE_ARGS); break;    \
    }
    switch (out) {
    case kOutLearned: NB_COARSE_LAUNCH(kOutLearned); break;
    case kOutRaw: hipLaunchKernelGGL((k_coarse64<kOutRaw, 1>), dim3(waves), dim3(64), 0, st, NB_COARSE_ARGS); break;
    case kOutFinish: NB_COARSE_LAUNCH(kOutFinish); break;
    default: return hipErrorInvalidValue;
    }
#undef NB_COARSE_LAUNCH
    return hipGetLastError();
}

hipError_t launch_pair_records(const Dev &d, const int *groups, int ngroups, float4 *rec, hipStream_t st)
{
    if (ngroups <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_pair_records, dim3((ngroups * 64 + 255) / 256), dim3(256), 0, st, d, groups, ngroups * 64, rec);
    return hipGetLastError();
}

hipError_t launch_pairs(const Dev &d, const Learn &L, const int *groups, int ngroups, const float4 *rec,
                        float *xraw, float4 *frame_out, float4 *acc_out, hipStream_t st)
{
    if (ngroups <= 0) return hipSuccess;
    const int fmode = 0;
    hipLaunchKernelGGL(k_pairs, dim3(2 * ngroups), dim3(64), 0, st, NB_COARSE_ARGS);
#undef NB_COARSE_ARGS
    return hipGetLastError();
}

// Test path: raw features -> normalized BF16 rows in LDS -> network -> y.
__global__ __launch_bounds__(256) void k_mlp_rows(Mlp m, const float *__restrict__ x, int rows,
                                                  float *__restrict__ y)
{
    __shared__ __attribute__((aligned(16))) uint16_t fs[4][64 * kFeat];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int row = (blockIdx.x * 4 + wv) * 64 + lane;
#pragma unroll
    for (int i = 0; i < kFeat; ++i)
        fs[wv][lane * kFeat + i] = row < rows ? to_bf16(clipz((x[(size_t)row * kFeat + i] - m.xmu[i]) * m.xrs[i])) : 0;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    float y0, y1, y2;
    mlp_wave(fs[wv], m, lane, y0, y1, y2);
    if (row < rows) {
        y[(size_t)row * 3 + 0] = y0;
        y[(size_t)row * 3 + 1] = y1;
        y[(size_t)row * 3 + 2] = y2;
    }
}

hipError_t launch_mlp_rows(const Learn &L, const float *xraw, int rows, float *y, hipStream_t st)
{
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_mlp_rows, dim3((rows + 255) / 256), dim3(256), 0, st, L.mlp, xraw, rows, y);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Training pairs
// ---------------------------------------------------------------------------
__global__ void k_make_target(const float4 *__restrict__ frame, const float4 *__restrict__ afine, int rows,
                              float *__restrict__ t)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= rows) return;
    const float4 f0 = frame[2 * (size_t)i], f1 = frame[2 * (size_t)i + 1];
    const float4 af = afine[i];
    float t0 = 0.f, t1 = 0.f, t2 = 0.f;
    if (f0.w > 0.f) {
        const float inv = 1.0f / f0.w;
        const float e1x = f0.x * inv, e1y = f0.y * inv, e1z = f0.z * inv;
        const float e2x = f1.x * inv, e2y = f1.y * inv, e2z = f1.z * inv;
        const float e3x = e1y * e2z - e1z * e2y, e3y = e1z * e2x - e1x * e2z, e3z = e1x * e2y - e1y * e2x;
        const float rx = af.x - f0.x, ry = af.y - f0.y, rz = af.z - f0.z;
        t0 = (rx * e1x + ry * e1y + rz * e1z) * inv;
        t1 = (rx * e2x + ry * e2y + rz * e2z) * inv;
        t2 = (rx * e3x + ry * e3y + rz * e3z) * inv;
    }
    t[3 * (size_t)i + 0] = t0;
    t[3 * (size_t)i + 1] = t1;
    t[3 * (size_t)i + 2] = t2;
}

hipError_t launch_make_target(const float4 *frame, const float4 *afine, int rows, float *t, hipStream_t st)
{
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_make_target, dim3((rows + 255) / 256), dim3(256), 0, st, frame, afine, rows, t);
    return hipGetLastError();
}

// One block per column; FP64 sums in a fixed order. Bound by the latency of the
// strided loads: a thread has kStatLoads in flight and adds them in order
// (163,840 rows of 24 columns: 186 -> 125 us).
constexpr int kStatLoads = 16;

__global__ __launch_bounds__(256) void k_colstats(const float *__restrict__ x, int rows, int cols,
                                                  float *__restrict__ mu, float *__restrict__ sd)
{
    __shared__ double s1[256], s2[256];
    const int c = blockIdx.x;
    double a = 0.0, b = 0.0;
    int r = threadIdx.x;
    for (; r + (kStatLoads - 1) * 256 < rows; r += kStatLoads * 256) {
        float q[kStatLoads];
#pragma unroll
        for (int u = 0; u < kStatLoads; ++u) q[u] = x[((size_t)r + u * 256) * cols + c];
#pragma unroll
        for (int u = 0; u < kStatLoads; ++u) {
            const double v = (double)q[u];
            a += v;
            b += v * v;
        }
    }
    for (; r < rows; r += 256) {
        const double v = (double)x[(size_t)r * cols + c];
        a += v;
        b += v * v;
    }
    s1[threadIdx.x] = a;
    s2[threadIdx.x] = b;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) {
            s1[threadIdx.x] += s1[threadIdx.x + o];
            s2[threadIdx.x] += s2[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double m = s1[0] / rows;
        const double var = fmax(s2[0] / rows - m * m, 0.0);
        const double s = sqrt(var);
        mu[c] = (float)m;
        sd[c] = s > 1e-12 ? (float)s : 1.0f;
    }
}

__global__ void k_apply_standardize(float *__restrict__ x, int rows, int cols, const float *__restrict__ mu,
                                    const float *__restrict__ sd)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)rows * cols) return;
    const int c = (int)(i % cols);
    x[i] = clipz((x[i] - mu[c]) / sd[c]);
}

hipError_t launch_standardize(float *x, int rows, int cols, float *mu, float *sd, hipStream_t st)
{
    if (rows <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_colstats, dim3(cols), dim3(256), 0, st, x, rows, cols, mu, sd);
    const size_t total = (size_t)rows * cols;
    hipLaunchKernelGGL(k_apply_standardize, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, x, rows,
                       cols, (const float *)mu, (const float *)sd);
    return hipGetLastError();
}

__global__ void k_gather_acc(const float4 *__restrict__ acc, const int *__restrict__ idx, int ns,
                             float4 *__restrict__ out)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < ns) out[i] = acc[idx[i]];
}

hipError_t launch_gather_acc(const Dev &d, const int *idx, int ns, float4 *out, hipStream_t st)
{
    if (ns <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_gather_acc, dim3((ns + 255) / 256), dim3(256), 0, st, (const float4 *)d.acc4, idx, ns,
                       out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// FP32 training: forward, backward, Adam
// ---------------------------------------------------------------------------
__device__ __forceinline__ int batch_row(uint64_t seed, int it, int r, int S)
{
    if (seed == 0) return r; // the whole dataset in order
    uint64_t z = seed + 0x9e3779b97f4a7c15ull * (((uint64_t)it << 32) + (uint64_t)r + 1ull);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    z ^= z >> 31;
    return (int)(z % (uint64_t)S);
}

// ---------------------------------------------------------------------------
// One training iteration: forward, backward and weight gradients of the batch
// in one kernel, the gradient's sum over the blocks and the Adam step in a
// second.
//
// The products run on the FP32 matrix instruction v_mfma_f32_16x16x4_f32 (FP32
// operands, products and sums). Operand layout, lane l with m = l % 16 and
// g = l / 16: A row m, k = g; B column m, k = g; D column m, rows 4 g .. 4 g + 3.
// The order of k is free as long as A and B agree, so a group of 16 k's is
// taken as k = 4 g + s in step s = 0 .. 3.
//
// The network runs in the transposed form Z^T = W^T X^T, the rows of the batch
// being the columns: a lane's D registers are four hidden units of one row. A
// block has 32 rows at a time, two waves for each 16, each of them with half of
// every layer's units; a layer's activations go to LDS as [unit][row], where the
// two waves take all of them as the next layer's B operands, forward and
// backward. The weights come straight from the parameters (they sit in the
// caches: every wave reads the same 24 KB). The weight gradients contract over
// the rows, which are spread over the lanes: they read the same LDS rows, of
// kTrainLd floats (a 16-byte read holds four steps of an operand), each of the
// block's four waves a quarter of the gradient's tiles. A block loops over tiles
// of 32 rows and keeps its gradient in accumulators; there are at most
// kGradBlocks blocks, so the partial gradients stay within 6 MB. All sums have a
// fixed order.
//
// Bound: the matrix unit of the CUs that have a block (a batch of 4,096 rows is
// 128 blocks; about 150 matrix instructions of 32 cycles per wave) and the
// latency of the layers. An iteration of 4,096 rows takes 11.8 + 4.7 us; with 64
// rows per block, a wave having 16 of them with all units in its registers, 17.6
// + 4.8 us (half as many CUs with twice the chain); as twelve launches that
// passed every layer's activations through memory and re-read the batch for
// each row of weights it took 130 us.
// ---------------------------------------------------------------------------
constexpr int kTrainRows = kTrainTile;     // rows per tile: two waves for each 16
constexpr int kTrainLd = kTrainRows + 4;   // LDS row length
static_assert(kFeat == 24 && kHid == 64 && kOut == 3 && kTrainRows == 32, "the tiling below");

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// gelu and its derivative from one tanh
__device__ __forceinline__ float gelu_both(float x, float &grad)
{
    const float x2 = x * x;
    const float t = tanh_fast(kGeluC * (x + kGeluA * x2 * x));
    grad = 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * kGeluC * (1.0f + 3.0f * kGeluA * x2);
    return 0.5f * x * (1.0f + t);
}

__global__ __launch_bounds__(256) void k_train_grad(const float *__restrict__ P, const float *__restrict__ X,
                                                    const float *__restrict__ T, uint64_t seed, int it, int S, int B,
                                                    float *__restrict__ gpart, float *__restrict__ loss_part)
{
    __shared__ __attribute__((aligned(16))) float xs[kFeat][kTrainLd], h1s[kHid][kTrainLd], d1s[kHid][kTrainLd];
    __shared__ __attribute__((aligned(16))) float h2s[kHid][kTrainLd], d2s[kHid][kTrainLd], dys[kOut][kTrainLd];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int m = lane & 15, g = lane >> 4;
    const float *W1 = P, *b1 = P + kOffB1, *W2 = P + kOffW2, *b2 = P + kOffB2, *W3 = P + kOffW3, *b3 = P + kOffB3;
    const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
    // this wave's gradient tiles: dW2 rows 16 w .., all columns; dW1 all rows
    // (two tiles of 16, the second half empty), columns 16 w ..; dW3 rows 16 w ..;
    // the biases' columns 16 w .. (b3: wave 0)
    f32x4 gw2[4] = {z4, z4, z4, z4}, gw1[2] = {z4, z4}, gw3 = z4;
    float gb1 = 0.f, gb2 = 0.f, gb3 = 0.f, loss = 0.f;
    const float sc = 2.0f / (3.0f * (float)B);
    const int ntiles = (B + kTrainRows - 1) / kTrainRows;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int rl = 16 * (w & 1) + m, r = tile * kTrainRows + rl; // this lane's row (column of the products)
        const int t0 = w & 2; // this wave's tiles of units: t0, t0 + 1
        const bool in = r < B;
        const size_t row = in ? (size_t)batch_row(seed, it, r, S) : 0;
        f32x4 x0 = z4, x1 = z4; // features 4 g .., and 16 + 4 g .. (g < 2)
        if (in) {
            x0 = *reinterpret_cast<const f32x4 *>(X + row * kFeat + 4 * g);
            if (g < 2) x1 = *reinterpret_cast<const f32x4 *>(X + row * kFeat + 16 + 4 * g);
        }
        float y0 = 0.f, y1 = 0.f, y2 = 0.f;
        if (in && g == 0) {
            y0 = T[row * kOut];
            y1 = T[row * kOut + 1];
            y2 = T[row * kOut + 2];
        }
        // this wave's units 16 (t0 + i) + 4 g + v into a layer's LDS rows, and all
        // four tiles of the layer out of them
        auto put = [&](float (*u)[kTrainLd], const f32x4 (&h)[2]) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int v = 0; v < 4; ++v) u[16 * (t0 + i) + 4 * g + v][rl] = h[i][v];
            __syncthreads();
        };
        auto all = [&](float (*u)[kTrainLd], f32x4 (&h)[4]) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) h[t][v] = u[16 * t + 4 * g + v][rl];
        };
        f32x4 h[2], p1[2], p2[2], in4[4]; // activations, their derivatives; a layer's input
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int t = t0 + i;
            f32x4 z = *reinterpret_cast<const f32x4 *>(b1 + 16 * t + 4 * g);
#pragma unroll
            for (int q = 0; q < 4; ++q) z = mfma4(W1[(4 * g + q) * kHid + 16 * t + m], x0[q], z);
#pragma unroll
            for (int q = 0; q < 4; ++q) z = mfma4(g < 2 ? W1[(16 + 4 * g + q) * kHid + 16 * t + m] : 0.f, x1[q], z);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float d;
                h[i][v] = gelu_both(z[v], d);
                p1[i][v] = d;
            }
        }
        __syncthreads(); // the last tile's gradients have been read
        if (w < 2) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                xs[4 * g + v][rl] = x0[v];
                if (g < 2) xs[16 + 4 * g + v][rl] = x1[v];
            }
        }
        put(h1s, h);
        all(h1s, in4);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int t = t0 + i;
            f32x4 z = *reinterpret_cast<const f32x4 *>(b2 + 16 * t + 4 * g);
#pragma unroll
            for (int rb = 0; rb < 4; ++rb)
#pragma unroll
                for (int q = 0; q < 4; ++q) z = mfma4(W2[(16 * rb + 4 * g + q) * kHid + 16 * t + m], in4[rb][q], z);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float d;
                h[i][v] = gelu_both(z[v], d);
                p2[i][v] = d;
            }
        }
        put(h2s, h);
        all(h2s, in4);
        // outputs 0 .. 2 of row r in lane m (g = 0); both waves of the rows work
        // them out
        f32x4 y = z4;
        if (g == 0) y = f32x4{b3[0], b3[1], b3[2], 0.f};
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
            for (int q = 0; q < 4; ++q) y = mfma4(m < kOut ? W3[(16 * rb + 4 * g + q) * kOut + m] : 0.f, in4[rb][q], y);
        float e0 = 0.f, e1 = 0.f, e2 = 0.f;
        if (in && g == 0) {
            e0 = y[0] - y0;
            e1 = y[1] - y1;
            e2 = y[2] - y2;
            if (w < 2) loss += e0 * e0 + e1 * e1 + e2 * e2;
        }
        e0 *= sc;
        e1 *= sc;
        e2 *= sc;
        // output g's gradient of row r in lane (m, g)
        const float s0 = __shfl(e0, m), s1 = __shfl(e1, m), s2 = __shfl(e2, m);
        const float dy = g == 0 ? s0 : g == 1 ? s1 : g == 2 ? s2 : 0.f;
        if (w < 2 && g < kOut) dys[g][rl] = dy;
#pragma unroll
        for (int i = 0; i < 2; ++i) h[i] = mfma4(g < kOut ? W3[(16 * (t0 + i) + m) * kOut + g] : 0.f, dy, z4) * p2[i];
        put(d2s, h);
        all(d2s, in4);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            f32x4 z = z4;
#pragma unroll
            for (int rb = 0; rb < 4; ++rb) {
                const f32x4 a = *reinterpret_cast<const f32x4 *>(W2 + (16 * (t0 + i) + m) * kHid + 16 * rb + 4 * g);
#pragma unroll
                for (int q = 0; q < 4; ++q) z = mfma4(a[q], in4[rb][q], z);
            }
            h[i] = z * p1[i];
        }
        put(d1s, h);
#pragma unroll
        for (int c = 0; c < kTrainRows / 16; ++c) {
            const int k0 = 16 * c + 4 * g; // this lane's rows of the chunk
            auto frag = [&](float (*u)[kTrainLd], int unit) { return *reinterpret_cast<const f32x4 *>(&u[unit][k0]); };
            const f32x4 a2 = frag(h1s, 16 * w + m), a3 = frag(h2s, 16 * w + m);
            const f32x4 a1 = frag(xs, m), a1b = m < 8 ? frag(xs, 16 + (m & 7)) : z4;
            const f32x4 c1 = frag(d1s, 16 * w + m), c3 = m < kOut ? frag(dys, m < kOut ? m : 0) : z4;
            gb1 += (c1[0] + c1[1]) + (c1[2] + c1[3]);
            gb3 += (c3[0] + c3[1]) + (c3[2] + c3[3]);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const f32x4 c2 = frag(d2s, 16 * t + m);
                if (t == w) gb2 += (c2[0] + c2[1]) + (c2[2] + c2[3]);
#pragma unroll
                for (int q = 0; q < 4; ++q) gw2[t] = mfma4(a2[q], c2[q], gw2[t]);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                gw1[0] = mfma4(a1[q], c1[q], gw1[0]);
                gw1[1] = mfma4(a1b[q], c1[q], gw1[1]);
                gw3 = mfma4(a3[q], c3[q], gw3);
            }
        }
    }
    float *o = gpart + (size_t)blockIdx.x * kMlpParams;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int i = 4 * g + v;
#pragma unroll
        for (int t = 0; t < 4; ++t) o[kOffW2 + (16 * w + i) * kHid + 16 * t + m] = gw2[t][v];
        o[i * kHid + 16 * w + m] = gw1[0][v];
        if (i < 8) o[(16 + i) * kHid + 16 * w + m] = gw1[1][v];
        if (m < kOut) o[kOffW3 + (16 * w + i) * kOut + m] = gw3[v];
    }
    // the biases: the four lanes of a column hold a quarter of the rows each
    auto over_g = [](float v) {
        v += __shfl_xor(v, 16);
        return v + __shfl_xor(v, 32);
    };
    gb1 = over_g(gb1);
    gb2 = over_g(gb2);
    gb3 = over_g(gb3);
    if (g == 0) {
        o[kOffB1 + 16 * w + m] = gb1;
        o[kOffB2 + 16 * w + m] = gb2;
        if (w == 0 && m < kOut) o[kOffB3 + m] = gb3;
    }
#pragma unroll
    for (int k = 1; k < 16; k <<= 1) loss += __shfl_xor(loss, k);
    __syncthreads();
    if (lane == 0) xs[0][w] = loss;
    __syncthreads();
    if (threadIdx.x == 0) loss_part[blockIdx.x] = (xs[0][0] + xs[0][1]) + (xs[0][2] + xs[0][3]);
}

// The gradient: the blocks' partial gradients added in order (four threads per
// parameter, a quarter of the blocks each), then the Adam step. Block 0 also
// adds the loss.
__global__ __launch_bounds__(256) void k_train_adam(float *__restrict__ P, float *__restrict__ G,
                                                    float *__restrict__ M, float *__restrict__ V,
                                                    const float *__restrict__ gpart, int nparts, float lr, float b1,
                                                    float b2, float eps, float c1, float c2,
                                                    const float *__restrict__ loss_part, int B,
                                                    float *__restrict__ loss_out, bool step)
{
    __shared__ float red[4][64];
    const int j = threadIdx.x & 63, q = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + j;
    float v = 0.f;
    if (i < kMlpParams) {
        const int k0 = nparts * q / 4, k1 = nparts * (q + 1) / 4;
#pragma unroll 8
        for (int k = k0; k < k1; ++k) v += gpart[(size_t)k * kMlpParams + i];
    }
    red[q][j] = v;
    if (blockIdx.x == 0 && q == 3) {
        // lane j the parts j, j + 64, ..., then the lanes in order of a tree
        float s = 0.f;
        for (int k = j; k < nparts; k += 64) s += loss_part[k];
#pragma unroll
        for (int k = 1; k < 64; k <<= 1) s += __shfl_xor(s, k);
        if (j == 0) *loss_out = s / (3.0f * (float)B);
    }
    __syncthreads();
    if (q != 0 || i >= kMlpParams) return;
    const float grad = (red[0][j] + red[1][j]) + (red[2][j] + red[3][j]);
    G[i] = grad;
    if (!step) return;
    const float mm = b1 * M[i] + (1.0f - b1) * grad;
    const float vv = b2 * V[i] + (1.0f - b2) * grad * grad;
    M[i] = mm;
    V[i] = vv;
    P[i] -= lr * (mm * c1) / (sqrtf(vv * c2) + eps);
}

hipError_t launch_train_iter(const Train &t, int B, int it, uint64_t seed, bool adam, float lr, float beta1,
                             float beta2, float eps, float c1, float c2, hipStream_t st)
{
    if (B <= 0) return hipErrorInvalidValue;
    const int nparts = train_parts(B);
    hipLaunchKernelGGL(k_train_grad, dim3(nparts), dim3(256), 0, st, (const float *)t.P, t.X, t.T, seed, it, t.S, B,
                       t.gpart, t.loss_part);
    hipLaunchKernelGGL(k_train_adam, dim3((kMlpParams + 63) / 64), dim3(256), 0, st, t.P, t.G, t.M, t.V,
                       (const float *)t.gpart, nparts, lr, beta1, beta2, eps, c1, c2, (const float *)t.loss_part, B,
                       t.loss_hist + it, adam);
    return hipGetLastError();
}

} // namespace nb
