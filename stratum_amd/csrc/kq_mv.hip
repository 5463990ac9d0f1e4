// kq_mv.hip -- exact MULTISEQ (gfx950): M streams through one pass over N rows.
//
// y_j[r] = row r . x_j, every stream bit-identical to the single-stream
// kernel (kq_segs_kernel): the same binary32 products and sequential sums
// per sub-block, the same binary64 terms, phases and tree.
//
// What bounds it is VALU issue: a rounded product and a rounded sum per
// weight and stream.  Measured per wave64 instruction and SIMD:
//   v_mul_f32, v_add_f32, v_and_b32 (32-bit encodings)       2.3 clk, two
//     waves issuing together (4.7 when a SIMD holds one wave)
//   v_mul_f32 with a byte select (the single-stream products) 5.2 clk
//   v_cvt_f32_ubyte, bit field, permute, DPP and binary64      4.3 clk
//   v_mfma_f32_4x4x1 (products on the matrix cores)            8.3 clk for
//     four multiplies' work, and no VALU issue overlaps it
//   ds_read_b128, conflict-free                     4 clk of the CU's LDS
// So each weight is converted once (4.3) for S = 2, 3 or 4 streams whose
// products are plain multiplies, 4.7 + 4.3 / S clk per weight and stream,
// against 7.5 for the byte-select form.  x needs no scaling window here: a
// quant is converted, not read as a denormal.
// The x tiles go from L2 to LDS without registers (global_load_lds), which
// with S = 4 leaves 128 VGPRs, four waves per SIMD.  The S = 4 forms of Q6_K
// and Q5_K do not quite fit them: 5 to 8 VGPRs spill, 24 to 36 bytes a lane
// (with S = 3 nothing does, and 5120 x 17408 B = 64 takes 620 us instead of
// 485).
//
// Measured against the multi-x kernel (kq_mx_kernel, byte-select products, x
// staged through registers), weights past the cache, us at B = 2 / 4 / 8 / 16
// / 64:
//   17408 x 5120  Q4_K 32 / 41 / 80 / 151 / 572 -> 28 / 35 / 51 / 94 / 337
//                 Q6_K 64 / 69 / 91 / 171 / 651 -> 39 / 50 / 70 / 113 / 418
//                 Q5_K 32 / 47 / 88 / 171 / 664 -> 30 / 45 / 61 / 115 / 409
//                 Q3_K 41 / 51 / 98 / 190 / 745 -> 34 / 45 / 65 / 110 / 380
//                 Q8_0 33 / 40 / 77 / 145 / 553 -> 30 / 38 / 57 / 97 / 354
//                 Q2_K 26.7 / 40 / 70 / 133 / 509 -> 27.2 / 36 / 52 / 95 / 341
//                 type 42 31 / 40 / 75 / 141 / 535 -> 28 / 37 / 53 / 97 / 347
//   5120 x 17408  Q4_K 30 / 59 / 108 / 205 / 788 -> 26 / 43 / 70 / 135 / 460
//                 Q6_K 57 / 70 / 132 / 256 / 997 -> 38 / 52 / 73 / 141 / 485
//                 Q2_K 31 / 46 / 85 / 163 / 634 -> 25 / 41 / 60 / 116 / 477
// Over 16 shapes, 13 B and the seven types 1.4 to 1.9 times (geometric means by
// type); slower in two of the 1456: Q8_0 17408 x 5120 B = 5 (46.8 -> 49.2) and
// Q2_K 17408 x 5120 B = 2.  At B = 8 on the gate the SIMDs issue 32 K VALU
// instructions each, about all of the kernel's clocks.
// The same kernel with its products on the matrix cores (K = 1 MFMAs, C = 0,
// which round like the multiply) took 59 and 104 us at B = 8 and 16.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kq_blocks.h"
#include "kq_launch.h"

#pragma clang fp contract(off)

namespace {

// ------------------------------------------------ chunk terms of S streams
// x of a unit's streams: the LDS byte address a of the lane's chunk for the
// first stream (float4 slot i at a ^ 16 i: slots are exchanged within a chunk
// by its number), the next streams xm bytes on each.
struct MvX {
    uint32_t a;
    int xm;
    __device__ __forceinline__ f32x4 get(int i, int s) const {
        return *reinterpret_cast<const f32x4 __attribute__((address_space(3)))*>(
            (a ^ (uint32_t)(16 * i)) + (uint32_t)(s * xm));
    }
};

// the four quants at mask m of v's bytes (in place: m = 0xf0 gives 16 q)
__device__ __forceinline__ void mv_quants(uint32_t v, uint32_t m, float (&q)[4]) {
    ubytes(v & (m * 0x01010101u), q[0], q[1], q[2], q[3]);
}

// a[s] += q . x of slot i of stream s, in order
template <int S>
__device__ __forceinline__ void mv_dot4(const float (&q)[4], const MvX& xc, int i, float (&a)[S]) {
    f32x4 x[S];
#pragma unroll
    for (int s = 0; s < S; s++) x[s] = xc.get(i, s);
#pragma unroll
    for (int s = 0; s < S; s++) a[s] = a[s] + q[0] * x[s].x;
#pragma unroll
    for (int s = 0; s < S; s++) a[s] = a[s] + q[1] * x[s].y;
#pragma unroll
    for (int s = 0; s < S; s++) a[s] = a[s] + q[2] * x[s].z;
#pragma unroll
    for (int s = 0; s < S; s++) a[s] = a[s] + q[3] * x[s].w;
    // bounds the live ranges: the compiler would hoist every read and product
#pragma unroll
    for (int s = 0; s < S; s++) asm volatile("" : "+v"(a[s]));
    __builtin_amdgcn_sched_barrier(0);
}

// run(): part[s] += the chunk term of stream s (x sums at xs[s], chunk c),
// in the operation order of term_q4k and its peers (kq_kernels.hip).
template <int TYPE, int S> struct MvTerms;

template <int S> struct MvTerms<T_Q4K, S> {
    static __device__ __forceinline__ void run(const RawQ4& r, int j, const MvX& xc,
                                               const float* const (&xs)[S], int c,
                                               double (&part)[S]) {
        float a1[S], a2[S];
#pragma unroll
        for (int s = 0; s < S; s++) a1[s] = a2[s] = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t v = k < 4 ? dw_of(r.qa, k) : dw_of(r.qb, k - 4);
            float q[4];
            mv_quants(v, 0x0fu, q);
            mv_dot4<S>(q, xc, k, a1);
            mv_quants(v, 0xf0u, q);             // 16 q: d2 is used divided by 16
            mv_dot4<S>(q, xc, 8 + k, a2);
        }
        const float d = f16_bits_to_f32(r.hd.x & 0xffffu);
        const float dmin = f16_bits_to_f32(r.hd.x >> 16);
        uint32_t sc1, n1, sc2, n2;
        scale_min_pair(r.hd.y, r.hd.z, r.hd.w, j, sc1, n1, sc2, n2);
        const float d1 = d * (float)sc1, d2 = (d * (float)sc2) * 0.0625f;
        const float m1 = dmin * (float)n1, m2 = dmin * (float)n2;
#pragma unroll
        for (int s = 0; s < S; s++) {
            const float2 sx = reinterpret_cast<const float2*>(xs[s])[c];
            const float t1 = d1 * a1[s] - m1 * sx.x;
            const float t2 = d2 * a2[s] - m2 * sx.y;
            part[s] = part[s] + ((double)t1 + (double)t2);
        }
    }
};

template <int S> struct MvTerms<T_Q5K, S> {
    static __device__ __forceinline__ void run(const RawQ5& r, int j, const MvX& xc,
                                               const float* const (&xs)[S], int c,
                                               double (&part)[S]) {
        float a1[S], a2[S];
#pragma unroll
        for (int s = 0; s < S; s++) a1[s] = a2[s] = 0.0f;
        const uint32_t b1 = 2u * (uint32_t)j;
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t v = k < 4 ? dw_of(r.qa, k) : dw_of(r.qb, k - 4);
            const uint32_t h = (k < 4 ? dw_of(r.h0, k) : dw_of(r.h1, k - 4)) >> b1;
            const uint32_t vl = (v & 0x0f0f0f0fu) | ((h << 4) & 0x10101010u);
            const uint32_t vh = ((v >> 4) & 0x0f0f0f0fu) | ((h << 3) & 0x10101010u);
            float q[4];
            mv_quants(vl, 0x1fu, q);
            mv_dot4<S>(q, xc, k, a1);
            mv_quants(vh, 0x1fu, q);
            mv_dot4<S>(q, xc, 8 + k, a2);
        }
        const float d = f16_bits_to_f32(r.hd.x & 0xffffu);
        const float dmin = f16_bits_to_f32(r.hd.x >> 16);
        uint32_t sc1, n1, sc2, n2;
        scale_min_pair(r.hd.y, r.hd.z, r.hd.w, j, sc1, n1, sc2, n2);
        const float d1 = d * (float)sc1, d2 = d * (float)sc2;
        const float m1 = dmin * (float)n1, m2 = dmin * (float)n2;
#pragma unroll
        for (int s = 0; s < S; s++) {
            const float2 sx = reinterpret_cast<const float2*>(xs[s])[c];
            const float t = ((d1 * a1[s] - m1 * sx.x) + d2 * a2[s]) - m2 * sx.y;
            part[s] = part[s] + (double)t;
        }
    }
};

template <int S> struct MvTerms<T_Q2K, S> {
    static __device__ __forceinline__ void run(const RawQ2& r, int u, const MvX& xc,
                                               const float* const (&xs)[S], int c,
                                               double (&part)[S]) {
        const float d = f16_bits_to_f32(r.dd & 0xffffu);
        const float dmin = f16_bits_to_f32(r.dd >> 16);
        const uint32_t S0 = r.s.x >> (8 * (u & 1)), S1 = r.s.y >> (8 * (u & 1));
        double acc[S];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float a[S];
#pragma unroll
            for (int s = 0; s < S; s++) a[s] = 0.0f;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t v = dw_of(r.q, k);
                float q[4];
                mv_quants(v, 0x03u << (2 * j), q);   // 4^j q
                mv_dot4<S>(q, xc, 4 * j + k, a);
            }
            const uint32_t sc = ((j < 2 ? S0 : S1) >> (16 * (j & 1))) & 0xffu;
            const float inv = j == 0 ? 1.0f : j == 1 ? 0.25f : j == 2 ? 0.0625f : 0.015625f;
            const float dl = (d * (float)(sc & 15u)) * inv, ml = dmin * (float)(sc >> 4);
#pragma unroll
            for (int s = 0; s < S; s++) {
                const float t = dl * a[s] - ml * xs[s][4 * c + j];
                acc[s] = (j ? acc[s] : 0.0) + (double)t;
            }
        }
#pragma unroll
        for (int s = 0; s < S; s++) part[s] = part[s] + acc[s];
    }
};

template <int S> struct MvTerms<T_NIB, S> {
    static __device__ __forceinline__ void run(const RawNB& r, int, const MvX& xc,
                                               const float* const (&xs)[S], int c,
                                               double (&part)[S]) {
        const float d = f16_bits_to_f32(r.dd & 0xffffu);
        const float dmin = f16_bits_to_f32(r.dd >> 16);
        double acc[S];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float a[S];
#pragma unroll
            for (int s = 0; s < S; s++) a[s] = 0.0f;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t v = dw_of(j < 2 ? r.qa : r.qb, k);
                float q[4];
                mv_quants(v, j & 1 ? 0xf0u : 0x0fu, q);
                mv_dot4<S>(q, xc, 4 * j + k, a);
            }
            const uint32_t sc = (r.s >> (8 * j)) & 0xffu;
            const float dl = (d * (float)(sc & 15u)) * (j & 1 ? 0.0625f : 1.0f);
            const float ml = dmin * (float)(sc >> 4);
#pragma unroll
            for (int s = 0; s < S; s++) {
                const float t = dl * a[s] - ml * xs[s][4 * c + j];
                acc[s] = (j ? acc[s] : 0.0) + (double)t;
            }
        }
#pragma unroll
        for (int s = 0; s < S; s++) part[s] = part[s] + acc[s];
    }
};

// Signed quants are converted (a signed byte has no such denormal): Q6_K's
// four runs step by step, their conversions shared by the streams.
template <int S> struct MvTerms<T_Q6K, S> {
    static __device__ __forceinline__ void run(const RawQ6& r, int u, const MvX& xc,
                                               const float* const (&)[S], int,
                                               double (&part)[S]) {
        float a[4][S];
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int s = 0; s < S; s++) a[t][s] = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            uint32_t y[4];
            q6k_words(r, k, y);
#pragma unroll
            for (int t = 0; t < 4; t++) {
                const float q[4] = {i8f(y[t], 0), i8f(y[t], 1), i8f(y[t], 2), i8f(y[t], 3)};
                mv_dot4<S>(q, xc, 4 * t + k, a[t]);
            }
        }
#pragma unroll
        for (int s = 0; s < S; s++) {
            const float as[4] = {a[0][s], a[1][s], a[2][s], a[3][s]};
            part[s] = part[s] + q6k_combine(r, u, as, 0.25);
        }
    }
};

template <int S> struct MvTerms<T_Q3K, S> {
    static __device__ __forceinline__ void run(const RawQ3& r, int u, const MvX& xc,
                                               const float* const (&)[S], int,
                                               double (&part)[S]) {
        const int sh2 = u >> 1, h = u & 1;
        const uint32_t sh = r.sh;
        const float d = f16_bits_to_f32(r.d);
        const uint32_t S0 = __builtin_amdgcn_alignbit(r.s[1], r.s[0], sh);
        const uint32_t S1 = __builtin_amdgcn_alignbit(r.s[2], r.s[1], sh);
        const uint32_t S2 = __builtin_amdgcn_alignbit(r.s[3], r.s[2], sh);
        uint32_t Q[4], M[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            Q[k] = __builtin_amdgcn_alignbit(r.q[k + 1], r.q[k], sh);
            M[k] = ~(__builtin_amdgcn_alignbit(r.m[k + 1], r.m[k], sh) >> (4 * sh2));
        }
        double acc[S];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float a[S];
#pragma unroll
            for (int s = 0; s < S; s++) a[s] = 0.0f;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t lo2 = (Q[k] >> (2 * j)) & 0x03030303u;
                const uint32_t neg = ((M[k] >> j) & 0x01010101u) << 2;
                const uint32_t y = (lo2 | neg) << 5;          // int8 32 * q3 per byte
                const float q[4] = {i8f(y, 0), i8f(y, 1), i8f(y, 2), i8f(y, 3)};
                mv_dot4<S>(q, xc, 4 * j + k, a);
            }
            // 6-bit scale of group 8s + 2j + h, as in term_q3k
            const uint32_t bi = 8u * (uint32_t)(2 * (j & 1) + h);
            const uint32_t w = (uint32_t)(2 * sh2 + (j >> 1));
            const uint32_t nib = bfe((w & 1u) ? S1 : S0, bi + ((w & 2u) ? 4u : 0u), 4);
            const uint32_t hi2 = bfe(S2, bi + 2u * w, 2);
            const float dl = (d * (float)((int)(nib | (hi2 << 4)) - 32)) * 0.03125f;
#pragma unroll
            for (int s = 0; s < S; s++) acc[s] = (j ? acc[s] : 0.0) + (double)(dl * a[s]);
        }
#pragma unroll
        for (int s = 0; s < S; s++) part[s] = part[s] + acc[s];
    }
};

template <int S> struct MvTerms<T_Q80, S> {
    static __device__ __forceinline__ void run(const RawQ8& r, int, const MvX& xc,
                                               const float* const (&)[S], int,
                                               double (&part)[S]) {
        double acc[S];
#pragma unroll
        for (int half = 0; half < 2; half++) {
            const float d = f16_bits_to_f32(half ? (r.w[8] >> 16) : (r.w[0] & 0xffffu));
            float a[S];
#pragma unroll
            for (int s = 0; s < S; s++) a[s] = 0.0f;
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const uint32_t v =
                    half ? r.w[9 + k] : __builtin_amdgcn_alignbit(r.w[k + 1], r.w[k], 16);
                const float q[4] = {i8f(v, 0), i8f(v, 1), i8f(v, 2), i8f(v, 3)};
                mv_dot4<S>(q, xc, 8 * half + k, a);
            }
#pragma unroll
            for (int s = 0; s < S; s++) acc[s] = (half ? acc[s] : 0.0) + (double)(d * a[s]);
        }
#pragma unroll
        for (int s = 0; s < S; s++) part[s] = part[s] + acc[s];
    }
};


// a unit's width as a type
template <int V> struct MvInt { static constexpr int v = V; };

template <int TYPE> struct MvRaw;
#define KQ_MV_RAW(T_, R_, F_)                                                                \
    template <> struct MvRaw<T_> {                                                           \
        using Raw = R_;                                                                      \
        static __device__ __forceinline__ Raw load(wptr blk, int u) { return F_(blk, u); }   \
    };
KQ_MV_RAW(T_Q4K, RawQ4, load_q4k)
KQ_MV_RAW(T_Q6K, RawQ6, load_q6k)
KQ_MV_RAW(T_Q2K, RawQ2, load_q2k)
KQ_MV_RAW(T_NIB, RawNB, load_nib)
KQ_MV_RAW(T_Q5K, RawQ5, load_q5k)
KQ_MV_RAW(T_Q3K, RawQ3, load_q3k)
KQ_MV_RAW(T_Q80, RawQ8, load_q80)
#undef KQ_MV_RAW

// ------------------------------------------------------------- the kernel
constexpr int MV_ME = 8;          // streams staged together
constexpr int MV_TW = 2;          // tasks per wave, at most
constexpr long MV_LANES = 1L << 32;   // of a launch (HIP refuses this many)

struct MvArg {
    const uint8_t* w;
    const float* X;
    float* Y;
    long x_stride, y_stride;      // floats
    int M, N, K;
    int ng, nblk;                 // row groups per item, items per stream chunk
    int nmc, mc;                  // stream chunks, streams per chunk (<= MV_ME)
    int nitems;
};

// x position (floats, within four chunks = one super-block) of float4 slot
// t of chunk c
template <bool LINEAR>
__device__ __forceinline__ int mv_pos(int c, int t) {
    if (LINEAR) return 64 * c + 4 * t;
    return 128 * (c >> 1) + 16 * (c & 1) + 32 * (t >> 2) + 4 * (t & 3);
}

// Pieces that a task of S streams is cut into when `rem` tasks are left for W
// waves
__host__ __device__ __forceinline__ int mv_cut(int S, int rem, int W) {
    return S * rem <= W ? S : S == 4 && 2 * rem <= W ? 2 : 1;
}

// Where a task of streams m0 .. m0 + n - 1 starts: one that would read past the
// last x slot (S = 3: streams 6, 7 and 8 of 8) takes the last n slots, and does
// not store the streams before m0.
__host__ __device__ __forceinline__ int mv_x0(int m0, int n) {
    return m0 < MV_ME - n ? m0 : MV_ME - n;
}

// A copy the optimiser takes for new values: the variants of a unit would
// otherwise have their common decode hoisted above the branch, all at once.
template <typename R> __device__ __forceinline__ R mv_opaque(const R& r) {
    struct Words { uint32_t w[sizeof(R) / 4]; };
    Words v = __builtin_bit_cast(Words, r);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(R) / 4); i++) asm volatile("" : "+v"(v.w[i]));
    return __builtin_bit_cast(R, v);
}

// H = 1: rows of at most 128 chunks, 8 phases; H = 2: longer rows, 32.
template <int H> struct MvShape {
    static constexpr int T = 512 * H, W = T / 64;
    static constexpr int GP = H == 1 ? 8 : 32, RPT = 64 / GP;      // phases, rows of a task
    static constexpr int TCH = 16 * H;                            // chunks per x tile
    static constexpr int XM = TCH * 256;                          // LDS bytes per stream
};

// One wave's tasks (wave-uniform): row group grp[k], streams m0[k] ..; tasks
// kb .. ke-1, task 0 a piece of n0 streams, the others S wide.
struct MvTasks {
    int grp[MV_TW], m0[MV_TW];
    int kb, ke, n0;
};

template <int TYPE, int H, int S>
__global__ __launch_bounds__((MvShape<H>::T)) __attribute__((amdgpu_waves_per_eu(4)))
void kq_mv_kernel(MvArg A) {
    using TI = TypeInfo<TYPE>;
    using Sh = MvShape<H>;
    constexpr int T = Sh::T, W = Sh::W, GP = Sh::GP, RPT = Sh::RPT, TCH = Sh::TCH;
    constexpr int XPC = TI::XS_PER_CHUNK, G4 = XPC == 2 ? 8 : 4;   // float4 per x sum
    extern __shared__ __align__(256) uint8_t smem[];               // two x buffers, sums
    float* sums = reinterpret_cast<float*>(smem + 2 * MV_ME * Sh::XM);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(uint8_t __attribute__((address_space(3)))*)smem;
    const int tid = threadIdx.x, lane = tid & 63, p = lane & (GP - 1), lr = lane / GP, u = p & 3;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int K = A.K, NC = K >> 6, N = A.N, ntile = (NC + TCH - 1) / TCH;
    const size_t rbytes = (size_t)(K >> 8) * TI::BB;
    // XCD-major items (workgroup i runs on XCD i % 8): the stream chunks of
    // one row block, which read the same weights, share an L2
    const int lb = (int)(blockIdx.x & 7) * ((int)gridDim.x >> 3) + (int)(blockIdx.x >> 3);
    if (lb >= A.nitems) return;
    const int blk = lb / A.nmc, m0 = (lb - blk * A.nmc) * A.mc;
    const int Mc = min(A.mc, A.M - m0);
    const int r0 = blk * A.ng * RPT, rows = min(A.ng * RPT, N - r0);

    // Tasks (row group, S streams): every wave takes `full` of them; the
    // `rem` left over are cut into pieces of fewer streams, one to a wave, so
    // that the last turn of few waves is a short one.
    const int nsg = (Mc + S - 1) / S, ntask = ((rows + RPT - 1) / RPT) * nsg;
    const int full = ntask / W, rem = ntask - full * W;
    const int cut = mv_cut(S, rem, W);
    // odd workgroups fill their waves from the other end
    const int w0 = (blockIdx.x >> 3) & 1 ? W - 1 - wave : wave;
    MvTasks tk;
    [[maybe_unused]] int own[MV_TW];               // the first stream to store (mv_x0)
    tk.kb = w0 < rem * cut ? 0 : 1;
    tk.ke = full + 1;
    tk.n0 = S / cut;
#pragma unroll
    for (int k = 0; k < MV_TW; k++) {
        const int t = k ? rem + w0 + (k - 1) * W : w0 / cut;
        tk.grp[k] = t / nsg;
        tk.m0[k] = (t - tk.grp[k] * nsg) * S + (k ? 0 : (w0 % cut) * tk.n0);
        if constexpr (MV_ME % S != 0) {
            own[k] = tk.m0[k];
            tk.m0[k] = mv_x0(own[k], k ? S : tk.n0);
        }
    }
    const wptr gw = to_global(A.w);
    auto wrow = [&](int k) {
        return gw + (size_t)min(r0 + RPT * tk.grp[k] + lr, r0 + rows - 1) * rbytes;
    };
    auto wload = [&](wptr row, int c) {            // chunk c (clamped: same u) of a row
        return MvRaw<TYPE>::load(row + (size_t)(min(c, NC - 4 + u) >> 2) * TI::BB, u);
    };
    const wptr wf = tk.kb ? wrow(1) : wrow(0);     // the row of the wave's first task
    typename MvRaw<TYPE>::Raw nxt = wload(wf, p);

    // x tiles go straight to LDS (global_load_lds, no registers): a wave's
    // load i takes super-block cg of the tile of stream j = wave / SB + 2 i,
    // lane l to slot l % 16 of chunk 4 cg + l / 16.  A lane reads float4 t of
    // chunk c at slot t ^ (c % 16): the chunks of a 16-lane read phase are
    // distinct mod 16 (8 phases: mod 8), so no two meet in a bank.
    constexpr int SB = TCH / 4;
    const int cg = wave % SB, jw = wave / SB;
    const int lc = 4 * cg + (lane >> 4);
    const uint32_t voff =
        4u * (uint32_t)(256 * cg + mv_pos<TI::LINEAR>(lane >> 4, (lane & 15) ^ (lc & 15)));
    auto xtile = [&](int ti) {
        if (ti * TCH + 4 * cg < NC) {              // uniform: a super-block is whole or past K
#pragma unroll
            for (int i = 0; i < MV_ME / 2; i++) {
                const int j = jw + 2 * i;
                if (j < Mc) {
                    const float* src = A.X + (size_t)(m0 + j) * A.x_stride + (size_t)ti * TCH * 64;
                    const uint32_t dst =
                        lds0 + (uint32_t)((ti & 1) * MV_ME + j) * Sh::XM + 1024u * cg;
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\t"
                                 "global_load_lds_dwordx4 %1, %2"
                                 :: "s"(dst), "v"(voff), "s"(src) : "memory", "m0");
                }
            }
        }
    };
    xtile(0);

    const int per = XPC ? K / (4 * G4) : 0;
    if constexpr (XPC != 0) {
        // the x sums of every sub-block, in the reference's sequential order
        for (int q = tid; q < Mc * per; q += T) {
            const int j = q / per, gi = q - j * per;
            const f32x4* src = reinterpret_cast<const f32x4*>(A.X + (size_t)(m0 + j) * A.x_stride) +
                               (size_t)gi * G4;
            f32x4 v[G4];
#pragma unroll
            for (int k = 0; k < G4; k++) v[k] = src[k];
            float acc = 0.0f;
#pragma unroll
            for (int k = 0; k < G4; k++) {
                acc = acc + v[k].x; acc = acc + v[k].y; acc = acc + v[k].z; acc = acc + v[k].w;
            }
            int xsi = gi;
            if (!TI::LINEAR) {                     // Q2_K: 16 gi = block, half, run, 16-sub
                const int x = 16 * gi, pp = x & 255;
                xsi = 4 * (4 * (x >> 8) + 2 * (pp >> 7) + ((pp >> 4) & 1)) + ((pp >> 5) & 3);
            }
            sums[j * per + xsi] = acc;
        }
    }

    double part[MV_TW][S];
#pragma unroll
    for (int k = 0; k < MV_TW; k++)
#pragma unroll
        for (int s = 0; s < S; s++) part[k][s] = 0.0;

    auto unit = [&](auto nn, int k, const typename MvRaw<TYPE>::Raw& cur, int ti, int c, int cl) {
        constexpr int n = decltype(nn)::v;
        const float* xs[n];
        double t[n];
        const MvX x = {lds0 + (uint32_t)(((ti & 1) * MV_ME + tk.m0[k]) * Sh::XM + 256 * cl +
                                         16 * (cl & 15)),
                       Sh::XM};
#pragma unroll
        for (int s = 0; s < n; s++) {
            // a stream past the last: its slots hold anything, its results are not stored
            xs[s] = sums + min(tk.m0[k] + s, Mc - 1) * per;
            t[s] = part[k][s];
        }
        MvTerms<TYPE, n>::run(mv_opaque(cur), u, x, xs, c, t);
#pragma unroll
        for (int s = 0; s < n; s++) part[k][s] = t[s];
    };

    for (int ti = 0; ti < ntile; ti++) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's part of the tile is in LDS
        __syncthreads();                                  // and everyone's; the other buffer is free
        if (ti + 1 < ntile) xtile(ti + 1);
#pragma unroll
        for (int j = 0; j < TCH / GP; j++) {
            const int cl = GP * j + p, c = ti * TCH + cl;
            // unconditional loads: one under a branch would make the
            // compiler wait for it at the join
#pragma unroll
            for (int k = 0; k < MV_TW; k++) {
                const typename MvRaw<TYPE>::Raw cur = nxt;
                const bool wrap = k + 1 >= tk.ke || k + 1 >= MV_TW;
                nxt = wload(wrap ? wf : wrow(1), c + (wrap ? GP : 0));
                if (k >= tk.kb && k < tk.ke && c < NC) {
                    if (k > 0 || tk.n0 == S) unit(MvInt<S>(), k, cur, ti, c, cl);
                    else if (S == 4 && tk.n0 == 2) unit(MvInt<2>(), 0, cur, ti, c, cl);
                    else unit(MvInt<1>(), 0, cur, ti, c, cl);
                }
            }
        }
    }

#pragma unroll
    for (int k = 0; k < MV_TW; k++)
        if (k >= tk.kb && k < tk.ke) {
#pragma unroll
            for (int s = 0; s < S; s++) {
                const double v = phase_tree(part[k][s], GP);
                const int m = tk.m0[k] + s, rr = RPT * tk.grp[k] + lr;
                if (p == 0 && rr < rows && m < Mc && (k > 0 || s < tk.n0) &&
                    (MV_ME % S == 0 || m >= own[k]))
                    A.Y[(size_t)(m0 + m) * A.y_stride + r0 + rr] = (float)v;
            }
        }
}

typedef void (*mv_fn)(MvArg);
#define KQ_MV_ROW(T_)                                                                   \
    {{&kq_mv_kernel<T_, 1, 2>, &kq_mv_kernel<T_, 1, 3>, &kq_mv_kernel<T_, 1, 4>},       \
     {&kq_mv_kernel<T_, 2, 2>, &kq_mv_kernel<T_, 2, 3>, &kq_mv_kernel<T_, 2, 4>}}
const int k_mv_types[7] = {T_Q4K, T_Q6K, T_Q2K, T_NIB, T_Q5K, T_Q3K, T_Q80};
const mv_fn k_mv[7][2][3] = {KQ_MV_ROW(T_Q4K), KQ_MV_ROW(T_Q6K), KQ_MV_ROW(T_Q2K), KQ_MV_ROW(T_NIB),
                          KQ_MV_ROW(T_Q5K), KQ_MV_ROW(T_Q3K), KQ_MV_ROW(T_Q80)};

int mv_type(int type) {
    for (int i = 0; i < 7; i++)
        if (k_mv_types[i] == type) return i;
    return -1;
}

int mv_xpc(int type) {
    return type == T_Q4K || type == T_Q5K ? 2 : type == T_Q2K || type == T_NIB ? 4 : 0;
}

}  // namespace

extern "C" {

// Plan of an exact MULTISEQ launch: plan[] = streams per chunk, stream
// chunks, row groups per item, items per stream chunk, S.  Returns the LDS
// bytes, or -1 when the kernel does not take it: x sums that leave no room for
// the tiles, or more workgroups than a launch holds (fewer streams may fit).
long kqk_mv_plan(int type, int N, int K, int M, int n_cu, int lds_max, int* plan) {
    if (mv_type(type) < 0 || N < 1 || M < 1 || K <= 0 || (K & 255)) return -1;
    const int NC = K >> 6, H = kq_phases(NC) == 32 ? 2 : 1;
    const int W = 8 * H, TCH = 16 * H, RPT = H == 1 ? 8 : 2, GP = 64 / RPT;
    const int xpc = mv_xpc(type);
    const long xsum = xpc ? (long)(K / (xpc == 2 ? 32 : 16)) * 4 : 0;   // LDS bytes per stream
    const long tiles = 2L * MV_ME * TCH * 256;
    if (tiles + xsum > lds_max) return -1;
    const int Q = (N + RPT - 1) / RPT, nstep = (NC + GP - 1) / GP;
    // clocks of a unit, counted from the generated code at the measured issue
    // rates: dec once, mem per stream
    const double dec = type == T_Q6K ? 620 : type == T_Q3K ? 800 : type == T_Q5K ? 600
                     : type == T_Q80 ? 420 : 480;
    const double mem = xpc == 4 || type == T_Q6K ? 370 : 340;
    double best = 1e300;
    long best_lds = -1;
    int best_wgs = 0;
    int nmc0 = (M + MV_ME - 1) / MV_ME;
    while (nmc0 < M && tiles + (M + nmc0 - 1) / nmc0 * xsum > lds_max) nmc0++;
    for (int nmc = nmc0; nmc <= M && nmc <= nmc0 + 1; nmc++) {
        const int mc = (M + nmc - 1) / nmc;
        if ((M + mc - 1) / mc != nmc) continue;
        const long lds = tiles + mc * xsum;
        if (lds > lds_max) continue;
        int res = (int)(lds_max / lds);
        if (res > 2 / H) res = 2 / H;
        for (int S = 2; S <= 4; S++) {
            const int nsg = (mc + S - 1) / S;
            for (int ng = 1; ng * nsg < W * MV_TW; ng++) {
                const long items = (long)((Q + ng - 1) / ng) * nmc, slots = (long)res * n_cu;
                if ((items + 7) * 512 * H >= MV_LANES) continue;
                const long rounds = (items + slots - 1) / slots, last = items - (rounds - 1) * slots;
                const int nt = ng * nsg, full = nt / W, rem = nt - full * W, cut = mv_cut(S, rem, W);
                // one group of four streams of Q5_K, whose S = 4 form spills,
                // unless every wave of two workgroups a CU has one: 17408 x 5120
                // 48.1 us (44.4 as two groups of two), 11007 x 4096 30.6 (25.1);
                // 32000 x 768, 500 items of 8 tasks, 16.2 (16.9)
                if (type == T_Q5K && M == 4 && S == 4 && (rem || items <= n_cu)) continue;
                // a turn of n waves on a SIMD takes max(2, n) of a wave's
                // clocks at the full issue rate, which needs two waves
                auto turn = [&](int wgs, int waves, int s) {
                    const int n = wgs * ((waves + 3) / 4);
                    return (n < 2 ? 2 : n) * (dec + mem * s);
                };
                auto round_cost = [&](int wgs) {
                    const double t =
                        full * turn(wgs, W, S) + (rem ? turn(wgs, rem * cut, S / cut) : 0.0);
                    // a CU's only workgroup with half its waves idle waits out
                    // its loads: 2560 x 9728 Q8_0 B = 3 in 6 waves of three
                    // streams 21.6 us, in 15 of one 17.7 (the model: even)
                    const bool few = H == 2 && !full && 2 * rem * cut <= W;
                    return nstep * (few ? 1.3 * t : t) + 12000.0;
                };
                const int wgs = (int)((last + n_cu - 1) / n_cu);
                const double cost = (rounds - 1) * round_cost(res) + round_cost(wgs);
                // at one cost (the same pieces in a SIMD), fewer workgroups on a
                // CU: each stages x for itself.  4096 x 4096 Q5_K B = 4 in 512
                // items of one row group 22.9 us, in 256 of two 17.2.  Not where
                // that leaves a turn of few waves: 11007 x 4096 Q2_K B = 5, 459
                // items of 6 tasks 29.4, 230 of 12 on 8 waves 31.8
                if (cost < best ||
                    (cost == best && S == plan[4] && wgs < best_wgs && (!full || !rem))) {
                    best = cost;
                    best_wgs = wgs;
                    best_lds = lds;
                    plan[0] = mc; plan[1] = nmc; plan[2] = ng; plan[3] = (Q + ng - 1) / ng;
                    plan[4] = S;
                }
            }
        }
    }
    return best_lds;
}

// x slots that the tasks of a plan's launch read (MV_ME are staged): every
// group of S streams of its stream chunks, whole and in pieces
int kqk_mv_slots(const int* plan, int M) {
    const int S = plan[4];
    int top = 0;
    for (int c = 0; c < plan[1]; c++) {
        const int Mc = c + 1 < plan[1] ? plan[0] : M - c * plan[0];
        for (int m0 = 0; m0 < Mc; m0 += S)
            for (int n = 1; n <= S; n++)
                for (int i = 0; S % n == 0 && i < S; i += n) {
                    const int t = (MV_ME % S ? mv_x0(m0 + i, n) : m0 + i) + n;
                    if (t > top) top = t;
                }
    }
    return top;
}

int kqk_mv_set_max_lds(int bytes) {
    for (int t = 0; t < 7; t++)
        for (int i = 0; i < 6; i++) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_mv[t][i / 3][i % 3]),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
            if (e != hipSuccess) return (int)e;
        }
    return 0;
}

int kqk_launch_mv(int type, const int* plan, long lds, const void* w, const float* X, long x_stride,
                  float* Y, long y_stride, int M, int N, int K, hipStream_t st) {
    const int ts = mv_type(type);
    if (ts < 0) return (int)hipErrorInvalidValue;
    const int H = kq_phases(K >> 6) == 32 ? 2 : 1;
    MvArg a;
    a.w = static_cast<const uint8_t*>(w);
    a.X = X; a.Y = Y;
    a.x_stride = x_stride; a.y_stride = y_stride;
    a.M = M; a.N = N; a.K = K;
    a.mc = plan[0]; a.nmc = plan[1]; a.ng = plan[2]; a.nblk = plan[3];
    a.nitems = a.nblk * a.nmc;
    const int grid = (a.nitems + 7) & ~7;
    hipLaunchKernelGGL(k_mv[ts][H - 1][plan[4] - 2], dim3(grid), dim3(512 * H), (size_t)lds, st, a);
    return (int)hipGetLastError();
}

}  // extern "C"
