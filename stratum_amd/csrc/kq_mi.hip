// kq_mi.hip -- int8 MULTISEQ of Q4_K and Q6_K (st_linear_multix under
// use_sdot) on the int8 matrix cores (gfx950).
//
// The reference's multix pack arithmetic, bit for bit:
//  Q4_K (q4k_dot_rows2_sdot_multix_pack, stratum_q4k_neon.h:870-948): per
//   sub-block the binary32 term fl(fl(fl(d sc) fl(fl(L) scl)) - fl(fl(dmin m)
//   fl(fl(S) scl))), L the exact dot, S the group's sum of x, added to a
//   binary64 sum in element order;
//  Q6_K (q6k_dot_rows2_sdot_multix_pack, stratum_q6k_neon.h:627-700): per
//   16-group ((double)d sc (double)scl) (double)A, A the exact dot of q - 32.
// The binary64 sum is grouped by K-part (kqk_mi8_parts: by the row length).
//
// One v_mfma_i32_16x16x32_i8 takes 16 streams x 32 positions against 16 rows:
// D[stream 4q + i][row l % 16] in lane l = 16 q + r, so a lane's four results
// are its row's dots with four streams.  Its operands are 8 bytes a lane: a
// sub-block of the row, and x laid out by the prep launch so that a lane's 8
// bytes of two sub-blocks are one 16-byte read.  (Q6_K's groups are half of
// the 32 positions: the other half of the weights is zeroed, twice.)
//
// What bounds it.  At 64 streams VALU issue: 17408 x 5120 Q4_K 24.6 K
// instructions a SIMD, 98 K clk of 58 us.  At 16 and fewer neither the weight
// stream (50 MB, 10 us) nor VALU (6.1 K instructions a SIMD, 10 to 12 us of
// 22.4): with two waves a SIMD, a wave waits in 37 % of its life for a step's
// loads, which are asked for one super-block ahead and all awaited at the
// step's barrier.  With the weights a row to a lane, as the MFMA wants its
// operand, every lane of a load is a cache access of its own (11 M a call at
// 16 streams, which held it at 26 to 30 us).  So all loads go to
// LDS without registers (global_load_lds) in address order, neighbouring lanes
// reading neighbouring bytes: one record per super-block and 16 streams,
// shared by the workgroup's row blocks, and each wave's 16 weight blocks, a
// step ahead.  Measured with the prep launch against the kernel before it,
// whose waves each loaded their operands to registers: 17408 x 5120 Q4_K B = 2
// / 8 / 16 / 32 / 64 26.0 / 27.4 / 35.6 / 54 / 91 -> 22.7 / 23.9 / 23.8 / 34.3
// / 56.0 us; 5120 x 17408 Q6_K B = 8 / 16 / 32 / 64 80 / 110 / 172 / 328 -> 53
// / 53 / 82 / 125 us; 4096 x 4096 Q4_K B = 4 13.5 -> 13.2 us.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kq_blocks.h"
#include "kq_launch.h"

#pragma clang fp contract(off)

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));

// A record: the quantized x of 16 streams at one super-block, then their
// coefficients.  x: 16 bytes at 1024 j + 16 (16 q + s): stream s, positions
// 64 j + 8 q .. +7 and 64 j + 32 + 8 q .. +7.  Coefficients: Q4_K float2
// {scl, fl(fl(S) scl)} [8 sub-blocks][16 streams]; Q6_K double scl [16
// groups][16 streams].
template <int TYPE> struct MiRec;
template <> struct MiRec<T_Q4K_I8> { static constexpr int G = 32, CF = 1024, BYTES = 4096 + CF; };
template <> struct MiRec<T_Q6K_I8> { static constexpr int G = 16, CF = 2048, BYTES = 4096 + CF; };

// One lane per (stream, group): the quantizer (q4k_quantize_x_q8,
// stratum_q4k_neon.h:229-275; q6k_quantize_x_q8_g16, stratum_q6k_neon.h:
// 117-133), into records; streams past B are zero.
template <int TYPE>
__global__ __launch_bounds__(64) void kq_mi_prep_kernel(const float* x, long x_stride, int K, int B,
                                                        int nset, uint8_t* rec) {
    using R = MiRec<TYPE>;
    constexpr int G = R::G;
    const int ng = K / G, g = blockIdx.y * 64 + threadIdx.x, s = blockIdx.x;
    if (g >= ng) return;
    f32x4 v[G / 4];
    const f32x4* src =
        reinterpret_cast<const f32x4*>(x + (size_t)min(s, B - 1) * x_stride) + (size_t)g * (G / 4);
#pragma unroll
    for (int k = 0; k < G / 4; k++) v[k] = s < B ? src[k] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float amax = 0.0f;
#pragma unroll
    for (int k = 0; k < G / 4; k++)
        amax = fmaxf(fmaxf(fmaxf(amax, fabsf(v[k].x)), fmaxf(fabsf(v[k].y), fabsf(v[k].z))),
                     fabsf(v[k].w));
    const float scale = __fdiv_rn(amax, 127.0f);
    const float inv = scale > 0.0f ? __fdiv_rn(1.0f, scale) : 0.0f;
    int sum = 0;
    uint32_t w[G / 4];
#pragma unroll
    for (int k = 0; k < G / 4; k++) {
        const float e[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
        w[k] = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int iv = min(127, max(-128, __float2int_rn(e[i] * inv)));
            sum += iv;
            w[k] |= ((uint32_t)iv & 0xffu) << (8 * i);
        }
    }
    const int p0 = g * G, sb = p0 >> 8, pp = p0 & 255, set = s >> 4, st = s & 15;
    uint8_t* r = rec + ((size_t)sb * nset + set) * R::BYTES;
    uint8_t* d = r + 1024 * (pp >> 6) + 8 * ((pp >> 5) & 1) + 16 * st;
    const int q0 = (pp & 31) >> 3;
#pragma unroll
    for (int k = 0; k < G / 8; k++)
        *reinterpret_cast<uint2*>(d + 256 * (q0 + k)) = make_uint2(w[2 * k], w[2 * k + 1]);
    if (G == 32)
        reinterpret_cast<float2*>(r + 4096)[16 * (g & 7) + st] = make_float2(scale, (float)sum * scale);
    else
        reinterpret_cast<double*>(r + 4096)[16 * (g & 15) + st] = (double)scale;
}

struct MiArg {
    const uint8_t* w;             // N rows of K weights
    const uint8_t* rec;           // records [super-block][set]
    float* y;                     // y[s * y_stride + r]
    long y_stride;
    int N, K, B, nset;
    int walign;                   // weights 16-byte aligned
};

// LDS bytes of 16 weight blocks (Q6_K: 14 loads of 64 dwords)
constexpr int mi_wb(bool q4) { return q4 ? 16 * 144 : 14 * 256; }

// a barrier that leaves the loads in flight (__syncthreads waits for them)
__device__ __forceinline__ void mi_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// A workgroup: 4 waves = RB 16-row blocks x KS K-parts; a wave 16
// streams (one set: two sets a wave, sharing the weights, leave a CU fewer
// waves and ran 54 against 44 us at B = 32 and 68 against 59 at B = 64).
// Step t is super-block t of each K-part, its records and each
// wave's 16 weight blocks loaded to one of two LDS buffers a step ahead.
template <int TYPE, int KS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
void kq_mi_kernel(MiArg A) {
    constexpr bool Q4 = TYPE == T_Q4K_I8;
    constexpr int RB = 4 / KS, REC = MiRec<TYPE>::BYTES, BB = Q4 ? 144 : 210;
    constexpr int XT = KS * REC, WB = mi_wb(Q4);   // LDS bytes of a step: records,
    constexpr int TILE = XT + 4 * WB;                   // and each wave's weights
    constexpr int DM = Q4 ? 1024 : 0;               // per wave: d sc, dmin m of 16 rows
    extern __shared__ __align__(16) uint8_t smem[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(uint8_t __attribute__((address_space(3)))*)smem;
    const int tid = threadIdx.x, lane = tid & 63, q = lane >> 4, jr = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int kp = wave % KS;
    asm volatile("" : "+s"(kp));                 // KS = 1: not a constant, or the loop is unrolled into spills
    // XCD-major (workgroup i runs on XCD i % 8): the sets of one group of row
    // blocks, which read the same weights, share an L2
    const int nset = A.nset, lb = (int)(blockIdx.x & 7) * ((int)gridDim.x >> 3) + (int)(blockIdx.x >> 3);
    const int rg = lb / nset, set = lb - rg * nset, rb = rg * RB + wave / KS;
    if (rg * RB * 16 >= A.N) return;               // uniform: the grid is rounded up
    const int N = A.N, nb = A.K >> 8, nbp = (nb + KS - 1) / KS;
    const int row = min(rb * 16 + jr, N - 1);
    uint8_t* dml = smem + 2 * TILE + wave * DM;

    // The records of step t in pieces of 1 KB, CP to a wave (a piece past the
    // last is the last again).
    constexpr int PC = REC / 1024, NP = KS * PC, CP = (NP + 3) / 4;
    // The wave's 16 blocks in address order, so that neighbouring lanes read
    // neighbouring bytes (read a row to a lane, every lane is a cache access
    // of its own: 320 and 770 a step against 40 and 70).  Q4_K: 9 x 16 bytes a
    // row; Q6_K, whose odd blocks start 2 bytes off: the dwords that hold the
    // block (53; 54 if it starts 3 off, in a tensor at an odd address: the
    // places past the 53rd hold the block's last dword), 55 to a row, an odd
    // count for the LDS banks.
    constexpr int NW = Q4 ? 3 : 14, PW = Q4 ? 9 : 55;
    uint32_t wo[NW], wd[Q4 ? 1 : NW];
#pragma unroll
    for (int i = 0; i < NW; i++) {
        const int c = min(lane + 64 * i, 16 * PW - 1), r = c / PW;
        wo[i] = (uint32_t)(min(rb * 16 + r, N - 1) - min(rb * 16, N - 1)) * (uint32_t)(nb * BB);
        if (Q4) wo[i] += 16u * (c - PW * r);
        else {
            const int k = c - PW * r;
            wd[Q4 ? 0 : i] = 4u * min(k, 52);
            wo[i] += k > 52;                       // 3 off: rounds down to the 54th
        }
    }
    const uint8_t* w0 = A.w + (size_t)min(rb * 16, N - 1) * ((size_t)nb * BB);   // uniform
    auto glds = [&](uint32_t dst, uint32_t off, const uint8_t* src) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :: "s"(dst), "v"(off), "s"(src) : "memory", "m0");
    };
    auto stage = [&](int t, int buf) {
#pragma unroll
        for (int i = 0; i < CP; i++) {
            const int p = min(wave + 4 * i, NP - 1);   // uniform
            const int pc = p % PC, k = p / PC, sb = min(k * nbp + t, nb - 1);
            glds(lds0 + (uint32_t)(buf * TILE + 1024 * p), 16u * lane,
                 A.rec + ((size_t)sb * nset + set) * REC + 1024 * pc);
        }
        const uint8_t* src = w0 + (size_t)min(kp * nbp + t, nb - 1) * BB;
        const uint32_t dst = lds0 + (uint32_t)(buf * TILE + XT + wave * WB);
        if constexpr (Q4) {
            if (A.walign) {                        // uniform
                glds(dst, wo[0], src);
                glds(dst + 1024, wo[1], src);
                if (lane < 16) glds(dst + 2048, wo[2], src);
            } else {                               // weights not 16-byte aligned: through registers
#pragma unroll
                for (int i = 0; i < 3; i++) {
                    const uint4 v = ld16(to_global(src) + wo[i]);
                    if (i < 2 || lane < 16)
                        *reinterpret_cast<uint4*>(smem + (dst - lds0) + 1024 * i + 16 * lane) = v;
                }
            }
        } else {
            const uint32_t mis = (uint32_t)(uintptr_t)src & 3u;
            const uint8_t* al = src - mis;
#pragma unroll
            for (int i = 0; i < NW; i++)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                             :: "s"(dst + 256u * i), "v"(((wo[i] + mis) & ~3u) + wd[Q4 ? 0 : i]), "s"(al)
                             : "memory", "m0");
        }
    };

    double acc[4];
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = 0.0;
    const i32x4 zero = {0, 0, 0, 0};
    stage(0, 0);
    for (int t0 = 0; t0 < nbp; t0 += 2) {
#pragma unroll
        for (int p = 0; p < 2; p++) {
            const int t = t0 + p;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wave's part of the step is in
            mi_barrier();                          // everyone's is; the other buffer is free
            if (t + 1 < nbp) stage(t + 1, 1 - p);
            if (t >= nbp || kp * nbp + t >= nb) continue;          // uniform
            const uint8_t* rec = smem + p * TILE + kp * REC;
            if constexpr (Q4) {
                const uint8_t* wl = smem + p * TILE + XT + wave * WB + 144 * jr;
                const uint4 hd = *reinterpret_cast<const uint4*>(wl);
                const float d = f16_bits_to_f32(hd.x & 0xffffu);
                const float dmin = f16_bits_to_f32(hd.x >> 16);
                uint32_t sc1, mn1, sc2, mn2;
                // lane group q decodes sub-blocks 2q, 2q+1 of its row for all
                scale_min_pair(hd.y, hd.z, hd.w, q, sc1, mn1, sc2, mn2);
                *reinterpret_cast<float4*>(dml + 16 * (16 * q + jr)) =
                    make_float4(d * (float)sc1, dmin * (float)mn1, d * (float)sc2, dmin * (float)mn2);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float4 dm = *reinterpret_cast<const float4*>(dml + 16 * (16 * j + jr));
                    const uint2 v = *reinterpret_cast<const uint2*>(wl + 16 + 32 * j + 8 * q);
                    const uint64_t lo = (uint64_t)(v.x & 0x0f0f0f0fu) | (uint64_t)(v.y & 0x0f0f0f0fu) << 32;
                    const uint64_t hi =
                        (uint64_t)((v.x >> 4) & 0x0f0f0f0fu) | (uint64_t)((v.y >> 4) & 0x0f0f0f0fu) << 32;
                    const ulonglong2 xa =
                        *reinterpret_cast<const ulonglong2*>(rec + 1024 * j + 16 * lane);
                    const i32x4 L = __builtin_amdgcn_mfma_i32_16x16x32_i8((long)xa.x, (long)lo, zero, 0, 0, 0);
                    const i32x4 H = __builtin_amdgcn_mfma_i32_16x16x32_i8((long)xa.y, (long)hi, zero, 0, 0, 0);
                    const float4* cl = reinterpret_cast<const float4*>(rec + 4096 +
                                                                      128 * (2 * j) + 32 * q);
                    const float4 c0 = cl[0], c1 = cl[1], e0 = cl[8], e1 = cl[9];
                    const float sl[4] = {c0.x, c0.z, c1.x, c1.z}, ml[4] = {c0.y, c0.w, c1.y, c1.w};
                    const float sh[4] = {e0.x, e0.z, e1.x, e1.z}, mh[4] = {e0.y, e0.w, e1.y, e1.w};
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float tl = dm.x * ((float)L[i] * sl[i]) - dm.y * ml[i];
                        acc[i] = acc[i] + (double)tl;
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const float th = dm.z * ((float)H[i] * sh[i]) - dm.w * mh[i];
                        acc[i] = acc[i] + (double)th;
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                // this row's block starts mis bytes into its dwords
                const uint8_t* wl = smem + p * TILE + XT + wave * WB + 220 * jr;
                const uint32_t sh = 8u * (((uint32_t)(uintptr_t)A.w +
                                           ((uint32_t)row * (uint32_t)nb + (uint32_t)(kp * nbp + t)) * 210u) & 3u);
                auto dw = [&](int o) { return *reinterpret_cast<const uint32_t*>(wl + o); };
                const double d = (double)f16_bits_to_f32(
                    __builtin_amdgcn_alignbit(dw(212), dw(208), sh) & 0xffffu);
                uint32_t S[4];
#pragma unroll
                for (int k = 0; k < 4; k++)
                    S[k] = __builtin_amdgcn_alignbit(dw(196 + 4 * k), dw(192 + 4 * k), sh);
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    // the bytes q - 32 of run-pairs t = 0..3 (positions 128h + 32t + 8q ..)
                    uint32_t bw[4][2];
#pragma unroll
                    for (int k = 0; k < 2; k++) {
                        const int o = 8 * q + 4 * k;
                        const uint32_t H = __builtin_amdgcn_alignbit(dw(132 + 32 * h + o), dw(128 + 32 * h + o), sh);
#pragma unroll
                        for (int t = 0; t < 4; t++) {
                            const int ol = o + 64 * h + 32 * (t & 1);
                            const uint32_t L = __builtin_amdgcn_alignbit(dw(ol + 4), dw(ol), sh);
                            const uint32_t v = ((L >> (4 * (t >> 1))) & 0x0f0f0f0fu) |
                                               (((H >> (2 * t)) & 0x03030303u) << 4);
                            bw[t][k] = ((v | 0x80808080u) - 0x20202020u) ^ 0x80808080u;
                        }
                    }
#pragma unroll
                    for (int is = 0; is < 2; is++) {
                        const bool on = (q >> 1) == is;        // the group's half of the positions
#pragma unroll
                        for (int t = 0; t < 4; t++) {
                            const int g = 8 * h + is + 2 * t;
                            const double ds = d * (double)(int8_t)(uint8_t)(S[g >> 2] >> (8 * (g & 3)));
                            const uint64_t bo = on ? (uint64_t)bw[t][0] | (uint64_t)bw[t][1] << 32 : 0;
                            const uint64_t xa = *reinterpret_cast<const uint64_t*>(
                                rec + 1024 * (2 * h + (t >> 1)) + 16 * lane + 8 * (t & 1));
                            const i32x4 D = __builtin_amdgcn_mfma_i32_16x16x32_i8((long)xa, (long)bo, zero, 0, 0, 0);
                            const double2* cs = reinterpret_cast<const double2*>(
                                rec + 4096 + 128 * g + 32 * q);
                            const double2 c0 = cs[0], c1 = cs[1];
                            const double c[4] = {c0.x, c0.y, c1.x, c1.y};
#pragma unroll
                            for (int i = 0; i < 4; i++)
                                acc[i] = acc[i] + ds * c[i] * (double)D[i];
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
        }
    }
    // the K-parts' sums, added in K-part order by the first part's wave
    if (KS > 1) {
        double* part = reinterpret_cast<double*>(smem);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (kp) {
#pragma unroll
            for (int i = 0; i < 4; i++) part[(wave * 4 + i) * 64 + lane] = acc[i];
        }
        __syncthreads();
        if (kp) return;
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int k = 1; k < KS; k++)
                acc[i] = acc[i] + part[((wave + k) * 4 + i) * 64 + lane];
    }
    if (rb * 16 + jr < N) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int s = 16 * set + 4 * q + i;
            if (s < A.B) A.y[(size_t)s * A.y_stride + rb * 16 + jr] = (float)acc[i];
        }
    }
}

typedef void (*mi_fn)(MiArg);
#define KQ_MI_ROW(T_) {&kq_mi_kernel<T_, 1>, &kq_mi_kernel<T_, 2>, &kq_mi_kernel<T_, 4>}
const mi_fn k_mi[2][3] = {KQ_MI_ROW(T_Q4K_I8), KQ_MI_ROW(T_Q6K_I8)};

long mi_rec(int type) { return type == T_Q4K_I8 ? MiRec<T_Q4K_I8>::BYTES : MiRec<T_Q6K_I8>::BYTES; }

long mi_lds(int type, int ks) {
    return 2 * (ks * mi_rec(type) + 4 * mi_wb(type == T_Q4K_I8)) + (type == T_Q4K_I8 ? 4 * 1024 : 0);
}

}  // namespace

extern "C" {

// Bytes of the records of B streams, or -1.
long kqk_mi_workspace(int type, int B, int K) {
    if ((type != T_Q4K_I8 && type != T_Q6K_I8) || B < 1 || K < 256 || (K & 255)) return -1;
    return (long)(K >> 8) * ((B + 15) / 16) * mi_rec(type);
}

int kqk_mi_set_max_lds(int bytes) {
    for (int t = 0; t < 2; t++)
        for (int i = 0; i < 3; i++) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_mi[t][i]),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
            if (e != hipSuccess) return (int)e;
        }
    return 0;
}

// Most streams of one launch, in whole sets: HIP refuses 2^32 lanes (2^24
// workgroups of 256); 2^16 sets also bound the prep launch
int kqk_mi_streams(int N, int K) {
    const int rb = 4 / kqk_mi8_parts(K);
    const long groups = ((N + 15L) / 16 + rb - 1) / rb, sets = ((1L << 24) - 8) / groups;
    return (int)(16 * (sets < 1 ? 1 : sets > 1 << 16 ? 1 << 16 : sets));
}

int kqk_launch_mi(int type, const float* xs, long x_stride, const void* w, float* ys, long y_stride,
                  int B, int N, int K, void* ws, hipStream_t st) {
    const int ks = kqk_mi8_parts(K), nset = (B + 15) / 16;
    if (kqk_mi_workspace(type, B, K) < 0 || N < 1 || B < 1 || (x_stride & 3) || x_stride < K ||
        y_stride < N || ((uintptr_t)xs & 15) || ((uintptr_t)ws & 255) || ks > 4 ||
        B > kqk_mi_streams(N, K))
        return (int)hipErrorInvalidValue;
    uint8_t* rec = static_cast<uint8_t*>(ws);
    if (type == T_Q4K_I8)
        hipLaunchKernelGGL(kq_mi_prep_kernel<T_Q4K_I8>, dim3(16 * nset, (K / 32 + 63) / 64), dim3(64), 0,
                           st, xs, x_stride, K, B, nset, rec);
    else
        hipLaunchKernelGGL(kq_mi_prep_kernel<T_Q6K_I8>, dim3(16 * nset, (K / 16 + 63) / 64), dim3(64), 0,
                           st, xs, x_stride, K, B, nset, rec);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return (int)e;
    MiArg a;
    a.w = static_cast<const uint8_t*>(w);
    a.rec = rec;
    a.y = ys; a.y_stride = y_stride;
    a.N = N; a.K = K; a.B = B; a.nset = nset;
    a.walign = ((uintptr_t)w & 15) == 0;
    const int rb = 4 / ks;
    const long wgs = ((N + 15L) / 16 + rb - 1) / rb * nset;
    hipLaunchKernelGGL(k_mi[type == T_Q6K_I8][ks == 4 ? 2 : ks - 1], dim3((unsigned)((wgs + 7) & ~7L)),
                       dim3(256), (size_t)mi_lds(type, ks), st, a);
    return (int)hipGetLastError();
}

}  // extern "C"
