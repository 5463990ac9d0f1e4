// kq_blocks.h -- the k-quant super-block formats on the device: type traits,
// raw weight loads, field extraction and the row reduction's phase rule,
// shared by the kernels' translation units (internal linkage: each has its
// own copy).
#ifndef KQ_BLOCKS_H
#define KQ_BLOCKS_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#pragma clang fp contract(off)

namespace {

constexpr int T_Q80 = 8;
constexpr int T_Q2K = 10;
constexpr int T_Q3K = 11;
constexpr int T_Q4K = 12;
constexpr int T_Q5K = 13;
constexpr int T_Q6K = 14;
constexpr int T_NIB = 42;
// the int8-activation mode (the reference's SDOT path) of Q4_K, Q6_K,
// Q5_K, Q3_K and Q8_0: the type id with this bit set
constexpr int T_I8 = 0x100;
constexpr int T_Q4K_I8 = T_I8 | T_Q4K;
constexpr int T_Q6K_I8 = T_I8 | T_Q6K;
constexpr int T_Q5K_I8 = T_I8 | T_Q5K;
constexpr int T_Q3K_I8 = T_I8 | T_Q3K;
constexpr int T_Q80_I8 = T_I8 | T_Q80;
// float4 slots per chunk in the int8 x layout: 64 bytes padded to 80
// (chunk c at byte 80c; 16-byte reads by consecutive chunks hit distinct
// banks)
constexpr int XPAD_I8 = 5;

constexpr int XPAD = 17;  // float4 slots per 64-weight chunk in LDS (16 + 1 pad)

typedef float f32x4 __attribute__((ext_vector_type(4)));

// BB: bytes per 256 weights; LINEAR: a chunk is 64 consecutive x values
// (else 4 runs of 16, spaced 32 apart); XS_PER_CHUNK: x sums per chunk for
// min terms; SCALED: products by the byte-select multiply on x staged as
// x * 2^KSC (the other types read x as staged and fold the factor into
// their scale).
// I8: the int8-activation mode (x quantized per group, XSTRIDE float4
// slots per chunk of int8 x; XS_PER_CHUNK floats hold each group's scale
// and integer sum).
template <int TYPE> struct TypeInfo;
template <> struct TypeInfo<T_Q4K> { static constexpr int BB = 144; static constexpr bool LINEAR = true;  static constexpr int XS_PER_CHUNK = 2; static constexpr bool SCALED = true; };
template <> struct TypeInfo<T_Q4K_I8> { static constexpr int BB = 144; static constexpr bool LINEAR = true;  static constexpr int XS_PER_CHUNK = 4; static constexpr bool SCALED = false; };
template <> struct TypeInfo<T_Q6K_I8> { static constexpr int BB = 210; static constexpr bool LINEAR = false; static constexpr int XS_PER_CHUNK = 8; static constexpr bool SCALED = false; };
template <> struct TypeInfo<T_Q5K_I8> { static constexpr int BB = 176; static constexpr bool LINEAR = true;  static constexpr int XS_PER_CHUNK = 4; static constexpr bool SCALED = false; };
template <> struct TypeInfo<T_Q80_I8> { static constexpr int BB = 272; static constexpr bool LINEAR = true;  static constexpr int XS_PER_CHUNK = 4; static constexpr bool SCALED = false; };
template <> struct TypeInfo<T_Q3K_I8> { static constexpr int BB = 110; static constexpr bool LINEAR = false; static constexpr int XS_PER_CHUNK = 8; static constexpr bool SCALED = false; };
template <> struct TypeInfo<T_Q6K> { static constexpr int BB = 210; static constexpr bool LINEAR = false; static constexpr int XS_PER_CHUNK = 0; static constexpr bool SCALED = false; };
template <> struct TypeInfo<T_Q2K> { static constexpr int BB = 84;  static constexpr bool LINEAR = false; static constexpr int XS_PER_CHUNK = 4; static constexpr bool SCALED = true; };
template <> struct TypeInfo<T_NIB> { static constexpr int BB = 148; static constexpr bool LINEAR = true;  static constexpr int XS_PER_CHUNK = 4; static constexpr bool SCALED = true; };
template <> struct TypeInfo<T_Q5K> { static constexpr int BB = 176; static constexpr bool LINEAR = true;  static constexpr int XS_PER_CHUNK = 2; static constexpr bool SCALED = true; };
template <> struct TypeInfo<T_Q3K> { static constexpr int BB = 110; static constexpr bool LINEAR = false; static constexpr int XS_PER_CHUNK = 0; static constexpr bool SCALED = false; };
template <> struct TypeInfo<T_Q80> { static constexpr int BB = 272; static constexpr bool LINEAR = true;  static constexpr int XS_PER_CHUNK = 0; static constexpr bool SCALED = false; };


__device__ __forceinline__ float f16_bits_to_f32(uint32_t h) {
    _Float16 v = __builtin_bit_cast(_Float16, (uint16_t)h);
    return (float)v;  // v_cvt_f32_f16: exact widening incl. subnormals
}

// the four bytes of v as floats (v_cvt_f32_ubyte0..3).  The empty asm
// hides the masked value's known bits from the optimiser, which would
// otherwise re-extract every field with v_bfe before converting.
__device__ __forceinline__ void ubytes(uint32_t v, float& a, float& b, float& c, float& d) {
    asm volatile("" : "+v"(v));
    a = (float)(v & 0xffu);
    b = (float)((v >> 8) & 0xffu);
    c = (float)((v >> 16) & 0xffu);
    d = (float)(v >> 24);
}

__device__ __forceinline__ uint32_t bfe(uint32_t v, uint32_t off, uint32_t w) {
    return __builtin_amdgcn_ubfe(v, off, w);
}

// v of the lane selected by DPP control CTRL (both 32-bit halves moved).
// Used only with every lane of the 8-lane group active.
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const int lo = __double2loint(v), hi = __double2hiint(v);
    const int l2 = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xf, 0xf, false);
    const int h2 = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xf, 0xf, false);
    return __hiloint2double(h2, l2);
}

// The row reduction's phase count: a row's chunk terms are summed as G
// partials (partial p: chunks p, p+G, ... in order, binary64 from 0),
// combined by the pairwise tree below.  G depends on the row length only
// (8, or 32 for rows longer than 128 chunks, whose long chains would
// otherwise leave few lanes per row busy), so every kernel reproduces it.
__host__ __device__ __forceinline__ int kq_phases(int NC) { return NC > 128 ? 32 : 8; }

// v of lane ^ 16 (both halves)
__device__ __forceinline__ double xor16_f64(double v) {
    const int lo = __shfl_xor(__double2loint(v), 16);
    const int hi = __shfl_xor(__double2hiint(v), 16);
    return __hiloint2double(hi, lo);
}

// Pairwise tree over the G = 8 or 32 partials held by consecutive lanes
// (every lane of the group active):
//   8: ((P0 + P1) + (P2 + P3)) + ((P4 + P5) + (P6 + P7))
//  32: ((S0 + S1) + (S2 + S3)) over the 8-lane sums S0..S3.
// A butterfly: each addition is commutative, so every lane of the group
// ends with the same bits.
__device__ __forceinline__ double phase_tree(double s, int G) {
    s = s + dpp_f64<0xB1>(s);    // quad_perm [1,0,3,2]: lane ^ 1
    s = s + dpp_f64<0x4E>(s);    // quad_perm [2,3,0,1]: lane ^ 2
    s = s + dpp_f64<0x141>(s);   // row_half_mirror: lane i <-> 7 - i (8 lanes)
    if (G == 32) {
        s = s + dpp_f64<0x140>(s);   // row_mirror: 8-lane halves of a 16-lane row
        s = s + xor16_f64(s);        // 16-lane rows 0 <-> 1, 2 <-> 3
    }
    return s;
}

// ------------------------------------------------------------ raw loads
// Weight bytes are read through explicit global-address-space pointers.
// A generic pointer (e.g. one read back from the LDS weight-base table)
// would make the compiler emit FLAT loads, which count against lgkmcnt as
// well as vmcnt: every LDS wait in the loop would then also wait for the
// whole weight prefetch.
#define KQ_GLOBAL __attribute__((address_space(1)))
typedef const uint8_t KQ_GLOBAL* wptr;

__device__ __forceinline__ wptr to_global(const uint8_t* p) { return (wptr)p; }

// 128-bit vectors: 16-byte aligned (Q4_K blocks are 144 B) and 4-byte
// aligned (Q6_K/Q2_K/type-42 blocks are only dword aligned;
// global_load_dwordx4 needs dword alignment only).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4a __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2a __attribute__((ext_vector_type(2), aligned(4)));

// Weight loads use the default cache policy.  The nontemporal policy
// (global_load ... nt) lifts a plain read stream on this GPU from about 6.4
// to 7.1 TB/s, but here neighbouring lanes read one cache line through
// different load instructions (a block's header and the two quant vectors
// of a 64-weight chunk), and with nt each of them fetches the line again:
// measured 2x slower for Q6_K, 1.2x for Q4_K.
template <typename V>
__device__ __forceinline__ V wload(wptr p) {
    return *reinterpret_cast<const KQ_GLOBAL V*>(p);
}

__device__ __forceinline__ uint4 ld16(wptr p) {
    const u32x4 v = wload<u32x4>(p);
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint4 ld16a4(wptr p) {
    const u32x4a v = wload<u32x4a>(p);
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint2 ld8a4(wptr p) {
    const u32x2a v = wload<u32x2a>(p);
    return make_uint2(v.x, v.y);
}
__device__ __forceinline__ uint32_t ld4(wptr p) {
    return wload<uint32_t>(p);
}
__device__ __forceinline__ uint32_t ld2(wptr p) {
    return wload<uint16_t>(p);
}

struct RawQ4 { uint4 hd, qa, qb; };
struct RawQ6 { uint32_t l[5], h[5], q[5], s[3], d; uint32_t sh; };
struct RawQ2 { uint4 q; uint2 s; uint32_t dd; };
struct RawNB { uint4 qa, qb; uint32_t s, dd; };
struct RawQ5 { uint4 hd, h0, h1, qa, qb; };
struct RawQ3 { uint32_t q[5], m[5], s[4]; uint32_t d, sh; };
struct RawQ8 { uint32_t w[17]; };

__device__ __forceinline__ RawQ4 load_q4k(wptr blk, int j) {
    RawQ4 r;
    r.hd = ld16(blk);
    r.qa = ld16(blk + 16 + 32 * j);
    r.qb = ld16(blk + 32 + 32 * j);
    return r;
}

// Q6_K blocks are 210 B, so odd blocks start 2 bytes off a dword.  Loads
// are dword-aligned and realigned with v_alignbit (shift 0 or 16).
__device__ __forceinline__ void load5(wptr p, uint32_t* o) {
    const uint4 v = ld16a4(p);
    o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
    o[4] = ld4(p + 16);
}

__device__ __forceinline__ RawQ6 load_q6k(wptr blk, int u) {
    RawQ6 r;
    const int h = u >> 1, is = u & 1;
    // realign by pointer arithmetic, which keeps the global address space
    const uint32_t mis = (uint32_t)reinterpret_cast<uintptr_t>(blk) & 3u;
    r.sh = mis * 8u;
    const wptr b4 = blk - mis;
    load5(b4 + 64 * h + 16 * is, r.l);
    load5(b4 + 64 * h + 32 + 16 * is, r.h);
    load5(b4 + 128 + 32 * h + 16 * is, r.q);
    // scales: 8 bytes from 192 + 8h.  A third dword is needed only when the
    // block is 2 bytes off; when aligned, dword 1 is re-read instead so the
    // last block of a tensor never reads past its 210 bytes.
    const wptr sp = b4 + 192 + 8 * h;
    r.s[0] = ld4(sp); r.s[1] = ld4(sp + 4); r.s[2] = ld4(sp + (r.sh ? 8 : 4));
    r.d = ld2(blk + 208);
    return r;
}

__device__ __forceinline__ RawQ2 load_q2k(wptr blk, int u) {
    RawQ2 r;
    const int s = u >> 1, h = u & 1;
    r.q = ld16a4(blk + 16 + 32 * s + 16 * h);
    r.s = ld8a4(blk + 8 * s);
    r.dd = ld4(blk + 80);
    return r;
}

// Q5_K (176 B, 16-byte aligned): header (d, dmin, scales), all of qh, and
// the 32 qs bytes of chunk j
__device__ __forceinline__ RawQ5 load_q5k(wptr blk, int j) {
    RawQ5 r;
    r.hd = ld16(blk);
    r.h0 = ld16(blk + 16);
    r.h1 = ld16(blk + 32);
    r.qa = ld16(blk + 48 + 32 * j);
    r.qb = ld16(blk + 64 + 32 * j);
    return r;
}

// Q3_K (110 B, blocks 2-byte aligned): chunk u = (s, h) reads 16 qs bytes
// at 32 + 32s + 16h, 16 hmask bytes at 16h, the 12 scale bytes at 96 and d
// at 108.  Dword-aligned loads realigned by v_alignbit; the fourth scale
// dword is needed only when the block is 2 bytes off (else dword 2 is read
// again), so the last block of a tensor is never read past its end.
__device__ __forceinline__ RawQ3 load_q3k(wptr blk, int u) {
    RawQ3 r;
    const int s = u >> 1, h = u & 1;
    const uint32_t mis = (uint32_t)reinterpret_cast<uintptr_t>(blk) & 3u;
    r.sh = mis * 8u;
    const wptr b4 = blk - mis;
    load5(b4 + 32 + 32 * s + 16 * h, r.q);
    load5(b4 + 16 * h, r.m);
    r.s[0] = ld4(b4 + 96); r.s[1] = ld4(b4 + 100); r.s[2] = ld4(b4 + 104);
    r.s[3] = ld4(b4 + (mis ? 108 : 104));
    r.d = ld2(blk + 108);
    return r;
}

// Q8_0: a 256-weight unit is eight 34-byte blocks (272 B, 16-byte aligned);
// chunk u is blocks 2u, 2u+1: 68 bytes from the dword-aligned offset 68u
__device__ __forceinline__ RawQ8 load_q80(wptr blk, int u) {
    RawQ8 r;
    const wptr p = blk + 68 * u;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint4 v = ld16a4(p + 16 * k);
        r.w[4 * k] = v.x; r.w[4 * k + 1] = v.y; r.w[4 * k + 2] = v.z; r.w[4 * k + 3] = v.w;
    }
    r.w[16] = ld4(p + 64);
    return r;
}

__device__ __forceinline__ RawNB load_nib(wptr blk, int u) {
    RawNB r;
    r.qa = ld16a4(blk + 16 + 32 * u);
    r.qb = ld16a4(blk + 32 + 32 * u);
    r.s = ld4(blk + 4 * u);
    r.dd = ld4(blk + 144);
    return r;
}

__device__ __forceinline__ uint32_t dw_of(const uint4& v, int k) {
    return k == 0 ? v.x : k == 1 ? v.y : k == 2 ? v.z : v.w;
}

__device__ __forceinline__ float i8f(uint32_t v, int e) {
    return (float)(int32_t)(int8_t)(uint8_t)(v >> (8 * e));
}

// The four words of step k (16 weights of each of the 4 runs of the chunk):
// byte = ((q ^ 0x20) << 2) = int8 4*(q - 32), q = lo4 | hi2 << 4.
__device__ __forceinline__ void q6k_words(const RawQ6& r, int k, uint32_t (&y)[4]) {
    const uint32_t sh = r.sh;
    const uint32_t L = __builtin_amdgcn_alignbit(r.l[k + 1], r.l[k], sh);
    const uint32_t H = __builtin_amdgcn_alignbit(r.h[k + 1], r.h[k], sh);
    const uint32_t Q = __builtin_amdgcn_alignbit(r.q[k + 1], r.q[k], sh) ^ 0xaaaaaaaau;
    y[0] = ((L << 2) & 0x3c3c3c3cu) | ((Q << 6) & 0xc0c0c0c0u);
    y[1] = ((H << 2) & 0x3c3c3c3cu) | ((Q << 4) & 0xc0c0c0c0u);
    y[2] = ((L >> 2) & 0x3c3c3c3cu) | ((Q << 2) & 0xc0c0c0c0u);
    y[3] = ((H >> 2) & 0x3c3c3c3cu) | (Q & 0xc0c0c0c0u);
}

// Q4_K / Q5_K 6-bit scale and min of sub-blocks 2j, 2j+1 from the 12
// scale bytes in words s0..s2 (stratum_q4k.h:57-65)
__device__ __forceinline__ void scale_min_pair(uint32_t s0, uint32_t s1, uint32_t s2, int j,
                                               uint32_t& sc1, uint32_t& m1, uint32_t& sc2,
                                               uint32_t& m2) {
    const bool lo = j < 2;
    const uint32_t ob = (uint32_t)((2 * j) & 3) * 8u;
    const uint32_t a_sc = lo ? s0 : s2;
    const uint32_t a_m = lo ? s1 : s2;
    const uint32_t w6 = lo ? 6u : 4u;
    const uint32_t om = lo ? 0u : 4u;
    const uint32_t wh = lo ? 0u : 2u;
    sc1 = bfe(a_sc, ob, w6) | (bfe(s0, ob + 6, wh) << 4);
    m1 = bfe(a_m, ob + om, w6) | (bfe(s1, ob + 6, wh) << 4);
    sc2 = bfe(a_sc, ob + 8, w6) | (bfe(s0, ob + 14, wh) << 4);
    m2 = bfe(a_m, ob + 8 + om, w6) | (bfe(s1, ob + 14, wh) << 4);
}

// The chunk term from the four 16-weight sums: d * s[t] * a_t in binary64.
__device__ __forceinline__ double q6k_combine(const RawQ6& r, int u, const float (&a)[4],
                                              double f6) {
    const int is = u & 1;
    const uint32_t sh = r.sh;
    // scales s[8h + is + 2t] sit at bytes is + 2t of the realigned pair
    const uint32_t S0 = __builtin_amdgcn_alignbit(r.s[1], r.s[0], sh);
    const uint32_t S1 = __builtin_amdgcn_alignbit(r.s[2], r.s[1], sh);
    const uint32_t dh = r.d;
    const double dq = (double)f16_bits_to_f32(dh) * f6;  // exact
    const uint32_t Sa = is ? (S0 >> 8) : S0;
    const uint32_t Sb = is ? (S1 >> 8) : S1;
    const double t0 = (dq * (double)(int8_t)(uint8_t)(Sa)) * (double)a[0];
    const double t1 = (dq * (double)(int8_t)(uint8_t)(Sa >> 16)) * (double)a[1];
    const double t2 = (dq * (double)(int8_t)(uint8_t)(Sb)) * (double)a[2];
    const double t3 = (dq * (double)(int8_t)(uint8_t)(Sb >> 16)) * (double)a[3];
    return (t0 + t1) + (t2 + t3);
}

}  // namespace

#endif  // KQ_BLOCKS_H
