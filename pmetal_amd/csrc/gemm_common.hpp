// Device code shared by the dequant-fused GEMM kernels (gemm.hip, gemm_kw.hip): operand types, direct global -> LDS copies,
// and the exact f16 operands built from the packed quants of each format.
#pragma once

#include "internal.hpp"

namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kGroups = 18;    // 16-byte items per activation row and half super-block
constexpr int kBlockBytes = 144;
// FMT 0: Q4_K (144 bytes: d, dmin, 12 scale bytes, 128 quant bytes); FMT 1: Q5_K (176 bytes: the same header, then 32 bytes
// qh with the fifth bits, then the 128 quant bytes; crates/pmetal-gguf/src/k_quants.rs:407-462)
template <int FMT>
struct BlockFmt {
    static constexpr int kBytes = FMT ? 176 : 144, kQs = FMT ? 48 : 16;
};

#define PMH_GPTR(p) ((const __attribute__((address_space(1))) void *)(p))
#define PMH_LPTR(p) ((__attribute__((address_space(3))) void *)(p))

// 16 bytes per lane from global memory to LDS: lane l lands at dst + 16 l (dst is wave-uniform).
__device__ __forceinline__ void dma16(const void *src, uint4 *dst) {
    __builtin_amdgcn_global_load_lds(PMH_GPTR(src), PMH_LPTR(dst), 16, 0, 0);
}

// Workgroup barrier that leaves the newest `keep` vector-memory requests in flight.  (__syncthreads() carries a
// release fence, which waits for every direct-to-LDS copy.)  The copies that the other waves will read are older
// than those, and this wave's own LDS reads have returned (lgkmcnt(0)) before another wave may refill a stage.
template <int KEEP>
__device__ __forceinline__ void barrier_keep() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070 | KEEP);  // vmcnt(KEEP) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ float f16_bits_to_f32(uint32_t h) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}
// The same where it multiplies a tile: behind the barrier the compiler multiplies and adds f32 numbers (v_fmac_f32, which two waves of a SIMD
// can issue at a time: 2.3 cycles each by two waves) and does not take d from its f16 bits in each of them (v_fma_mix_f32, 8 bytes long: 3.4).
__device__ __forceinline__ float tile_scale(float d) {
    asm("" : "+v"(d));
    return d;
}
__device__ __forceinline__ float bf16_to_f32(uint32_t h) { return __builtin_bit_cast(float, h << 16); }

__device__ __forceinline__ uint32_t bf16_rne_bits(const float v) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    return ((u & 0x7FFFFFFFu) > 0x7F800000u) ? ((u >> 16) | 0x40u) : ((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}

// 8 quants of one dword (low nibbles, then high nibbles) times their integer scales -> 8 exact f16 values:
// 0x6400 | q is the f16 1024 + q, and (1024 + q) * sc - 1024 * sc is exact in a packed f16 fma.  Built in four
// pieces, so that the pieces can be placed between matrix instructions.  k-step t selects the
// scales: GGML order multiplies the low nibbles by the first and the high nibbles by the second sub-block scale,
// REF order both by the scale of sub-block t / 4.
struct Dq {
    uint32_t lo, hi;
    half2_t r[4];
    __device__ __forceinline__ half8_t value() const { return half8_t{r[0][0], r[0][1], r[1][0], r[1][1], r[2][0], r[2][1], r[3][0], r[3][1]}; }
};
// Q5_K (FMT 1): bit 4 of every quant comes from `hq`.  GGML order: hq is the qh dword of the same four bytes, shifted so
// that bits 0 and 1 of each of its bytes belong to the low and the high nibble of the quant byte at the same place.  REF
// order: hq is the one qh byte whose bits 0..7 belong to the eight consecutive elements of this k-step (even elements =
// low nibbles): a multiplication spreads bits 0, 2, 4, 6 to bit 4 of bytes 0..3 (bit 2 i lands on 2 i + 4 + 6 i; the
// other partial products meet at most in pairs on bits that the mask drops, and their carries stop there).  Values up to
// 31 times scales up to 63 stay below 2048: exact in f16 like Q4_K's.
template <int ORDER, int FMT = 0>
__device__ __forceinline__ void dq_chunk(const int c, const int t, const uint32_t w, const half2_t (&sc2)[2], const half2_t (&off2)[2], Dq &d,
                                         const uint32_t hq = 0) {
    const int lo_s = ORDER == 0 ? (t >> 2) : 0, hi_s = ORDER == 0 ? (t >> 2) : 1;
    if (FMT == 1 && c == 0) {
        const uint32_t bit = ORDER == 0 ? ((hq & 0x55u) * 0x00410410u) & 0x10101010u : (hq & 0x01010101u) << 4;
        d.lo = (w & 0x0F0F0F0Fu) | bit;
        d.r[0] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, d.lo, 0x04010400u)), sc2[lo_s], off2[lo_s]);
    } else if (FMT == 1 && c == 1) {
        d.r[1] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, d.lo, 0x04030402u)), sc2[lo_s], off2[lo_s]);
        const uint32_t bit = ORDER == 0 ? (((hq >> 1) & 0x55u) * 0x00410410u) & 0x10101010u : (hq & 0x02020202u) << 3;
        d.hi = ((w >> 4) & 0x0F0F0F0Fu) | bit;
    } else if (c == 0) {
        d.lo = w & 0x0F0F0F0Fu;
        d.r[0] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, d.lo, 0x04010400u)), sc2[lo_s], off2[lo_s]);
    } else if (c == 1) {
        d.r[1] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, d.lo, 0x04030402u)), sc2[lo_s], off2[lo_s]);
        d.hi = (w >> 4) & 0x0F0F0F0Fu;
    } else if (c == 2) {
        d.r[2] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, d.hi, 0x04010400u)), sc2[hi_s], off2[hi_s]);
    } else {
        d.r[3] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, d.hi, 0x04030402u)), sc2[hi_s], off2[hi_s]);
    }
}

// -(dmin * mn) split exactly into an f16 head and tail (dmin has 11 significant bits, mn 6).
__device__ __forceinline__ void neg_min_split(const float dmin, const uint32_t mn, _Float16 &h, _Float16 &l) {
    const float p = -(dmin * (float)mn);  // exact in fp32
    h = (_Float16)p;
    l = (_Float16)(p - (float)h);
}

// Integers below 64, a byte each, as the f16 pair of the two that `pick` names: 0x64bb is 1024 + bb, so `bias` is -1024 (- 32: signed).
// The compiler reads halves of a pair by operand selection, so a scale for all lanes of a packed operation costs no move.
__device__ __forceinline__ half2_t byte_pair(const uint32_t bytes, const uint32_t pick, const float bias = -1024.0f) {
    return __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, bytes, pick)) + half2_t{(_Float16)bias, (_Float16)bias};
}
// m0 k and m1 k as f16 heads and tails (h0, h0, l0, l0, h1, h1, l1, l1), the operand that meets the activations' (H, L, H, L).  Exact: k has
// eleven bits and |m| at most seven, and what the head leaves is a multiple of k's last bit, which the fma keeps.
__device__ __forceinline__ half8_t heads_and_tails(const half2_t m, const half2_t k) {
    const half2_t h = m * k, l = __builtin_elementwise_fma(m, k, -h);
    return half8_t{h[0], h[0], l[0], l[0], h[1], h[1], l[1], l[1]};
}
__device__ __forceinline__ half2_t f16_twice(const uint32_t bits16) {  // of the low half
    return __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(bits16, bits16, 0x01000100u));
}
// (Decoding a lane's two scales and mins one by one in f32 took some 45 vector instructions a half super-block and row group, this takes
// 16: with the copies of a half spread over its k-steps the row kernels' 128-row forms take, us of a call at 14336 x 4096 M = 2048 before ->
// after, Q4_K 290 -> 280, Q5_K 318 -> 300, Q3_K 349 -> 325, Q2_K 316 -> 302; of the two the copies are 5 of Q4_K's 10.)
// Q4_K and Q5_K: the scales and mins of four sub-blocks (half H of the super-block), a byte each, from the twelve bytes y, z, w
// (6-bit fields, crates/pmetal/src/commands/quantize.rs:844-855).
template <int H>
__device__ __forceinline__ uint32_t scale_bytes(const uint32_t y, const uint32_t w) {
    return H == 0 ? y & 0x3F3F3F3Fu : (w & 0x0F0F0F0Fu) | ((y >> 2) & 0x30303030u);
}
template <int H>
__device__ __forceinline__ uint32_t min_bytes(const uint32_t z, const uint32_t w) {
    return H == 0 ? z & 0x3F3F3F3Fu : ((w >> 4) & 0x0F0F0F0Fu) | ((z >> 2) & 0x30303030u);
}

constexpr int kGroups16 = 20;  // activation items per row and half super-block: 16 operands and four of sub-block sums
template <int FMT>
struct Block16 {  // FMT 2: Q3_K, 3: Q2_K
    static constexpr int kBytes = FMT == 3 ? 84 : 110, kQs = FMT == 3 ? 16 : 32;
    static constexpr int kHdrPieces = FMT == 3 ? 2 : 3;           // per row and super-block
    static constexpr int kHdrRounds = (32 * kHdrPieces + 63) / 64;  // whole-wave copies
    static constexpr int kHdrStage = 64 * kHdrRounds;              // items of a wave's header stage
    static __device__ __forceinline__ uint32_t piece_off(int p) { return FMT == 3 ? (p == 0 ? 0u : 68u) : (p == 2 ? 94u : 16u * (uint32_t)p); }
};

constexpr int kQ6Bytes = 210, kQ6Groups = 16, kQ6Stage = 192;  // LDS items of a wave's quant stage: 128 ql + 64 qh

// The two operands of one k-step, built in eight pieces that are placed between matrix instructions: 1/32 of sc * nib and of
// 16 sc * (hi2 - 2), so that every multiplier and offset of a packed f16 fma is a number f16 holds (the kernels multiply d by 32).
// 0x6400 | nib is the f16 1024 + nib: times sc / 32, less 32 sc.  0x40 | hi2 as the upper byte is the f16 2 + hi2 / 2: times sc,
// less 3 sc.  All of it exact for |sc| <= 128.  22 vector instructions a k-step; an addition and a multiplication a pair, with the
// unscaled values, were 30.  The row kernel is bound by in-order issue at two waves a SIMD, the tile kernel by memory: us of a call, 30 -> 22,
// 4096 x 14336 M = 2048 419 -> 407, 14336 x 4096 M = 512 116 -> 113, M = 128 51.8 -> 50.0, M = 64 30.0 -> 29.4.
struct Dq6 {
    uint32_t nlo, nhi, hlo, hhi;
    half2_t r1[4], r2[4];
    __device__ __forceinline__ half8_t b1() const { return half8_t{r1[0][0], r1[0][1], r1[1][0], r1[1][1], r1[2][0], r1[2][1], r1[3][0], r1[3][1]}; }
    __device__ __forceinline__ half8_t b2() const { return half8_t{r2[0][0], r2[0][1], r2[1][0], r2[1][1], r2[2][0], r2[2][1], r2[3][0], r2[3][1]}; }
};
constexpr float kQ6OperandScale = 32.0f;
struct Q6Scales {  // of the low-nibble and of the high-nibble elements of four k-steps
    half2_t sc[2], sc32[2], off[2], off3[2];
    __device__ __forceinline__ void set(const half2_t lo, const half2_t hi) {
        const half2_t c32 = {(_Float16)0.03125f, (_Float16)0.03125f}, m32 = {(_Float16)-32.0f, (_Float16)-32.0f}, m3 = {(_Float16)-3.0f, (_Float16)-3.0f};
        sc[0] = lo, sc[1] = hi;
#pragma unroll
        for (int i = 0; i < 2; i++) sc32[i] = sc[i] * c32, off[i] = sc[i] * m32, off3[i] = sc[i] * m3;
    }
};
// qlw: the ql dword of the k-step; qhw: its qh dword already shifted by 2 g
__device__ __forceinline__ void dq6_chunk(const int c, const uint32_t qlw, const uint32_t qhw, const Q6Scales &s, Dq6 &d) {
    if (c == 0) d.nlo = qlw & 0x0F0F0F0Fu;
    if (c == 2) d.nhi = (qlw >> 4) & 0x0F0F0F0Fu;
    if (c == 4) d.hlo = (qhw & 0x03030303u) | 0x40404040u;
    if (c == 6) d.hhi = ((qhw >> 4) & 0x03030303u) | 0x40404040u;
    if (c < 4) {  // bytes (b0, b1) resp. (b2, b3) -> 0x64bb pairs
        const uint32_t v = __builtin_amdgcn_perm(0x64646464u, c < 2 ? d.nlo : d.nhi, (c & 1) ? 0x04030402u : 0x04010400u);
        d.r2[c] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, v), s.sc32[c >> 1], s.off[c >> 1]);
    } else {  // ... -> 0xbb00 pairs (selector 12 is a zero byte)
        const uint32_t v = __builtin_amdgcn_perm(0u, c < 6 ? d.hlo : d.hhi, (c & 1) ? 0x030C020Cu : 0x010C000Cu);
        d.r1[c - 4] = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, v), s.sc[(c - 4) >> 1], s.off3[(c - 4) >> 1]);
    }
}

// 8 int8 -> 8 exact f16: q + 128 as an unsigned byte b, 0x6400 | b is the f16 1024 + b, minus 1152.
__device__ __forceinline__ half8_t q8_operand(const uint32_t w0, const uint32_t w1) {
    const half2_t m1152 = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    const uint32_t u0 = w0 ^ 0x80808080u, u1 = w1 ^ 0x80808080u;
    const half2_t r0 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, u0, 0x04010400u)) + m1152;
    const half2_t r1 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, u0, 0x04030402u)) + m1152;
    const half2_t r2 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, u1, 0x04010400u)) + m1152;
    const half2_t r3 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, u1, 0x04030402u)) + m1152;
    return half8_t{r0[0], r0[1], r1[0], r1[1], r2[0], r2[1], r3[0], r3[1]};
}

typedef float float4_t __attribute__((ext_vector_type(4)));

// Two weights in one launch: the workgroups from second.first on belong to the second one.  Whether there is one is a bit of an
// argument that arrives with the wave (kHasSecond in `mode`, `flags` or `ybf16`): the kernel of a single weight asks for nothing more.
constexpr int kHasSecond = 256;
__device__ __forceinline__ void take_weight(const pmh::GemmSecond &second, int &flags, int &bx, const uint8_t *__restrict__ &W, void *__restrict__ &y,
                                            int &N) {
    if (flags & kHasSecond) {
        flags &= kHasSecond - 1;
        if (bx >= second.first) bx -= second.first, W = second.w, y = second.y, N = second.n;
    }
}

}  // namespace
