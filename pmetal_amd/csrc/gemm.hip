// Dequant-fused Q4_K, Q5_K, Q6_K and Q8_0 GEMM  Y[m,n] = sum_k X[m,k] * W[n,k]  on the gfx950 matrix cores, every wave
// owning its weight rows.  The text below describes Q4_K (Q5_K is the same kernel with the fifth bit of every quant
// taken from the block's qh bytes: FMT = 1); the Q6_K and Q8_0 kernels further down note their differences.
//
// W is the packed GGUF stream [n, k] of 144-byte super-blocks; a weight's value is what the reference's
// dequantize_q4k yields (crates/pmetal-gguf/src/k_quants.rs:358-404; element order REF or GGML as for the
// GEMV).  The reference has no fused kernel (it dequantizes on the CPU at load,
// crates/pmetal-models/src/weight_format.rs:299-303, and multiplies densely); this kernel is checked against
// exactly that, dequantize-then-matmul, to 1e-3.
//
// A wave owns 32 weight rows and dequantizes them straight into MFMA operand registers (no shared weight tile
// in LDS, no LDS writes by the waves at all); only the activations are shared by the waves of a workgroup.  A
// launch is cut along N, M and, for short activation batches, K into enough workgroups to fill the machine.
// The arithmetic is exact up to the fp32 accumulation: rounding d*sc*q - dmin*m to f16 or bf16 leaves a relative
// error per product that fails the element-wise 1e-3 gate on small outputs, so the MFMA multiplies integer tiles
// sc * q in f16 (<= 63 * 15 = 945; f16 holds integers to 2048) with activations scaled per row by a power of two
// into the f16 range (bf16 activations are exact there), the per-super-block factor d is applied to the fp32
// partial sums, and the min term is a K = 32 MFMA product of exact head + tail splits.
//
// Data movement uses direct global -> LDS loads only (no staging registers, no ds_write):
//   * activations: a pre-pass writes 16-byte items (8 f16) in the order the MFMA wants them,
//     xs[(2 sb + h) * 18 + grp][Mp], per half super-block h 16 operand groups (k-step t, lane half g) and two
//     groups of sub-block sums; a workgroup copies the 18 x BM items of a half super-block into one of two
//     LDS stages while it computes on the other (one barrier per half super-block);
//   * weights: each wave copies the 64 quant bytes per row of a half super-block (coalesced: four lanes per
//     row) two half super-blocks ahead, and the 16-byte headers one super-block ahead, into its private LDS
//     region; then every lane (row n = lane % 32, half g = lane / 32) reads back the 32 bytes it multiplies:
//     dword t of them holds the eight 4-bit quants of MFMA k-step t.  Which k they are is a property of the
//     element order, matched by the pre-pass:
//         GGML: k = 64 (2h + g) + 4t + e (low nibbles, sub-block 4h+2g), + 32 (high nibbles, sub-block 4h+2g+1)
//         REF : k = 32 (4h + 2g + t/4) + 4 (t%4) + e (low), + 16 (high), both sub-block 4h + 2g + t/4
// With a K split (grid.z > 1) the workgroups write fp32 partial tiles and a small kernel adds them in a fixed
// order, so the result does not depend on scheduling.
//
// What bounds it: every matrix instruction reads its 1 KiB activation fragment from LDS (a wave cannot reuse a
// fragment for a second group of weight rows without doubling the dequantization work per matrix instruction,
// which measured slower, as did one wave per SIMD with a 128 x 64 tile), so a 128-row workgroup is bound by the
// LDS read rate at about 60 % of the matrix peak.
#include "gemm_common.hpp"
#include "../../include/pmetal_hip.h"

namespace {


// ------------------------------------------------------------------------------------------------
// Pre-pass: a workgroup takes R activation rows m < Mp (R = 1: 512 threads on one row, for few rows; otherwise 1024 / R threads
// per row with the row index fastest across lanes, so that R lanes write 16 R contiguous bytes of every item row).  Bound by
// latency for few rows and by its scattered stores and the reads for many: the elements are read once and held (with a second read
// for the conversion, k = 14336, bf16: M = 16 6.0 -> 4.7 us, M = 512 18.1 -> 9.8, M = 2048 30.2 -> 26.5; f32 M = 2048 43 -> 30).
// rowscale[m] = 2^e with the row maximum * 2^-e in [2^9, 2^10) (bf16 activations are then exact in f16 and block sums stay below 2^15); rows >= M are zero.
// One thread per operand item: chunk u = 64 elements = sub-blocks 2u, 2u+1 (u = 4 sb + 2 h + g), k-step t.
// ORDER 0 / 1: Q4_K element orders REF / GGML (1 is also Q5_K's GGML order); ORDER 2: the Q6_K layout, ORDER 3: the
// natural order (Q8_0), both without block sums; ORDER 4: Q5_K's REF order, whose sub-block j holds its 32 elements as
// consecutive nibbles of 16 bytes, so k-step t of a chunk is elements 8 t .. 8 t + 7, the even ones (low nibbles) first;
// ORDER 5: Q2_K / Q3_K, whose qs byte 32 h + l holds elements 128 h + l + 32 s at bit 2 s: k-step t of lane half g is dword
// t / 2 of the bytes 16 g .. 16 g + 15 of a half with the shifts s = 2 (t % 2) (first run) and 2 (t % 2) + 1 (second run), and
// the sums are those of the four 16-element sub-blocks 4 (t % 2) + 2 (run) + g of the half: 20 items per half.
// ------------------------------------------------------------------------------------------------
template <bool XF32>
struct PrepRaw {  // the eight elements of an item as they lie in memory
    uint4 a, b;   // (bf16: all in a)
};

// NI > 0: k <= 8 NI NT / R; a thread's items stay in registers between the row maximum and the conversion.  NI = 0: any k.
template <bool XF32, int ORDER, int R, int NI>
__global__ __launch_bounds__(R == 1 ? 512 : 1024) void k_prep_rw(const void *__restrict__ xg, int64_t k, int M, int Mp,
                                                                  float *__restrict__ rowscale, uint4 *__restrict__ xs, uint32_t *__restrict__ clear,
                                                                  int n_clear) {  // (n_clear: at most 512 words)
    constexpr int NT = R == 1 ? 512 : 1024, JN = NT / R, NWV = NT / 64;
    constexpr int kGroups = ORDER == 5 ? 20 : (ORDER == 2 || ORDER == 3 ? 16 : 18);  // items per half super-block and row (shadows the Q4_K constant)
    const int tid = threadIdx.x, lane = tid & 63, r = tid % R, j = tid / R;
    const int m = blockIdx.x * R + r;
    const bool live = m < M;
    const int64_t items = k / 8;
    if (blockIdx.x == 0 && tid < n_clear) clear[tid] = 0;
    // an item's two runs of four elements (lo, hi), its half super-block and its operand group
    auto place = [&](const int64_t q, int64_t &lo, int64_t &hi, int64_t &half, int &t, int &g) __attribute__((always_inline)) {
        if (ORDER == 2 || ORDER == 3) {  // half = 128 elements, 16 items
            half = q >> 4;
            t = (int)(q & 15) >> 1, g = (int)q & 1;
            if (ORDER == 2) {  // Q6_K: low nibbles at 32 g + 4 t, high nibbles 64 further
                lo = 128 * half + 32 * g + 4 * t;
                hi = lo + 64;
            } else {  // Q8_0: the natural order, 8 consecutive elements
                lo = 128 * half + 16 * t + 8 * g;
                hi = lo + 4;
            }
        } else {
            const int64_t u = q >> 3;
            t = (int)(q & 7), g = (int)u & 1;
            half = u >> 1;
            lo = ORDER == 5   ? 128 * half + 64 * (t & 1) + 16 * g + 4 * (t >> 1)
                 : ORDER == 4 ? 64 * u + 8 * t
                              : (ORDER == 0 ? 64 * u + 32 * (t >> 2) + 4 * (t & 3) : 64 * u + 4 * t);
            hi = lo + (ORDER == 4 ? 4 : (ORDER == 0 ? 16 : 32));
        }
    };
    auto fetch = [&](const int64_t q) __attribute__((always_inline)) {
        int64_t lo, hi, half;
        int t, g;
        place(q, lo, hi, half, t, g);
        PrepRaw<XF32> w;
        if (XF32) {
            const float *row = reinterpret_cast<const float *>(xg) + (int64_t)m * k;
            w.a = *reinterpret_cast<const uint4 *>(row + lo), w.b = *reinterpret_cast<const uint4 *>(row + hi);
        } else {
            const uint16_t *row = reinterpret_cast<const uint16_t *>(xg) + (int64_t)m * k;
            const uint2 a = *reinterpret_cast<const uint2 *>(row + lo), b = *reinterpret_cast<const uint2 *>(row + hi);
            w.a = make_uint4(a.x, a.y, b.x, b.y);
        }
        return w;
    };
    auto widen = [&](const PrepRaw<XF32> &w, float (&v)[8]) __attribute__((always_inline)) {
        const uint32_t a[8] = {w.a.x, w.a.y, w.a.z, w.a.w, XF32 ? w.b.x : 0u, XF32 ? w.b.y : 0u, XF32 ? w.b.z : 0u, XF32 ? w.b.w : 0u};
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = XF32 ? __builtin_bit_cast(float, a[i]) : bf16_to_f32(i & 1 ? a[i / 2] >> 16 : a[i / 2] & 0xFFFFu);
    };
    auto max_with = [&](float amax, const PrepRaw<XF32> &w) __attribute__((always_inline)) {
        float v[8];
        widen(w, v);
#pragma unroll
        for (int i = 0; i < 8; i++) amax = __builtin_fmaxf(amax, __builtin_fabsf(v[i]));
        return amax;
    };
    __shared__ float red[NWV][R];
    float amax = 0.0f;
    constexpr int kHeld = NI > 0 ? NI : 1;
    PrepRaw<XF32> held[kHeld];
    if (live) {
        if (NI > 0) {
#pragma unroll
            for (int i = 0; i < kHeld; i++) {
                const int64_t q = j + i * JN;
                held[i] = fetch(q < items ? q : items - 1);  // (past the row: its last item again, which does not change the maximum)
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < kHeld; i++) amax = max_with(amax, held[i]);
        } else {
            for (int64_t q = j; q < items; q += JN) amax = max_with(amax, fetch(q));
        }
    }
    for (int off = 32; off >= R; off >>= 1) amax = __builtin_fmaxf(amax, __shfl_xor(amax, off));
    if (lane < R) red[tid >> 6][lane] = amax;
    __syncthreads();
    amax = red[0][r];
#pragma unroll
    for (int w = 1; w < NWV; w++) amax = __builtin_fmaxf(amax, red[w][r]);
    const int eb = (int)((__builtin_bit_cast(uint32_t, amax) >> 23) & 0xFFu);  // amax in [2^(eb-127), 2^(eb-126))
    int e = eb - 126 - 10;
    e = e < -126 ? -126 : (e > 126 ? 126 : e);
    if (eb == 255) e = 0;  // inf / NaN: let them through
    const float up = __builtin_bit_cast(float, (uint32_t)(127 + e) << 23);
    if (j == 0) rowscale[m] = up;
    const float down = live ? 1.0f / up : 0.0f;  // exact: a power of two

    auto emit = [&](const int64_t q, const PrepRaw<XF32> &raw) __attribute__((always_inline)) {
        int64_t lo, hi, half;
        int t, g;
        place(q, lo, hi, half, t, g);
        float v[8];
        if (live) {
            widen(raw, v);
        } else {
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = 0.0f;
        }
        if (ORDER == 4) {  // eight consecutive elements: the even ones, then the odd ones
            const float e[8] = {v[0], v[2], v[4], v[6], v[1], v[3], v[5], v[7]};
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = e[i];
        }
        half8_t h;
        float slo = 0.0f, shi = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            h[i] = (_Float16)(v[i] * down);
            if (i < 4) slo += (float)h[i];
            else shi += (float)h[i];
        }
        const size_t base = (size_t)(half * kGroups) * Mp + m;
        xs[base + (size_t)(t * 2 + g) * Mp] = __builtin_bit_cast(uint4, h);
        if (ORDER == 2 || ORDER == 3) return;  // Q6_K and Q8_0 have no min term: no block sums
        // sums of the two sub-blocks of the chunk over its 8 k-steps (8 lanes, R apart)
        float s0, s1;
        if (ORDER == 5) {
            // the first runs of the k-steps of one parity are one 16-element sub-block, their second runs another:
            // k-step 0 ends up with the sums for t % 2 == 0 (item 16 + g), k-step 1 with those for t % 2 == 1 (item 18 + g)
            slo += __shfl_xor(slo, 2 * R), shi += __shfl_xor(shi, 2 * R);
            slo += __shfl_xor(slo, 4 * R), shi += __shfl_xor(shi, 4 * R);
            if (t < 2) {
                const _Float16 h0 = (_Float16)slo, h1 = (_Float16)shi;
                const _Float16 l0 = (_Float16)(slo - (float)h0), l1 = (_Float16)(shi - (float)h1);
                const half8_t item = {h0, l0, h0, l0, h1, l1, h1, l1};
                xs[base + (size_t)(16 + 2 * t + g) * Mp] = __builtin_bit_cast(uint4, item);
            }
            return;
        }
        if (ORDER == 0 || ORDER == 4) {  // sub-block 2u: k-steps 0..3 (low and high nibbles), 2u+1: k-steps 4..7
            float s = slo + shi;
            s += __shfl_xor(s, R);
            s += __shfl_xor(s, 2 * R);
            s0 = s;
            s1 = __shfl_down(s, 4 * R);
        } else {  // sub-block 2u: the low nibbles of all k-steps, 2u+1: the high nibbles
            slo += __shfl_xor(slo, R), shi += __shfl_xor(shi, R);
            slo += __shfl_xor(slo, 2 * R), shi += __shfl_xor(shi, 2 * R);
            slo += __shfl_xor(slo, 4 * R), shi += __shfl_xor(shi, 4 * R);
            s0 = slo, s1 = shi;
        }
        if (t == 0) {  // exact head + tail split of each sum; item (H0, L0, H0, L0, H1, L1, H1, L1)
            const _Float16 h0 = (_Float16)s0, h1 = (_Float16)s1;
            const _Float16 l0 = (_Float16)(s0 - (float)h0), l1 = (_Float16)(s1 - (float)h1);
            const half8_t item = {h0, l0, h0, l0, h1, l1, h1, l1};
            xs[base + (size_t)(16 + g) * Mp] = __builtin_bit_cast(uint4, item);
        }
    };
    if (NI > 0) {
#pragma unroll
        for (int i = 0; i < kHeld; i++) {
            const int64_t q = j + i * JN;
            if (q < items) emit(q, held[i]);  // (the eight threads of a chunk together)
        }
    } else {
        for (int64_t q = j; q < items; q += JN) emit(q, live ? fetch(q) : PrepRaw<XF32>{});
    }
}

// ------------------------------------------------------------------------------------------------
// main kernel
// ------------------------------------------------------------------------------------------------
// Epilogue shared by the kernels below: a workgroup's BM x 32 NW tile of Y (256 columns for 8 waves) goes through LDS so that it leaves as
// whole rows (16 bytes per lane, 512 bytes or 1 KiB contiguous per row) instead of 2- or 4-byte pieces per lane.
// Every wave holds 32 columns (lane % 32) of all BM rows: C layout of v_mfma_f32_32x32x*: rows
// 8 (r / 4) + 4 (lane / 32) + r % 4 of block i.  mode 0: y f32, 1: y bf16 (both scaled by rowscale), 2: fp32
// partial tile of split z.  Must be reached by all threads of the workgroup, with no copies into LDS in flight.
constexpr int kTilePad = 16;  // bytes added to an LDS row: rows 4 apart (the two lane halves) then lie in different banks
template <int MB, int NW = 8>
constexpr size_t tile_lds_bytes() {
    return (size_t)32 * MB * (32 * NW * 4 + kTilePad);
}


struct __attribute__((packed, aligned(2))) u32x4_a2 {
    uint32_t x, y, z, w;
};

template <int MB, int NW = 8>
__device__ __forceinline__ void store_tile(const float16_t (&acc)[MB], uint4 *smem, const int wave, const int col, const int g,
                                           const int m0, const int n0, const int M, const int N, const int Mp,
                                           const float *__restrict__ rowscale, void *__restrict__ yg,
                                           float *__restrict__ partial, const int mode, const int z) {
    constexpr int BM = 32 * MB;
    constexpr int kCols = 32 * NW;                    // weight rows of the workgroup = columns of its tile of Y
    constexpr int kRowStride = kCols * 4 + kTilePad;  // the LDS tile is fp32, not yet scaled
    uint8_t *tile = reinterpret_cast<uint8_t *>(smem);
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int ml = 32 * i + 8 * (r >> 2) + 4 * g + (r & 3);
            *reinterpret_cast<float *>(tile + ml * kRowStride + (32 * wave + col) * 4) = acc[i][r];
        }
    __syncthreads();
    // one 16-byte store per trip and lane: 4 (fp32) or 8 (bf16) consecutive outputs of one row
    const int per = mode == 1 ? 8 : 4, chunks = kCols / per, esize = mode == 1 ? 2 : 4;
    uint8_t *out = mode == 2 ? reinterpret_cast<uint8_t *>(partial) + (size_t)z * Mp * N * 4 : reinterpret_cast<uint8_t *>(yg);
    const bool rows_aligned = ((size_t)N * esize) % 16 == 0;
    for (int idx = threadIdx.x; idx < BM * chunks; idx += blockDim.x) {
        const int ml = idx / chunks, c = idx % chunks;
        const int m = m0 + ml, n = n0 + c * per;
        if (m >= M || n >= N) continue;
        const float scale = mode == 2 ? 1.0f : rowscale[m];
        const float4 *src = reinterpret_cast<const float4 *>(tile + ml * kRowStride + c * per * 4);
        float v[8];
        const float4 lo = src[0];
        v[0] = lo.x * scale, v[1] = lo.y * scale, v[2] = lo.z * scale, v[3] = lo.w * scale;
        uint4 pack;
        if (mode == 1) {
            const float4 hi = src[1];
            v[4] = hi.x * scale, v[5] = hi.y * scale, v[6] = hi.z * scale, v[7] = hi.w * scale;
            pack = make_uint4(bf16_rne_bits(v[0]) | (bf16_rne_bits(v[1]) << 16), bf16_rne_bits(v[2]) | (bf16_rne_bits(v[3]) << 16),
                              bf16_rne_bits(v[4]) | (bf16_rne_bits(v[5]) << 16), bf16_rne_bits(v[6]) | (bf16_rne_bits(v[7]) << 16));
        } else {
            pack = make_uint4(__builtin_bit_cast(uint32_t, v[0]), __builtin_bit_cast(uint32_t, v[1]),
                              __builtin_bit_cast(uint32_t, v[2]), __builtin_bit_cast(uint32_t, v[3]));
        }
        uint8_t *dst = out + ((size_t)m * N + n) * esize;
        if (rows_aligned && n + per <= N) {
            // Y is not read again by this launch: a streaming store keeps it from pushing the activation items and the
            // other row blocks' weights out of the caches (a partial tile is read back by the reduction: an ordinary store)
            if (mode == 2) *reinterpret_cast<uint4 *>(dst) = pack;
            else __builtin_nontemporal_store(u32x4{pack.x, pack.y, pack.z, pack.w}, reinterpret_cast<u32x4 *>(dst));
        } else if (n + per <= N) {  // rows that start off 16-byte boundaries (N ragged): the same store at the alignment of an output
            *reinterpret_cast<u32x4_a2 *>(dst) = u32x4_a2{pack.x, pack.y, pack.z, pack.w};
        } else {
            for (int e = 0; e < per && n + e < N; e++) {
                if (mode == 1) reinterpret_cast<uint16_t *>(dst)[e] = (uint16_t)bf16_rne_bits(v[e]);
                else reinterpret_cast<float *>(dst)[e] = v[e];
            }
        }
    }
}

// per-thread constants of the copy roles; a wave owns NR groups of 32 weight rows
template <int MB, int NR, int NW>
struct Lane {
    static constexpr int BM = 32 * MB, kThreads = 64 * NW;
    static constexpr int kARounds = (kGroups * BM + kThreads - 1) / kThreads;
    int wave, col, g;
    uint32_t q_off[NR][2];     // byte offset of this lane's quant piece of round r from the workgroup's first row
    uint32_t h_off[NR];        // ... of this lane's header
    uint32_t qh_off[NR];       // ... of this lane's piece of the fifth bits (Q5_K: row lane / 2, piece lane % 2)
    uint32_t a_off[kARounds];  // item offset of this lane's activation item of round i from (group 0, row m0)
};

template <int MB, int NR>
struct Acc {
    float16_t acc[NR][MB], part[NR][MB];
    u32x4 hdr[NR];  // headers of the current super-block: d | dmin << 16, then the 12 scale bytes
    uint32_t qh[NR][8];  // Q5_K: the 32 qh bytes of the current super-block of this lane's row
};


// One half super-block H of one wave.  The restrict qualifiers say what the copies in flight cannot touch:
// operand reads from a_cur / q_cur need not wait for the direct loads into a_nxt / q_nxt / hb.
//   a_cur / a_nxt: activation stages (18 x BM items)      q_cur / q_nxt: this wave's quant pieces (NR x 128 items)
//   hb: this wave's headers (NR x 64 items)       qhs: Q5_K, this wave's fifth bits (NR x 32 rows x 2 items)
//   xs_nxt: item (group 0, row m0) of the next half super-block    wq_nxt / wh_nxt: first row of the workgroup at
//   the next half's quant bytes / the next super-block's header
template <int ORDER, int MB, int NR, int NW, int H, int FMT>
__device__ __forceinline__ void rw_half(const uint4 *__restrict__ a_cur, uint4 *__restrict__ a_nxt,
                                        const uint4 *__restrict__ q_cur, uint4 *__restrict__ q_nxt, uint4 *__restrict__ hb,
                                        uint4 *__restrict__ qhs, const uint4 *__restrict__ xs_nxt, const uint8_t *__restrict__ wq_nxt,
                                        const uint8_t *__restrict__ wh_nxt, const Lane<MB, NR, NW> &L, Acc<MB, NR> &R) {
    constexpr int BM = 32 * MB, kThreads = 64 * NW;
    const int col = L.col, g = L.g;
    if (H == 0) {
#pragma unroll
        for (int rg = 0; rg < NR; rg++) {
            const uint4 hv = hb[rg * 64 + col];
            R.hdr[rg] = u32x4{hv.x, hv.y, hv.z, hv.w};
            if (FMT == 1) {  // both halves of the super-block take their fifth bits from these registers
                const uint4 ha = qhs[rg * 64 + 2 * col], hb2 = qhs[rg * 64 + 2 * col + 1];
                R.qh[rg][0] = ha.x, R.qh[rg][1] = ha.y, R.qh[rg][2] = ha.z, R.qh[rg][3] = ha.w;
                R.qh[rg][4] = hb2.x, R.qh[rg][5] = hb2.y, R.qh[rg][6] = hb2.z, R.qh[rg][7] = hb2.w;
            }
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the headers are in registers before their buffer is refilled
    }
    // The copies for the next half super-block in five steps, of which 128 rows take one behind each of the first k-steps: all at the start of
    // a half they held its waves up for 610 to 970 of 3930 cycles (a copy passes the address unit in 16, and a workgroup issues 56), and no matrix
    // instruction ran meanwhile.  Fewer rows have no k-steps to spare behind which the copies could come back.  The quant copies must be the newest
    // requests of this half: the barrier at its end waits for all but them.
    auto copies = [&](const int step) __attribute__((always_inline)) {
        if (step < 3) {
#pragma unroll
            for (int i = 2 * step; i < 2 * step + 2; i++)
                if (i < Lane<MB, NR, NW>::kARounds && i * kThreads + L.wave * 64 < kGroups * BM) dma16(xs_nxt + L.a_off[i], a_nxt + i * kThreads + L.wave * 64);
        }
        if (H == 0 && step == 2) {
#pragma unroll
            for (int rg = 0; rg < NR; rg++) {
                dma16(wh_nxt + L.h_off[rg], hb + rg * 64);
                if (FMT == 1) dma16(wh_nxt + L.qh_off[rg], qhs + rg * 64);
            }
        }
        if (step >= 3) {
#pragma unroll
            for (int rg = 0; rg < NR; rg++) dma16(wq_nxt + L.q_off[rg][step - 3], q_nxt + rg * 128 + (step - 3) * 64);
        }
    };
    static_assert(Lane<MB, NR, NW>::kARounds <= 6, "two rounds of activation copies a step");
    if (MB < 4) {
#pragma unroll
        for (int step = 0; step < 5; step++) {
            if (step == 3) __builtin_amdgcn_sched_barrier(0);  // (what follows is quant copies)
            copies(step);
        }
        __builtin_amdgcn_sched_barrier(0);
    }

    // Scales and mins of sub-blocks j0 = 4 H + 2 g and j0 + 1.  The min term: (-h, -h, -l, -l) against the activations' (H, L, H, L), all four cross products of the exact head + tail
    // splits, straight into the accumulators (after the eight k-steps).
    const uint32_t pick = g ? 0x04030402u : 0x04010400u;
    const half2_t m1024 = {(_Float16)-1024.0f, (_Float16)-1024.0f};
    half2_t sc2[NR][2], off2[NR][2];
    half8_t br[NR];
    uint32_t qd[NR][8];
    // this lane's 32 quant bytes per row group: pieces 2g and 2g+1 of row col (the copy swizzles the four pieces of
    // a row by (row / 4) % 4 so that 16 consecutive rows read conflict-free)
    const int sw = (col >> 2) & 3;
#pragma unroll
    for (int rg = 0; rg < NR; rg++) {
        const uint4 qa = q_cur[rg * 128 + col * 4 + ((2 * g) ^ sw)], qb = q_cur[rg * 128 + col * 4 + ((2 * g + 1) ^ sw)];
        qd[rg][0] = qa.x, qd[rg][1] = qa.y, qd[rg][2] = qa.z, qd[rg][3] = qa.w;
        qd[rg][4] = qb.x, qd[rg][5] = qb.y, qd[rg][6] = qb.z, qd[rg][7] = qb.w;
        const u32x4 h = R.hdr[rg];
        const half2_t sc = byte_pair(scale_bytes<H>(h.y, h.w), pick), mn = byte_pair(min_bytes<H>(h.z, h.w), pick);
        sc2[rg][0] = half2_t{sc[0], sc[0]}, sc2[rg][1] = half2_t{sc[1], sc[1]};
        off2[rg][0] = sc2[rg][0] * m1024, off2[rg][1] = sc2[rg][1] * m1024;  // exact: sc <= 63
        br[rg] = heads_and_tails(mn, -f16_twice(h.x >> 16));
    }

    // Q5_K: where k-step t finds its fifth bits.  GGML order: qh dword t (the same four bytes as quant dword t), bits
    // j0 = 4 H + 2 g (low nibbles) and j0 + 1 (high nibbles) of every byte.  REF order: byte 4 j0 + t of qh.
    auto fifth = [&](int rg, int t) -> uint32_t {
        if (FMT == 0) return 0u;
        if (ORDER == 1) return R.qh[rg][t] >> (uint32_t)(4 * H + 2 * g);
        const uint32_t dw = g ? R.qh[rg][4 * H + 2 + (t >> 2)] : R.qh[rg][4 * H + (t >> 2)];
        return dw >> (8 * (t & 3));  // (the decoder masks the byte)
    };

    // Software pipeline, written in issue order (a wave issues in order, so the order here is the schedule):
    // the activation fragments of k-step t + 1 are requested before the products of k-step t, and the weights of
    // k-step t + 1 are dequantized in pieces between those products.
    constexpr int kSlots = MB * NR, kChunks = 4 * NR;
    half8_t af[2][MB];
    Dq dq[NR];
#pragma unroll
    for (int i = 0; i < MB; i++) af[0][i] = __builtin_bit_cast(half8_t, a_cur[g * BM + 32 * i + col]);
#pragma unroll
    for (int rg = 0; rg < NR; rg++)
#pragma unroll
        for (int c = 0; c < 4; c++) dq_chunk<ORDER, FMT>(c, 0, qd[rg][0], sc2[rg], off2[rg], dq[rg], fifth(rg, 0));
#pragma unroll
    for (int t = 0; t < 8; t++) {
        half8_t b[NR];
#pragma unroll
        for (int rg = 0; rg < NR; rg++) b[rg] = dq[rg].value();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int rg = 0; rg < NR; rg++) {
                const half8_t a = af[t & 1][i];
                if (H == 0 && t == 0) {  // first product of a super-block starts from zero
                    float16_t z;
#pragma unroll
                    for (int r = 0; r < 16; r++) z[r] = 0.0f;
                    R.part[rg][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b[rg], z, 0, 0, 0);
                } else {
                    R.part[rg][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b[rg], R.part[rg][i], 0, 0, 0);
                }
                if (t < 7) {
                    const int slot = i * NR + rg;
#pragma unroll
                    for (int ch = slot * kChunks / kSlots; ch < (slot + 1) * kChunks / kSlots; ch++)
                        dq_chunk<ORDER, FMT>(ch % 4, t + 1, qd[ch / 4][t + 1], sc2[ch / 4], off2[ch / 4], dq[ch / 4], fifth(ch / 4, t + 1));
                }
                if (i == 0 && rg == 0) {
                    // the next step's fragments are requested behind the first product of this step: the wait in
                    // front of that product then covers only fragments requested a whole step ago
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int ii = 0; ii < MB; ii++)
                        af[(t + 1) & 1][ii] = __builtin_bit_cast(half8_t, a_cur[(t < 7 ? (t + 1) * 2 + g : 16 + g) * BM + 32 * ii + col]);
                }
                if (MB >= 4 && i == MB - 1 && rg == NR - 1 && t < 5) copies(t);
                __builtin_amdgcn_sched_barrier(0);
            }
    }
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int rg = 0; rg < NR; rg++) R.acc[rg][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[0][i], br[rg], R.acc[rg][i], 0, 0, 0);
    if (H == 1) {
#pragma unroll
        for (int rg = 0; rg < NR; rg++) {
            const float d = f16_bits_to_f32(R.hdr[rg].x & 0xFFFFu);
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) R.acc[rg][i][r] = __builtin_fmaf(d, R.part[rg][i][r], R.acc[rg][i][r]);
        }
    }
}

// grid (ceil(N / (32 NR NW)), Mp / BM, splits); workgroup z works on super-blocks [z * chunk, min(spr, (z + 1) * chunk)).
// mode 0: y f32 [M][N], 1: y bf16, 2: fp32 partial tiles [splits][Mp][N] (not yet scaled by rowscale)
//
// Copies in flight: the activation stage of the next half super-block (it comes from L2) and the quant pieces of
// the next two (they come from HBM): three quant stages per wave, rotated.  Within a half super-block the
// activation copies are requested before the quant copies, so waiting until only the 2 NR newest requests are
// outstanding leaves exactly the quant copies for the half after next in flight.
template <int ORDER, int MB, int NR, int NW, int FMT = 0>
__global__ __launch_bounds__(64 * NW, MB * NR <= 1 && NW <= 8 ? 2 : 1) void k_qgemm_rw(
    const uint8_t *__restrict__ W, const uint4 *__restrict__ xs, const float *__restrict__ rowscale, void *__restrict__ yg,
    float *__restrict__ partial, int M, int Mp, int N, int spr, int chunk, int mode, const pmh::GemmSecond second) {
    constexpr int BM = 32 * MB, kThreads = 64 * NW, kRows = 32 * NR * NW;
    constexpr int kBlockBytes = BlockFmt<FMT>::kBytes, kQs = BlockFmt<FMT>::kQs;
    extern __shared__ uint4 smem[];
    uint4 *a0 = smem, *a1 = a0 + kGroups * BM, *qbase = a1 + kGroups * BM, *hb = qbase + 3 * NW * NR * 128;
    uint4 *qhb = hb + NW * NR * 64;  // Q5_K only
    const int tid = threadIdx.x;
    Lane<MB, NR, NW> L;
    L.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    L.col = lane & 31, L.g = lane >> 5;
    int bx = (int)blockIdx.x;
    take_weight(second, mode, bx, W, yg, N);
    const int n0 = bx * kRows, m0 = blockIdx.y * BM;
    const int nw0 = n0 + 32 * NR * L.wave;  // first weight row of this wave
    const int sb0 = blockIdx.z * chunk;
    const int cnt = spr - sb0 < chunk ? spr - sb0 : chunk;
    const uint32_t row_bytes = (uint32_t)spr * kBlockBytes;
    auto row_off = [&](int row) {  // byte offset of a row of this wave from the workgroup's first row; rows past N repeat the last
        int n = nw0 + row;
        n = n < N ? n : N - 1;
        return (uint32_t)(n - n0) * row_bytes;
    };
#pragma unroll
    for (int rg = 0; rg < NR; rg++) {
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int row = 16 * r + (lane >> 2);
            L.q_off[rg][r] = row_off(32 * rg + row) + 16u * (uint32_t)((lane & 3) ^ ((row >> 2) & 3));
        }
        L.h_off[rg] = row_off(32 * rg + (lane & 31));
        L.qh_off[rg] = row_off(32 * rg + (lane >> 1)) + 16u + 16u * (uint32_t)(lane & 1);
    }
#pragma unroll
    for (int i = 0; i < Lane<MB, NR, NW>::kARounds; i++) {
        const int idx = tid + i * kThreads;
        L.a_off[i] = (uint32_t)((idx / BM) * Mp + idx % BM);
    }
    // this wave's three quant stages (rotated: qa is read, qb is next, qc receives the copies) and its headers
    uint4 *qa = qbase + L.wave * (NR * 128), *qb = qa + NW * NR * 128, *qc = qb + NW * NR * 128;
    uint4 *hw = hb + L.wave * (NR * 64), *qhw = qhb + L.wave * (NR * 64);
    const uint8_t *wblk = W + (size_t)n0 * row_bytes;

    Acc<MB, NR> R;
#pragma unroll
    for (int rg = 0; rg < NR; rg++)
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) R.acc[rg][i][r] = 0.0f, R.part[rg][i][r] = 0.0f;

    // prologue: headers, both halves' quant pieces and the first activation stage of super-block sb0
    {
        const uint8_t *blk = wblk + (size_t)sb0 * kBlockBytes;
#pragma unroll
        for (int rg = 0; rg < NR; rg++) {
            dma16(blk + L.h_off[rg], hw + rg * 64);
            if (FMT == 1) dma16(blk + L.qh_off[rg], qhw + rg * 64);
#pragma unroll
            for (int r = 0; r < 2; r++) {
                dma16(blk + kQs + L.q_off[rg][r], qa + rg * 128 + r * 64);
                dma16(blk + kQs + 64 + L.q_off[rg][r], qb + rg * 128 + r * 64);
            }
        }
        const uint4 *xa = xs + (size_t)(sb0 * 2 * kGroups) * Mp + m0;
#pragma unroll
        for (int i = 0; i < Lane<MB, NR, NW>::kARounds; i++)
            if (i * kThreads + L.wave * 64 < kGroups * BM) dma16(xa + L.a_off[i], a0 + i * kThreads + L.wave * 64);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();

    for (int s = 0; s < cnt; s++) {
        const int sb = sb0 + s;
        const int sbn = sb + 1 < spr ? sb + 1 : spr - 1;  // the copies for "the next super-block" stay inside the matrix
        const uint8_t *blkn = wblk + (size_t)sbn * kBlockBytes;
        rw_half<ORDER, MB, NR, NW, 0, FMT>(a0, a1, qa, qc, hw, qhw, xs + (size_t)((sb * 2 + 1) * kGroups) * Mp + m0, blkn + kQs, blkn, L, R);
        barrier_keep<2 * NR>();
        rw_half<ORDER, MB, NR, NW, 1, FMT>(a1, a0, qb, qa, hw, qhw, xs + (size_t)(sbn * 2 * kGroups) * Mp + m0, blkn + kQs + 64, nullptr, L, R);
        barrier_keep<2 * NR>();
        // two half super-blocks on: (qa, qb, qc) <- (qc, qa, qb)
        uint4 *t = qc;
        qc = qb, qb = qa, qa = t;
    }
    // the last copies (for a half super-block past the end) have landed and every wave is done with the stages
    static_assert(NR == 1, "the tile store takes one group of weight rows per wave");
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();
    store_tile<MB, NW>(R.acc[0], smem, L.wave, L.col, L.g, m0, n0, M, N, Mp, rowscale, yg, partial, mode, blockIdx.z);
}

// ------------------------------------------------------------------------------------------------
// Q2_K and Q3_K (crates/pmetal-gguf/src/k_quants.rs:230-266, :281-355): sixteen 16-element sub-blocks per super-block,
// two-bit quants, qs byte 32 h + l = elements 128 h + l + 32 s at bit 2 s.  The Q4_K kernel's structure with these
// differences:
//   * a half super-block of a row is 32 bytes of qs: lane (n, g) takes bytes 16 g .. 16 g + 15; dword t / 2 of them gives
//     k-step t its eight values, four at shift 4 (t % 2) (sub-block 8 h + 4 (t % 2) + g) and four at 4 (t % 2) + 2
//     (sub-block 8 h + 4 (t % 2) + 2 + g): four scales per lane and half, one quant copy per wave and half;
//   * Q2_K: value d (sc & 15) q - dmin (sc >> 4), q in 0..3: the B tile is (sc & 15) q, and the min terms of the lane's
//     four sub-blocks are two K = 16 products of exact head + tail splits (activation items 16 + g and 18 + g);
//   * Q3_K: value d s' (q3 - 4) with s' = sc6 - 32 and q3 = q | hbit << 2, hbit = bit 4 h + s of hmask[l]: the B tile is
//     s' q3 = (1024 + q3) s' - 1024 s' (1028 s' would not be an f16 number), and the - 4 d s' of every element leaves with the
//     sub-block sums of the activations, exactly as Q2_K's mins do (coefficient 4 d s' in place of dmin m);
//   * blocks are 84 / 110 bytes, so rows start at 4- / 2-byte aligned addresses (the direct-to-LDS loads take them); the
//     header pieces of a row are Q2_K: bytes 0..15 (scales) and 68..83 (d, dmin in the last dword); Q3_K: 0..31 (hmask) and
//     94..109 (scales in bytes 2..13 of the piece, d in 14..15).
// ------------------------------------------------------------------------------------------------

template <int FMT, int MB, int H>
__device__ __forceinline__ void rw16_half(const uint4 *__restrict__ a_cur, uint4 *__restrict__ a_nxt, const uint4 *__restrict__ q_cur,
                                          uint4 *__restrict__ q_nxt, uint4 *__restrict__ hs, const uint4 *__restrict__ xs_nxt,
                                          const uint8_t *__restrict__ wq_nxt, const uint8_t *__restrict__ wh_nxt, const int wave,
                                          const int col, const int g, const uint32_t q_off, const uint32_t (&h_off)[Block16<FMT>::kHdrRounds],
                                          const uint32_t *a_off, float16_t (&acc)[MB], float16_t (&part)[MB], uint32_t (&hdr)[8],
                                          uint32_t (&hm)[4], uint32_t &dbits) {
    using B = Block16<FMT>;
    constexpr int BM = 32 * MB, kThreads = 512, kARounds = (kGroups16 * BM + kThreads - 1) / kThreads;
    if (H == 0) {
        // this row's header pieces into registers, then their stage is refilled with the next super-block's
        if (FMT == 3) {
            const uint4 sc = hs[col * 2], dd = hs[col * 2 + 1];
            hdr[0] = sc.x, hdr[1] = sc.y, hdr[2] = sc.z, hdr[3] = sc.w;
            dbits = dd.w;  // d | dmin << 16
        } else {
            const uint4 m0 = hs[col * 3], m1 = hs[col * 3 + 1], sd = hs[col * 3 + 2];
            // the lane's hmask bytes 16 g + 4 dw .. + 3 (both halves of the super-block use them)
            hm[0] = g ? m1.x : m0.x, hm[1] = g ? m1.y : m0.y, hm[2] = g ? m1.z : m0.z, hm[3] = g ? m1.w : m0.w;
            // the twelve scale bytes as three dwords (they start two bytes into the piece), d behind them
            hdr[0] = __builtin_amdgcn_alignbit(sd.y, sd.x, 16), hdr[1] = __builtin_amdgcn_alignbit(sd.z, sd.y, 16);
            hdr[2] = __builtin_amdgcn_alignbit(sd.w, sd.z, 16);
            dbits = sd.w >> 16;
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    }
    // in steps behind k-steps or all at the start, as in the Q4_K kernel; the quant copy must be the newest request of this half
    auto copies = [&](const int step) __attribute__((always_inline)) {
        if (step < 3) {
#pragma unroll
            for (int i = 2 * step; i < 2 * step + 2; i++)
                if (i < kARounds && i * kThreads + wave * 64 < kGroups16 * BM) dma16(xs_nxt + a_off[i], a_nxt + i * kThreads + wave * 64);
        }
        if (H == 0 && step == 2) {
#pragma unroll
            for (int r = 0; r < B::kHdrRounds; r++) dma16(wh_nxt + h_off[r], hs + 64 * r);
        }
        if (step == 3) dma16(wq_nxt + q_off, q_nxt);
    };
    static_assert(kARounds <= 6, "two rounds of activation copies a step");
    if (MB < 4) {
#pragma unroll
        for (int step = 0; step < 4; step++) {
            if (step == 3) __builtin_amdgcn_sched_barrier(0);  // (what follows is quant copies)
            copies(step);
        }
        __builtin_amdgcn_sched_barrier(0);
    }

    // this lane's 16 quant bytes: piece g of row col
    const uint4 qv = q_cur[col * 2 + g];
    const uint32_t qd[4] = {qv.x, qv.y, qv.z, qv.w};
    // scales (and mins) of the lane's four sub-blocks j = 8 H + 4 sp + 2 lh + g, index 2 sp + lh
    half2_t sc2[4], off2[4];
    half8_t br[2];  // what a sub-block subtracts per unit of its activation sum, negated: -dmin m (Q2_K), -4 d s' (Q3_K)
    const uint32_t pick = g ? 0x04030401u : 0x04020400u;  // bytes g and g + 2
    const half2_t m1024 = {(_Float16)-1024.0f, (_Float16)-1024.0f}, m4 = {(_Float16)-4.0f, (_Float16)-4.0f};
#pragma unroll
    for (int sp = 0; sp < 2; sp++) {
        half2_t sc;
        if (FMT == 3) {  // byte j of the sixteen: low nibble scale, high nibble min
            sc = byte_pair(hdr[2 * H + sp] & 0x0F0F0F0Fu, pick);
            br[sp] = heads_and_tails(byte_pair((hdr[2 * H + sp] >> 4) & 0x0F0F0F0Fu, pick), -f16_twice(dbits >> 16));
        } else {
            // sc6 of sub-block j: low nibble (j < 8) or high nibble (j >= 8) of byte j % 8, bits 4..5 = bits
            // 2 (j / 4) of byte 8 + j % 4
            sc = byte_pair(((hdr[sp] >> (4 * H)) & 0x0F0F0F0Fu) | (((hdr[2] >> (2 * (2 * H + sp))) & 0x03030303u) << 4), pick, -1056.0f);
            br[sp] = heads_and_tails(sc * m4, f16_twice(dbits));
        }
        sc2[2 * sp] = half2_t{sc[0], sc[0]}, sc2[2 * sp + 1] = half2_t{sc[1], sc[1]};
        off2[2 * sp] = sc2[2 * sp] * m1024, off2[2 * sp + 1] = sc2[2 * sp + 1] * m1024;  // exact: |sc| <= 32
    }
    // operand of k-step t: dword t / 2, the two-bit fields at 4 (t % 2) and 4 (t % 2) + 2 (Q3_K: bit 2 from hmask)
    auto operand = [&](int t) -> half8_t {
        const int dw = t >> 1, sp = t & 1;
        uint32_t lo = (qd[dw] >> (4 * sp)) & 0x03030303u, hi = (qd[dw] >> (4 * sp + 2)) & 0x03030303u;
        if (FMT == 2) {
            const uint32_t m = hm[dw] >> (4 * H + 2 * sp);
            lo |= (m & 0x01010101u) << 2, hi |= (m & 0x02020202u) << 1;
        }
        const half2_t r0 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, lo, 0x04010400u)), sc2[2 * sp], off2[2 * sp]);
        const half2_t r1 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, lo, 0x04030402u)), sc2[2 * sp], off2[2 * sp]);
        const half2_t r2 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, hi, 0x04010400u)), sc2[2 * sp + 1], off2[2 * sp + 1]);
        const half2_t r3 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, hi, 0x04030402u)), sc2[2 * sp + 1], off2[2 * sp + 1]);
        return half8_t{r0[0], r0[1], r1[0], r1[1], r2[0], r2[1], r3[0], r3[1]};
    };
    half8_t af[2][MB];
#pragma unroll
    for (int i = 0; i < MB; i++) af[0][i] = __builtin_bit_cast(half8_t, a_cur[g * BM + 32 * i + col]);
    half8_t b = operand(0);
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const half8_t bt = b;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < MB; i++) {
            const half8_t a = af[t & 1][i];
            if (H == 0 && t == 0) {  // first product of a super-block starts from zero
                float16_t z;
#pragma unroll
                for (int r = 0; r < 16; r++) z[r] = 0.0f;
                part[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, bt, z, 0, 0, 0);
            } else {
                part[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, bt, part[i], 0, 0, 0);
            }
            if (i == 0) {
                // the next step's fragments (after the last step: the first sums item) and its operand
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int ii = 0; ii < MB; ii++)
                    af[(t + 1) & 1][ii] = __builtin_bit_cast(half8_t, a_cur[(t < 7 ? (t + 1) * 2 + g : 16 + g) * BM + 32 * ii + col]);
                if (t < 7) b = operand(t + 1);
            }
            if (MB >= 4 && i == MB - 1 && t < 4) copies(t);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    {
        // sum terms of the lane's four sub-blocks: exact head + tail splits (h, h, l, l) against the sums' (H, L, H, L), pairs
        // (sp, 0), (sp, 1)
#pragma unroll
        for (int sp = 0; sp < 2; sp++) {
#pragma unroll
            for (int i = 0; i < MB; i++) {
                const half8_t a = sp == 0 ? af[0][i] : __builtin_bit_cast(half8_t, a_cur[(18 + g) * BM + 32 * i + col]);
                acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, br[sp], acc[i], 0, 0, 0);
            }
        }
    }
    if (H == 1) {
        const float d = f16_bits_to_f32(dbits & 0xFFFFu);
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][r] = __builtin_fmaf(d, part[i][r], acc[i][r]);
    }
}

// grid and modes as k_qgemm_rw; eight waves of 32 weight rows
template <int FMT, int MB>
__global__ __launch_bounds__(512, MB <= 1 ? 2 : 1) void k_qgemm_rw16(const uint8_t *__restrict__ W, const uint4 *__restrict__ xs,
                                                                      const float *__restrict__ rowscale, void *__restrict__ yg,
                                                                      float *__restrict__ partial, int M, int Mp, int N, int spr, int chunk,
                                                                      int mode, const pmh::GemmSecond second) {
    using B = Block16<FMT>;
    constexpr int BM = 32 * MB, NW = 8, kThreads = 512, kRows = 256, kARounds = (kGroups16 * BM + kThreads - 1) / kThreads;
    extern __shared__ uint4 smem[];
    uint4 *a0 = smem, *a1 = a0 + kGroups16 * BM, *qbase = a1 + kGroups16 * BM, *hb = qbase + 3 * NW * 64;
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63, col = lane & 31, g = lane >> 5;
    int bx = (int)blockIdx.x;
    take_weight(second, mode, bx, W, yg, N);
    const int n0 = bx * kRows, m0 = blockIdx.y * BM;
    const int nw0 = n0 + 32 * wave;  // first weight row of this wave
    const int sb0 = blockIdx.z * chunk;
    const int cnt = spr - sb0 < chunk ? spr - sb0 : chunk;
    const uint32_t row_bytes = (uint32_t)spr * B::kBytes;
    auto row_off = [&](int row) {  // byte offset of a row of this wave from the workgroup's first row; rows past N repeat the last
        int n = nw0 + row;
        n = n < N ? n : N - 1;
        return (uint32_t)(n - n0) * row_bytes;
    };
    // quant copy: lane -> (row lane / 2, piece lane % 2); header copies: item lane + 64 r -> (row item / P, piece item % P)
    const uint32_t q_off = row_off(lane >> 1) + 16u * (uint32_t)(lane & 1);
    uint32_t h_off[B::kHdrRounds];
#pragma unroll
    for (int r = 0; r < B::kHdrRounds; r++) {
        int item = lane + 64 * r;
        item = item < 32 * B::kHdrPieces ? item : 32 * B::kHdrPieces - 1;  // (the copies past the last item repeat it into the stage's padding)
        h_off[r] = row_off(item / B::kHdrPieces) + B::piece_off(item % B::kHdrPieces);
    }
    uint32_t a_off[kARounds];
#pragma unroll
    for (int i = 0; i < kARounds; i++) {
        const int idx = tid + i * kThreads;
        a_off[i] = (uint32_t)((idx / BM) * Mp + idx % BM);
    }
    uint4 *qa = qbase + wave * 64, *qb = qa + NW * 64, *qc = qb + NW * 64;
    uint4 *hw = hb + wave * B::kHdrStage;
    const uint8_t *wblk = W + (size_t)n0 * row_bytes;

    float16_t acc[MB], part[MB];
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = 0.0f, part[i][r] = 0.0f;
    uint32_t hdr[8] = {0, 0, 0, 0, 0, 0, 0, 0}, hm[4] = {0, 0, 0, 0}, dbits = 0;

    {  // prologue: headers, both halves' quant pieces and the first activation stage of super-block sb0
        const uint8_t *blk = wblk + (size_t)sb0 * B::kBytes;
#pragma unroll
        for (int r = 0; r < B::kHdrRounds; r++) dma16(blk + h_off[r], hw + 64 * r);
        dma16(blk + B::kQs + q_off, qa);
        dma16(blk + B::kQs + 32 + q_off, qb);
        const uint4 *xa = xs + (size_t)(sb0 * 2 * kGroups16) * Mp + m0;
#pragma unroll
        for (int i = 0; i < kARounds; i++)
            if (i * kThreads + wave * 64 < kGroups16 * BM) dma16(xa + a_off[i], a0 + i * kThreads + wave * 64);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();

    for (int s = 0; s < cnt; s++) {
        const int sb = sb0 + s;
        const int sbn = sb + 1 < spr ? sb + 1 : spr - 1;  // the copies for "the next super-block" stay inside the matrix
        const uint8_t *blkn = wblk + (size_t)sbn * B::kBytes;
        rw16_half<FMT, MB, 0>(a0, a1, qa, qc, hw, xs + (size_t)((sb * 2 + 1) * kGroups16) * Mp + m0, blkn + B::kQs, blkn, wave, col, g, q_off,
                              h_off, a_off, acc, part, hdr, hm, dbits);
        barrier_keep<1>();
        rw16_half<FMT, MB, 1>(a1, a0, qb, qa, hw, xs + (size_t)(sbn * 2 * kGroups16) * Mp + m0, blkn + B::kQs + 32, nullptr, wave, col, g, q_off,
                              h_off, a_off, acc, part, hdr, hm, dbits);
        barrier_keep<1>();
        uint4 *t = qc;  // two half super-blocks on: (qa, qb, qc) <- (qc, qa, qb)
        qc = qb, qb = qa, qa = t;
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();
    store_tile<MB, NW>(acc, smem, wave, col, g, m0, n0, M, N, Mp, rowscale, yg, partial, mode, blockIdx.z);
}

template <int FMT, int MB>
constexpr size_t rw16_lds_bytes() {
    const size_t stages = (size_t)(2 * kGroups16 * 32 * MB + 8 * (3 * 64 + Block16<FMT>::kHdrStage)) * 16;
    return stages > tile_lds_bytes<MB, 8>() ? stages : tile_lds_bytes<MB, 8>();
}

// ------------------------------------------------------------------------------------------------
// Q6_K (crates/pmetal-gguf/src/k_quants.rs:474-496: 210-byte super-blocks: ql[128] low nibbles, qh[64] top two
// bits, 16 int8 scales, f16 d; value d * sc * (q - 32)).  Same structure as the Q4_K kernel, with these differences:
//   * sc * (q - 32) can reach 4096 and is not always exact in f16, so it is split where the storage splits it,
//     q - 32 = 16 (hi2 - 2) + nib, into two exact tiles  B1 = (16 sc) (hi2 - 2)  and  B2 = sc * nib  (1/32 of each) that multiply
//     the same activation fragment one after the other (a fragment read from LDS feeds two matrix instructions);
//   * no min term; one scale per 16 elements;
//   * a half super-block of a row is 64 bytes of ql and 32 of qh; lane (n, g) multiplies ql bytes 32 g .. 32 g + 31
//     (dword t: low nibbles = elements 32 g + 4 t + e of the half, high nibbles 64 further) with the qh bytes
//     4 t + e (two-bit field g for the low, 2 + g for the high nibbles);
//   * super-blocks are only 2-byte aligned; the direct-to-LDS loads take such addresses.
// ------------------------------------------------------------------------------------------------

template <int MB>
struct LaneQ6 {
    static constexpr int BM = 32 * MB, kThreads = 512;
    static constexpr int kARounds = kQ6Groups * BM / kThreads;
    static_assert(kQ6Groups * BM % kThreads == 0, "the activation stage must divide among the threads");
    int wave, col, g;
    uint32_t ql_off[2], qh_off, h_off;  // byte offsets of this lane's pieces from the workgroup's first row
    uint32_t a_off[kARounds];
};

template <int MB>
struct AccQ6 {
    float16_t acc[MB], part[MB];
    u32x4 sc;    // the 16 int8 scales of the current super-block
    uint32_t d;  // f16 bits of d
};


template <int MB, int H>
__device__ __forceinline__ void rw_half_q6(const uint4 *__restrict__ a_cur, uint4 *__restrict__ a_nxt,
                                           const uint4 *__restrict__ q_cur, uint4 *__restrict__ q_nxt, uint4 *__restrict__ hb,
                                           const uint4 *__restrict__ xs_nxt, const uint8_t *__restrict__ wq_nxt,
                                           const uint8_t *__restrict__ wh_nxt, const LaneQ6<MB> &L, AccQ6<MB> &R) {
    constexpr int BM = 32 * MB, kThreads = 512;
    const int col = L.col, g = L.g;
    if (H == 0) {
        const uint4 sv = hb[col], dv = hb[32 + col];  // bytes 192..207 and 194..209 of the super-block
        R.sc = u32x4{sv.x, sv.y, sv.z, sv.w};
        R.d = dv.w >> 16;
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the header is in registers before its buffer is refilled
    }
    // In steps behind k-steps or all at the start, as in the Q4_K kernel.  The three quant copies, two half super-blocks ahead (ql bytes
    // 64 H .., qh bytes 128 + 32 H .. of that super-block), stay the newest requests (see barrier_keep).
    auto copies = [&](const int step) __attribute__((always_inline)) {
        if (step < 2) {
#pragma unroll
            for (int i = 2 * step; i < 2 * step + 2; i++)
                if (i < LaneQ6<MB>::kARounds) dma16(xs_nxt + L.a_off[i], a_nxt + i * kThreads + L.wave * 64);
        }
        if (H == 0 && step == 2) dma16(wh_nxt + L.h_off, hb);
        if (step == 3 || step == 4) dma16(wq_nxt + 64 * H + L.ql_off[step - 3], q_nxt + (step - 3) * 64);
        if (step == 5) dma16(wq_nxt + 32 * H + L.qh_off, q_nxt + 128);
    };
    static_assert(LaneQ6<MB>::kARounds <= 4, "two rounds of activation copies a step");
    if (MB < 4) {
#pragma unroll
        for (int step = 0; step < 6; step++) {
            if (step == 3) __builtin_amdgcn_sched_barrier(0);  // (what follows is quant copies)
            copies(step);
        }
        __builtin_amdgcn_sched_barrier(0);
    }

    // this lane's 32 ql bytes and the 32 qh bytes of its row (pieces swizzled by the copy for conflict-free reads)
    const int sw = (col >> 2) & 3, sw2 = (col >> 3) & 1;
    const uint4 qa = q_cur[col * 4 + ((2 * g) ^ sw)], qb = q_cur[col * 4 + ((2 * g + 1) ^ sw)];
    const uint4 ha = q_cur[128 + col * 2 + sw2], hc = q_cur[128 + col * 2 + (1 ^ sw2)];
    const uint32_t qd[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
    const uint32_t hs = 2u * (uint32_t)g;
    const uint32_t hd[8] = {ha.x >> hs, ha.y >> hs, ha.z >> hs, ha.w >> hs, hc.x >> hs, hc.y >> hs, hc.z >> hs, hc.w >> hs};
    // scales 8 H + 2 g + t / 4 (low nibbles) and 8 H + 4 + 2 g + t / 4 (high nibbles)
    const uint32_t wlo = (H == 0 ? R.sc.x : R.sc.z) >> (16u * (uint32_t)g), whi = (H == 0 ? R.sc.y : R.sc.w) >> (16u * (uint32_t)g);
    half2_t sc[2][2];  // [k-step / 4][low, high]
#pragma unroll
    for (int th = 0; th < 2; th++) {
        const _Float16 lo = (_Float16)(float)(int)(int8_t)(wlo >> (8 * th)), hi = (_Float16)(float)(int)(int8_t)(whi >> (8 * th));
        sc[th][0] = half2_t{lo, lo}, sc[th][1] = half2_t{hi, hi};
    }
    Q6Scales sv;
    sv.set(sc[0][0], sc[0][1]);

    // software pipeline in issue order, as in the Q4_K kernel; every fragment feeds two matrix instructions
    constexpr int kSlots = 2 * MB;
    half8_t af[2][MB];
    Dq6 dq;
#pragma unroll
    for (int i = 0; i < MB; i++) af[0][i] = __builtin_bit_cast(half8_t, a_cur[g * BM + 32 * i + col]);
#pragma unroll
    for (int c = 0; c < 8; c++) dq6_chunk(c, qd[0], hd[0], sv, dq);
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const half8_t b1 = dq.b1(), b2 = dq.b2();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int slot = 0; slot < kSlots; slot++) {
            const int i = slot >> 1;
            const half8_t a = af[t & 1][i];
            if (H == 0 && t == 0 && (slot & 1) == 0) {  // first product of a super-block starts from zero
                float16_t z;
#pragma unroll
                for (int r = 0; r < 16; r++) z[r] = 0.0f;
                R.part[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b1, z, 0, 0, 0);
            } else {
                R.part[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, (slot & 1) ? b2 : b1, R.part[i], 0, 0, 0);
            }
            if (t < 7) {
#pragma unroll
                for (int ch = slot * 8 / kSlots; ch < (slot + 1) * 8 / kSlots; ch++) {
                    if (t == 3 && ch == 0) sv.set(sc[1][0], sc[1][1]);
                    dq6_chunk(ch, qd[t + 1], hd[t + 1], sv, dq);
                }
                if (slot == 0) {
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int ii = 0; ii < MB; ii++)
                        af[(t + 1) & 1][ii] = __builtin_bit_cast(half8_t, a_cur[((t + 1) * 2 + g) * BM + 32 * ii + col]);
                }
            }
            if (MB >= 4 && slot == kSlots - 1 && t < 6) copies(t);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (H == 1) {
        const float d = kQ6OperandScale * f16_bits_to_f32(R.d);
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) R.acc[i][r] = __builtin_fmaf(d, R.part[i][r], R.acc[i][r]);
    }
}

// grid and modes as for k_qgemm_rw; 8 waves = 256 weight rows per workgroup
template <int MB>
__global__ __launch_bounds__(512, 1) void k_qgemm_rw_q6(const uint8_t *__restrict__ W, const uint4 *__restrict__ xs,
                                                         const float *__restrict__ rowscale, void *__restrict__ yg,
                                                         float *__restrict__ partial, int M, int Mp, int N, int spr, int chunk,
                                                         int mode, const pmh::GemmSecond second) {
    constexpr int BM = 32 * MB, kThreads = 512, NW = 8;
    extern __shared__ uint4 smem[];
    uint4 *a0 = smem, *a1 = a0 + kQ6Groups * BM, *qbase = a1 + kQ6Groups * BM, *hb = qbase + 3 * NW * kQ6Stage;
    const int tid = threadIdx.x;
    LaneQ6<MB> L;
    L.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    L.col = lane & 31, L.g = lane >> 5;
    int bx = (int)blockIdx.x;
    take_weight(second, mode, bx, W, yg, N);
    const int n0 = bx * 256, m0 = blockIdx.y * BM;
    const int nw0 = n0 + 32 * L.wave;
    const int sb0 = blockIdx.z * chunk;
    const int cnt = spr - sb0 < chunk ? spr - sb0 : chunk;
    const uint32_t row_bytes = (uint32_t)spr * kQ6Bytes;
    auto row_off = [&](int row) {  // rows past N repeat the last
        int n = nw0 + row;
        n = n < N ? n : N - 1;
        return (uint32_t)(n - n0) * row_bytes;
    };
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const int row = 16 * r + (lane >> 2);
        L.ql_off[r] = row_off(row) + 16u * (uint32_t)((lane & 3) ^ ((row >> 2) & 3));
    }
    {
        const int row = lane >> 1;
        L.qh_off = row_off(row) + 128u + 16u * (uint32_t)((lane & 1) ^ ((row >> 3) & 1));
    }
    L.h_off = row_off(lane & 31) + (lane < 32 ? 192u : 194u);
#pragma unroll
    for (int i = 0; i < LaneQ6<MB>::kARounds; i++) {
        const int idx = tid + i * kThreads;
        L.a_off[i] = (uint32_t)((idx / BM) * Mp + idx % BM);
    }
    uint4 *qa = qbase + L.wave * kQ6Stage, *qb = qa + NW * kQ6Stage, *qc = qb + NW * kQ6Stage;
    uint4 *hw = hb + L.wave * 64;
    const uint8_t *wblk = W + (size_t)n0 * row_bytes;

    AccQ6<MB> R;
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) R.acc[i][r] = 0.0f, R.part[i][r] = 0.0f;

    {
        const uint8_t *blk = wblk + (size_t)sb0 * kQ6Bytes;
        dma16(blk + L.h_off, hw);
#pragma unroll
        for (int r = 0; r < 2; r++) {
            dma16(blk + L.ql_off[r], qa + r * 64);
            dma16(blk + 64 + L.ql_off[r], qb + r * 64);
        }
        dma16(blk + L.qh_off, qa + 128);
        dma16(blk + 32 + L.qh_off, qb + 128);
        const uint4 *xa = xs + (size_t)(sb0 * 2 * kQ6Groups) * Mp + m0;
#pragma unroll
        for (int i = 0; i < LaneQ6<MB>::kARounds; i++) dma16(xa + L.a_off[i], a0 + i * kThreads + L.wave * 64);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();

    for (int s = 0; s < cnt; s++) {
        const int sb = sb0 + s;
        const int sbn = sb + 1 < spr ? sb + 1 : spr - 1;
        const uint8_t *blkn = wblk + (size_t)sbn * kQ6Bytes;
        rw_half_q6<MB, 0>(a0, a1, qa, qc, hw, xs + (size_t)((sb * 2 + 1) * kQ6Groups) * Mp + m0, blkn, blkn, L, R);
        barrier_keep<3>();
        rw_half_q6<MB, 1>(a1, a0, qb, qa, hw, xs + (size_t)(sbn * 2 * kQ6Groups) * Mp + m0, blkn, nullptr, L, R);
        barrier_keep<3>();
        uint4 *t = qc;
        qc = qb, qb = qa, qa = t;
    }

    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the last copies (past the end) have landed
    __syncthreads();
    store_tile<MB>(R.acc, smem, L.wave, L.col, L.g, m0, n0, M, N, Mp, rowscale, yg, partial, mode, blockIdx.z);
}

// ------------------------------------------------------------------------------------------------
// Q8_0 (crates/pmetal-gguf/src/quantize.rs:268-300: 34-byte blocks of 32: f16 d, 32 int8; value d * q).  The int8
// quants are exact in f16, so the B tile is q itself and d, one per 32 elements, multiplies the fp32 partial
// sum of two k-steps.  That is 16 fp32 FMAs per matrix instruction pair and output block: this kernel is bound
// by its VALU work, not by the matrix pipe.  A block is 34 bytes, so nothing in a row is aligned to more than
// 2 bytes: every lane (row n, half g) loads its own 8 quants per k-step and the scales straight from global
// memory into registers, one half super-block (four blocks) ahead; the activations go through LDS as in the
// kernels above (natural element order).
// ------------------------------------------------------------------------------------------------
struct __attribute__((packed, aligned(2))) q8_u32x2 {
    uint32_t x, y;
};
typedef uint16_t q8_u16 __attribute__((aligned(2)));

struct Q8Half {       // one lane's share of four blocks
    uint32_t q[4][2][2];  // [block][k-step of the block][dword]
    uint32_t d[4];        // f16 bits
};

__device__ __forceinline__ void q8_load(const uint8_t *p, const int g, Q8Half &h) {  // p: the lane's row at the half
#pragma unroll
    for (int b = 0; b < 4; b++) {
        h.d[b] = *reinterpret_cast<const q8_u16 *>(p + 34 * b);
#pragma unroll
        for (int tt = 0; tt < 2; tt++) {
            const q8_u32x2 v = *reinterpret_cast<const q8_u32x2 *>(p + 34 * b + 2 + 16 * tt + 8 * g);
            h.q[b][tt][0] = v.x, h.q[b][tt][1] = v.y;
        }
    }
}


template <int MB>
__device__ __forceinline__ void rw_half_q8(const uint4 *__restrict__ a_cur, uint4 *__restrict__ a_nxt,
                                           const uint4 *__restrict__ xs_nxt, const uint8_t *w_nxt, const Q8Half &cur,
                                           Q8Half &nxt, const LaneQ6<MB> &L, float16_t (&acc)[MB]) {
    constexpr int BM = 32 * MB, kThreads = 512;
    const int col = L.col, g = L.g;
    // `cur` was requested a whole half super-block ago and is the only thing still outstanding; waiting for it
    // here, before the new requests go out, keeps that wait from covering them too
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
#pragma unroll
    for (int i = 0; i < LaneQ6<MB>::kARounds; i++) dma16(xs_nxt + L.a_off[i], a_nxt + i * kThreads + L.wave * 64);
    __builtin_amdgcn_sched_barrier(0);  // the 12 register loads below stay the newest requests (see barrier_keep)
    q8_load(w_nxt, g, nxt);
    __builtin_amdgcn_sched_barrier(0);

    half8_t af[2][MB];
#pragma unroll
    for (int i = 0; i < MB; i++) af[0][i] = __builtin_bit_cast(half8_t, a_cur[g * BM + 32 * i + col]);
#pragma unroll
    for (int b = 0; b < 4; b++) {
        float16_t part[MB];
#pragma unroll
        for (int tt = 0; tt < 2; tt++) {
            const int t = 2 * b + tt;
            const half8_t bop = q8_operand(cur.q[b][tt][0], cur.q[b][tt][1]);
#pragma unroll
            for (int i = 0; i < MB; i++) {
                if (tt == 0) {
                    float16_t z;
#pragma unroll
                    for (int r = 0; r < 16; r++) z[r] = 0.0f;
                    part[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[t & 1][i], bop, z, 0, 0, 0);
                } else {
                    part[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[t & 1][i], bop, part[i], 0, 0, 0);
                }
                if (i == 0 && t < 7) {  // the next step's fragments, behind the first product of this step
#pragma unroll
                    for (int ii = 0; ii < MB; ii++)
                        af[(t + 1) & 1][ii] = __builtin_bit_cast(half8_t, a_cur[((t + 1) * 2 + g) * BM + 32 * ii + col]);
                }
            }
        }
        const float d = tile_scale(f16_bits_to_f32(cur.d[b]));
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][r] = __builtin_fmaf(d, part[i][r], acc[i][r]);
    }
}

// grid and modes as for k_qgemm_rw; 8 waves = 256 weight rows per workgroup; LDS holds the two activation stages
template <int MB>
__global__ __launch_bounds__(512, 1) void k_qgemm_rw_q8(const uint8_t *__restrict__ W, const uint4 *__restrict__ xs,
                                                         const float *__restrict__ rowscale, void *__restrict__ yg,
                                                         float *__restrict__ partial, int M, int Mp, int N, int spr, int chunk,
                                                         int mode, const pmh::GemmSecond second) {
    constexpr int BM = 32 * MB, kThreads = 512;
    extern __shared__ uint4 smem[];
    uint4 *a0 = smem, *a1 = a0 + kQ6Groups * BM;
    const int tid = threadIdx.x;
    LaneQ6<MB> L;
    L.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    L.col = lane & 31, L.g = lane >> 5;
    int bx = (int)blockIdx.x;
    take_weight(second, mode, bx, W, yg, N);
    const int n0 = bx * 256, m0 = blockIdx.y * BM;
    const int n = n0 + 32 * L.wave + L.col;
    const int sb0 = blockIdx.z * chunk;
    const int cnt = spr - sb0 < chunk ? spr - sb0 : chunk;
    const size_t row_bytes = (size_t)spr * 272;
    // this lane's row (rows past N repeat the last) at the first block of super-block sb0, and at its last half
    const uint8_t *wp = W + (size_t)(n < N ? n : N - 1) * row_bytes + (size_t)sb0 * 272;
    const uint8_t *wlast = W + (size_t)(n < N ? n : N - 1) * row_bytes + (size_t)(spr * 2 - 1) * 136;
#pragma unroll
    for (int i = 0; i < LaneQ6<MB>::kARounds; i++) {
        const int idx = tid + i * kThreads;
        L.a_off[i] = (uint32_t)((idx / BM) * Mp + idx % BM);
    }
    float16_t acc[MB];
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[i][r] = 0.0f;

    Q8Half ha, hb;
    q8_load(wp, L.g, ha);
    {
        const uint4 *xa = xs + (size_t)(sb0 * 2 * kQ6Groups) * Mp + m0;
#pragma unroll
        for (int i = 0; i < LaneQ6<MB>::kARounds; i++) dma16(xa + L.a_off[i], a0 + i * kThreads + L.wave * 64);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __syncthreads();

    for (int s = 0; s < cnt; s++) {
        const int sb = sb0 + s;
        const int sbn = sb + 1 < spr ? sb + 1 : spr - 1;  // the copies for "the next super-block" stay inside the matrix
        const uint8_t *w1 = wp + 136, *w2 = wp + 272;
        rw_half_q8<MB>(a0, a1, xs + (size_t)((sb * 2 + 1) * kQ6Groups) * Mp + m0, w1, ha, hb, L, acc);
        barrier_keep<12>();
        rw_half_q8<MB>(a1, a0, xs + (size_t)(sbn * 2 * kQ6Groups) * Mp + m0, w2 < wlast ? w2 : wlast, hb, ha, L, acc);
        barrier_keep<12>();
        wp = w2;
    }

    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the last register loads and copies (past the end) are done
    __syncthreads();
    store_tile<MB>(acc, smem, L.wave, L.col, L.g, m0, n0, M, N, Mp, rowscale, yg, partial, mode, blockIdx.z);
}

// ------------------------------------------------------------------------------------------------
// Q4_K with at most 16 activation rows (a decode batch, a speculative window) and rows of at most 16 super-blocks: the
// weights are read once, at the pace of the GEMV, and (rows of at most eight super-blocks, see SmallX) no other kernel runs.
//   * v_mfma_f32_16x16x32_f16: 16 activation rows x 16 weight rows x 32 k.  Lane (r = lane % 16, kg = lane / 16) holds
//     the eight k of k-group kg for activation row r (first operand) resp. weight row r (second operand); the output
//     tile has column lane % 16 (weight row) and rows 4 (lane / 16) + 0..3 (activation rows).
//   * A wave owns one or two super-block columns of W (wave w: super-blocks w and w + 8) and walks the row tiles of its
//     workgroup.  Its activation operands for those super-blocks -- per super-block eight items (k-step t, k-group kg)
//     and the item of sub-block sums, as a pre-pass arranges them -- are converted or loaded once and stay in registers.
//   * Per row tile the wave copies its one or two super-blocks of the 16 rows (144 or 288 contiguous bytes per row)
//     through registers into its own piece of LDS with whole-wave 16-byte loads, a row tile ahead (every load
//     unconditional, so the outstanding loads are counted exactly); a lane then takes the 16-byte header of its weight
//     row and the 32 quant bytes of sub-blocks 2 kg and 2 kg + 1 (dword t of them is its operand of k-step t) out of
//     LDS.  LDS executes a wave's instructions in order, so the copy needs no barrier.  (Each lane loading its own three
//     pieces from global memory -- 16-byte pieces 32 bytes apart, 16 rows per request -- was 4 % slower per call.)
//     Arithmetic as in the large kernel: exact integer tiles sc * q, d on the fp32 sum of a super-block, the min term as
//     one more matrix instruction over exact head + tail splits.
//   * The waves' 16 x 16 partial tiles (one per super-block column) are added through LDS in wave order by the first
//     wave (one barrier per row tile, no partial tiles in global memory, no reduction kernel; the result does not
//     depend on scheduling) and collected in LDS; the workgroup stores its columns of y after its last row tile, scaled
//     by the rows' powers of two.  No store and no other load is issued inside the streaming loop: on this target stores
//     share the loads' counter, and one of them in flight turns every counted wait into a wait for everything.
// ------------------------------------------------------------------------------------------------
constexpr int kSmallWaves = 8;  // waves per workgroup (fewer when a row has fewer super-blocks); 16 waves of one super-block each run alike
constexpr int kSmallDepth = 2;  // row tiles in flight per wave (four are slower: 16.5 against 12.7 us at 14336 x 4096)
constexpr int kSmallMaxM = 16, kSmallMaxSpr = 16;
constexpr int kSmallMaxM2 = 32;  // Q4_K, Q5_K and Q8_0: two 16-row blocks of activations per weight operand

// The two steps the short-batch kernels share.  A row tile's 16 x 16 partial tiles, one per wave: every wave leaves its
// own in LDS, and after one barrier the first wave adds them in wave order and keeps the sum as finished tile `ti` (the
// next tile writes the other buffer; the one after that comes behind the next barrier).
//
// A workgroup with few tiles (at most kSmallKeepTiles) keeps every wave's partial tile of every row tile instead
// ([tile][wave][lane]) and adds them after the last one, in the same wave order: its waves then meet at one
// barrier, not at one per tile.
// `red`, `keep`, behind the finished tiles: two buffers of a partial tile per wave, or those.  (All of it in dynamic LDS and as long as the
// workgroup's waves need: with the buffers of eight waves beside what activations pass through before the first tile, fewer workgroups of
// rows of one to four super-blocks fit a compute unit than the launch counts on, and the last ones of a round waited for the others:
// f32, three Q4_K weights of 24737 x 256, M = 9, 20.0 -> 14.3 us; Q6_K 33017 and 8456 x 1024, M = 6, 22.2 -> 16.1.)
constexpr int kSmallKeepTiles = 8;
// UNROLL: of the sum over the waves of one tile after the other.  Written out eight times it moves the rest of the kernel about: weights from
// memory, M = 16, 14336 x 4096, us with 8 / 1: Q4_K 13.26 / 12.99, 60000 x 2048, M = 8, 21.24 / 21.16, Q3_K 17.67 / 17.61, Q2_K 13.43 / 13.35, but Q6_K 18.24 / 18.54, and 9000 x 3584,
// M = 7, 19.3 / 21.4.
template <int UNROLL>
__device__ __forceinline__ void small_add_waves(float4_t *red, float4_t *keep, int ti, int wave, int nwaves, int lane, const float4_t acc,
                                                float4_t *out_tiles) {
    if (keep) {  // workgroup-uniform
        keep[(ti * nwaves + wave) * 64 + lane] = acc;
        return;
    }
    const int buf = (ti & 1) * nwaves;
    red[(buf + wave) * 64 + lane] = acc;
    __syncthreads();
    if (wave == 0) {
        float4_t v = red[buf * 64 + lane];
#pragma unroll UNROLL
        for (int q = 1; q < nwaves; q++) {
            const float4_t u = red[(buf + q) * 64 + lane];
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] += u[r];
        }
        out_tiles[ti * 64 + lane] = v;
    }
}

__device__ __forceinline__ void small_add_kept(const float4_t *keep, int n_tiles, int wave, int nwaves, int lane, float4_t *out_tiles) {
    if (!keep) return;
    __syncthreads();
    for (int ti = wave; ti < n_tiles; ti += nwaves) {
        float4_t v = keep[(ti * nwaves) * 64 + lane];
        for (int q = 1; q < nwaves; q++) {
            const float4_t u = keep[(ti * nwaves + q) * 64 + lane];
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] += u[r];
        }
        out_tiles[ti * 64 + lane] = v;
    }
}

// After the last tile: the finished tiles leave; or, when a long row is cut into runs over the grid's second dimension, as the fp32
// partial tile of this run for k_rw_reduce.  Of at most 16 rows every wave has scaled its tiles (`rs` is 1, k_rw_reduce is given no scales).
// Of two blocks of rows they are scaled by the rows' powers of two, here or by k_rw_reduce (`rs`: that of row `lane`, requested when the
// kernel starts: asked for here it would be a trip to memory at the kernel's end).  A thread takes a lane slot: four rows of one column.
// (mt: 16-row blocks of activations per row tile of weights; the finished tile of block b of row tile ti is slot ti * mt + b)
__device__ __forceinline__ float small_row_scale(const float *__restrict__ rowscale) { return rowscale[threadIdx.x & 31]; }

__device__ __forceinline__ void small_store(const float4_t *out_tiles, int t0, int t1, int M, int Mp, int N, const float rs,
                                            void *__restrict__ yg, int ybf16, float *__restrict__ partial, const int mt = 1) {
    __shared__ float4_t scales[8];  // (of the type that is read back: only that aligns an LDS object to 16 bytes)
    if (threadIdx.x < 32) reinterpret_cast<float *>(scales)[threadIdx.x] = rs;
    __syncthreads();
    for (int idx = (int)threadIdx.x; idx < (t1 - t0) * mt * 64; idx += (int)blockDim.x) {
        const int tile = mt == 1 ? idx >> 6 : idx >> 7, b = mt == 1 ? 0 : (idx >> 6) & 1, l = idx & 63;
        const int n = (t0 + tile) * 16 + (l & 15), m = 16 * b + 4 * (l >> 4);
        const float4_t v = out_tiles[idx], o = v * scales[m / 4];
        if (n >= N) continue;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if (m + r >= M) break;
            if (partial) partial[((size_t)blockIdx.y * Mp + m + r) * N + n] = v[r];
            else if (ybf16) reinterpret_cast<uint16_t *>(yg)[(size_t)(m + r) * N + n] = (uint16_t)bf16_rne_bits(o[r]);
            else reinterpret_cast<float *>(yg)[(size_t)(m + r) * N + n] = o[r];
        }
    }
}

// ------------------------------------------------------------------------------------------------
// At most 16 activation rows: every wave converts the activations it multiplies.  A pre-pass for so few rows is 16 workgroups and a
// chain of latencies (3 to 4 us of 15) in front of a kernel whose waves then wait for their first weights; here the
// conversion runs while those are on their way.  A wave's super-block of the 16 rows comes in whole-wave 16-byte loads, goes through the
// wave's own LDS (piece p of row r at piece p ^ r: neither the writes nor the reads collide), and a lane takes its eight items:
// two runs of four elements each, of row lane % 16, where the pre-pass's order of the same number puts them.  The power of two that
// takes a row into [2^9, 2^10) is that of the wave's part of it and not of the whole row: its inverse multiplies the wave's tiles,
// exactly, before they are added, so nothing is rounded that a pre-pass would not round.
// Measured (us a call, weights from memory, with a pre-pass in front -> so): 14336 x 4096, M = 10, bf16 Q4_K 14.5 -> 12.8, Q5_K 16.1 -> 15.3, Q6_K
// 18.0 -> 17.3, Q8_0 18.3 -> 18.1, Q3_K 17.9 -> 17.5, Q2_K 14.2 -> 12.9; M = 16, f32 Q4_K 14.7 -> 14.2; 4096 x 14336, M = 12, f32 Q4_K 18.8 -> 16.1,
// Q6_K 22.4 -> 19.7.  1.13 times as fast over 42 shapes of 1 to 16 rows.
// ------------------------------------------------------------------------------------------------
constexpr int kSmallXItems = 512;  // 16-byte items of LDS for a super-block of 16 rows in bf16; f32: twice as many
template <bool XF32, int ORDER, int NSB>
struct SmallX {
    static constexpr int kPieces = XF32 ? 64 : 32, kLoads = 16 * kPieces / 64;  // per row and super-block; per lane
    u32x4 piece[NSB][kLoads];
    // Past the last row, and of a super-block past the end of the row (valid false), the buffer returns zeros.
    __device__ __forceinline__ void request(const int i, const __amdgpu_buffer_rsrc_t r, const uint32_t row_bytes, const int sb, const bool valid, const int lane) {
        uint32_t base = valid ? (uint32_t)sb * (16u * kPieces) : 0x7F000000u;
        asm("" : "+s"(base));  // (opaque: a choice the compiler sees becomes a branch around each load, with a wait for it)
        base += 16u * ((uint32_t)lane % kPieces) + (XF32 ? 0u : ((uint32_t)lane >> 5) * row_bytes);
#pragma unroll
        for (int j = 0; j < kLoads; j++)
            piece[i][j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, base + (XF32 ? j : 2 * j) * row_bytes, 0, 0));
    }
    // first element of the two runs of item t of k-group kg
    static __device__ __forceinline__ void runs(const int t, const int kg, int &lo, int &hi) {
        if (ORDER == 2) lo = 128 * (t >> 2) + 32 * (t & 1) + 16 * ((t >> 1) & 1) + 4 * kg, hi = lo + 64;  // t = 4 hh + 2 lh + gp
        else if (ORDER == 3) lo = 32 * t + 8 * kg, hi = lo + 4;
        else if (ORDER == 5) lo = 128 * (kg >> 1) + 64 * (t & 1) + 16 * (kg & 1) + 4 * (t >> 1), hi = lo + 32;
        else if (ORDER == 4) lo = 64 * kg + 8 * t, hi = lo + 4;
        else if (ORDER == 0) lo = 64 * kg + 32 * (t >> 2) + 4 * (t & 3), hi = lo + 16;
        else lo = 64 * kg + 4 * t, hi = lo + 32;
    }
    // af: the items; up: 2^e of the rows 4 kg .. 4 kg + 3 (the rows of the lane's part of a product tile).  (In instructions that two
    // waves of a SIMD can issue at a time: packed ones and v_fma_mix would end that)
    __device__ __forceinline__ void convert(u32x4 *stage, const int lane, half8_t *const (&af)[NSB], float4_t &up) const {
        convert(stage, lane, af, up, [](float most) { return most; });
    }
    // join: the largest magnitude of the row over what other waves hold of it, too
    template <class Join>
    __device__ __forceinline__ void convert(u32x4 *stage, const int lane, half8_t *const (&af)[NSB], float4_t &up, const Join &join) const {
        const int nl = lane & 15, kg = lane >> 4;
        const u32x4 *mine = stage + nl * kPieces;
        uint32_t raw[NSB][8][XF32 ? 8 : 4];
        float most[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // the largest magnitudes of the row (a NaN does not count)
        // An infinity in the high half of a word, with what lies in the low one, is a signalling NaN.  In IEEE mode (bit 9) a maximum with one is
        // a quiet NaN, and the next maximum drops that together with the word's other element; without it the NaN alone is dropped.
        // (Clearing the low half instead, or 16-bit maxima, cost 0.15 to 0.6 us a call.)
        if (!XF32) asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 9, 1), 0" : "+v"(most[0]), "+v"(most[1]), "+v"(most[2]), "+v"(most[3]));
#pragma unroll
        for (int i = 0; i < NSB; i++) {
#pragma unroll
            for (int j = 0; j < kLoads; j++) {
                const int row = XF32 ? j : 2 * j + (lane >> 5), p = lane % kPieces;
                stage[row * kPieces + (p ^ row)] = piece[i][j];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 8; t++) {
                int lo, hi;
                runs(t, kg, lo, hi);
                uint32_t (&w)[XF32 ? 8 : 4] = raw[i][t];
                if (XF32) {
                    const u32x4 a = mine[(lo >> 2) ^ nl], b = mine[(hi >> 2) ^ nl];
#pragma unroll
                    for (int c = 0; c < 4; c++) w[c] = a[c], w[XF32 ? 4 + c : 0] = b[c];
                } else if (hi == lo + 4) {
                    const u32x4 a = mine[(lo >> 3) ^ nl];
#pragma unroll
                    for (int c = 0; c < 4; c++) w[c] = a[c];
                } else {
                    const uint2 a = reinterpret_cast<const uint2 *>(mine + ((lo >> 3) ^ nl))[(lo >> 2) & 1], b = reinterpret_cast<const uint2 *>(mine + ((hi >> 3) ^ nl))[(hi >> 2) & 1];
                    w[0] = a.x, w[1] = a.y, w[2] = b.x, w[3] = b.y;
                }
            }
#pragma unroll
            for (int t = 0; t < 8; t++)
#pragma unroll
                for (int c = 0; c < 4; c++)  // (bf16: the low half's bits do not change the exponent of the high one)
                    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(most[c]) : "v"(raw[i][t][c]), "v"(XF32 ? raw[i][t][XF32 ? 4 + c : 0] : raw[i][t][c] << 16));
        }
        if (!XF32) asm volatile("s_setreg_imm32_b32 hwreg(HW_REG_MODE, 9, 1), 1" : "+v"(most[0]), "+v"(most[1]), "+v"(most[2]), "+v"(most[3]));
        float amax = __builtin_fmaxf(__builtin_fmaxf(most[0], most[1]), __builtin_fmaxf(most[2], most[3]));
        amax = __builtin_fmaxf(amax, __shfl_xor(amax, 16));
        amax = join(__builtin_fmaxf(amax, __shfl_xor(amax, 32)));
        const int eb = (int)((__builtin_bit_cast(uint32_t, amax) >> 23) & 0xFFu);  // it lies in [2^(eb-127), 2^(eb-126))
        int e = eb - 126 - 10;
        e = e < -126 ? -126 : (e > 126 ? 126 : e);
        if (eb == 255) e = 0;  // inf: let them through
        const float down = __builtin_bit_cast(float, (uint32_t)(127 - e) << 23), mine_up = __builtin_bit_cast(float, (uint32_t)(127 + e) << 23);
#pragma unroll
        for (int q = 0; q < 4; q++) up[q] = __shfl(mine_up, 4 * kg + q);  // (lane r holds row r)
#pragma unroll
        for (int i = 0; i < NSB; i++)
#pragma unroll
            for (int t = 0; t < 8; t++) {
                float v[8];
#pragma unroll
                for (int c = 0; c < 8; c++)
                    v[c] = down * __builtin_bit_cast(float, XF32 ? raw[i][t][XF32 ? c : 0] : c & 1 ? raw[i][t][c / 2] & 0xFFFF0000u : raw[i][t][c / 2] << 16);
                half8_t h;
#pragma unroll
                for (int c = 0; c < 8; c++) {  // (ORDER 4: eight consecutive elements, the even ones first)
                    float a = v[ORDER == 4 ? 2 * (c & 3) + (c >> 2) : c];
                    asm("" : "+v"(a));  // (the product and its rounding apart, not one v_fma_mix.  The conversion itself is not written as asm:
                                        // what reads its result has to wait, which the compiler sees to for instructions it knows)
                    h[c] = (_Float16)a;
                }
                af[i][t] = h;
            }
    }
};

// The sums of the sub-blocks over the converted activations, as head + tail items (H0, L0, H0, L0, H1, L1, H1, L1) like the pre-pass's: ORDER 5
// two of them (k-steps of one parity: their first runs are one sub-block, their second runs another), the others one (its sub-blocks
// 2 kg and 2 kg + 1).  A product with a matrix of zeros and ones adds them up over lanes that hold parts of them; it leaves
// the sum of column c for row 4 kg + r in lane (c, kg), and LDS takes it to the lane of its row.
template <int ORDER>
__device__ __forceinline__ void small_sums(const half8_t (&af)[8], float *stage, const int lane, half8_t (&sums)[ORDER == 5 ? 2 : 1]) {
    const int nl = lane & 15, kg = lane >> 4;
    float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const int lo = ORDER == 5 ? 4 * kg + 2 * (t & 1) : ORDER == 1 ? 2 * kg : 2 * kg + (t >> 2), hi = ORDER == 5 || ORDER == 1 ? lo + 1 : lo;
        const _Float16 a = (_Float16)(nl == lo ? 1.0f : 0.0f), b = (_Float16)(nl == hi ? 1.0f : 0.0f);
        const half8_t ones = {a, a, a, a, b, b, b, b};
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[t], ones, acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) stage[(4 * kg + r) * 17 + nl] = acc[r];
    constexpr int kSums = ORDER == 5 ? 2 : 1;
#pragma unroll
    for (int i = 0; i < kSums; i++) {
        const float s0 = stage[nl * 17 + 2 * kSums * kg + 2 * i], s1 = stage[nl * 17 + 2 * kSums * kg + 2 * i + 1];
        const _Float16 h0 = (_Float16)s0, h1 = (_Float16)s1;
        const _Float16 l0 = (_Float16)(s0 - (float)h0), l1 = (_Float16)(s1 - (float)h1);
        sums[i] = half8_t{h0, l0, h0, l0, h1, l1, h1, l1};
    }
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t small_x_buffer(const void *x, const int M, const uint32_t row_bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(x), 0, M * (int)row_bytes, 0x00027000);
}
// Before a wave's LDS takes another use that other waves share: its own reads have returned, and everyone is here.  (Requests for
// weights stay in flight; __syncthreads() would wait for them.)
__device__ __forceinline__ void barrier_lds() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Where several launches multiply the same activations by rows of more than eight super-blocks, a workgroup per pair of them converts
// them ahead, by the same code (the results do not depend on who converts): per pair the items, the sums' items and the scales, an
// item per lane and 64 items, 1 KiB, at a time.
template <int ORDER>
constexpr int kPairItems = 2 * (8 + (ORDER == 2 || ORDER == 3 ? 0 : ORDER == 5 ? 2 : 1)) + 1;
template <bool XF32, int ORDER>
__global__ __launch_bounds__(128) void k_prep_pairs(const void *__restrict__ x, int M, int spr, uint4 *__restrict__ out) {  // a wave per super-block
    __shared__ u32x4 stages[2][(XF32 ? 2 : 1) * kSmallXItems];
    __shared__ float most[2][16];
    constexpr int kSums = ORDER == 2 || ORDER == 3 ? 0 : ORDER == 5 ? 2 : 1;
    const int lane = threadIdx.x & 63, i = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), sb = 2 * (int)blockIdx.x + i;
    const uint32_t x_row = (uint32_t)spr * (XF32 ? 1024u : 512u);
    const __amdgpu_buffer_rsrc_t xr = small_x_buffer(x, M, x_row);
    SmallX<XF32, ORDER, 1> X;
    X.request(0, xr, x_row, sb, sb < spr, lane);
    half8_t af[8];
    half8_t *const to[1] = {af};
    float4_t up;
    X.convert(stages[i], lane, to, up, [&](float v) {
        if (lane < 16) most[i][lane] = v;
        __syncthreads();
        return __builtin_fmaxf(most[0][lane & 15], most[1][lane & 15]);
    });
    uint4 *mine = out + (size_t)blockIdx.x * (64 * kPairItems<ORDER>) + lane;
#pragma unroll
    for (int t = 0; t < 8; t++) mine[64 * (8 * i + t)] = __builtin_bit_cast(uint4, af[t]);
    if (i == 0) mine[64 * (kPairItems<ORDER> - 1)] = __builtin_bit_cast(uint4, up);
    if constexpr (kSums > 0) {
        half8_t sums[kSums];
        small_sums<ORDER>(af, reinterpret_cast<float *>(stages[i]), lane, sums);
#pragma unroll
        for (int c = 0; c < kSums; c++) mine[64 * (16 + kSums * i + c)] = __builtin_bit_cast(uint4, sums[c]);
    }
}
// A wave's pair, or zeros where the row has ended (valid false).  item: of super-block i number t (from 8 on: its sums)
template <int ORDER>
struct SmallPair {
    const uint4 *at;
    uint32_t keep;
    __device__ __forceinline__ SmallPair(const void *ws, const int sb, const bool valid, const int lane)
        : at(reinterpret_cast<const uint4 *>(ws) + (size_t)(sb >> 1) * (64 * kPairItems<ORDER>) + lane), keep(valid ? 0xFFFFFFFFu : 0u) {}
    __device__ __forceinline__ u32x4 get(const int n) const {
        const u32x4 v = *reinterpret_cast<const u32x4 *>(at + 64 * n);
        return v & u32x4{keep, keep, keep, keep};
    }
    __device__ __forceinline__ half8_t item(const int i, const int t) const {
        constexpr int kSums = (kPairItems<ORDER> - 17) / 2;
        return __builtin_bit_cast(half8_t, get(t < 8 ? 8 * i + t : 16 + kSums * i + t - 8));
    }
    __device__ __forceinline__ float4_t up() const { return __builtin_bit_cast(float4_t, get(kPairItems<ORDER> - 1)); }
};

template <int NSB, int FMT = 0>
struct SmallRun {
    static constexpr int kPerSb = BlockFmt<FMT>::kBytes / 16;  // 16-byte pieces of a super-block: 9 (Q4_K) or 11 (Q5_K)
    static constexpr int kPieces = 16 * kPerSb * NSB;          // ... of a row tile's NSB super-blocks
    static constexpr int kLoads = (kPieces + 63) / 64;         // per lane: 5 or 3 (Q5_K: 6 or 3)
    u32x4 piece[kLoads];  // (a vector type: copies of it are loads and stores that stay in registers)
};

// FMT 1: Q5_K -- eleven pieces per super-block (header, two of qh, eight of quants); a lane takes the qh bytes of its two
// sub-blocks out of its stage as well and ors the fifth bits into the quant dwords as in the large kernel.
// MT: 16-row blocks of activations (1: at most 16 rows, 2: at most 32); a weight operand then feeds MT matrix instructions.
// XT: what xg is: 0 the pre-pass's items (MT = 2: twice the rows to convert would not hide behind the first weights), 1 and 2 the
// activations themselves in bf16 and in f32, 3 the pairs of super-blocks that k_prep_pairs has converted (NSB = 2).
template <int ORDER, int NSB, int FMT, int MT, int XT>
__global__ __launch_bounds__(64 * kSmallWaves) void k_qgemm_small(const uint8_t *__restrict__ W, const void *__restrict__ xg,
                                                                   const float *__restrict__ rowscale, void *__restrict__ yg, int M,
                                                                   int Mp, int N, int spr, int tiles, int tiles_per_wg, int ybf16,
                                                                   float *__restrict__ partial, const pmh::GemmSecond second) {
    int bx = (int)blockIdx.x;
    if (ybf16 & kHasSecond) {
        take_weight(second, ybf16, bx, W, yg, N);
        tiles = (N + 15) / 16;
    }
    extern __shared__ float4_t dyn[];  // out_tiles [tiles_per_wg rounded up to whole rounds][64]: lane slots of the finished tiles; the waves' partial tiles; then the waves' stages
    const float rs = XT ? 1.0f : small_row_scale(rowscale);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nwaves = (int)(blockDim.x >> 6);
    const int nl = lane & 15, kg = lane >> 4;
    const uint32_t low = kg < 2 ? 0xFFFFFFFFu : 0u;
    const int rounds = (tiles_per_wg + kSmallDepth - 1) / kSmallDepth;
    float4_t *out_tiles = dyn;
    float4_t *red = dyn + rounds * kSmallDepth * MT * 64, *keep = tiles_per_wg * MT <= kSmallKeepTiles ? red : nullptr;
    u32x4 *stage = reinterpret_cast<u32x4 *>(dyn + (rounds * kSmallDepth * MT * (keep ? 1 + nwaves : 1) + (keep ? 0 : 2 * nwaves)) * 64) + wave * SmallRun<NSB, FMT>::kPieces;
    int sbi[NSB];
    bool sbv[NSB];  // wave-uniform
#pragma unroll
    for (int i = 0; i < NSB; i++) {
        sbi[i] = (int)blockIdx.y * (NSB * nwaves) + NSB * wave + i;  // adjacent super-blocks: one contiguous piece of every row per wave; workgroup row blockIdx.y of the grid takes the blockIdx.y-th run of NSB * waves super-blocks of a long row
        sbv[i] = sbi[i] < spr;
        sbi[i] = sbv[i] ? sbi[i] : 0;
    }
    // activation operands of this wave's super-blocks: item (2 sb + kg / 2, group 2 t + kg % 2) of rows nl (and 16 + nl), and the sums item
    half8_t af[NSB][MT][8], asum[NSB][MT];
    constexpr int kXOrder = ORDER == 1 ? 1 : FMT ? 4 : 0;
    constexpr bool kOwn = XT == 1 || XT == 2;
    SmallX<XT == 2, kXOrder, NSB> X;
    float4_t up;
    const uint32_t x_row = (uint32_t)spr * (XT == 2 ? 1024u : 512u);
    const __amdgpu_buffer_rsrc_t xr = small_x_buffer(xg, M, x_row);
    if constexpr (kOwn) {
#pragma unroll
        for (int i = 0; i < NSB; i++) X.request(i, xr, x_row, sbi[i], sbv[i], lane);
        __builtin_amdgcn_sched_barrier(0);
    } else if constexpr (XT == 3) {
        const SmallPair<kXOrder> pair(xg, sbi[0], sbv[0], lane);
#pragma unroll
        for (int i = 0; i < NSB; i++) {
#pragma unroll
            for (int t = 0; t < 8; t++) af[i][0][t] = pair.item(i, t);
            asum[i][0] = pair.item(i, 8);
        }
        up = pair.up();
    } else {
        const uint4 *xs = reinterpret_cast<const uint4 *>(xg);
#pragma unroll
        for (int i = 0; i < NSB; i++)
#pragma unroll
            for (int b = 0; b < MT; b++) {
                const uint4 *base = xs + (size_t)((2 * sbi[i] + (kg >> 1)) * kGroups) * Mp + 16 * b + nl;
#pragma unroll
                for (int t = 0; t < 8; t++) af[i][b][t] = __builtin_bit_cast(half8_t, base[(size_t)(2 * t + (kg & 1)) * Mp]);
                asum[i][b] = __builtin_bit_cast(half8_t, base[(size_t)(16 + (kg & 1)) * Mp]);
                if (!sbv[i]) {  // a super-block past the end of the row multiplies zeros (no branch in the streaming loop)
                    const half8_t z = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                    for (int t = 0; t < 8; t++) af[i][b][t] = z;
                    asum[i][b] = z;
                }
            }
    }
    const int t0 = bx * tiles_per_wg;
    const int t1 = t0 + tiles_per_wg < tiles ? t0 + tiles_per_wg : tiles;  // t1 > t0 by the launch geometry
    constexpr int kPerSb = SmallRun<NSB, FMT>::kPerSb, kBlockBytes = BlockFmt<FMT>::kBytes, kQ0 = FMT ? 3 : 1;  // kQ0: first quant piece
    const uint32_t row_bytes = (uint32_t)spr * (uint32_t)kBlockBytes;
    // piece j of this lane: index lane + 64 j of the tile's 16 rows x 9 NSB pieces (a load past the last piece repeats it
    // and is dropped); a super-block past the end of the row is replaced by the row's first
    constexpr int kLoads = SmallRun<NSB, FMT>::kLoads, kPieces = SmallRun<NSB, FMT>::kPieces;
    uint32_t piece_row[kLoads], piece_off[kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; j++) {
        int idx = lane + 64 * j;
        idx = idx < kPieces ? idx : kPieces - 1;
        const int p = idx % (kPerSb * NSB);
        piece_row[j] = (uint32_t)(idx / (kPerSb * NSB));
        piece_off[j] = (uint32_t)(NSB == 2 && p >= kPerSb ? sbi[NSB - 1] : sbi[0]) * (uint32_t)kBlockBytes + 16u * (uint32_t)(p % kPerSb);
    }
    auto issue = [&](int ti, SmallRun<NSB, FMT> &w) __attribute__((always_inline)) {
        int tile = t0 + ti;
        tile = tile < t1 ? tile : t1 - 1;  // past the end: the last tile again (loaded, not used)
#pragma unroll
        for (int j = 0; j < kLoads; j++) {
            int n = tile * 16 + (int)piece_row[j];
            n = n < N ? n : N - 1;
            w.piece[j] = *reinterpret_cast<const u32x4 *>(W + ((uint32_t)n * row_bytes + piece_off[j]));  // the tensor is smaller than 4 GiB (checked by the launcher)
        }
    };
    const u32x4 *mine = stage + nl * (kPerSb * NSB);  // this lane's weight row in the stage
    auto consume = [&](int ti, const SmallRun<NSB, FMT> &w) __attribute__((always_inline)) {
        float4_t acc[MT];
#pragma unroll
        for (int b = 0; b < MT; b++) acc[b] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < kLoads; j++)
            if (lane + 64 * j < kPieces) stage[lane + 64 * j] = w.piece[j];
        // LDS executes a wave's instructions in order: the reads below see the writes above, and the next tile's
        // writes come after these reads
#pragma unroll
        for (int i = 0; i < NSB; i++) {
            const u32x4 hv = mine[kPerSb * i], qav = mine[kPerSb * i + kQ0 + 2 * kg], qbv = mine[kPerSb * i + kQ0 + 1 + 2 * kg];
            const uint4 hdr = make_uint4(hv.x, hv.y, hv.z, hv.w);
            // scales and mins of sub-blocks 2 kg and 2 kg + 1 (6-bit fields, crates/pmetal-gguf/src/quantize.rs:844-855)
            const uint32_t sh = 16u * (uint32_t)(kg & 1);
            const uint32_t yv = hdr.y >> sh, zv = hdr.z >> sh, wv = hdr.w >> sh;
            // sub-blocks 0..3 (kg < 2) and 4..7 store them differently; both forms are computed and one is picked by a
            // per-lane bit mask (a branch here would be taken by half of every wave)
            const uint32_t sc0 = ((yv & 63u) & low) | (((wv & 0xFu) | ((yv >> 2) & 0x30u)) & ~low);
            const uint32_t sc1 = (((yv >> 8) & 63u) & low) | ((((wv >> 8) & 0xFu) | ((yv >> 10) & 0x30u)) & ~low);
            const uint32_t mn0 = ((zv & 63u) & low) | ((((wv >> 4) & 0xFu) | ((zv >> 2) & 0x30u)) & ~low);
            const uint32_t mn1 = (((zv >> 8) & 63u) & low) | ((((wv >> 12) & 0xFu) | ((zv >> 10) & 0x30u)) & ~low);
            const _Float16 s0 = (_Float16)(float)sc0, s1 = (_Float16)(float)sc1;
            const _Float16 o0 = (_Float16)(-1024.0f * (float)sc0), o1 = (_Float16)(-1024.0f * (float)sc1);  // exact: sc <= 63
            const half2_t sc2[2] = {half2_t{s0, s0}, half2_t{s1, s1}}, off2[2] = {half2_t{o0, o0}, half2_t{o1, o1}};
            const uint32_t qd[8] = {qav.x, qav.y, qav.z, qav.w, qbv.x, qbv.y, qbv.z, qbv.w};
            // Q5_K: the fifth bits of k-step t.  GGML order: qh dword t (the same four bytes as quant dword t), bits 2 kg and
            // 2 kg + 1 of every byte.  REF order: byte 4 (2 kg + t / 4) + t % 4 of qh, i.e. of the lane's two qh dwords.
            uint32_t qh[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            if (FMT == 1) {
                if (ORDER == 1) {
                    const u32x4 ha = mine[kPerSb * i + 1], hb = mine[kPerSb * i + 2];
                    const uint32_t h8[8] = {ha.x, ha.y, ha.z, ha.w, hb.x, hb.y, hb.z, hb.w};
#pragma unroll
                    for (int t = 0; t < 8; t++) qh[t] = h8[t] >> (2 * kg);
                } else {
                    const uint2 hp = *reinterpret_cast<const uint2 *>(reinterpret_cast<const uint8_t *>(mine + kPerSb * i + 1) + 8 * kg);
#pragma unroll
                    for (int t = 0; t < 8; t++) qh[t] = (t < 4 ? hp.x : hp.y) >> (8 * (t & 3));
                }
            }
            float4_t part[MT];
#pragma unroll
            for (int b = 0; b < MT; b++) part[b] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int t = 0; t < 8; t++) {
                Dq d;
#pragma unroll
                for (int c = 0; c < 4; c++) dq_chunk<ORDER, FMT>(c, t, qd[t], sc2, off2, d, qh[t]);
                const half8_t bv = d.value();
#pragma unroll
                for (int b = 0; b < MT; b++) part[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i][b][t], bv, part[b], 0, 0, 0);
            }
            // (of a super-block past the end of the row only zeros may enter the sums, whatever bytes were loaded for it)
            const float dmin = sbv[i] ? f16_bits_to_f32(hdr.x >> 16) : 0.0f, dd = sbv[i] ? f16_bits_to_f32(hdr.x & 0xFFFFu) : 0.0f;
            _Float16 h0, l0, h1, l1;
            neg_min_split(dmin, mn0, h0, l0);
            neg_min_split(dmin, mn1, h1, l1);
            const half8_t br = {h0, h0, l0, l0, h1, h1, l1, l1};
#pragma unroll
            for (int b = 0; b < MT; b++) {
                acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(asum[i][b], br, acc[b], 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; r++) acc[b][r] = __builtin_fmaf(dd, part[b][r], acc[b][r]);
            }
        }
        if (XT) acc[0] *= up;
#pragma unroll
        for (int b = 0; b < MT; b++) small_add_waves<1>(red, keep, ti * MT + b, wave, nwaves, lane, acc[b], out_tiles);
    };
    static_assert(kSmallDepth == 2, "the ring is written out as two tiles");
    SmallRun<NSB, FMT> ring0, ring1;
    issue(0, ring0);
    if (XT != 2 || NSB == 1) issue(1, ring1);
    if constexpr (kOwn) {  // while the first weights are on their way
        __builtin_amdgcn_sched_barrier(0);
        u32x4 *x_stage = reinterpret_cast<u32x4 *>(dyn) + wave * ((XT == 2 ? 2 : 1) * kSmallXItems);
        half8_t *to[NSB];
#pragma unroll
        for (int i = 0; i < NSB; i++) to[i] = af[i][0];
        X.convert(x_stage, lane, to, up);
#pragma unroll
        for (int i = 0; i < NSB; i++) {
            half8_t sums[1];
            small_sums<kXOrder>(af[i][0], reinterpret_cast<float *>(x_stage), lane, sums);
            asum[i][0] = sums[0];
        }
        barrier_lds();
        if (XT == 2 && NSB == 2) issue(1, ring1);  // (in f32 two super-blocks' activations leave no registers for it before)
    }
    // Whole rounds of two tiles, with nothing conditional around the loads, so that the outstanding loads are counted
    // exactly at every wait; the tiles past the workgroup's last one are computed on repeated data and dropped.
    for (int rd = 0; rd < rounds; rd++) {
        consume(2 * rd, ring0);
        issue(2 * rd + 2, ring0);
        consume(2 * rd + 1, ring1);
        issue(2 * rd + 3, ring1);
    }
    small_add_kept(keep, rounds * kSmallDepth * MT, wave, nwaves, lane, out_tiles);
    small_store(out_tiles, t0, t1, M, Mp, N, rs, yg, ybf16, partial, MT);
}

// ------------------------------------------------------------------------------------------------
// The same for Q8_0 (34-byte blocks: f16 d, 32 int8).  A k-step of v_mfma_f32_16x16x32_f16 is one block: lane (r, kg)
// holds the eight quants 8 kg .. 8 kg + 7 of the block of weight row r, exact in f16, and the block's d multiplies the
// fp32 product tile of that one k-step.  A wave owns one or two runs of eight blocks (256 elements = 272 bytes) of every
// row, as the Q4_K kernel owns super-blocks.  Nothing in a row of 34-byte blocks is aligned to more than two bytes, and
// loads at such addresses are slow, so the wave copies the 16 x 272 bytes of a row tile's run -- 16-byte aligned at both
// ends -- through registers into its own piece of LDS with whole-wave 16-byte loads (the ring holds these pieces) and
// every lane takes its quants and scales out of LDS: aligned dwords, those of the even blocks shifted by two bytes.  LDS
// executes a wave's instructions in order, so the copy needs no barrier.  Ring, reduction over the waves and epilogue
// as above.
// ------------------------------------------------------------------------------------------------
constexpr int kQ8RunBytes = 272, kQ8TileRunPieces = 16 * kQ8RunBytes / 16;  // 272 pieces of 16 bytes: 4.25 per lane

// (one run's pieces: a tile of two runs is two of these, kept apart so that each stays in registers)
struct SmallRunQ8 {
    u32x4 piece[5];  // (a vector type: copies of it are loads and stores that stay in registers)
};

template <int NSB, int MT, int XT>  // (XT as above)
__global__ __launch_bounds__(64 * kSmallWaves) void k_qgemm_small_q8(const uint8_t *__restrict__ W, const void *__restrict__ xg,
                                                                      const float *__restrict__ rowscale, void *__restrict__ yg, int M,
                                                                      int Mp, int N, int spr, int tiles, int tiles_per_wg, int ybf16,
                                                                   float *__restrict__ partial, const pmh::GemmSecond second) {
    int bx = (int)blockIdx.x;
    if (ybf16 & kHasSecond) {
        take_weight(second, ybf16, bx, W, yg, N);
        tiles = (N + 15) / 16;
    }
    extern __shared__ float4_t dyn[];  // out_tiles [tiles_per_wg rounded up to whole rounds][64], the waves' partial tiles, then the waves' stages
    const float rs = XT ? 1.0f : small_row_scale(rowscale);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nwaves = (int)(blockDim.x >> 6);
    const int nl = lane & 15, kg = lane >> 4;
    const int rounds = (tiles_per_wg + kSmallDepth - 1) / kSmallDepth;
    float4_t *out_tiles = dyn;
    float4_t *red = dyn + rounds * kSmallDepth * MT * 64, *keep = tiles_per_wg * MT <= kSmallKeepTiles ? red : nullptr;
    u32x4 *stage = reinterpret_cast<u32x4 *>(dyn + (rounds * kSmallDepth * MT * (keep ? 1 + nwaves : 1) + (keep ? 0 : 2 * nwaves)) * 64) + wave * (NSB * kQ8TileRunPieces);
    int sbi[NSB];
    bool sbv[NSB];  // wave-uniform
#pragma unroll
    for (int i = 0; i < NSB; i++) {
        sbi[i] = (int)blockIdx.y * (NSB * nwaves) + NSB * wave + i;
        sbv[i] = sbi[i] < spr;
        sbi[i] = sbv[i] ? sbi[i] : 0;
    }
    // activation operands: block b of run sb holds elements 256 sb + 32 b ..; the item of its k-group kg is item
    // 4 (b % 4) + kg of half 2 sb + b / 4 (the pre-pass writes 16 items of eight consecutive elements per 128)
    half8_t af[NSB][MT][8];  // (MT 16-row blocks of activations: rows nl, 16 + nl)
    constexpr bool kOwn = XT == 1 || XT == 2;
    SmallX<XT == 2, 3, NSB> X;
    float4_t up;
    const uint32_t x_row = (uint32_t)spr * (XT == 2 ? 1024u : 512u);
    const __amdgpu_buffer_rsrc_t xr = small_x_buffer(xg, M, x_row);
    if constexpr (kOwn) {
#pragma unroll
        for (int i = 0; i < NSB; i++) X.request(i, xr, x_row, sbi[i], sbv[i], lane);
        __builtin_amdgcn_sched_barrier(0);
    } else if constexpr (XT == 3) {
        const SmallPair<3> pair(xg, sbi[0], sbv[0], lane);
#pragma unroll
        for (int i = 0; i < NSB; i++)
#pragma unroll
            for (int b = 0; b < 8; b++) af[i][0][b] = pair.item(i, b);
        up = pair.up();
    } else {
        const uint4 *xs = reinterpret_cast<const uint4 *>(xg);
#pragma unroll
        for (int i = 0; i < NSB; i++)
#pragma unroll
            for (int mb = 0; mb < MT; mb++)
#pragma unroll
                for (int b = 0; b < 8; b++) {
                    const uint4 *item = xs + (size_t)((2 * sbi[i] + (b >> 2)) * kQ6Groups + 4 * (b & 3) + kg) * Mp + 16 * mb + nl;
                    af[i][mb][b] = __builtin_bit_cast(half8_t, *item);
                    if (!sbv[i]) af[i][mb][b] = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
                }
    }
    const int t0 = bx * tiles_per_wg;
    const int t1 = t0 + tiles_per_wg < tiles ? t0 + tiles_per_wg : tiles;
    const uint32_t row_bytes = (uint32_t)spr * (uint32_t)kQ8RunBytes;
    // piece j of this lane: index lane + 64 j of the tile's 272 (the fifth exists for the first 16 lanes; the others load
    // the last piece again and drop it)
    uint32_t piece_row[5], piece_off[5];
#pragma unroll
    for (int j = 0; j < 5; j++) {
        int idx = lane + 64 * j;
        idx = idx < kQ8TileRunPieces ? idx : kQ8TileRunPieces - 1;
        piece_row[j] = (uint32_t)(idx / 17), piece_off[j] = 16u * (uint32_t)(idx % 17);
    }
    auto issue = [&](int ti, SmallRunQ8 &wa, SmallRunQ8 &wb) __attribute__((always_inline)) {
        int tile = t0 + ti;
        tile = tile < t1 ? tile : t1 - 1;  // past the end: the last tile again (loaded, not used)
#pragma unroll
        for (int j = 0; j < 5; j++) {
            int n = tile * 16 + (int)piece_row[j];
            n = n < N ? n : N - 1;
            const uint8_t *p = W + ((uint32_t)n * row_bytes + piece_off[j]);  // the tensor is smaller than 4 GiB (checked by the launcher)
#pragma unroll
            for (int i = 0; i < NSB; i++) (i == 0 ? wa : wb).piece[j] = *reinterpret_cast<const u32x4 *>(p + (uint32_t)sbi[i] * (uint32_t)kQ8RunBytes);
        }
    };
    const uint32_t *mine = reinterpret_cast<const uint32_t *>(stage) + nl * (kQ8RunBytes / 4);  // this lane's weight row in the stage
    auto consume = [&](int ti, const SmallRunQ8 &wa, const SmallRunQ8 &wb) __attribute__((always_inline)) {
        float4_t acc[MT];
#pragma unroll
        for (int mb = 0; mb < MT; mb++) acc[mb] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
        const float4_t none = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < NSB; i++) {
            u32x4 *st = stage + i * kQ8TileRunPieces;
            const SmallRunQ8 &w = i == 0 ? wa : wb;
#pragma unroll
            for (int j = 0; j < 4; j++) st[lane + 64 * j] = w.piece[j];
            if (lane < kQ8TileRunPieces - 256) st[lane + 256] = w.piece[4];
            // LDS executes a wave's instructions in order: the reads below see the writes above, and the next tile's
            // writes come after these reads
            const uint32_t *row = mine + i * (kQ8TileRunPieces * 4);
#pragma unroll
            for (int b = 0; b < 8; b++) {
                // block b starts at byte 34 b of the run: on a dword boundary for even b (d in the low half of that dword,
                // the quants from its high half on), two bytes past one for odd b (d in the high half of the dword below)
                uint32_t q0, q1, dbits;
                if ((b & 1) == 0) {
                    const uint32_t *p = row + (34 * b) / 4 + 2 * kg;
                    const uint32_t w0 = p[0], w1 = p[1], w2 = p[2];
                    q0 = __builtin_amdgcn_alignbit(w1, w0, 16), q1 = __builtin_amdgcn_alignbit(w2, w1, 16);
                    dbits = row[(34 * b) / 4] & 0xFFFFu;
                } else {
                    const uint32_t *p = row + (34 * b + 2) / 4 + 2 * kg;
                    q0 = p[0], q1 = p[1];
                    dbits = row[(34 * b - 2) / 4] >> 16;
                }
                // (of a run past the end of the row only zeros may enter the sums, whatever bytes were loaded for it)
                const float d = sbv[i] ? f16_bits_to_f32(dbits) : 0.0f;
                const half8_t bv = q8_operand(q0, q1);
#pragma unroll
                for (int mb = 0; mb < MT; mb++) {
                    const float4_t part = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i][mb][b], bv, none, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[mb][r] = __builtin_fmaf(d, part[r], acc[mb][r]);
                }
            }
        }
        if (XT) acc[0] *= up;
#pragma unroll
        for (int mb = 0; mb < MT; mb++) small_add_waves<1>(red, keep, ti * MT + mb, wave, nwaves, lane, acc[mb], out_tiles);
    };
    static_assert(kSmallDepth == 2, "the ring is written out as two tiles");
    SmallRunQ8 ring0a, ring0b, ring1a, ring1b;  // (the b halves are unused with one run per wave)
    issue(0, ring0a, ring0b);
    if (XT != 2 || NSB == 1) issue(1, ring1a, ring1b);
    if constexpr (kOwn) {  // while the first weights are on their way
        __builtin_amdgcn_sched_barrier(0);
        u32x4 *x_stage = reinterpret_cast<u32x4 *>(dyn) + wave * ((XT == 2 ? 2 : 1) * kSmallXItems);
        half8_t *to[NSB];
#pragma unroll
        for (int i = 0; i < NSB; i++) to[i] = af[i][0];
        X.convert(x_stage, lane, to, up);
        barrier_lds();
        if (XT == 2 && NSB == 2) issue(1, ring1a, ring1b);  // (in f32 two super-blocks' activations leave no registers for it before)
    }
    for (int rd = 0; rd < rounds; rd++) {
        consume(2 * rd, ring0a, ring0b);
        issue(2 * rd + 2, ring0a, ring0b);
        consume(2 * rd + 1, ring1a, ring1b);
        issue(2 * rd + 3, ring1a, ring1b);
    }
    small_add_kept(keep, rounds * kSmallDepth * MT, wave, nwaves, lane, out_tiles);
    small_store(out_tiles, t0, t1, M, Mp, N, rs, yg, ybf16, partial, MT);
}

// ------------------------------------------------------------------------------------------------
// The same for Q6_K (210-byte super-blocks: ql[128], qh[64], 16 int8 scales, f16 d; value d sc (q - 32),
// crates/pmetal-gguf/src/k_quants.rs:474-496); first for rows of a multiple of eight super-blocks, which start on
// 16-byte boundaries.  A k-step of v_mfma_f32_16x16x16_f16 is one sub-block of 16 elements: lane (r, kg) holds the
// four quants 4 kg .. 4 kg + 3 of the sub-block of weight row r as exact f16 (q - 32), and d sc of the sub-block
// multiplies the fp32 product tile of that step.  Sub-block (hh, g, lh) -- elements 128 hh + 32 g + 16 lh .. of the
// super-block -- takes the low (g < 2) or high nibbles of the ql dword at 64 hh + 32 (g % 2) + 16 lh + 4 kg, bits 2 g of
// the qh dword at 32 hh + 16 lh + 4 kg and scale 8 hh + 2 g + lh; its activation operand is one half of the pre-pass
// item (t = 4 lh + kg, g % 2) of half hh, which holds elements 32 (g % 2) + 4 t .. and those 64 further.
// A wave owns one or two adjacent super-blocks of every row.  Their bytes start (210 NSB wave) % 16 bytes into a
// 16-byte piece: the wave copies the pieces that cover them, row by row, through registers into its own LDS with
// whole-wave 16-byte loads (never past the piece that holds the tensor's last byte), and the lanes read aligned dwords;
// the fields of a super-block sit a wave-uniform 0 or 2 bytes off a dword boundary and are shifted into place.
// ------------------------------------------------------------------------------------------------
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
template <int NSB, bool ANY = false>
struct SmallQ6 {
    // 16-byte pieces that cover 210 NSB bytes from where a wave's super-blocks start in their piece: any even byte for one
    // super-block per wave or rows of any length (ANY), a multiple of four for pairs of super-blocks in rows that start
    // on 16-byte boundaries
    static constexpr int kRowPieces = NSB == 2 ? (ANY ? 28 : 27) : 14;
    static constexpr int kLoads = (16 * kRowPieces + 63) / 64;        // pieces per lane and row tile: 7 or 4
    static constexpr int kStageDwords = 16 * kRowPieces * 4 + 4;      // (+ one piece: the shifted reads look one dword ahead)
};
template <int NSB>
struct SmallRunQ6 {
    u32x4 piece[SmallQ6<NSB>::kLoads];  static_assert(SmallQ6<NSB, true>::kLoads == SmallQ6<NSB, false>::kLoads, "one ring for both forms");  // (a vector type: copies of it are loads and stores that stay in registers)
};

// ANY: rows of any number of super-blocks.  A row then starts at any even address, so where a wave's super-blocks lie in
// their first piece, and whether their fields sit two bytes off a dword boundary, differs from row to row (per lane); the
// last wave with work may own one super-block where the others own two.
template <int NSB, bool ANY, int XT>  // (XT as above)
__global__ __launch_bounds__(64 * kSmallWaves) void k_qgemm_small_q6(const uint8_t *__restrict__ W, const void *__restrict__ xg,
                                                                      void *__restrict__ yg, int M,
                                                                      int Mp, int N, int spr, int tiles, int tiles_per_wg, int ybf16,
                                                                      uint32_t w_last, float *__restrict__ partial, const pmh::GemmSecond second) {
    int bx = (int)blockIdx.x;
    if (ybf16 & kHasSecond) {
        take_weight(second, ybf16, bx, W, yg, N);
        tiles = (N + 15) / 16;
        w_last = (uint32_t)(((uint64_t)N * (uint64_t)spr * 210u - 1) & ~(uint64_t)15);
    }
    constexpr int P = SmallQ6<NSB, ANY>::kRowPieces, kLoads = SmallQ6<NSB, ANY>::kLoads;
    extern __shared__ float4_t dyn[];  // out_tiles [tiles_per_wg rounded up to whole rounds][64], the waves' partial tiles, then the waves' stages
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nwaves = (int)(blockDim.x >> 6);
    const int nl = lane & 15, kg = lane >> 4;
    const int rounds = (tiles_per_wg + kSmallDepth - 1) / kSmallDepth;
    float4_t *out_tiles = dyn;
    float4_t *red = dyn + rounds * kSmallDepth * 64, *keep = tiles_per_wg <= kSmallKeepTiles ? red : nullptr;
    uint32_t *stage = reinterpret_cast<uint32_t *>(dyn + (rounds * kSmallDepth * (keep ? 1 + nwaves : 1) + (keep ? 0 : 2 * nwaves)) * 64) + wave * SmallQ6<NSB, ANY>::kStageDwords;
    // this wave's super-blocks sb0 .. sb0 + NSB - 1 (rows are whole multiples of eight super-blocks, so the NSB of a wave
    // exist together or not at all; a wave past the end of a long row's last run works on the row's first super-blocks
    // with zero activations and zero scales)
    const int sb_here = (int)blockIdx.y * (NSB * nwaves) + NSB * wave;
    bool sbv[NSB];  // wave-uniform; without ANY all of a wave's super-blocks exist or none
#pragma unroll
    for (int i = 0; i < NSB; i++) sbv[i] = sb_here + i < spr;
    const int sb0 = sbv[0] ? sb_here : 0;
    const uint32_t run_start = 210u * (uint32_t)sb0, delta = run_start & 15u;
    // activation operands: item (t = 4 lh + kg, gp) of half 2 sb + hh; index 4 hh + 2 lh + gp
    half8_t af[NSB][8];
    constexpr bool kOwn = XT == 1 || XT == 2;
    SmallX<XT == 2, 2, NSB> X;
    float4_t up;
    const uint32_t x_row = (uint32_t)spr * (XT == 2 ? 1024u : 512u);
    const __amdgpu_buffer_rsrc_t xr = small_x_buffer(xg, M, x_row);
    if constexpr (kOwn) {
#pragma unroll
        for (int i = 0; i < NSB; i++) X.request(i, xr, x_row, sb0 + i, sbv[i], lane);
        __builtin_amdgcn_sched_barrier(0);
    } else {
        const SmallPair<2> pair(xg, sb0, sbv[0], lane);
#pragma unroll
        for (int i = 0; i < NSB; i++)
#pragma unroll
            for (int t = 0; t < 8; t++) af[i][t] = pair.item(i, t);
        up = pair.up();
    }
    const int t0 = bx * tiles_per_wg;
    const int t1 = t0 + tiles_per_wg < tiles ? t0 + tiles_per_wg : tiles;
    const uint32_t row_bytes = (uint32_t)spr * 210u;
    uint32_t piece_row[kLoads], piece_off[kLoads];
#pragma unroll
    for (int j = 0; j < kLoads; j++) {
        int idx = lane + 64 * j;
        idx = idx < 16 * P ? idx : 16 * P - 1;  // (the last load of a lane may not exist: it repeats the last piece and is dropped)
        piece_row[j] = (uint32_t)(idx / P), piece_off[j] = (ANY ? 0u : run_start & ~15u) + 16u * (uint32_t)(idx % P);
    }
    auto issue = [&](int ti, SmallRunQ6<NSB> &w) __attribute__((always_inline)) {
        int tile = t0 + ti;
        tile = tile < t1 ? tile : t1 - 1;  // past the end: the last tile again (loaded, not used)
#pragma unroll
        for (int j = 0; j < kLoads; j++) {
            int n = tile * 16 + (int)piece_row[j];
            n = n < N ? n : N - 1;
            uint32_t a = (uint32_t)n * row_bytes + piece_off[j];  // the tensor is smaller than 4 GiB (checked by the launcher)
            if (ANY) a = (((uint32_t)n * row_bytes + run_start) & ~15u) + piece_off[j];  // from the piece that holds the run's first byte in this row
            a = a < w_last ? a : w_last;  // a piece past the one with the tensor's last byte holds nothing of this run
            w.piece[j] = *reinterpret_cast<const u32x4 *>(W + a);
        }
    };
    const uint32_t *mine = stage + nl * (P * 4);  // this lane's weight row in the stage (dwords)
    auto consume = [&](int ti, const SmallRunQ6<NSB> &w) __attribute__((always_inline)) {
        float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
        const float4_t none = {0.0f, 0.0f, 0.0f, 0.0f};
        u32x4 *st = reinterpret_cast<u32x4 *>(stage);
#pragma unroll
        for (int j = 0; j < kLoads; j++)
            if (lane + 64 * j < 16 * P) st[lane + 64 * j] = w.piece[j];
        // LDS executes a wave's instructions in order: the reads below see the writes above, and the next tile's
        // writes come after these reads
        uint32_t delta_row = delta;
        if (ANY) {  // of the row this lane reads, as issue() took it
            int tile = t0 + ti;
            tile = tile < t1 ? tile : t1 - 1;
            int n = tile * 16 + nl;
            n = n < N ? n : N - 1;
            delta_row = ((uint32_t)n * row_bytes + run_start) & 15u;
        }
#pragma unroll
        for (int i = 0; i < NSB; i++) {
            const uint32_t at = delta_row + 210u * (uint32_t)i;  // byte of the super-block in the lane's staged row (wave-uniform without ANY)
            const uint32_t sh = 8u * (at & 2u);
            const uint32_t *blk = mine + (at >> 2);
            auto field = [&](int dword) -> uint32_t {  // the dword at byte 4 * dword of the super-block
                return __builtin_amdgcn_alignbit(blk[dword + 1], blk[dword], sh);
            };
            uint32_t sc[4];
#pragma unroll
            for (int q = 0; q < 4; q++) sc[q] = field(48 + q);
            const float d = sbv[i] ? f16_bits_to_f32(field(52) & 0xFFFFu) : 0.0f;
#pragma unroll
            for (int hh = 0; hh < 2; hh++)
#pragma unroll
                for (int lh = 0; lh < 2; lh++) {
                    const uint32_t qh = field(32 + 8 * hh + 4 * lh + kg);
#pragma unroll
                    for (int gp = 0; gp < 2; gp++) {
                        const uint32_t ql = field(16 * hh + 8 * gp + 4 * lh + kg);
                        const half8_t a8 = af[i][4 * hh + 2 * lh + gp];
#pragma unroll
                        for (int up = 0; up < 2; up++) {  // group g = gp + 2 up: the low, then the high nibbles
                            const int g = gp + 2 * up;
                            const uint32_t v = ((ql >> (4 * up)) & 0x0F0F0F0Fu) | (((qh >> (2 * g)) & 0x03030303u) << 4);
                            // 0x6400 | q is the f16 1024 + q; minus 1056 leaves q - 32, exact
                            const half2_t m1056 = {(_Float16)-1056.0f, (_Float16)-1056.0f};
                            const half2_t b01 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)) + m1056;
                            const half2_t b23 = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)) + m1056;
                            const half4_t b4 = {b01[0], b01[1], b23[0], b23[1]};
                            const half4_t a4 = up ? half4_t{a8[4], a8[5], a8[6], a8[7]} : half4_t{a8[0], a8[1], a8[2], a8[3]};
                            const float4_t part = __builtin_amdgcn_mfma_f32_16x16x16f16(a4, b4, none, 0, 0, 0);
                            const int si = 8 * hh + 2 * g + lh;  // the sub-block's scale byte
                            const float s = d * (float)((int)(sc[si >> 2] << (24 - 8 * (si & 3))) >> 24);
#pragma unroll
                            for (int r = 0; r < 4; r++) acc[r] = __builtin_fmaf(s, part[r], acc[r]);
                        }
                    }
                }
        }
        acc *= up;
        small_add_waves<8>(red, keep, ti, wave, nwaves, lane, acc, out_tiles);
    };
    static_assert(kSmallDepth == 2, "the ring is written out as two tiles");
    SmallRunQ6<NSB> ring0, ring1;
    issue(0, ring0);
    if (XT != 2 || NSB == 1) issue(1, ring1);
    if constexpr (kOwn) {  // while the first weights are on their way
        __builtin_amdgcn_sched_barrier(0);
        u32x4 *x_stage = reinterpret_cast<u32x4 *>(dyn) + wave * ((XT == 2 ? 2 : 1) * kSmallXItems);
        half8_t *to[NSB];
#pragma unroll
        for (int i = 0; i < NSB; i++) to[i] = af[i];
        X.convert(x_stage, lane, to, up);
        barrier_lds();
        if (XT == 2 && NSB == 2) issue(1, ring1);  // (in f32 two super-blocks' activations leave no registers for it before)
    }
    for (int rd = 0; rd < rounds; rd++) {
        consume(2 * rd, ring0);
        issue(2 * rd + 2, ring0);
        consume(2 * rd + 1, ring1);
        issue(2 * rd + 3, ring1);
    }
    small_add_kept(keep, rounds * kSmallDepth, wave, nwaves, lane, out_tiles);
    small_store(out_tiles, t0, t1, M, Mp, N, 1.0f, yg, ybf16, partial);
}

__global__ __launch_bounds__(256) void k_copy16(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t items) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < items) dst[i] = src[i];
}

// y[m][n] = rowscale[m] * (partial[0][m][n] + partial[1][m][n] + ...), added in this order (rowscale NULL: the tiles are scaled already).  A thread takes PER consecutive
// outputs of the row-major result, whatever the row length: eight, in 16-byte accesses (rows of a length that is no multiple
// of 8 went one output per thread: with the tile store's wide form for them 4674 x 1024 at M = 829 39.8 -> 29.9 us a call), or
// one where the result is small and the kernel is the time of one trip to memory (7 x 1661: 1.5 us longer with eight).
template <bool YBF16, int PER>
__global__ __launch_bounds__(256) void k_rw_reduce(const float *__restrict__ partial, int splits, int M, int Mp, int N,
                                                    const float *__restrict__ rowscale, void *__restrict__ yg) {
    const size_t first = (size_t)blockIdx.x * (256 * PER), total = (size_t)M * N, idx = first + threadIdx.x * PER;
    if (idx >= total) return;
    // the row of the first output, and how far into it (the 64-bit division once per workgroup, in scalar registers)
    const uint32_t m_first = (uint32_t)(first / (uint32_t)N);
    const uint32_t at = (uint32_t)(first - (size_t)m_first * (uint32_t)N) + threadIdx.x * PER;
    const uint32_t m = m_first + at / (uint32_t)N, col = at % (uint32_t)N;
    const size_t plane = (size_t)Mp * N;
    auto one = [&](const int e) {  // output idx + e: its row may be a later one
        float t = partial[idx + e];
        for (int z = 1; z < splits; z++) t += partial[(size_t)z * plane + idx + e];
        if (rowscale) t *= rowscale[m + (col + e) / (uint32_t)N];
        if (YBF16) reinterpret_cast<uint16_t *>(yg)[idx + e] = (uint16_t)bf16_rne_bits(t);
        else reinterpret_cast<float *>(yg)[idx + e] = t;
    };
    if (PER == 1) {
        one(0);
    } else if (total - idx < 8 || N < 8) {
        for (int e = 0; e < 8 && idx + e < total; e++) one(e);
    } else {
        const float s0 = rowscale ? rowscale[m] : 1.0f, s1 = rowscale ? rowscale[m + 1 < (uint32_t)M ? m + 1 : m] : 1.0f;  // at most one row ends among the eight
        float4 a = reinterpret_cast<const float4 *>(partial + idx)[0], b = reinterpret_cast<const float4 *>(partial + idx)[1];
        for (int z = 1; z < splits; z++) {
            const float4 *q = reinterpret_cast<const float4 *>(partial + (size_t)z * plane + idx);
            const float4 c = q[0], d = q[1];
            a.x += c.x, a.y += c.y, a.z += c.z, a.w += c.w;
            b.x += d.x, b.y += d.y, b.z += d.z, b.w += d.w;
        }
        float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] *= col + e < (uint32_t)N ? s0 : s1;
        if (YBF16) {
            *reinterpret_cast<uint4 *>(reinterpret_cast<uint16_t *>(yg) + idx) =
                make_uint4(bf16_rne_bits(v[0]) | (bf16_rne_bits(v[1]) << 16), bf16_rne_bits(v[2]) | (bf16_rne_bits(v[3]) << 16),
                           bf16_rne_bits(v[4]) | (bf16_rne_bits(v[5]) << 16), bf16_rne_bits(v[6]) | (bf16_rne_bits(v[7]) << 16));
        } else {
            float4 *o = reinterpret_cast<float4 *>(reinterpret_cast<float *>(yg) + idx);
            o[0] = make_float4(v[0], v[1], v[2], v[3]);
            o[1] = make_float4(v[4], v[5], v[6], v[7]);
        }
    }
}

template <int MB, int NR, int NW, int FMT = 0>
constexpr size_t rw_lds_bytes() {
    const size_t stages = (size_t)(2 * kGroups * 32 * MB + NW * NR * (3 * 128 + 64 + (FMT ? 64 : 0))) * 16;
    return stages > tile_lds_bytes<MB, NW>() ? stages : tile_lds_bytes<MB, NW>();
}

// ------------------------------------------------------------------------------------------------
// The same for Q3_K and Q2_K (sixteen 16-element sub-blocks).  Lane (r, kg) of v_mfma_f32_16x16x32_f16 stands where lane
// (n, g) of half h stands in the large kernel, with h = kg / 2 and g = kg % 2: the 16 bytes 16 kg .. of the 64 quant bytes
// of weight row r, whose dword t / 2 gives k-step t its eight values, against the pre-pass's item (2 sb + h, 2 t + g); four
// scales per lane; the sub-block sums of the activations (items 16 + g and 18 + g of the half) against the negated min
// coefficients in two further matrix instructions.  Blocks are 84 / 110 bytes and a lane needs few of them, so every lane
// loads its own: Q2_K rows start at multiples of four bytes, the quant piece, the scale bytes of its half and the d / dmin
// dword are plain loads; Q3_K blocks start at any even address, so a lane loads the aligned dwords that cover its pieces
// (quants and hmask: five; scales and d: four -- every one of them holds bytes of the block, none lies wholly past it) and
// shifts them by the block's 0 or 16 bits.  Ring, reduction over the waves and epilogue as above.
// ------------------------------------------------------------------------------------------------
struct __attribute__((packed, aligned(4))) u32x4_a4 {  // sixteen bytes at a 4-byte aligned address
    uint32_t x, y, z, w;
};
struct __attribute__((packed, aligned(4))) u32x2_a4 {
    uint32_t x, y;
};
__device__ __forceinline__ u32x4 load16_a4(const uint8_t *p) {
    const u32x4_a4 v = *reinterpret_cast<const u32x4_a4 *>(p);
    return u32x4{v.x, v.y, v.z, v.w};
}

template <int FMT, int NSB>
struct SmallRun16 {  // what a lane holds of a row tile
    u32x4 q[NSB];          // quant piece (Q3_K: from the dword boundary below it)
    uint32_t qx[NSB];      // Q3_K: the dword behind it
    u32x4 hm[NSB];         // Q3_K: hmask bytes 16 g ..
    uint32_t hmx[NSB];
    u32x4 sc[NSB];         // Q3_K: scales and d; Q2_K: x, y = scale bytes 8 h .., z = d | dmin << 16
};

template <int FMT, int NSB, int XT>  // (XT as above)
__global__ __launch_bounds__(64 * kSmallWaves) void k_qgemm_small16(const uint8_t *__restrict__ W, const void *__restrict__ xg,
                                                                     void *__restrict__ yg, int M,
                                                                     int Mp, int N, int spr, int tiles, int tiles_per_wg, int ybf16,
                                                                     float *__restrict__ partial, const pmh::GemmSecond second) {
    int bx = (int)blockIdx.x;
    if (ybf16 & kHasSecond) {
        take_weight(second, ybf16, bx, W, yg, N);
        tiles = (N + 15) / 16;
    }
    using B = Block16<FMT>;
    extern __shared__ float4_t dyn[];  // out_tiles [tiles_per_wg rounded up to whole rounds][64], then the waves' partial tiles
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nwaves = (int)(blockDim.x >> 6);
    const int nl = lane & 15, kg = lane >> 4;
    const uint32_t h = (uint32_t)(kg >> 1), g = (uint32_t)(kg & 1);
    const int rounds = (tiles_per_wg + kSmallDepth - 1) / kSmallDepth;
    float4_t *out_tiles = dyn;
    float4_t *red = dyn + rounds * kSmallDepth * 64, *keep = tiles_per_wg <= kSmallKeepTiles ? red : nullptr;
    int sbi[NSB];
    bool sbv[NSB];  // wave-uniform
#pragma unroll
    for (int i = 0; i < NSB; i++) {
        sbi[i] = (int)blockIdx.y * (NSB * nwaves) + NSB * wave + i;
        sbv[i] = sbi[i] < spr;
        sbi[i] = sbv[i] ? sbi[i] : 0;
    }
    half8_t af[NSB][8], asum[NSB][2];
    constexpr bool kOwn = XT == 1 || XT == 2;
    SmallX<XT == 2, 5, NSB> X;
    float4_t up;
    const uint32_t x_row = (uint32_t)spr * (XT == 2 ? 1024u : 512u);
    const __amdgpu_buffer_rsrc_t xr = small_x_buffer(xg, M, x_row);
    if constexpr (kOwn) {
#pragma unroll
        for (int i = 0; i < NSB; i++) X.request(i, xr, x_row, sbi[i], sbv[i], lane);
        __builtin_amdgcn_sched_barrier(0);
    } else {
        const SmallPair<5> pair(xg, sbi[0], sbv[0], lane);
#pragma unroll
        for (int i = 0; i < NSB; i++) {
#pragma unroll
            for (int t = 0; t < 8; t++) af[i][t] = pair.item(i, t);
            asum[i][0] = pair.item(i, 8), asum[i][1] = pair.item(i, 9);
        }
        up = pair.up();
    }
    const int t0 = bx * tiles_per_wg;
    const int t1 = t0 + tiles_per_wg < tiles ? t0 + tiles_per_wg : tiles;  // t1 > t0 by the launch geometry
    const uint32_t row_bytes = (uint32_t)spr * (uint32_t)B::kBytes;
    auto block_at = [&](int ti, int i) -> uint32_t {  // byte offset of super-block sbi[i] of this lane's row of tile ti (the tensor is smaller than 4 GiB)
        int tile = t0 + ti;
        tile = tile < t1 ? tile : t1 - 1;  // past the end: the last tile again (loaded, not used)
        int n = tile * 16 + nl;
        n = n < N ? n : N - 1;
        return (uint32_t)n * row_bytes + (uint32_t)sbi[i] * (uint32_t)B::kBytes;
    };
    auto issue = [&](int ti, SmallRun16<FMT, NSB> &w) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NSB; i++) {
            const uint32_t blk = block_at(ti, i);
            if (FMT == 3) {
                w.q[i] = load16_a4(W + (blk + 16u + 16u * (uint32_t)kg));
                const u32x2_a4 s2 = *reinterpret_cast<const u32x2_a4 *>(W + (blk + 8u * h));
                const uint32_t dd = *reinterpret_cast<const uint32_t *>(W + (blk + 80u));
                w.sc[i] = u32x4{s2.x, s2.y, dd, 0u};
            } else {
                const uint32_t lo = blk & ~3u;  // (the pieces' offsets inside the block are multiples of four)
                w.q[i] = load16_a4(W + (lo + 32u + 16u * (uint32_t)kg));
                w.qx[i] = *reinterpret_cast<const uint32_t *>(W + (lo + 48u + 16u * (uint32_t)kg));
                w.hm[i] = load16_a4(W + (lo + 16u * g));
                w.hmx[i] = *reinterpret_cast<const uint32_t *>(W + (lo + 16u + 16u * g));
                w.sc[i] = load16_a4(W + (lo + 96u));
            }
        }
    };
    auto consume = [&](int ti, const SmallRun16<FMT, NSB> &w) __attribute__((always_inline)) {
        float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < NSB; i++) {
            uint32_t qd[4], hm[4] = {0, 0, 0, 0}, s8[3], dbits;
            if (FMT == 3) {
                qd[0] = w.q[i][0], qd[1] = w.q[i][1], qd[2] = w.q[i][2], qd[3] = w.q[i][3];
                s8[0] = w.sc[i][0], s8[1] = w.sc[i][1], s8[2] = 0;
                dbits = w.sc[i][2];  // d | dmin << 16
            } else {
                const uint32_t sh = (block_at(ti, i) & 2u) * 8u;  // the block starts two bytes past a dword boundary, or on one
                qd[0] = __builtin_amdgcn_alignbit(w.q[i][1], w.q[i][0], sh), qd[1] = __builtin_amdgcn_alignbit(w.q[i][2], w.q[i][1], sh);
                qd[2] = __builtin_amdgcn_alignbit(w.q[i][3], w.q[i][2], sh), qd[3] = __builtin_amdgcn_alignbit(w.qx[i], w.q[i][3], sh);
                hm[0] = __builtin_amdgcn_alignbit(w.hm[i][1], w.hm[i][0], sh), hm[1] = __builtin_amdgcn_alignbit(w.hm[i][2], w.hm[i][1], sh);
                hm[2] = __builtin_amdgcn_alignbit(w.hm[i][3], w.hm[i][2], sh), hm[3] = __builtin_amdgcn_alignbit(w.hmx[i], w.hm[i][3], sh);
                s8[0] = __builtin_amdgcn_alignbit(w.sc[i][1], w.sc[i][0], sh), s8[1] = __builtin_amdgcn_alignbit(w.sc[i][2], w.sc[i][1], sh);
                s8[2] = __builtin_amdgcn_alignbit(w.sc[i][3], w.sc[i][2], sh);
                dbits = (w.sc[i][3] >> sh) & 0xFFFFu;
            }
            // (of a super-block past the end of the row only zeros may enter the sums, whatever bytes were loaded for it)
            const float d = sbv[i] ? f16_bits_to_f32(dbits & 0xFFFFu) : 0.0f;
            const float dmin = sbv[i] ? f16_bits_to_f32(dbits >> 16) : 0.0f;
            // scales (and mins) of the lane's four sub-blocks j = 8 h + 4 sp + 2 lh + g, index 2 sp + lh
            half2_t sc2[4], off2[4];
            float nm[4];
#pragma unroll
            for (int sp = 0; sp < 2; sp++)
#pragma unroll
                for (int lh = 0; lh < 2; lh++) {
                    float scf;
                    if (FMT == 3) {  // s8[sp]: bytes 8 h + 4 sp .. of the sixteen; low nibble scale, high nibble min
                        const uint32_t b = (s8[sp] >> (8u * g + 16u * lh)) & 0xFFu;
                        scf = (float)(b & 15u);
                        nm[2 * sp + lh] = -(dmin * (float)(b >> 4));
                    } else {
                        const uint32_t lo4 = (s8[sp] >> (8u * g + 16u * lh + 4u * h)) & 15u;
                        const uint32_t hi2 = (s8[2] >> (8u * g + 16u * lh + 2u * (2u * h + sp))) & 3u;
                        scf = (float)((int)(lo4 | (hi2 << 4)) - 32);
                        nm[2 * sp + lh] = -(d * (4.0f * scf));
                    }
                    const _Float16 s16 = (_Float16)scf, o16 = (_Float16)(-1024.0f * scf);  // exact: |sc| <= 32
                    sc2[2 * sp + lh] = half2_t{s16, s16}, off2[2 * sp + lh] = half2_t{o16, o16};
                }
            float4_t part = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const int dw = t >> 1, sp = t & 1;
                uint32_t lo = (qd[dw] >> (4 * sp)) & 0x03030303u, hi = (qd[dw] >> (4 * sp + 2)) & 0x03030303u;
                if (FMT == 2) {
                    const uint32_t m = hm[dw] >> (4u * h + 2u * sp);
                    lo |= (m & 0x01010101u) << 2, hi |= (m & 0x02020202u) << 1;
                }
                const half2_t r0 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, lo, 0x04010400u)), sc2[2 * sp], off2[2 * sp]);
                const half2_t r1 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, lo, 0x04030402u)), sc2[2 * sp], off2[2 * sp]);
                const half2_t r2 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, hi, 0x04010400u)), sc2[2 * sp + 1], off2[2 * sp + 1]);
                const half2_t r3 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, hi, 0x04030402u)), sc2[2 * sp + 1], off2[2 * sp + 1]);
                const half8_t b = half8_t{r0[0], r0[1], r1[0], r1[1], r2[0], r2[1], r3[0], r3[1]};
                part = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i][t], b, part, 0, 0, 0);
            }
#pragma unroll
            for (int sp = 0; sp < 2; sp++) {
                const _Float16 h0 = (_Float16)nm[2 * sp], h1 = (_Float16)nm[2 * sp + 1];
                const _Float16 l0 = (_Float16)(nm[2 * sp] - (float)h0), l1 = (_Float16)(nm[2 * sp + 1] - (float)h1);
                const half8_t br = half8_t{h0, h0, l0, l0, h1, h1, l1, l1};
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(asum[i][sp], br, acc, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) acc[r] = __builtin_fmaf(d, part[r], acc[r]);
        }
        acc *= up;
        small_add_waves<1>(red, keep, ti, wave, nwaves, lane, acc, out_tiles);
    };
    static_assert(kSmallDepth == 2, "the ring is written out as two tiles");
    SmallRun16<FMT, NSB> ring0, ring1;
    issue(0, ring0);
    if (XT != 2 || NSB == 1) issue(1, ring1);
    if constexpr (kOwn) {  // while the first weights are on their way
        __builtin_amdgcn_sched_barrier(0);
        u32x4 *x_stage = reinterpret_cast<u32x4 *>(dyn) + wave * ((XT == 2 ? 2 : 1) * kSmallXItems);
        half8_t *to[NSB];
#pragma unroll
        for (int i = 0; i < NSB; i++) to[i] = af[i];
        X.convert(x_stage, lane, to, up);
#pragma unroll
        for (int i = 0; i < NSB; i++) small_sums<5>(af[i], reinterpret_cast<float *>(x_stage), lane, asum[i]);
        barrier_lds();
        if (XT == 2 && NSB == 2) issue(1, ring1);  // (in f32 two super-blocks' activations leave no registers for it before)
    }
    for (int rd = 0; rd < rounds; rd++) {  // whole rounds of two tiles, nothing conditional around the loads
        consume(2 * rd, ring0);
        issue(2 * rd + 2, ring0);
        consume(2 * rd + 1, ring1);
        issue(2 * rd + 3, ring1);
    }
    small_add_kept(keep, rounds * kSmallDepth, wave, nwaves, lane, out_tiles);
    small_store(out_tiles, t0, t1, M, Mp, N, 1.0f, yg, ybf16, partial);
}

}  // namespace

namespace pmh {

static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// The fused kernels for at most 16 activation rows.  Rows of more than 16 super-blocks are cut into runs of 16, one
// workgroup row of the grid each, whose partial tiles k_rw_reduce adds (qgemm_plan sets splits and chunk to match).
constexpr int kSmallMaxRuns = 8;  // k <= 32768
// Super-blocks of a row that one short-batch workgroup takes (a longer row goes in runs of that many); 0: no such kernel.
// Up to 16 rows: eight waves of two super-blocks.  17 to 32 rows (two 16-row blocks of activations per weight operand), where
// the tile kernel does not take them: Q4_K / Q5_K hold two super-blocks' activations per wave, Q8_0 one.
static int small_run_spr(uint32_t type, int64_t m) {
    const bool any = type == kTypeQ4K || type == kTypeQ5K || type == kTypeQ6K || type == kTypeQ8_0 || type == kTypeQ3K || type == kTypeQ2K;
    if (m <= kSmallMaxM) return any ? kSmallMaxSpr : 0;
    if (m > kSmallMaxM2) return 0;
    if (type == kTypeQ4K || type == kTypeQ5K) return kSmallMaxSpr;
    if (type == kTypeQ8_0) return kSmallWaves;
    return 0;
}
static bool qgemm_small_applies(uint32_t type, int64_t m, int64_t n, int64_t k) {
    const int64_t spr = k / 256;
    const int run = small_run_spr(type, m);
    if (run == 0 || spr > (int64_t)run * kSmallMaxRuns) return false;
    if (type == kTypeQ4K) return (uint64_t)n * (uint64_t)spr * 144u < (1ull << 32);
    if (type == kTypeQ5K) return (uint64_t)n * (uint64_t)spr * 176u < (1ull << 32);
    if (type == kTypeQ8_0) return (uint64_t)n * (uint64_t)spr * 272u < (1ull << 32);
    if (type == kTypeQ6K) return (uint64_t)n * (uint64_t)spr * 210u < (1ull << 32);
    if (type == kTypeQ3K) return (uint64_t)n * (uint64_t)spr * 110u < (1ull << 32);
    if (type == kTypeQ2K) return (uint64_t)n * (uint64_t)spr * 84u < (1ull << 32);
    return false;
}

// Row tiles of a short-batch workgroup: one workgroup per compute unit (of fewer waves: as many as have eight together) over all runs of a
// long row, each of which then walks several row tiles with its activation operands in registers (one tile per workgroup and four times the
// workgroups: 35 against 27 us at M = 16, 4096 x 14336).  second_n: rows of the launch's second weight; a workgroup's tiles are of one weight.
// The finished tiles wait in LDS, 1 KiB each, beside the waves' stages (at most 70 KiB, Q8_0) and at most 16 KiB of the
// reduction buffers: 64 of them keep the workgroup within 160 KiB for every type.
static int small_tiles_per_wg(const GemmPlan &p, int64_t m, int64_t n, int64_t second_n, int64_t k) {
    const int spr = (int)(k / 256), nwaves = spr < kSmallWaves ? spr : kSmallWaves, most = m > kSmallMaxM ? 32 : 64;
    int64_t slots = (int64_t)compute_units() * (kSmallWaves / nwaves) / p.splits;
    slots = slots < 1 ? 1 : slots;
    const int tiles = (int)((n + 15) / 16), tiles1 = (int)((second_n + 15) / 16);
    const int n_wg = (int)(tiles + tiles1 < slots ? tiles + tiles1 : slots);
    int per = (tiles + tiles1 + n_wg - 1) / n_wg;
    if (tiles1 > 0 && (tiles + per - 1) / per + (tiles1 + per - 1) / per > n_wg) per++;
    return per < most ? per : most;
}

// (Who converts does not change a bit of the result: k_prep_pairs does as the waves do.)
// Up to eight super-blocks a row a wave converts one, which its first weights hide.  Of longer rows it converts two, which costs 1 to 3 us of
// the pre-pass's 4: not where several launches share one pre-pass (us for three bf16 weights of 4096, 1024 and 1024 x 4096, M = 16, two launches,
// with one / without: Q4_K 17.1 / 18.3, Q3_K 21.3 / 24.3; of 2048 x 2048 12.6 / 12.4), and not f32 activations of Q8_0 and Q3_K, 128 registers of
// them, behind which the second row tile has to be asked for (M = 16, 14336 x 4096: Q8_0 18.4 / 19.3; Q3_K, M = 4, 1024 x 4096 11.9 / 12.2, M = 9,
// 4096 x 3328 11.9 / 12.4; Q4_K 14.9 / 14.5, 9.7 / 9.5, 10.6 / 10.2) or two Q3_K weights in one launch (14336 x 4096, M = 16, 24.6 / 25.1: their sums
// of sixteen elements take the longest to make).  Nor of Q3_K and Q8_0 where a workgroup walks so many row tiles that its waves meet at each: the
// kernels that convert take longer over a tile (bf16, a pre-pass / without: Q3_K 16908 x 5120 36.2 / 38.6, 47394 x 2304 36.5 / 40.5, 28582 x
// 10496 68.6 / 75.1, Q8_0 36966 x 5376 66.0 / 67.1; with five tiles Q3_K 18833 x 4096 23.1 / 22.9, with ten Q4_K, Q5_K and Q6_K within 1 %).
bool qgemm_small_rows(const GemmPlan &p, int64_t m) { return p.kernel == GemmKernel::kSmall && m <= kSmallMaxM; }
bool qgemm_converts_itself(const GemmPlan &p, uint32_t type, int64_t m, int64_t n, int64_t second_n, int64_t k, uint32_t x_dtype, bool shared) {
    if (!qgemm_small_rows(p, m)) return false;
    if (k <= kSmallWaves * 256) return true;
    if (shared) return false;
    if (type == kTypeQ3K && second_n > 0) return false;
    return (type != kTypeQ8_0 && type != kTypeQ3K) || (x_dtype != kDtypeF32 && small_tiles_per_wg(p, m, n, second_n, k) <= kSmallKeepTiles);
}

bool qgemm_fits(uint32_t type, int64_t m, int64_t n, int64_t k) {
    // byte offsets inside a workgroup's rows and item offsets inside the activation copy are 32-bit
    return (type == kTypeQ4K || type == kTypeQ5K || type == kTypeQ6K || type == kTypeQ8_0 || type == kTypeQ3K || type == kTypeQ2K) && m >= 1 && m <= (int64_t)1 << 22 && n >= 1 && k >= 256 && k % 256 == 0 && k <= (int64_t)1 << 22 && n <= 0x7FFFFF00;
}

// Waves of a workgroup of the tile kernel: eight while the tiles fill the machine at most once, four, two workgroups to a compute unit, above.  Two
// workgroups are at different places of their tiles, so that one multiplies while the other waits for its first weights, adds its
// waves' tiles or stores; alone on a compute unit four waves wait longer for memory than eight.  Four against eight, times
// as long over 1400 drawn shapes, by tile and rounds of 256 workgroups:
//   32 x 32: 1.02 up to half a round (Q6_K, Q8_0 and Q2_K 1.05), 1.01 up to one, 0.98 up to two, 0.95 above
//   64 x 32: 0.98 to 0.99 up to one, 0.88 above (by registers twelve waves of it fit a compute unit, three workgroups of four or one of eight)
//   64 x 64: 1.02 up to 0.8, 0.99 up to one (Q6_K and Q8_0 1.00 and, with rows of 12 to 40 super-blocks, up to 1.17), 0.92 up to
//     two, 0.89 up to three, 0.84 above; 32 x 64 alike
// They decide the order in which a result is summed: a launch of two weights has the waves that either has alone.
static int kw_waves(int mb, int nr, double rounds, uint32_t type) {
    if (mb == 2 && nr == 1) return 4;
    const bool late = mb * nr < 4 || type == kTypeQ6K || type == kTypeQ8_0;
    return rounds <= (late ? 1.0 : 0.8) ? 8 : 4;
}
// Workgroups eight apart are on one die, whose cache holds an eighth of the larger operand's tiles and all of the other's.
bool kw_by_m(int64_t mblocks, int64_t tiles, int mb, int nr, int64_t block_bytes) {
    return mblocks >= 8 && mblocks * mb * 2 * 256 > tiles * nr * block_bytes;
}
// Rounds are the busiest die's workgroups of eight waves by what its 32 compute units hold of them: one each, two of 32 x 32 tiles.
KwMixed kw_mixed(int64_t mblocks, int64_t of_four, int64_t of_eight, bool by_m, int mb, int nr) {
    auto rounds = [&](int64_t columns) {
        const int64_t outer = by_m ? mblocks : columns, inner = by_m ? columns : mblocks;
        return (double)((outer + 7) / 8 * inner) / (mb * nr == 1 ? 64.0 : 32.0);
    };
    const double alone = rounds(of_four + of_eight), twos = rounds((of_four + 1) / 2 + of_eight);
    const bool by_twos = __builtin_ceil(twos) < __builtin_ceil(alone);
    return {by_twos, by_twos ? twos : alone};
}
static int64_t block_bytes(uint32_t type) {  // of a super-block of 256 elements
    return type == kTypeQ4K ? 144 : type == kTypeQ5K ? 176 : type == kTypeQ6K ? 210 : type == kTypeQ8_0 ? 272 : type == kTypeQ3K ? 110 : 84;
}

// The tile kernel's best tile and K split for a shape, and the microseconds it is expected to take behind the pre-pass, the gap in front
// of its launch (2.7 us) included, with eight waves.  Fitted to times of 1500 shapes (rms 12 %; 14 % over 150 others, drawn from 2 to 700 activation
// rows and timed by kernel trace; with the waves that it gets, the tile chosen is within 2 % of the best one on average over 1380 drawn shapes of more
// than 32 rows): per round of 256 workgroups a wave's super-blocks cost 1/124 us per KB of activations and
// 1/34 us per KB of weights the workgroup takes in, plus 0.8 us per 32 x 32 tile (Q6_K has twice the matrix instructions).
struct KwChoice {
    int mb, nr, splits, nw;
    double us, rounds;
};
static KwChoice kw_choice(int64_t m, int64_t n, int64_t spr, uint32_t type) {
    const double block = (double)block_bytes(type);
    const double items = type == kTypeQ3K || type == kTypeQ2K ? 40 : type == kTypeQ6K || type == kTypeQ8_0 ? 32 : 36;  // per row and super-block
    const double cost = type == kTypeQ6K ? 1.35 : 0.79;
    KwChoice best = {1, 1, 1, 8, 0.0, 0.0};
    bool have = false;
    for (int mb = 1; mb <= (m <= 32 ? 1 : 2); mb++)
        for (int nr = 1; nr <= 2; nr++) {
            if (m > 32 && mb == 1 && nr == 2) continue;  // never the best tile
            const int64_t tiles = ((n + 32 * nr - 1) / (32 * nr)) * ((m + 32 * mb - 1) / (32 * mb));
            for (int splits = 1; splits <= 4 && splits <= spr; splits *= 2) {
                if (splits > 1 && (tiles * splits > 256 || (m <= 32 && nr == 2))) break;  // only to fill the machine
                const int64_t chunk = (spr + splits - 1) / splits, per = (chunk + 7) / 8, wgs = tiles * splits;
                const double rounds = ((double)wgs / 256.0 + (double)((wgs + 255) / 256)) / 2;
                const double nwaves = m <= kSmallMaxM2 && spr < 8 ? (double)spr : 8.0;  // (a short row's workgroup has a wave per super-block)
                const double one = (double)per * nwaves * (mb * 32 * items * 16 / 1e3 / 124.0 + nr * 32 * block / 1e3 / 34.0) + cost * mb * nr * per;
                const double us = 5.9 + (1.0 + (rounds - 1.0) * 0.78) * one + (splits > 1 ? 2.5 + splits * (double)m * (double)n * 8.0 * 0.7 / 4.0e6 : 0.0);
                if (!have || us < best.us) best = {mb, nr, splits, kw_waves(mb, nr, (double)wgs / 256.0, type), us, (double)wgs / 256.0}, have = true;
            }
        }
    return best;
}

// The same for the row kernels, whose tile and K split are the plan's.
static double rows_us(const GemmPlan &p, int64_t m, int64_t n, uint32_t type) {
    const double half = type == kTypeQ4K ? 1.17 : type == kTypeQ5K ? 1.47 : type == kTypeQ6K ? 1.98 : type == kTypeQ8_0 ? 2.88 : type == kTypeQ3K ? 1.52 : 1.31;
    const int64_t wgs = (n + 255) / 256 * (p.mp / (32 * p.mb)) * p.splits;
    return 9.6 + (double)((wgs + 255) / 256) * 2.0 * p.chunk * half * (p.mb == 4 ? 1.45 : 1.0) +
           (p.splits > 1 ? 5.5 + (double)p.splits * (double)m * (double)n * 8.0 * 0.32 / 4.0e6 : 0.0);
}

// Both again for calls of more than 64 activation rows of three super-blocks or more, the pre-pass included, fitted to 1380 drawn shapes (33 to 2048
// rows, 400 to 20000 weight rows of 2 to 56 super-blocks; rms 8 to 10 %, row kernels 11 %).  A round of 256 workgroups costs a
// tile's start and end and so much a super-block; what the last round lacks saves `part` of its share, and a machine less than
// half full saves up to `few` of the round.
struct KwFit {
    double call, round, part, few, split, split_us;  // (split_us: per million partial sums)
    double sb[6];                                    // Q4_K, Q5_K, Q6_K, Q8_0, Q3_K, Q2_K
};
constexpr KwFit kKwFits[3] = {{7.93, 0.0, 0.41, 0.25, 2.96, 3.61, {0.334, 0.407, 0.477, 0.415, 0.406, 0.341}},    // 32 x 32
                              {7.90, 0.13, 0.29, 0.22, 2.58, 4.52, {0.528, 0.603, 0.679, 0.621, 0.615, 0.564}},   // 64 x 32
                              {8.24, 1.33, 0.39, 0.26, 2.44, 3.66, {0.740, 0.881, 1.166, 0.974, 0.896, 0.767}}};  // 64 x 64
constexpr double kRowsFit[6] = {1.312, 1.460, 1.966, 2.444, 1.672, 1.472};  // half a super-block
static int fit_index(uint32_t type) {
    return type == kTypeQ4K ? 0 : type == kTypeQ5K ? 1 : type == kTypeQ6K ? 2 : type == kTypeQ8_0 ? 3 : type == kTypeQ3K ? 4 : 5;
}
// Whether the dies do not share the activations among them and each reads more of them than its cache holds.
static bool dies_read_all(int64_t m, int64_t spr, int mb, int nr, int64_t tiles, uint32_t type) {
    return m * spr * 512 > (int64_t)12 << 20 && !kw_by_m((m + 32 * mb - 1) / (32 * mb), tiles, mb, nr, block_bytes(type));
}
// Rounds are counted half way from the whole machine's to the busiest die's (even: the whole machine's): of nine blocks of the operand that the
// dies share one has two and the others one.  Without that 4 of 513 drawn shapes that went to the tiles took 1.27 to 1.33 times the rows'
// time: Q4_K 1276 x 8704 M = 615, ten blocks of activation rows; Q6_K 5344 x 9472 M = 153 62 -> 82 us, four dies with 33 workgroups for 32 compute units.
static double many_tiles_us(const KwChoice &kw, int64_t m, int64_t n, int64_t spr, uint32_t type, bool even = false) {
    const KwFit &f = kKwFits[kw.mb + kw.nr - 2];
    const int64_t mt = (m + 32 * kw.mb - 1) / (32 * kw.mb), nt = (n + 32 * kw.nr - 1) / (32 * kw.nr);
    const bool by_m = kw_by_m(mt, nt, kw.mb, kw.nr, block_bytes(type));
    const double busiest = (double)(((by_m ? mt : nt) + 7) / 8 * (by_m ? nt : mt) * kw.splits) / 32.0;
    const double r = even ? kw.rounds : (kw.rounds + busiest) / 2, whole = __builtin_ceil(r);
    const double rounds = r > 1.0 ? f.part * r + (1.0 - f.part) * whole : r < 0.5 ? 1.0 - f.few * (1.0 - 2.0 * r) : 1.0;
    const double us = f.call + rounds * (f.round + f.sb[fit_index(type)] * (double)((spr + kw.splits - 1) / kw.splits)) +
                      (kw.splits > 1 ? f.split + f.split_us * 1e-6 * kw.splits * (double)m * (double)n : 0.0);
    // (Q4_K 14336 x 4096: M = 1024, 8 MB of activations, 185 us as expected, M = 2048 590 for 377)
    return dies_read_all(m, spr, kw.mb, kw.nr, nt, type) ? us * 1.5 : us;
}
static double many_rows_us(const GemmPlan &p, int64_t m, int64_t n, uint32_t type) {
    const int64_t wgs = (n + 255) / 256 * (p.mp / (32 * p.mb)) * p.splits;
    return 10.25 + (double)((wgs + 255) / 256) * (1.84 + 2.0 * p.chunk * kRowsFit[fit_index(type)] * (p.mb == 4 ? 1.53 : 1.0)) +
           (p.splits > 1 ? 1.31 + 2.04e-6 * p.splits * (double)m * (double)n : 0.0);
}

// 17 to 32 activation rows, Q4_K, Q5_K and Q8_0: microseconds of a whole call with the tile kernel and with the short-batch kernel's
// two blocks of activations, fitted to 4900 drawn shapes of 200 to 60000 weight rows of 1 to 130 super-blocks that were timed with
// both (rms 9 and 9 %).  Both are staircases: the tile kernel's in the workgroups of the busiest compute unit, each as long as its share of
// a row, none faster than the weights come from memory (the 4-norm of the two times); the short-batch kernel's in the row
// tiles of a workgroup, taken in pairs, with a step where it no longer keeps all partial tiles to the end.
static double two_blocks_tile_us(const KwChoice &kw, int64_t m, int64_t n, int64_t spr, uint32_t type) {
    const double block = type == kTypeQ4K ? 144 : type == kTypeQ5K ? 176 : 272, work = type == kTypeQ4K ? 0.47 : type == kTypeQ5K ? 0.96 : 0.85;
    const int64_t chunk = (spr + kw.splits - 1) / kw.splits, per = (chunk + 7) / 8, wgs = (n + 32 * kw.nr - 1) / (32 * kw.nr) * kw.splits;
    const double one = 0.3 * kw.nr + (double)per * (0.79 + kw.nr * work) + 0.155 * kw.nr * (double)chunk;
    const double us = (1.0 + (kw.nr == 1 ? 0.65 : 1.0) * (double)((wgs + 255) / 256 - 1)) * one, mem = (double)n * (double)spr * block * 4.1e-7;
    return 5.1 + __builtin_sqrt(__builtin_sqrt(us * us * us * us + mem * mem * mem * mem)) +
           (kw.splits > 1 ? 2.5 + 3.7e-6 * kw.splits * (double)m * (double)n : 0.0);
}
static double two_blocks_small_us(int64_t m, int64_t n, int64_t spr, uint32_t type) {
    const int64_t run = small_run_spr(type, m), runs = (spr + run - 1) / run, tiles = (n + 15) / 16;
    const int64_t per_cu = kSmallWaves / (spr < kSmallWaves ? spr : kSmallWaves), room = 256 * per_cu / runs, slots = room < 1 ? 1 : room;
    const int64_t wgs = tiles < slots ? tiles : slots, want = (tiles + wgs - 1) / wgs, t = want < 32 ? want : 32;
    const int64_t rounds = ((tiles + t - 1) / t * runs + 256 * per_cu - 1) / (256 * per_cu);
    const bool pair = run > kSmallWaves && spr > kSmallWaves, q4 = type == kTypeQ4K, q8 = type == kTypeQ8_0;  // (two super-blocks a wave)
    const double first = pair ? (q4 ? 4.0 : 4.7) : 0.0, next = pair ? (q4 ? 4.8 : 5.9) : (q4 ? 3.2 : 3.7);
    return 8.0 + (double)rounds * (first + next * (double)((t + 1) / 2 - 1) + (2 * t > kSmallKeepTiles ? 1.6 : 0.0)) +
           (runs > 1 ? (q8 ? 2.0 : 0.6) + (q8 ? 0.63 : 1.16) * (double)runs + 6e-7 * (double)(runs * m) * (double)n : 0.0);
}

// The tile kernel's grid counts eighths of its row tiles along z, which holds 65535; tiles of 32 rows, and two ragged ends for a
// pair.  Only Q2_K at 17 to 32 rows, which takes the tile kernel at every size, has weights this tall (the row kernels take them).
constexpr int64_t kKwMaxRows = (int64_t)32 * 8 * 65534;

// the tile kernel requests up to six k-steps of items past the last one (32 bytes per row each): they lie in the workspace
static size_t kw_slack(const GemmPlan &p) { return p.kernel == GemmKernel::kWaves ? (size_t)p.mp * 256 : 0; }

// the pre-pass's items (the types without a min term have no block sums)
static size_t prep_bytes(uint32_t type, int64_t k, int mp) {
    const int groups = type == kTypeQ3K || type == kTypeQ2K ? kGroups16 : type == kTypeQ6K || type == kTypeQ8_0 ? kQ6Groups : kGroups;
    return align256((size_t)(k / 256) * 2 * groups * mp * 16);
}

static size_t plan_bytes(const GemmPlan &p, uint32_t type, int64_t n, int64_t k) {
    const size_t xs = prep_bytes(type, k, p.mp);
    const size_t part = p.splits > 1 ? align256((size_t)p.splits * p.mp * n * 4) : 0;
    return xs + align256((size_t)p.mp * 4) + part + kw_slack(p);
}

GemmPlan qgemm_plan(int64_t m, int64_t n, int64_t k, uint32_t type) {
    GemmPlan p;
    p.kernel = GemmKernel::kRows, p.nr = 1;
    // 32, 64 or 128 activation rows per workgroup; up to 192 rows 64-row blocks beat 128-row blocks (fewer K splits
    // for the same number of workgroups: 36.9 against 38.3 us at M = 128, 51.7 against 53.8 at M = 192, 14336x4096;
    // equal at 256, and from 320 rows on the larger block wins)
    p.mb = m <= 32 ? 1 : (m <= 192 ? 2 : 4);
    // few tiles (a narrow weight: k / v projections of 1024 or 2048 rows): 64-row blocks double them and halve the K
    // splits (M = 512: 1024 x 4096 28.7 -> 25.3 us, 2048 x 4096 33.8 -> 30.5; equal from 64 tiles on)
    if (p.mb == 4 && ((n + 255) / 256) * ((m + 127) / 128) <= 32) p.mb = 2;
    p.mp = (m + 32 * p.mb - 1) / (32 * p.mb) * (32 * p.mb);
    p.nw = 8;
    const int64_t spr = k / 256;
    const int64_t rows = 32 * p.nw;
    const int64_t base = (n + rows - 1) / rows * (p.mp / (32 * p.mb));
    // K split: more workgroups fill more of the machine, but every split writes and re-reads an fp32 tile of Y.
    // Estimated time = (time on a full machine) / (fraction of workgroup slots in use) + partial-tile traffic;
    // rates as measured on MI355X (about 700 TFLOP/s of this kernel, 4 TB/s for the weight stream and for the
    // partial tiles, 3 us for the extra launch).
    const double slots = 256.0;  // one workgroup per compute unit keeps the weight stream busy
    const double flops = 2.0 * (double)p.mp * (double)n * (double)k, wbytes = (double)n * (double)k * 0.5625;
    const double t_full = flops / 7.0e14 > wbytes / 4.0e12 ? flops / 7.0e14 : wbytes / 4.0e12;
    double best = 0.0;
    p.splits = 1, p.chunk = (int)spr;
    for (int64_t want = 1; want <= spr; want *= 2) {
        const int64_t chunk = (spr + want - 1) / want, splits = (spr + chunk - 1) / chunk;
        const double groups = (double)(base * splits);
        const double rounds = (double)(int64_t)((groups + slots - 1) / slots);
        const double t = t_full * rounds * slots / groups +
                         (splits > 1 ? (double)splits * (double)m * (double)n * 8.0 / 4.0e12 + 3.0e-6 : 0.0);
        if (want == 1 || t < best) best = t, p.splits = (int)splits, p.chunk = (int)chunk;
    }
    // The tile kernel (gemm_kw.hip) needs no second pass over partial tiles and no barrier per step, but reads the activations
    // once per 32 or 64 weight rows: the better one for few activation rows and for narrow weights.
    KwChoice kw = kw_choice(m, n, spr, type);
    const int run = small_run_spr(type, m);
    const bool small = qgemm_small_applies(type, m, n, k);
    bool waves;
    if (m <= kSmallMaxM) {
        // The short-batch kernels' workgroups walk 16 super-blocks of a row at a time however few of them there are, and add the
        // runs of a longer row in a launch behind; the tile kernel's waves share what there is.  Tile kernel against them, us at
        // M = 12 and how many times faster (both behind a pre-pass, 1 to 3 us of which a short-batch launch of its own no longer takes):
        //   rows of 9 to 12 super-blocks, without a K split, so that a second weight can share the launch: ahead for every type up to
        //     7168 rows of nine and 4096 of twelve (1.05 to 1.33; two weights of 4096 rows of ten together 1.07 to 1.18).  Above, the
        //     types part: 12288 rows of nine Q3_K 16.1 -> 12.9, Q5_K 15.8 -> 15.2, 9216 rows Q8_0 15.7 -> 16.3; 8192 rows of twelve
        //     Q6_K 16.7 -> 14.5, Q8_0 12.8 -> 13.6; 12288 rows Q4_K 14.6 -> 16.6
        //   rows of 17 to 20: up to 14336 rows (Q4_K 8192 x 5120 15.9 -> 13.6, Q6_K 14336 x 5120 41.4 -> 28.7).  Above, Q4_K, Q5_K and
        //     Q8_0 are behind (27648 x 5120 34.3 -> 38.8, 41.9 -> 47.0, 47.4 -> 51.5), Q3_K and Q2_K at 20480 rows (34.2 -> 40.5, 30.7
        //     -> 34.5) and not at 27648 (43.3 -> 42.1, 38.4 -> 35.4); Q6_K alone stays ahead (75.4 -> 58.4)
        //   rows of 21 to 24 and of 33 to 36, where the tiles fill half or three quarters of the machine without a K split: 5008 and
        //     8192 rows of 24 1.07 to 1.31, 7008 rows of 36 1.04 to 1.42 (one Q5_K weight is behind there, 25.0 -> 27.0; two of 6208 x 8448 44.3 -> 38.0)
        // 13 to 16, 25 to 32 and longer rows leave the short-batch kernels little idle: 14336 rows of 14, 28 and 48 0.77 to 1.10.
        // Weights of 8193 to 12288 rows are one row of tiles too many for a round of 32-row tiles and fill less than three quarters
        // of one of 64-row tiles: a single one is behind for Q5_K and Q8_0 (10818 x 5120 23.3 -> 25.2, 25.2 -> 26.8) and, with rows of 24, for
        // Q4_K and Q6_K (1.06, 1.14 times as long).  They stay here for the launch that two of a batch share: Q8_0 8957 x 4352 43.5 -> 35.6
        // for two, Q6_K 9465 x 5632 56.6 -> 45.5.
        if (spr > 8 && spr <= 12) {
            waves = n <= (spr == 9 ? 7168 : 4096);
            if (waves) kw.splits = 1, kw.nr = 1, kw.nw = kw_waves(1, 1, (double)((n + 31) / 32) / 256.0, type);
        } else if (spr > 16 && spr <= 20) {
            waves = n <= 14336;
        } else {
            const double filled = spr > 20 && spr <= 24 ? 0.5 : spr > 32 && spr <= 36 && type != kTypeQ8_0 ? 0.75 : 1.0;
            waves = kw.splits == 1 && kw.rounds > filled && kw.rounds <= 1.0;
        }
    } else if (m <= kSmallMaxM2) {
        // 17 to 32 rows, against the short-batch kernels with two blocks of activations or, for the types without them, the
        // 32-row blocks: below 96 Mi elements (Q4_K 4096 x 4096 12.8 -> 10.9 us, Q6_K 21.9 -> 13.4, 14336 x 4096 29.2 -> 26.1; behind at
        // 128256 x 4096: Q4_K 87 -> 103, Q6_K 141 -> 154) and where a row is not whole runs (32000 x 5120: Q4_K 50.8 -> 40.5)
        waves = n * k < ((int64_t)96 << 20) || (small && spr > run && spr % run != 0 && type != kTypeQ8_0);
        waves = waves || (type == kTypeQ2K);  // (no short-batch form for two blocks; ahead at most sizes: 128256 x 4096 98 -> 90 us; 0.85 over 765 drawn shapes)
        // Not where the short-batch kernel's two blocks are expected to be clearly ahead: long rows, and rounds of workgroups that end soon
        // after they began (Q5_K 17096 x 19712 135.3 -> 83.7 us, 16796 x 22016 150.3 -> 98.8, 4355 x 26112 63.4 -> 44.9, Q4_K 17542 x
        // 14848 79.5 -> 59.4, Q8_0 37321 x 2048 35.8 -> 26.7).  By how much follows from the fits' errors and from the launch that two
        // weights of a batch share, which the short-batch kernel's runs cannot (two of Q8_0 6772 x 8192 39.8 us, in runs 50.5): closely
        // for the long rows of Q4_K and Q5_K, on which two weights gain nothing.
        if (small && spr > 2) {
            const double margin = spr > 32 && type != kTypeQ8_0 ? 1.05 : spr > run ? 1.25 : 1.2;
            waves = waves && two_blocks_tile_us(kw, m, n, spr, type) < margin * two_blocks_small_us(m, n, spr, type);
        }
    } else {
        // against the row kernels, by the times fitted to both over 1000...14336 weight rows of 1024...14336 elements and
        // 64...2048 activation rows (within 2 % of the better one there on average; over 1600 shapes drawn
        // up to 60000 rows of 130 super-blocks within 3 %, one in ten more than a tenth from it); from the third round of
        // workgroups on (Q6_K, two matrix instructions per step: the second; Q8_0, whose row kernel is the slowest: the
        // fifth) the row kernels, which read the activations once per 256 weight rows, are ahead
        const double t_rows = rows_us(p, m, n, type);
        waves = kw.rounds <= (type == kTypeQ6K ? 1.9 : type == kTypeQ8_0 ? 4.0 : type == kTypeQ3K || type == kTypeQ5K ? 2.1 : 2.6) && kw.us < t_rows;
        // With four waves to a workgroup the tiles stay ahead for longer: over the 1380 shapes 0.945 of the time that the line above
        // gives.  us of a call, rows -> tiles: Q4_K 4096 x 4096 M = 512 40 -> 35, 1024 x 4096 M = 2048 45 -> 37, Q8_0 14336 x 4096 M = 512
        // 143 -> 116; 14336 x 4096 Q4_K M = 512, 1792 tiles, stays with the rows, 79 to 94.  Not one block of rows, where the row
        // kernels read nothing twice, either, and not rows of one or two super-blocks, which leave half of the waves without work.
        if (!waves && m > 64 && spr > 2) {
            const double rows = 0.97 * many_rows_us(p, m, n, type);
            waves = many_tiles_us(kw, m, n, spr, type) < rows;
            // (but the tiles, if only uneven dies speak against them, where the rows' K split does not fit the scratch of the entry point that
            // allocates nothing: Q4_K 1605 x 8448 M = 636 66.8 us, 50.1 with 41 MB of scratch)
            if (!waves && plan_bytes(p, type, n, k) > PMETAL_HIP_NOALLOC_SCRATCH_BYTES) waves = many_tiles_us(kw, m, n, spr, type, true) < rows;
        }
    }
    if (small) {
        // short batches: rows longer than a run are cut into runs of 16 (or 8) super-blocks, these kernels' K split
        p.kernel = GemmKernel::kSmall;
        p.chunk = spr > run ? run : (int)spr, p.splits = (int)((spr + p.chunk - 1) / p.chunk);
    }
    if (waves && n <= kKwMaxRows) {
        GemmPlan t = p;
        t.kernel = GemmKernel::kWaves;
        t.mb = kw.mb, t.nr = kw.nr, t.nw = kw.nw, t.splits = kw.splits, t.chunk = (int)((spr + kw.splits - 1) / kw.splits);
        // (one padding for both block heights and for the row kernels of the batch's wider weights: they share their converted activations)
        t.mp = (int)(m <= 32 ? 32 : m <= 192 ? (m + 63) / 64 * 64 : (m + 127) / 128 * 128);
        // ... where that fits the array of the entry point that allocates nothing; the tiles themselves need whole blocks of 64
        if (m > 192 && plan_bytes(t, type, n, k) > PMETAL_HIP_NOALLOC_SCRATCH_BYTES) t.mp = (int)((m + 63) / 64 * 64);
        // its items past the end (and now and then more splits) take more scratch: not where only the other kernel's fits that array
        if (plan_bytes(t, type, n, k) <= PMETAL_HIP_NOALLOC_SCRATCH_BYTES || plan_bytes(p, type, n, k) > PMETAL_HIP_NOALLOC_SCRATCH_BYTES) p = t;
    }
    return p;
}

size_t qgemm_workspace_bytes(uint32_t type, int64_t m, int64_t n, int64_t k) { return plan_bytes(qgemm_plan(m, n, k, type), type, n, k); }

static bool pair_plan(int64_t m, int64_t n0, int64_t n1, int64_t k, uint32_t type, GemmPlan *plan, int *second_nw) {
    if (!qgemm_fits(type, m, n0 + n1, k)) return false;
    const GemmPlan p = qgemm_plan(m, n0, k, type), q = qgemm_plan(m, n1, k, type);
    // the same kernel for both and no K split: every result is then the sum, in the same order, that it is in a call of its own
    if (p.kernel != q.kernel || p.mp != q.mp || p.splits > 1 || q.splits > 1) return false;
    *plan = p, *second_nw = q.nw;
    // Short batches and wave tiles gain the second launch's start and the idle end of the first (us for two weights sharing their
    // activations, apart -> together: Q4_K 14336 x 4096 M = 16 27.2 -> 21.7, M = 64 41.9 -> 41.0; Q6_K 4096 x 4096 M = 16 21.9 ->
    // 13.4).  Row kernels, one workgroup per compute unit, only where a round of workgroups that neither weight fills goes
    // (Q4_K 14336 x 4096 M = 2048 566 -> 525; with as many rounds together 9728 x 2560 M = 512 was 86 -> 93).
    if (p.kernel == GemmKernel::kRows) {
        if (p.mb != q.mb) return false;
        auto rounds = [&](int64_t tiles) { return (tiles * (p.mp / (32 * p.mb)) + 255) / 256; };
        const int64_t t0 = (n0 + 255) / 256, t1 = (n1 + 255) / 256;
        return rounds(t0 + t1) < rounds(t0) + rounds(t1);
    }
    if (p.kernel == GemmKernel::kWaves) {
        if (n0 + n1 > kKwMaxRows) return false;
        const KwChoice kw = kw_choice(m, n0 + n1, k / 256, type);
        if (kw.splits == 1) plan->mb = kw.mb, plan->nr = kw.nr;
        // One weight's tiles have four waves, the other's eight: a launch of its own for each costs 4 to 6 us more, workgroups of eight waves
        // for both what two workgroups of four on a compute unit gain. us, together / apart: Q4_K 4096 and 1024 x 4096, M = 100 17.6 / 20.9, Q6_K M = 96 20.1 /
        // 28.0, Q8_0 2048 and 512 x 2048 M = 160 11.3 / 16.2; two and a half rounds of 64 x 32 tiles of Q8_0 2560 and 1280 x 2560 M = 300 30.6 / 26.9, Q4_K
        // 1008 and 504 x 5888 M = 720, twelve blocks of activation rows on eight dies, 51.1 / 39.3.
        // Times as long together as apart, by rounds, over 1150 drawn pairs with rows of more than four super-blocks (shorter ones have as many waves
        // either way): up to one 0.70 to 0.89; to one and a half 1.03 to 1.17, 32 x 32 tiles 0.88; to two 0.86 to 0.94; above 1.00 to 1.09. Over 500 others so
        // 0.83 (0.84 all together), ten of the 448 that are together 2 to 12 % longer.
        const int64_t spr = k / 256, nt0 = (n0 + 32 * plan->nr - 1) / (32 * plan->nr), nt1 = (n1 + 32 * plan->nr - 1) / (32 * plan->nr), nt = nt0 + nt1;
        if (p.nw != q.nw && spr > 4) {
            const int64_t mt = (m + 32 * plan->mb - 1) / (32 * plan->mb);
            const double rounds = kw_mixed(mt, p.nw == 4 ? nt0 : nt1, p.nw == 4 ? nt1 : nt0, kw_by_m(mt, nt, plan->mb, plan->nr, block_bytes(type)), plan->mb, plan->nr).rounds;
            if (rounds > 2.0 || (rounds > 1.0 && rounds <= 1.5 && plan->mb * plan->nr > 1)) return false;
        }
        // Tiles of which alone the dies share the activations, and together, more weight rows than activation rows then, the weights. That
        // costs from some 1300 activation rows on; Q8_0's tiles, which take longer, from 1900, Q6_K's nothing. us, together / apart, two
        // weights: Q4_K 4600 x 4096 M = 2048 390 / 232, 3322 x 4864 M = 1487 206 / 155, 2352 x 5888 M = 1081 111 / 139, Q2_K 5502 x 9216 M = 1709 927 / 533,
        // Q5_K 3032 and 1694 x 7168 M = 1456 224 / 193, Q8_0 2932 x 6912 M = 2004 373 / 329, 1891 x 7936 M = 1540 216 / 226, Q6_K 3366 x 4608 M = 2362 370 / 380.
        auto alone = [&](const GemmPlan &a, int64_t n) { return dies_read_all(m, spr, a.mb, a.nr, (n + 32 * a.nr - 1) / (32 * a.nr), type); };
        const int64_t most = type == kTypeQ6K ? m : type == kTypeQ8_0 ? 1900 : 1280;
        if (m > most && dies_read_all(m, spr, plan->mb, plan->nr, nt, type) && !(alone(p, n0) && alone(q, n1))) return false;
    }
    return true;
}

bool qgemm_pair_plan(int64_t m, int64_t n0, int64_t n1, int64_t k, uint32_t type, GemmPlan *plan) {
    int second_nw;
    return pair_plan(m, n0, n1, k, type, plan, &second_nw);
}

// Tiles of `rows` weight rows along the grid; with a second weight also where its tiles begin and the bit that says so.
static unsigned tiles_of_both(int64_t n, int rows, GemmSecond &second, int &mode) {
    const unsigned tiles = (unsigned)((n + rows - 1) / rows);
    if (second.n == 0) return tiles;
    second.first = (int)tiles, mode |= kHasSecond;
    return tiles + (unsigned)((second.n + rows - 1) / rows);
}

template <int ORDER, int MB, int NR, int NW, int FMT = 0>
static hipError_t launch_rw(hipStream_t s, const uint8_t *w, const uint4 *xs, const float *rowscale, void *y, float *partial,
                            int64_t m, int64_t n, int spr, const GemmPlan &p, int mode, GemmSecond second) {
    auto kern = k_qgemm_rw<ORDER, MB, NR, NW, FMT>;
    constexpr size_t lds = rw_lds_bytes<MB, NR, NW, FMT>();
    constexpr int kRows = 32 * NR * NW;
    if (lds > 64 * 1024) {
        hipError_t a = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (a != hipSuccess) return a;
    }
    const dim3 grid(tiles_of_both(n, kRows, second, mode), (unsigned)(p.mp / (32 * MB)), (unsigned)p.splits);
    hipLaunchKernelGGL(kern, grid, dim3(64 * NW), lds, s, w, xs, rowscale, y, partial, (int)m, (int)p.mp, (int)n, spr, p.chunk, mode, second);
    return hipGetLastError();
}

template <int FMT, int MB>
static hipError_t launch_rw16(hipStream_t s, const uint8_t *w, const uint4 *xs, const float *rowscale, void *y, float *partial, int64_t m,
                              int64_t n, int spr, const GemmPlan &p, int mode, GemmSecond second) {
    auto kern = k_qgemm_rw16<FMT, MB>;
    constexpr size_t lds = rw16_lds_bytes<FMT, MB>();
    if (lds > 64 * 1024) {
        hipError_t a = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (a != hipSuccess) return a;
    }
    const dim3 grid(tiles_of_both(n, 256, second, mode), (unsigned)(p.mp / (32 * MB)), (unsigned)p.splits);
    hipLaunchKernelGGL(kern, grid, dim3(512), lds, s, w, xs, rowscale, y, partial, (int)m, (int)p.mp, (int)n, spr, p.chunk, mode, second);
    return hipGetLastError();
}

template <int MB>
static hipError_t launch_rw_q6(hipStream_t s, const uint8_t *w, const uint4 *xs, const float *rowscale, void *y, float *partial,
                               int64_t m, int64_t n, int spr, const GemmPlan &p, int mode, GemmSecond second) {
    auto kern = k_qgemm_rw_q6<MB>;
    constexpr size_t stages = (size_t)(2 * kQ6Groups * 32 * MB + 8 * (3 * kQ6Stage + 64)) * 16;
    constexpr size_t lds = stages > tile_lds_bytes<MB>() ? stages : tile_lds_bytes<MB>();
    hipError_t a = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (a != hipSuccess) return a;
    const dim3 grid(tiles_of_both(n, 256, second, mode), (unsigned)(p.mp / (32 * MB)), (unsigned)p.splits);
    hipLaunchKernelGGL(kern, grid, dim3(512), lds, s, w, xs, rowscale, y, partial, (int)m, (int)p.mp, (int)n, spr, p.chunk, mode, second);
    return hipGetLastError();
}

template <int MB>
static hipError_t launch_rw_q8(hipStream_t s, const uint8_t *w, const uint4 *xs, const float *rowscale, void *y, float *partial,
                               int64_t m, int64_t n, int spr, const GemmPlan &p, int mode, GemmSecond second) {
    auto kern = k_qgemm_rw_q8<MB>;
    constexpr size_t stages = (size_t)(2 * kQ6Groups * 32 * MB) * 16;
    constexpr size_t lds = stages > tile_lds_bytes<MB>() ? stages : tile_lds_bytes<MB>();
    if (lds > 64 * 1024) {
        hipError_t a = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (a != hipSuccess) return a;
    }
    const dim3 grid(tiles_of_both(n, 256, second, mode), (unsigned)(p.mp / (32 * MB)), (unsigned)p.splits);
    hipLaunchKernelGGL(kern, grid, dim3(512), lds, s, w, xs, rowscale, y, partial, (int)m, (int)p.mp, (int)n, spr, p.chunk, mode, second);
    return hipGetLastError();
}

// LDS of a short-batch workgroup: the finished tiles, a partial tile per wave (of each of few tiles until the end, or two in turn) and the
// waves' stages; before the first tile the activations that the waves convert pass through the same.
size_t qgemm_small_lds(uint32_t type, int64_t m, int64_t k, int tiles_per_wg, bool own, bool xf32) {
    const int spr = (int)(k / 256), nwaves = spr < kSmallWaves ? spr : kSmallWaves, mt = m > kSmallMaxM ? 2 : 1;
    const bool two = small_run_spr(type, m) > kSmallWaves && spr > kSmallWaves;  // super-blocks a wave
    const int tiles = (tiles_per_wg + kSmallDepth - 1) / kSmallDepth * kSmallDepth * mt;
    size_t stage = 0;  // (Q3_K and Q2_K: none)
    if (type == kTypeQ4K) stage = 16 * (two ? SmallRun<2, 0>::kPieces : SmallRun<1, 0>::kPieces);
    else if (type == kTypeQ5K) stage = 16 * (two ? SmallRun<2, 1>::kPieces : SmallRun<1, 1>::kPieces);
    else if (type == kTypeQ6K) stage = 4 * (two ? SmallQ6<2, true>::kStageDwords : SmallQ6<1>::kStageDwords);
    else if (type == kTypeQ8_0) stage = 16 * (two ? 2 : 1) * kQ8TileRunPieces;
    const size_t work = (size_t)(tiles + (tiles_per_wg * mt <= kSmallKeepTiles ? tiles : 2) * nwaves) * 1024 + nwaves * stage;
    const size_t x_lds = own ? (size_t)nwaves * (xf32 ? 2 : 1) * kSmallXItems * 16 : 0;
    return work > x_lds ? work : x_lds;
}

hipError_t launch_copy_x(const void *x, size_t bytes, void *to, hipStream_t s) {
    const size_t items = bytes / 16;  // (whole super-blocks)
    hipLaunchKernelGGL(k_copy16, dim3((unsigned)((items + 255) / 256)), dim3(256), 0, s, reinterpret_cast<const uint4 *>(x), reinterpret_cast<uint4 *>(to), items);
    return hipGetLastError();
}

hipError_t launch_qgemm(uint32_t type, const uint8_t *w, int64_t n, int64_t k, const void *x, uint32_t x_dtype,
                                int64_t m, void *y, uint32_t y_dtype, uint32_t order, void *workspace, hipStream_t s, bool reuse_prepass,
                                const GemmSecond &second_weight, bool shared) {
    if (!qgemm_fits(type, m, n, k)) return hipErrorInvalidValue;
    GemmSecond second = second_weight;
    GemmPlan p;
    int second_nw = 0;  // kWaves: the waves of the second weight's tiles, as its own plan has them
    if (second.n == 0) p = qgemm_plan(m, n, k, type);
    else if (!pair_plan(m, n, second.n, k, type, &p, &second_nw)) return hipErrorInvalidValue;
    const int spr = (int)(k / 256);
    uint8_t *ws = reinterpret_cast<uint8_t *>(workspace);
    uint4 *xs = reinterpret_cast<uint4 *>(ws);
    const bool q23 = type == kTypeQ3K || type == kTypeQ2K;
    const size_t xs_bytes = prep_bytes(type, k, p.mp);
    float *rowscale = reinterpret_cast<float *>(ws + xs_bytes);
    float *partial = reinterpret_cast<float *>(ws + xs_bytes + align256((size_t)p.mp * 4));
    const bool xf32 = x_dtype == kDtypeF32, q6 = type == kTypeQ6K, q8 = type == kTypeQ8_0, q5 = type == kTypeQ5K, ref = order == kOrderRef;
    const int xorder = q23 ? 5 : (q8 ? 3 : (q6 ? 2 : (ref ? (q5 ? 4 : 0) : 1)));  // the element order the pre-pass lays the activations out for
    // Rows per workgroup: one for few rows (a chain of latencies: 512 threads on it), two from 384 rows on and four from 1024 on,
    // whose threads write 32 and 64 bytes at a place instead of 16 (us of the pre-pass with one / two / four rows, bf16, k = 14336:
    // M = 64 7.6 / 8.7 / 15.2, M = 512 15.1 / 9.8 / 14.0, M = 2048 56 / 35 / 27).  An item count beyond eight per thread is read twice.
    // Threads hold 1, 2, 3, 4, 6 or 8 items, the least that is enough: what a row does not fill is its last item again (bf16, k = 10240,
    // 2.5 or 5 items a thread held as 4 or 8: M = 2048 27.0 -> 19.5 us, k = 5120, M = 1500 14.2 -> 12.6; read twice 22.5, 12.7).
    const int per_wg = p.mp >= 1024 ? 4 : p.mp >= 384 ? 2 : 1;
    const int64_t ni = (k / 8 * per_wg + (per_wg == 1 ? 511 : 1023)) / (per_wg == 1 ? 512 : 1024);
#define PMH_PREP_N(F, O, R, NI)                                                                                              \
    hipLaunchKernelGGL((k_prep_rw<F, O, R, NI>), dim3((unsigned)p.mp / (R)), dim3((R) == 1 ? 512 : 1024), 0, s, x, k, (int)m, \
                       (int)p.mp, rowscale, xs, arrived, n_arrived)
#define PMH_PREP_R(F, O, R)                       \
    do {                                          \
        if (ni <= 1) PMH_PREP_N(F, O, R, 1);      \
        else if (ni <= 2) PMH_PREP_N(F, O, R, 2); \
        else if (ni <= 3) PMH_PREP_N(F, O, R, 3); \
        else if (ni <= 4) PMH_PREP_N(F, O, R, 4); \
        else if (ni <= 6) PMH_PREP_N(F, O, R, 6); \
        else if (ni <= 8) PMH_PREP_N(F, O, R, 8); \
        else PMH_PREP_N(F, O, R, 0);              \
    } while (0)
#define PMH_PREP(F, O)                          \
    do {                                        \
        if (per_wg == 4) PMH_PREP_R(F, O, 4);   \
        else if (per_wg == 2) PMH_PREP_R(F, O, 2); \
        else PMH_PREP_R(F, O, 1);               \
    } while (0)
    // The tile kernel adds the splits of K itself where this call's pre-pass has cleared its counters, at most 256 of them: they lie in the slack
    // behind the partial tiles, 8 KiB and more.
    const int64_t kw_tiles = ((n + 32 * p.nr - 1) / (32 * p.nr)) * ((m + 32 * p.mb - 1) / (32 * p.mb));
    const bool joined = p.kernel == GemmKernel::kWaves && p.splits > 1 && joins_splits(p.mb, p.nr) && !reuse_prepass && kw_tiles <= 256;
    uint32_t *const arrived = joined ? reinterpret_cast<uint32_t *>(ws + plan_bytes(p, type, n, k) - kw_slack(p)) : nullptr;
    const int n_arrived = joined ? (int)kw_tiles : 0;
    const bool own = qgemm_converts_itself(p, type, m, n, second.n, k, x_dtype, shared);
    if (own) {
        // Every wave converts what it multiplies.  Results over the activations would race with other workgroups' reads of them.
        const uintptr_t xb = reinterpret_cast<uintptr_t>(x), xe = xb + (size_t)m * k * (xf32 ? 4 : 2);
        auto over_x = [&](const void *out, int64_t rows) {
            const uintptr_t b = reinterpret_cast<uintptr_t>(out);
            return b < xe && xb < b + (size_t)m * rows * (y_dtype == kDtypeF32 ? 4 : 2);
        };
        if (over_x(y, n) || (second.n > 0 && over_x(second.y, second.n))) {  // (16 f32 rows are what 32 rows of items take)
            const hipError_t e = launch_copy_x(x, xe - xb, xs, s);
            if (e != hipSuccess) return e;
            x = xs;
        }
    } else if (reuse_prepass) {
        // the workspace still holds the converted activations of the previous call (same x, m, k and weight type)
    } else if (qgemm_small_rows(p, m)) {
#define PMH_PAIRS(F, O) hipLaunchKernelGGL((k_prep_pairs<F, O>), dim3((unsigned)((spr + 1) / 2)), dim3(128), 0, s, x, (int)m, spr, xs)
#define PMH_PAIRS_X(O)               \
    do {                             \
        if (xf32) PMH_PAIRS(true, O); \
        else PMH_PAIRS(false, O);    \
    } while (0)
        if (xorder == 0) PMH_PAIRS_X(0);
        else if (xorder == 1) PMH_PAIRS_X(1);
        else if (xorder == 2) PMH_PAIRS_X(2);
        else if (xorder == 3) PMH_PAIRS_X(3);
        else if (xorder == 4) PMH_PAIRS_X(4);
        else PMH_PAIRS_X(5);
#undef PMH_PAIRS_X
#undef PMH_PAIRS
    } else if (xf32) {
        if (xorder == 0) PMH_PREP(true, 0);
        else if (xorder == 1) PMH_PREP(true, 1);
        else if (xorder == 2) PMH_PREP(true, 2);
        else if (xorder == 3) PMH_PREP(true, 3);
        else if (xorder == 4) PMH_PREP(true, 4);
        else PMH_PREP(true, 5);
    } else {
        if (xorder == 0) PMH_PREP(false, 0);
        else if (xorder == 1) PMH_PREP(false, 1);
        else if (xorder == 2) PMH_PREP(false, 2);
        else if (xorder == 3) PMH_PREP(false, 3);
        else if (xorder == 4) PMH_PREP(false, 4);
        else PMH_PREP(false, 5);
    }
#undef PMH_PREP
#undef PMH_PREP_R
#undef PMH_PREP_N
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const bool ybf = y_dtype == kDtypeBf16;
    if (p.kernel == GemmKernel::kWaves) {
        e = launch_qgemm_kw(type, p, w, xs, rowscale, y, ybf, m, n, spr, order, partial, arrived, second, second_nw, s);
        if (e != hipSuccess || p.splits == 1 || joined) return e;
    } else if (p.kernel == GemmKernel::kSmall) {
        const int nwaves = spr < kSmallWaves ? spr : kSmallWaves;
        const int tiles = (int)((n + 15) / 16);
        const int run = small_run_spr(type, m);
        const int tiles1 = (second.n + 15) / 16;  // of the second weight
        const int tiles_per_wg = small_tiles_per_wg(p, m, n, second.n, k);
        const int mt = m > kSmallMaxM ? 2 : 1;  // 16-row blocks of activations
        // a long row: p.splits runs, one workgroup row of the grid each, partial tiles for k_rw_reduce
        const int runs = p.splits;
        float *const part_out = runs > 1 ? partial : nullptr;
        const int nsb = run > kSmallWaves && spr > kSmallWaves ? 2 : 1;
        second.first = (tiles + tiles_per_wg - 1) / tiles_per_wg;
        const int ybf16 = (ybf ? 1 : 0) | (tiles1 > 0 ? kHasSecond : 0);
        const dim3 grid((unsigned)(second.first + (tiles1 + tiles_per_wg - 1) / tiles_per_wg), (unsigned)runs), block((unsigned)(64 * nwaves));
        const size_t bytes = qgemm_small_lds(type, m, k, tiles_per_wg, own, xf32);
        // (LDS beyond the launch default has to be asked for)
        auto go = [&](auto kern, auto... args) {
            if (bytes > 48 * 1024) {
                const hipError_t a = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
                if (a != hipSuccess) return a;
            }
            hipLaunchKernelGGL(kern, grid, block, bytes, s, args...);
            return hipGetLastError();
        };
        const void *const xa = own ? x : (const void *)xs;
        if (q23) {
#define PMH_SMALL16(F, S, X) go(k_qgemm_small16<F, S, X>, w, xa, y, (int)m, (int)p.mp, (int)n, spr, tiles, tiles_per_wg, ybf16, part_out, second)
            if (type == kTypeQ2K) {
                if (nsb == 2) e = !own ? PMH_SMALL16(3, 2, 3) : xf32 ? PMH_SMALL16(3, 2, 2) : PMH_SMALL16(3, 2, 1);
                else e = xf32 ? PMH_SMALL16(3, 1, 2) : PMH_SMALL16(3, 1, 1);
            } else {
                if (nsb == 2) e = own ? PMH_SMALL16(2, 2, 1) : PMH_SMALL16(2, 2, 3);
                else e = xf32 ? PMH_SMALL16(2, 1, 2) : PMH_SMALL16(2, 1, 1);
            }
#undef PMH_SMALL16
        } else if (q6) {
            const bool any = spr % 8 != 0;  // rows that do not start on 16-byte boundaries
            const uint32_t w_last = (uint32_t)(((uint64_t)n * (uint64_t)spr * 210u - 1) & ~(uint64_t)15);
#define PMH_SMALL_Q6(S, A, X) go(k_qgemm_small_q6<S, A, X>, w, xa, y, (int)m, (int)p.mp, (int)n, spr, tiles, tiles_per_wg, ybf16, w_last, part_out, second)
            if (nsb == 2 && any) e = !own ? PMH_SMALL_Q6(2, true, 3) : xf32 ? PMH_SMALL_Q6(2, true, 2) : PMH_SMALL_Q6(2, true, 1);
            else if (nsb == 2) e = !own ? PMH_SMALL_Q6(2, false, 3) : xf32 ? PMH_SMALL_Q6(2, false, 2) : PMH_SMALL_Q6(2, false, 1);
            else if (any) e = xf32 ? PMH_SMALL_Q6(1, true, 2) : PMH_SMALL_Q6(1, true, 1);
            else e = xf32 ? PMH_SMALL_Q6(1, false, 2) : PMH_SMALL_Q6(1, false, 1);
#undef PMH_SMALL_Q6
        } else if (q8) {
#define PMH_SMALL_Q8(S, T, X) go(k_qgemm_small_q8<S, T, X>, w, xa, rowscale, y, (int)m, (int)p.mp, (int)n, spr, tiles, tiles_per_wg, ybf16, part_out, second)
            if (mt == 2) e = PMH_SMALL_Q8(1, 2, 0);  // (two blocks of activations: one run of eight blocks per wave)
            else if (nsb == 2) e = own ? PMH_SMALL_Q8(2, 1, 1) : PMH_SMALL_Q8(2, 1, 3);
            else e = xf32 ? PMH_SMALL_Q8(1, 1, 2) : PMH_SMALL_Q8(1, 1, 1);
#undef PMH_SMALL_Q8
        } else {
            static_assert(2 * kSmallWaves >= kSmallMaxSpr, "two super-blocks per wave must cover the longest row");
#define PMH_SMALL_X(O, S, F, T, X) go(k_qgemm_small<O, S, F, T, X>, w, xa, rowscale, y, (int)m, (int)p.mp, (int)n, spr, tiles, tiles_per_wg, ybf16, part_out, second)
#define PMH_SMALL_F(O, S, F) (mt == 2 ? PMH_SMALL_X(O, S, F, 2, 0) : xf32 ? PMH_SMALL_X(O, S, F, 1, 2) : PMH_SMALL_X(O, S, F, 1, 1))
#define PMH_SMALL_2(O, F) (mt == 1 && !own ? PMH_SMALL_X(O, 2, F, 1, 3) : PMH_SMALL_F(O, 2, F))
            if (spr > kSmallWaves) e = ref ? (q5 ? PMH_SMALL_2(0, 1) : PMH_SMALL_2(0, 0)) : (q5 ? PMH_SMALL_2(1, 1) : PMH_SMALL_2(1, 0));
            else e = ref ? (q5 ? PMH_SMALL_F(0, 1, 1) : PMH_SMALL_F(0, 1, 0)) : (q5 ? PMH_SMALL_F(1, 1, 1) : PMH_SMALL_F(1, 1, 0));
#undef PMH_SMALL_2
#undef PMH_SMALL_F
#undef PMH_SMALL_X
        }
        if (mt == 1) rowscale = nullptr;  // the tiles leave scaled
        if (e != hipSuccess || runs == 1) return e;
    } else {
    const int mode = p.splits > 1 ? 2 : (ybf ? 1 : 0);
#define PMH_RW_CASE(O, B, R, NWV) launch_rw<O, B, R, NWV>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second)
    if (q8) {
        e = p.mb == 1   ? launch_rw_q8<1>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second)
            : p.mb == 2 ? launch_rw_q8<2>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second)
                        : launch_rw_q8<4>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second);
    } else if (q6) {
        e = p.mb == 1   ? launch_rw_q6<1>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second)
            : p.mb == 2 ? launch_rw_q6<2>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second)
                        : launch_rw_q6<4>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second);
    } else if (q23) {
        e = type == kTypeQ2K ? (p.mb == 1   ? launch_rw16<3, 1>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second)
                                : p.mb == 2 ? launch_rw16<3, 2>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second)
                                            : launch_rw16<3, 4>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second))
                             : (p.mb == 1   ? launch_rw16<2, 1>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second)
                                : p.mb == 2 ? launch_rw16<2, 2>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second)
                                            : launch_rw16<2, 4>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second));
    } else if (q5) {
#define PMH_RW5_CASE(O, B) launch_rw<O, B, 1, 8, 1>(s, w, xs, rowscale, y, partial, m, n, spr, p, mode, second)
        e = p.mb == 1   ? (ref ? PMH_RW5_CASE(0, 1) : PMH_RW5_CASE(1, 1))
            : p.mb == 2 ? (ref ? PMH_RW5_CASE(0, 2) : PMH_RW5_CASE(1, 2))
                        : (ref ? PMH_RW5_CASE(0, 4) : PMH_RW5_CASE(1, 4));
#undef PMH_RW5_CASE
    } else if (p.mb == 1) {
        e = ref ? PMH_RW_CASE(0, 1, 1, 8) : PMH_RW_CASE(1, 1, 1, 8);
    } else if (p.mb == 2) {
        e = ref ? PMH_RW_CASE(0, 2, 1, 8) : PMH_RW_CASE(1, 2, 1, 8);
    } else {
        e = ref ? PMH_RW_CASE(0, 4, 1, 8) : PMH_RW_CASE(1, 4, 1, 8);
    }
#undef PMH_RW_CASE
    if (e != hipSuccess || p.splits == 1) return e;
    }
    // the partial tiles of a K split (of the large kernels or of the short-batch kernels' runs), added in split order
    const size_t total = (size_t)m * n;
    const bool few = total < ((size_t)1 << 17);
    const dim3 rgrid((unsigned)((total + (few ? 255 : 2047)) / (few ? 256 : 2048)));
#define PMH_REDUCE(B, P) hipLaunchKernelGGL((k_rw_reduce<B, P>), rgrid, dim3(256), 0, s, partial, p.splits, (int)m, (int)p.mp, (int)n, rowscale, y)
    if (ybf && few) PMH_REDUCE(true, 1);
    else if (ybf) PMH_REDUCE(true, 8);
    else if (few) PMH_REDUCE(false, 1);
    else PMH_REDUCE(false, 8);
#undef PMH_REDUCE
    return hipGetLastError();
}

}  // namespace pmh
