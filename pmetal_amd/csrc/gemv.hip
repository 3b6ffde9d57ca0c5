// Dequant-fused GEMV  y[n] = sum_k W[n,k] * x[k]  for Q6_K and Q8_0 weights on gfx950, and the
// dispatch over weight types (Q4_K lives in gemv_q4k.hip).
//
// W is the packed GGUF block stream, row-major [n, k]; the value of a weight is what the
// reference's dequantize yields (k_quants.rs:474-496 for Q6_K, dequant.rs:466-495 for Q8_0).  The
// reference has no fused kernel: it dequantizes on the CPU at load
// (crates/pmetal-models/src/weight_format.rs:299) and multiplies dense; these kernels are checked
// against exactly that (dequantize, then matmul), to 1e-3.
//
//  * A "team" of T lanes takes one weight row; for Q6_K 8 lanes share a 210-byte
//    super-block, for Q8_0 one lane owns a 34-byte block.  Blocks are only 2-byte aligned, so the
//    loads are unaligned dword loads, which the hardware supports.  T follows from the shape (row_teams), not from what divides the row:
//    us of a launch in a replayed sequence, teams that divide the row and two rows a team -> a team a row: Q6_K 1024 x 1024 3.1 -> 2.3,
//    1024 x 3072 4.9 -> 3.6 (f32 x 8.2 -> 4.1), 1024 x 3584 7.4 -> 3.6, 8192 x 1024 4.7 -> 4.0, 1024 x 11008 31 -> 7.2; Q8_0 3072 x 1024 f32 x
//    3.7 -> 3.1, 1024 x 3584 11.8 -> 3.5, 8192 x 1280 9.5 -> 5.3, 1024 x 11008 64 -> 6.9, 151936 x 1024 40 -> 37.5.
//  * Q6_K quants are assembled in registers into bf16 pairs: OR-ing the integer q' = q + 32 (shifted
//    by one) into the mantissa of bf16(64.0) gives exactly 64 + q', and one v_dot2c_f32_bf16
//    multiplies two of them with two activations, accumulating in fp32.  The offsets are removed
//    with per-group sums of x computed once.
//  * x is staged once per workgroup in LDS, already permuted into the pair order the unpacking
//    produces, laid out so that consecutive lanes read consecutive 16-byte words.  f32 activations
//    are split exactly into three bf16 planes (hi + mid + lo) and run through the same path thrice.
//  * The team's partial sums are reduced with DPP (quad_perm, row_half_mirror, row_mirror) and, for
//    teams wider than a 16-lane row, row broadcasts; the last lane of the team stores y[row].
#include "gemv_q6k_small.hpp"

namespace {

template <bool XF32>
__global__ __launch_bounds__(256) void k_qgemv_q6k(const uint8_t *__restrict__ W, const void *__restrict__ xg,
                                                    float *__restrict__ y, int n_rows, int spr) {
    extern __shared__ uint4 smem[];
    q6k_small_body<8, XF32>(W, xg, y, n_rows, spr, (int)blockIdx.x, (int)gridDim.x, 32, smem);
}

template <int T, bool XF32, int D>
__global__ __launch_bounds__(256) void k_qgemv_q6k_row(const uint8_t *__restrict__ W, const void *__restrict__ xg,
                                                        float *__restrict__ y, int n_rows, int spr) {
    extern __shared__ uint4 smem[];
    q6k_row_body<T, XF32, D>(W, xg, y, n_rows, spr, (int)(blockIdx.x * (blockDim.x / T) + threadIdx.x / T), smem);
}

// ------------------------------------------------------------------------------------------------
// Q8_0 (34-byte blocks of 32, 2-byte aligned).  One lane per block; 8-bit quants do not fit the
// bf16 mantissa trick, so each is sign-extended, converted and multiplied in fp32 with x held as f32
// in LDS (at 8.5 bits per weight the VALU budget per byte is twice that of Q4_K).
// LDS: xf[8][blocks] float4 (elements 32b + 4q .. +3).
// ------------------------------------------------------------------------------------------------
template <bool XF32>
__device__ __forceinline__ void stage_x_q8_0(const void *xg, int bpr, float4 *xf) {
    for (int b = threadIdx.x; b < bpr; b += blockDim.x) {
#pragma unroll
        for (int q = 0; q < 8; q++) {
            float4 v;
            if (XF32) {
                v = reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(xg) + (size_t)b * 32)[q];
            } else {
                const uint2 u =
                    reinterpret_cast<const uint2 *>(reinterpret_cast<const uint16_t *>(xg) + (size_t)b * 32)[q];
                v = make_float4(bf16_to_f32(u.x & 0xFFFFu), bf16_to_f32(u.x >> 16), bf16_to_f32(u.y & 0xFFFFu),
                                bf16_to_f32(u.y >> 16));
            }
            xf[q * bpr + b] = v;
        }
    }
}

struct Q8Raw {  // a block as it lies in memory
    u32x4_a2 a, b;
    uint32_t d;
};

__device__ __forceinline__ Q8Raw q8_0_load(const uint8_t *blk) {
    Q8Raw r;
    r.d = *reinterpret_cast<const u16_a2 *>(blk);
    r.a = *reinterpret_cast<const u32x4_a2 *>(blk + 2), r.b = *reinterpret_cast<const u32x4_a2 *>(blk + 18);
    return r;
}

__device__ __forceinline__ float q8_0_lane(const Q8Raw &raw, const float4 *xf, const int bpr, const int b) {
    const uint32_t w[8] = {raw.a.x, raw.a.y, raw.a.z, raw.a.w, raw.b.x, raw.b.y, raw.b.z, raw.b.w};
    float acc = 0.0f;
#pragma unroll
    for (int q = 0; q < 8; q++) {
        const float4 xv = xf[q * bpr + b];
        acc += (float)(int8_t)(w[q]) * xv.x;
        acc += (float)(int8_t)(w[q] >> 8) * xv.y;
        acc += (float)(int8_t)(w[q] >> 16) * xv.z;
        acc += (float)(int8_t)(w[q] >> 24) * xv.w;
    }
    return f16_bits_to_f32(raw.d) * acc;
}

// A team of T lanes takes one row, a lane a block of each chunk of T; as q6k_row_body, for the same reasons.
template <int T, bool XF32, int D>
__global__ __launch_bounds__(256) void k_qgemv_q8_0(const uint8_t *__restrict__ W, const void *__restrict__ xg,
                                                     float *__restrict__ y, int n_rows, int bpr) {
    extern __shared__ uint4 smem[];
    float4 *xf = reinterpret_cast<float4 *>(smem);
    const int lt = threadIdx.x & (T - 1), team = (int)(blockIdx.x * (blockDim.x / T) + threadIdx.x / T);
    const int iters = (bpr + T - 1) / T;
    const uint8_t *row = W + (size_t)(team < n_rows ? team : n_rows - 1) * ((size_t)bpr * 34);
    auto block_of = [&](int it) { return min(it * T + lt, bpr - 1); };
    Q8Raw c[D];
#pragma unroll
    for (int i = 0; i < D; i++) c[i] = q8_0_load(row + (uint32_t)block_of(i) * 34u);
    stage_x_q8_0<XF32>(xg, bpr, xf);
    __syncthreads();
    float acc = 0.0f;
    for (int first = 0; first < iters; first += D) {
#pragma unroll
        for (int i = 0; i < D; i++) {
            const int it = first + i;
            if (it < iters) {
                const float v = q8_0_lane(c[i], xf, bpr, block_of(it));
                acc += it * T + lt < bpr ? v : 0.0f;
                if (it + D < iters) c[i] = q8_0_load(row + (uint32_t)block_of(it + D) * 34u);
            }
        }
    }
    acc = T >= 8 ? team_sum_last<T>(acc) : team_sum<T>(acc);
    if (lt == T - 1 && team < n_rows) y[team] = acc;
}

// ------------------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------------------
constexpr int rows_per_team() { return 4; }

// Rows per team: rows_per_team() when that still leaves a workgroup for every compute unit, fewer otherwise
// (a small matrix is spread over the whole chip rather than streamed by a few workgroups).
unsigned grid_for_rows(int64_t n, int teams_per_wg, int64_t r = rows_per_team()) {
    const int64_t cus = compute_units();
    while (r > 1 && (n + teams_per_wg * r - 1) / (teams_per_wg * r) < cus) r /= 2;
    const int64_t per_wg = (int64_t)teams_per_wg * r;
    int64_t g = (n + per_wg - 1) / per_wg;
    if (g < 1) g = 1;
    if (g > (1 << 20)) g = 1 << 20;
    return (unsigned)g;
}

template <typename Kern>
hipError_t launch(Kern kern, unsigned grid, size_t lds, hipStream_t s, const uint8_t *w, const void *x, float *y,
                  int n, int units, unsigned threads = 256) {
    if (lds > kMaxLds) return hipErrorInvalidValue;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), lds, s, w, x, y, n, units);
    return hipGetLastError();
}

// Lanes of a team that takes one row of `lanes` lanes' work, by team_cost, and threads of a workgroup.
struct RowTeams {
    int team;
    unsigned threads;
};
RowTeams row_teams(int64_t n_rows, uint32_t lanes, size_t slots) {
    const uint32_t cus = (uint32_t)compute_units(), n = n_rows < (1 << 24) ? (uint32_t)n_rows : 1u << 24;
    RowTeams t{0, 256};
    uint32_t best = 0, whole = 0;
    for (uint32_t log = 6; log >= 3; log--) {
        const uint32_t cost = pmh::gemv::team_cost(n, lanes, log), fits = (lanes & ((1u << log) - 1)) == 0;
        // (as long either way: the one that the row fills)
        if (t.team == 0 || cost < best || (cost == best && fits > whole)) t.team = 1 << log, best = cost, whole = fits;
    }
    // Smaller workgroups where they spread the waves more evenly and one of them converts x in one go (us, 3072 x 1536: 192 workgroups of
    // 256 threads 3.9 us, 768 of 64 3.7; 2048 x 1280 4.8, 3.9).
    if (slots <= 128 && (uint64_t)n * t.team <= 512ull * 256 * cus) {
        auto waves_of_a_cu = [&](uint32_t threads) { return ((n * (uint32_t)t.team + threads - 1) / threads + cus - 1) / cus * (threads / 64); };
        uint32_t least = waves_of_a_cu(256);
        for (uint32_t threads = 128; threads >= 64 && threads >= slots && least <= 8; threads /= 2) {
            const uint32_t w = waves_of_a_cu(threads);
            if (w < least) t.threads = threads, least = w;
        }
    }
    return t;
}

// A launch for every 2^24 rows (a grid holds fewer than 2^32 threads).
template <typename Kern>
hipError_t launch_rows(Kern kern, RowTeams t, size_t lds, hipStream_t s, const uint8_t *w, size_t row_bytes, const void *x, float *y, int64_t n,
                       int units) {
    const int64_t most = (int64_t)1 << 24, per_wg = t.threads / t.team;
    for (int64_t r = 0; r < n; r += most) {
        const int64_t rows = n - r < most ? n - r : most;
        const hipError_t e = launch(kern, (unsigned)((rows + per_wg - 1) / per_wg), lds, s, w + (size_t)r * row_bytes, x, y + r, (int)rows, units, t.threads);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int T, bool XF32>
hipError_t launch_q6k(RowTeams t, size_t lds, hipStream_t s, const uint8_t *w, const void *x, float *y, int64_t n, int spr) {
    const size_t row = (size_t)spr * 210;
    switch ((spr + T / 8 - 1) / (T / 8)) {
    case 1: return launch_rows(k_qgemv_q6k_row<T, XF32, 1>, t, lds, s, w, row, x, y, n, spr);
    case 2: return launch_rows(k_qgemv_q6k_row<T, XF32, 2>, t, lds, s, w, row, x, y, n, spr);
    case 3: return launch_rows(k_qgemv_q6k_row<T, XF32, 3>, t, lds, s, w, row, x, y, n, spr);
    default: return launch_rows(k_qgemv_q6k_row<T, XF32, 4>, t, lds, s, w, row, x, y, n, spr);
    }
}

template <int T, bool XF32>
hipError_t launch_q8_0(RowTeams t, size_t lds, hipStream_t s, const uint8_t *w, const void *x, float *y, int64_t n, int bpr) {
    const size_t row = (size_t)bpr * 34;
    if (T < 8) return launch_rows(k_qgemv_q8_0<T, XF32, 1>, t, lds, s, w, row, x, y, n, bpr);  // (the whole row)
    switch ((bpr + T - 1) / T) {
    case 1: return launch_rows(k_qgemv_q8_0<T, XF32, 1>, t, lds, s, w, row, x, y, n, bpr);
    case 2: return launch_rows(k_qgemv_q8_0<T, XF32, T < 8 ? 1 : 2>, t, lds, s, w, row, x, y, n, bpr);
    case 3: return launch_rows(k_qgemv_q8_0<T, XF32, T < 8 ? 1 : 3>, t, lds, s, w, row, x, y, n, bpr);
    default: return launch_rows(k_qgemv_q8_0<T, XF32, T < 8 ? 1 : 4>, t, lds, s, w, row, x, y, n, bpr);
    }
}

}  // namespace

namespace pmh {

// Preconditions (checked by the C ABI layer): n > 0, k > 0 a multiple of the block size, n and
// k / block below 2^31, pointers 16-byte aligned, type/order/x_dtype valid.  Returns
// hipErrorInvalidValue when the staged activations do not fit the 160 KiB of LDS.
hipError_t launch_qgemv(uint32_t type, const uint8_t *w, int64_t n, int64_t k, const void *x, uint32_t x_dtype,
                        float *y, uint32_t order, hipStream_t s) {
    const bool xf32 = x_dtype == kDtypeF32;
    const int planes = xf32 ? 3 : 1;
    if (type == kTypeQ4K) return launch_qgemv_q4k(w, n, k, x, x_dtype, y, order, s);
    if (type == kTypeQ5K) return launch_qgemv_q5k(w, n, k, x, x_dtype, y, order, s);
    if (type == kTypeQ2K) return launch_qgemv_q2k(w, n, k, x, x_dtype, y, s);
    if (type == kTypeQ3K) return launch_qgemv_q3k(w, n, k, x, x_dtype, y, s);
    if (type == kTypeQ6K) {
        hipError_t chunk_err = hipSuccess;
        if (try_launch_qgemv_q6k_chunk(w, n, k, x, x_dtype, y, s, &chunk_err)) return chunk_err;
        const int spr = (int)(k / 256);
        const size_t slots = (size_t)spr * 8;
        const size_t lds = slots * 64 * planes + slots * 16;
        // Rows of five super-blocks, which no team but one of eight lanes takes whole, of a tall matrix: two rows a team at a time, x
        // converted by fewer workgroups (us, two rows / a row a team: 24000 x 1280 9.9 / 9.7, 32000 x 1280 10.3 / 11.7, 128256 x 1280 32.0 / 32.9
        // with 16 rows per team from 65536 rows on).  So are tall matrices of one or two super-blocks a row with f32 x, which is the most to convert:
        // 11733 x 512 6.1 / 4.0, 16826 6.5 / 6.7, 26787 6.9 / 7.9, 45517 10.2 / 9.9, 57437 10.5 / 14.7; 42519 x 256 6.4 / 6.5, 60965 6.8 / 8.1,
        // 76091 10.1 / 9.6, 115881 10.5 / 12.6.  Any other shape is faster with a team a row (three super-blocks, f32, 39488 x 768 12.8 / 10.9).
        if ((spr == 5 && n > 24576) || (xf32 && ((spr == 2 && n >= 16384) || (spr == 1 && n >= 49152)))) {
            const unsigned grid = grid_for_rows(n, 32, n >= 65536 ? 16 : rows_per_team());
            return xf32 ? launch(k_qgemv_q6k<true>, grid, lds, s, w, x, y, (int)n, spr) : launch(k_qgemv_q6k<false>, grid, lds, s, w, x, y, (int)n, spr);
        }
        const RowTeams t = row_teams(n, (uint32_t)slots, slots);
#define PMH_ROW(T) (xf32 ? launch_q6k<T, true>(t, lds, s, w, x, y, n, spr) : launch_q6k<T, false>(t, lds, s, w, x, y, n, spr))
        switch (t.team) {
        case 8: return PMH_ROW(8);
        case 16: return PMH_ROW(16);
        case 32: return PMH_ROW(32);
        default: return PMH_ROW(64);
        }
#undef PMH_ROW
    }
    if (type == kTypeQ8_0) {
        hipError_t chunk_err = hipSuccess;
        if (try_launch_qgemv_q8_0_chunk(w, n, k, x, x_dtype, y, s, &chunk_err)) return chunk_err;
        const int bpr = (int)(k / 32);
        const size_t lds = (size_t)bpr * 128;
        RowTeams t = row_teams(n, (uint32_t)bpr, (size_t)bpr);
        if (bpr <= 4) t = RowTeams{bpr == 3 ? 4 : bpr, 256};  // (k = 32 ... 128)
#define PMH_ROW(T) (xf32 ? launch_q8_0<T, true>(t, lds, s, w, x, y, n, bpr) : launch_q8_0<T, false>(t, lds, s, w, x, y, n, bpr))
        switch (t.team) {
        case 1: return PMH_ROW(1);
        case 2: return PMH_ROW(2);
        case 4: return PMH_ROW(4);
        case 8: return PMH_ROW(8);
        case 16: return PMH_ROW(16);
        case 32: return PMH_ROW(32);
        default: return PMH_ROW(64);
        }
#undef PMH_ROW
    }
    return hipErrorInvalidValue;
}

}  // namespace pmh
