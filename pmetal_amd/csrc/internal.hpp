// Internal declarations shared by the translation units of libpmetal_hip.so.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace pmh {

constexpr uint32_t kTypeQ8_0 = 8, kTypeQ2K = 10, kTypeQ3K = 11, kTypeQ4K = 12, kTypeQ5K = 13, kTypeQ6K = 14, kTypeQ8K = 15;
constexpr uint32_t kOrderRef = 0, kOrderGgml = 1;
constexpr uint32_t kDtypeF32 = 0, kDtypeBf16 = 1;

// compute units of the current device (256 on MI355X); falls back to 256 if the query fails
inline int compute_units() {
    static const int n = [] {
        int dev = 0, cu = 0;
        if (hipGetDevice(&dev) != hipSuccess) return 256;
        if (hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cu <= 0) return 256;
        return cu;
    }();
    return n;
}

// ---- codec.hip: bit-exact quantize / dequantize (compiled without fp contraction) ----
hipError_t launch_quantize_q8_0(const float *x, size_t n, uint8_t *dst, hipStream_t s);
hipError_t launch_quantize_legacy32(uint32_t type, const float *x, size_t n, uint8_t *dst, hipStream_t s);
hipError_t launch_dequantize_legacy32(uint32_t type, const uint8_t *src, size_t n, float *dst, hipStream_t s);
// Q4_K, Q5_K and Q6_K: up to kMaxTileTensors tensors of one type in one launch
struct TileTensor {
    const float *x;
    uint8_t *dst;
    size_t n;  // elements
};
constexpr int kMaxTileTensors = 64;
inline bool quantizes_in_tiles(uint32_t type) { return type == kTypeQ4K || type == kTypeQ5K || type == kTypeQ6K; }
hipError_t launch_quantize_tiles(uint32_t type, const TileTensor *tensors, int count, hipStream_t s);
hipError_t launch_quantize_q2k(const float *x, size_t n, uint8_t *dst, hipStream_t s);
hipError_t launch_quantize_q3k(const float *x, size_t n, uint8_t *dst, hipStream_t s);
hipError_t launch_dequantize_q8_0(const uint8_t *src, size_t n, float *dst, hipStream_t s);
hipError_t launch_dequantize_q4k(const uint8_t *src, size_t n, float *dst, uint32_t order, hipStream_t s);
hipError_t launch_dequantize_q5k(const uint8_t *src, size_t n, float *dst, uint32_t order, hipStream_t s);
hipError_t launch_dequantize_q2k(const uint8_t *src, size_t n, float *dst, hipStream_t s);
hipError_t launch_dequantize_q3k(const uint8_t *src, size_t n, float *dst, hipStream_t s);
hipError_t launch_dequantize_q6k(const uint8_t *src, size_t n, float *dst, hipStream_t s);

// ---- gemv.hip: dequant-fused y = W x ----
hipError_t launch_qgemv(uint32_t type, const uint8_t *w, int64_t n, int64_t k, const void *x, uint32_t x_dtype,
                        float *y, uint32_t order, hipStream_t s);

// ---- gemv_q4k.hip ----
constexpr int kMaxGemvGroup = 4;

// gemv_q5k.hip: the Q5_K GEMV (every shape with k a multiple of 256 that fits; hipErrorInvalidValue otherwise)
hipError_t launch_qgemv_q5k(const uint8_t *w, int64_t n, int64_t k, const void *x, uint32_t x_dtype, float *y, uint32_t order,
                            hipStream_t s);
// gemv_q23k.hip: the Q2_K and Q3_K GEMVs (every shape with k a multiple of 256 that fits; hipErrorInvalidValue otherwise)
hipError_t launch_qgemv_q2k(const uint8_t *w, int64_t n, int64_t k, const void *x, uint32_t x_dtype, float *y, hipStream_t s);
hipError_t launch_qgemv_q3k(const uint8_t *w, int64_t n, int64_t k, const void *x, uint32_t x_dtype, float *y, hipStream_t s);
// gemv_q6k.hip: the row-staging integer-dot kernel for large Q6_K matrices; false when the shape does not suit it
bool try_launch_qgemv_q6k_chunk(const uint8_t *w, int64_t n, int64_t k, const void *x, uint32_t x_dtype, float *y,
                                hipStream_t s, hipError_t *err);
// gemv_q8_0.hip: the row-staging integer-dot kernel for large Q8_0 matrices; false when the shape does not suit it
bool try_launch_qgemv_q8_0_chunk(const uint8_t *w, int64_t n, int64_t k, const void *x, uint32_t x_dtype, float *y,
                                 hipStream_t s, hipError_t *err);
hipError_t launch_qgemv_q4k(const uint8_t *w, int64_t n, int64_t k, const void *x, uint32_t x_dtype, float *y,
                            uint32_t order, hipStream_t s);
// Several small Q4_K matrices with the same k, x, x_dtype and order in one launch (count <= kMaxGemvGroup);
// launch_qgemv_q4k_pair: two large matrices (not groupable) that share k, x and the element order in one launch of the
// large-matrix kernel; hipErrorNotSupported when the pair does not suit it.
hipError_t launch_qgemv_q4k_pair(const uint8_t *w0, int64_t n0, float *y0, const uint8_t *w1, int64_t n1, float *y1, int64_t k,
                                 const void *x, uint32_t x_dtype, uint32_t order, hipStream_t s);
// qgemv_q4k_groupable tells whether a matrix is small enough to go into a group.
bool qgemv_q4k_groupable(int64_t n, int64_t k);
hipError_t launch_qgemv_q4k_q6k_group(const uint8_t *const *w, const int64_t *n, float *const *y, int count, const uint8_t *w6, int64_t n6,
                                      float *y6, int64_t k, const void *x, uint32_t x_dtype, uint32_t order, hipStream_t s);
hipError_t launch_qgemv_q4k_group(const uint8_t *const *w, const int64_t *n, float *const *y, int count, int64_t k,
                                  const void *x, uint32_t x_dtype, uint32_t order, hipStream_t s);

// ---- gemm.hip, gemm_kw.hip: dequant-fused Y = X W^T ----
enum class GemmKernel {
    kSmall,  // gemm.hip, k_qgemm_small*: the weights stream past activations held in registers (at most 32 rows)
    kWaves,  // gemm_kw.hip: a tile of Y per workgroup, K split between its waves
    kRows,   // gemm.hip, k_qgemm_rw*: every wave owns 32 weight rows, activations shared through LDS
};
// A second weight of the same type, element order and row length for the launch: its tiles lie behind the first weight's.
struct GemmSecond {
    const uint8_t *w;
    void *y;
    int n;      // weight rows; 0: no second weight
    int first;  // its first workgroup along the grid's x dimension (kWaves: its first tile, or pair of tiles)
};
struct GemmPlan {
    GemmKernel kernel;
    int mb;      // 32-row activation blocks per workgroup (kRows: 1, 2 or 4; kWaves: 1 or 2)
    int nr;      // kWaves: 32-row blocks of weights per workgroup (1 or 2)
    int mp;      // padded activation rows, a multiple of 32 mb
    int nw;      // waves per workgroup (kWaves: at most; a short row has fewer)
    int splits;  // workgroups along K (more than one: partial tiles, added by a reduction kernel or, kWaves, by the tile's last workgroup)
    int chunk;   // super-blocks per split
};
// Which operand's tiles the dies share among them in the tile kernel (true: the blocks of activation rows)
bool kw_by_m(int64_t mblocks, int64_t tiles, int mb, int nr, int64_t block_bytes);
// Two weights in one launch of the tile kernel, with workgroups of eight waves, tiles of four and of eight waves (columns of each): whether two tiles of four
// share a workgroup, and the rounds of workgroups that the launch takes
struct KwMixed {
    bool by_twos;
    double rounds;
};
KwMixed kw_mixed(int64_t mblocks, int64_t of_four, int64_t of_eight, bool by_m, int mb, int nr);
bool qgemm_fits(uint32_t type, int64_t m, int64_t n, int64_t k);
// (the padded row count mp follows m and the kernel, and the type and n only where the entry point that allocates nothing would be short of scratch)
GemmPlan qgemm_plan(int64_t m, int64_t n, int64_t k, uint32_t type = kTypeQ4K);
// Bytes of device workspace qgemm needs for a weight of `type` at (m, n, k); the caller provides it.
size_t qgemm_workspace_bytes(uint32_t type, int64_t m, int64_t n, int64_t k);
// Whether two weights of one type and element order that share their activations go in one launch (launch_qgemm with `second`), and
// the launch's plan: the padded rows and the workspace are those of either weight alone, as are the results to the bit.
bool qgemm_pair_plan(int64_t m, int64_t n0, int64_t n1, int64_t k, uint32_t type, GemmPlan *plan);
// Whether the plan's kernel takes at most 16 rows, converted per pair of super-blocks and not per row: no other kernel can use those.
bool qgemm_small_rows(const GemmPlan &plan, int64_t m);
// Whether the plan's kernel reads the activations as they are: a launch with it leaves no converted ones for the next.
// second_n: rows of the launch's second weight (0: none).  shared: another launch could use the converted ones.
bool qgemm_converts_itself(const GemmPlan &plan, uint32_t type, int64_t m, int64_t n, int64_t second_n, int64_t k, uint32_t x_dtype, bool shared);
// LDS bytes of a workgroup of the short-batch kernels (own: it converts the activations for itself), beside the 128 it always has.
size_t qgemm_small_lds(uint32_t type, int64_t m, int64_t k, int tiles_per_wg, bool own, bool xf32);
// `bytes` of activations, a multiple of 16, to where results that lie over them do not reach
hipError_t launch_copy_x(const void *x, size_t bytes, void *to, hipStream_t s);
// reuse_prepass: the workspace still holds the converted activations of the previous launch_qgemm on this stream with the same
// x, m, k and weight type (two weights that share their activations: the pre-pass runs once)
hipError_t launch_qgemm(uint32_t type, const uint8_t *w, int64_t n, int64_t k, const void *x, uint32_t x_dtype,
                        int64_t m, void *y, uint32_t y_dtype, uint32_t order, void *workspace, hipStream_t s,
                        bool reuse_prepass = false, const GemmSecond &second = GemmSecond{}, bool shared = false);

// Which tiles of the tile kernel's launch add their splits of K themselves (gemm_kw.hip).  Not 64 x 64 ones: four waves take in up to 64 KiB of
// partial sums then, which the launch behind reads with the whole machine (Q4_K 2048 x 8192 M = 120 21.2 us a call, 24.8 without it).
constexpr bool joins_splits(int mb, int nr) { return mb * nr < 4; }
// gemm_kw.hip (spr: super-blocks per row; partial: fp32 tiles [splits][mp][n] when plan.splits > 1, not scaled by rowscale; arrived: a
// cleared counter per tile of Y, where the launch adds the splits itself)
hipError_t launch_qgemm_kw(uint32_t type, const GemmPlan &plan, const uint8_t *w, const void *xs, const float *rowscale, void *y, bool y_bf16, int64_t m,
                           int64_t n, int spr, uint32_t order, float *partial, uint32_t *arrived, const GemmSecond &second, int second_nw, hipStream_t s);

// ---- q8k.hip: Q8_K activation blocks and the integer dot products over them ----
hipError_t launch_quantize_q8k(const float *x, size_t n, uint8_t *dst, hipStream_t s);
hipError_t launch_dequantize_q8k(const uint8_t *src, size_t n, float *dst, hipStream_t s);
// four f64 sums per workgroup (sum (a-b)^2, sum a^2, sum a b, sum b^2) into partial[4 * kl_sums_workgroups(n)]
int kl_sums_workgroups(size_t n);
hipError_t launch_kl_sums(const float *a, const float *b, size_t n, double *partial, hipStream_t s);
// the same sums between `original` and the first n elements decoded from k-quant blocks (never stored), into
// Exact re-blocking of Q5_K / Q3_K / Q2_K super-blocks into Q6_K ones (210 bytes each): W = A (+ B for the formats with
// mins).  reblock_q6k_parts: 2, 1, 2; 0 for any other type.  dst_b is not touched when there is one part.
int reblock_q6k_parts(uint32_t type);
hipError_t launch_reblock_q6k(uint32_t type, const uint8_t *src, size_t n_blocks, uint32_t order, uint8_t *dst_a, uint8_t *dst_b,
                              hipStream_t s);
// y[i] = a[i] + b[i], stored as f32 or bf16
hipError_t launch_add_store(const float *a, const float *b, size_t n, void *y, bool y_bf16, hipStream_t s);
// partial[4 * kl_sums_quantized_workgroups(n)]; hipErrorInvalidValue for a type that is not a k-quant
int kl_sums_quantized_workgroups(size_t n);
hipError_t launch_kl_sums_quantized(uint32_t type, const uint8_t *src, const float *original, size_t n, uint32_t order, double *partial,
                                    hipStream_t s);
// k a multiple of 256 and at most 32768 (the activation blocks live in LDS); type Q4_K or Q6_K
hipError_t launch_qgemv_q8k(uint32_t type, const uint8_t *w, int64_t n, int64_t k, const uint8_t *xq, float *y, hipStream_t s);

// ---- api.hip ----
size_t codec_chunk(size_t n);  // elements of a staging chunk of the host codec

// ---- util.hip ----
hipError_t launch_fill_normal(float *dst, size_t n, uint64_t seed, float std, float outlier_rate,
                              float outlier_mag, hipStream_t s);
hipError_t launch_f32_to_bf16(const float *src, uint16_t *dst, size_t n, hipStream_t s);
hipError_t launch_zero_bytes(uint8_t *dst, size_t bytes, hipStream_t s);
hipError_t launch_mfma_probe(int iters, int vary, int workgroups, float *sink, hipStream_t s);
hipError_t launch_read_probe(const void *src, size_t bytes, uint32_t *sink, hipStream_t s);

}  // namespace pmh
