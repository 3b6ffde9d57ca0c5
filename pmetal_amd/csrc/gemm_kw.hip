// Dequant-fused GEMM  Y[m,n] = sum_k X[m,k] * W[n,k]  for a few dozen activation rows, or few weight rows: the waves of a
// workgroup split K between them.
//
// The kernels of gemm.hip give every wave its own weight rows and fill the machine with a K split over workgroups, whose
// partial tiles a second launch adds: at M = 64 their loop has 0.5 us of matrix work per step and waits for memory in each,
// and prepare + multiply + add are three dependent launches.  Here a workgroup owns a tile of 32 MB activation rows x 32 NR
// weight rows for the whole of K.  Its waves, eight or four (the plan's kw_waves) and no more than there are super-blocks, take super-blocks in
// turn, run without a barrier from start to end, and their fp32 tiles are added through LDS in wave order: the result does not depend on
// scheduling, and there are no partial tiles in memory.  Only where a few long rows leave the machine empty does a tile have two or four
// workgroups, the last of which, or a launch behind, adds their sums (join_splits).  (Consecutive runs of super-blocks, which is what the waves took before, lie far apart in
// a row: 1 to 5 % slower, two Q4_K weights of 14336 x 4096 M = 64 38.6 -> 36.8 us, Q5_K 8192 x 4096 M = 100 24.6 -> 23.4.)
//   * Weights: a wave copies a unit of its rows (one or half a super-block of 32 NR rows) directly global -> LDS, one unit
//     ahead, into LDS of its own; a lane (row n = lane % 32, half g = lane / 32) reads its quants and scales back and
//     makes the exact f16 operands of gemm_common.hpp.
//   * Activations: the items of the pre-pass (k_prep_rw) are matrix operands as they lie in memory, so they are loaded
//     straight into registers, a ring of kDepth k-steps ahead.  Nothing is shared between waves, so LDS would not help.
//   * Requests return in order, so waiting for a fragment waits for the copies requested before it: the wait in front of a
//     unit is never longer than that for its first fragments.
//   * The operands of k-step s + 1 are made between the matrix instructions of step s.
//
// What bounds it: a compute unit's path to memory, through which weights and activations come in the order of their requests.  By time stamps
// (Q4_K 14336 x 4096 M = 64, 224 workgroups of 64 x 64), a wave's first requests are all issued 1.1 to 8.7 us after its start and its loop ends
// 8.8 to 15.2 us after it: what waits for weights from HBM holds up the activations behind it, 0.74 MB a workgroup at 26
// bytes a clock.  Adding the tiles takes 1.2 us of it.  The time goes in whole rounds of 256 workgroups, each as long as its share of the row: 7 us, launch and
// pre-pass included, and per round and eight super-blocks of a row 2.9 (Q2_K), 3.5 (Q4_K, Q3_K), 4.6 (Q5_K), 4.9 us (Q8_0, Q6_K) with 32 x
// 32 tiles (up to 32 activation rows, rows of 32 super-blocks and more); 0.6 to 0.8 of that where fewer than 64 workgroups run.  Inside, by
// counters (share of the waves' time that they issue / are ready and cannot issue / wait for memory, LDS or each other; share of the
// time that the matrix cores work):
//   Q4_K, two of 14336 x 4096, M = 64 (64 x 64, 448 workgroups of four waves)     28.6 us  31 / 55 / 15 %, matrix cores 32 %
//   Q8_0, 4999 x 3584, M = 203 (64 x 32, 628 of four)                             24.0 us  30 / 45 / 26 %, 23 % (LDS bank conflicts 22 %: rows of 144 bytes)
//   Q6_K, 4096 x 14336, M = 27 (32 x 32, two splits joined, 256 of eight)         21.5 us  26 / 44 / 30 %, 17 %
#include "gemm_common.hpp"

namespace {

template <int N>
__device__ __forceinline__ void wait_vm() {  // at most N vector-memory requests outstanding
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
    asm volatile("" ::: "memory");
}

// p + off with the offset kept in one 32-bit register: a uniform base and a lane offset are one address operand of a load.
// (Otherwise the compiler widens loop-invariant offsets to 64-bit pairs ahead of the loop: twice the registers.)
__device__ __forceinline__ const uint8_t *at(const uint8_t *p, uint32_t off) {
    asm("" : "+v"(off));
    return p + off;
}

// Neighbouring results of a row, which may begin at any of them.
template <class T, int ALIGN, int COUNT>
struct __attribute__((packed, aligned(ALIGN))) RowPiece {
    T v[COUNT > 0 ? COUNT : 1];
};

// 16 bytes per lane from a buffer to LDS (lane l lands at dst + 16 l).  The buffer form and not dma16(): the compiler takes a
// global load into LDS for an access to either memory and waits for everything outstanding at the next use of any load.
__device__ __forceinline__ void buf16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, uint4 *dst) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, PMH_LPTR(dst), 16, voff, soff, 0, 0);
}

// ------------------------------------------------------------------------------------------------
// Formats.  kUnitHalves: halves of a super-block that a unit of copies holds; kPieces: its 16-byte pieces per row, piece p
// at piece_off(p), moved by half_delta(p) for the second half; slot(p, row): where piece p of a row lies in the staged row
// (rows whose stride would put them on the same LDS banks are swizzled).  kSums: operand items of sub-block sums per half;
// kTiles: matrix instructions per fragment (Q6_K's exact split); kFlush: k-steps between two additions of scale * partial
// sum.
// ------------------------------------------------------------------------------------------------
template <int ORDER, int FMT>
struct KwQ45 {  // FMT 0: Q4_K, 1: Q5_K
    static constexpr int kBytes = BlockFmt<FMT>::kBytes, kUnitHalves = FMT ? 1 : 2, kPieces = FMT ? 7 : 9, kSums = 1, kTiles = 1,
                         kFlush = 16;
    static __device__ __forceinline__ uint32_t piece_off(int p) { return 16u * (uint32_t)p; }
    static __device__ __forceinline__ uint32_t half_delta(int p) { return FMT && p >= 3 ? 64u : 0u; }
    static __device__ __forceinline__ int slot(int p, int) { return p; }
    const uint4 *row_;
    int g_;
    uint32_t q[4], qh[4];  // of four k-steps
    half2_t scs, offs, mns;  // of the lane's two sub-blocks: scale, -1024 scale, min
    uint32_t dd;             // d | dmin << 16
    template <int H>
    __device__ __forceinline__ void load(const uint4 *st, int, const int g) {
        row_ = st, g_ = g;
        const uint4 hdr = st[0];
        // scales and mins of sub-blocks 4 H + 2 g and the next one
        const uint32_t pick = g ? 0x04030402u : 0x04010400u;
        const half2_t m1024 = {(_Float16)-1024.0f, (_Float16)-1024.0f};
        scs = byte_pair(scale_bytes<H>(hdr.y, hdr.w), pick), mns = byte_pair(min_bytes<H>(hdr.z, hdr.w), pick);
        offs = scs * m1024;  // exact: sc <= 63
        dd = hdr.x;
    }
    template <int H>
    __device__ __forceinline__ void operands(const int t, half8_t (&b)[1]) {
        if (t % 4 == 0) {
            const uint4 v = row_[(FMT ? 3 : 1 + 4 * H) + 2 * g_ + t / 4];
            q[0] = v.x, q[1] = v.y, q[2] = v.z, q[3] = v.w;
            if (FMT && ORDER) {  // qh dword t: the same four bytes as quant dword t
                const uint4 h = row_[1 + t / 4];
                const uint32_t sh = (uint32_t)(4 * H + 2 * g_);
                qh[0] = h.x >> sh, qh[1] = h.y >> sh, qh[2] = h.z >> sh, qh[3] = h.w >> sh;
            } else if (FMT) {  // qh byte 4 (4 H + 2 g) + t
                qh[0] = reinterpret_cast<const uint32_t *>(row_ + 1)[4 * H + 2 * g_ + t / 4];
            }
        }
        const uint32_t hq = !FMT ? 0u : ORDER ? qh[t % 4] : qh[0] >> (8 * (t & 3));
        const half2_t sc2[2] = {half2_t{scs[0], scs[0]}, half2_t{scs[1], scs[1]}}, off2[2] = {half2_t{offs[0], offs[0]}, half2_t{offs[1], offs[1]}};
        Dq v;
#pragma unroll
        for (int c = 0; c < 4; c++) dq_chunk<ORDER, FMT>(c, t, q[t % 4], sc2, off2, v, hq);
        b[0] = v.value();
    }
    // (made where they are used: the 64 x 64 tile has no registers to hold them over the half)
    __device__ __forceinline__ half8_t sums(int) const {
        uint32_t w = dd;
        asm("" : "+v"(w));  // (not earlier: 170 registers for Q4_K's 64 x 32 tile, two waves a SIMD, for 163, three, and a register of Q5_K's 64 x 64 in memory)
        return heads_and_tails(mns, -f16_twice(w >> 16));
    }
    __device__ __forceinline__ float scale(int) const { return f16_bits_to_f32(dd & 0xFFFFu); }
};

struct KwQ6 {
    static constexpr int kBytes = kQ6Bytes, kUnitHalves = 1, kPieces = 8, kSums = 0, kTiles = 2, kFlush = 16;
    // pieces 0..3: ql, 4, 5: qh, 6: bytes 192..207 (scales), 7: bytes 194..209 (d in the last two)
    static __device__ __forceinline__ uint32_t piece_off(int p) { return p < 4 ? 16u * (uint32_t)p : p < 6 ? 64u + 16u * (uint32_t)p : 180u + 2u * (uint32_t)p; }
    static __device__ __forceinline__ uint32_t half_delta(int p) { return p < 4 ? 64u : p < 6 ? 32u : 0u; }
    static __device__ __forceinline__ int slot(int p, int row) { return p ^ ((row >> 1) & 7); }
    const uint4 *row_;
    int i_, g_;
    uint32_t q[4], h[4];  // of four k-steps
    half2_t sc[2][2];  // [k-step / 4][low, high]
    Q6Scales s;
    float d;
    template <int H>
    __device__ __forceinline__ void load(const uint4 *st, const int row, const int g) {
        row_ = st, i_ = row, g_ = g;
        const uint4 sv = st[slot(6, row)];
        d = kQ6OperandScale * f16_bits_to_f32(reinterpret_cast<const uint32_t *>(st + slot(7, row))[3] >> 16);
        // scales 8 H + 2 g + t / 4 (low nibbles) and 8 H + 4 + 2 g + t / 4 (high nibbles)
        const uint32_t wlo = (H == 0 ? sv.x : sv.z) >> (16u * (uint32_t)g), whi = (H == 0 ? sv.y : sv.w) >> (16u * (uint32_t)g);
#pragma unroll
        for (int th = 0; th < 2; th++) {
            const _Float16 lo = (_Float16)(float)(int)(int8_t)(wlo >> (8 * th)), hi = (_Float16)(float)(int)(int8_t)(whi >> (8 * th));
            sc[th][0] = half2_t{lo, lo}, sc[th][1] = half2_t{hi, hi};
        }
    }
    template <int H>
    __device__ __forceinline__ void operands(const int t, half8_t (&b)[2]) {
        if (t % 4 == 0) {
            const uint4 v = row_[slot(2 * g_ + t / 4, i_)], w = row_[slot(4 + t / 4, i_)];
            const uint32_t hs = 2u * (uint32_t)g_;
            q[0] = v.x, q[1] = v.y, q[2] = v.z, q[3] = v.w;
            h[0] = w.x >> hs, h[1] = w.y >> hs, h[2] = w.z >> hs, h[3] = w.w >> hs;
            s.set(sc[t >> 2][0], sc[t >> 2][1]);
        }
        Dq6 v;
#pragma unroll
        for (int c = 0; c < 8; c++) dq6_chunk(c, q[t % 4], h[t % 4], s, v);
        b[0] = v.b1(), b[1] = v.b2();
    }
    __device__ __forceinline__ half8_t sums(int) const { return half8_t{0, 0, 0, 0, 0, 0, 0, 0}; }
    __device__ __forceinline__ float scale(int) const { return d; }
};

struct KwQ8 {  // eight 34-byte blocks stand for a super-block; a half (136 bytes) begins 8 bytes into its first piece when it is the second
    static constexpr int kBytes = 272, kUnitHalves = 1, kPieces = 9, kSums = 0, kTiles = 1, kFlush = 2;
    static __device__ __forceinline__ uint32_t piece_off(int p) { return 16u * (uint32_t)p; }
    static __device__ __forceinline__ uint32_t half_delta(int) { return 128u; }
    static __device__ __forceinline__ int slot(int p, int) { return p; }
    const uint32_t *p_;
    int g_;
    float ds[2];
    template <int H>
    __device__ __forceinline__ void load(const uint4 *st, int, const int g) { p_ = reinterpret_cast<const uint32_t *>(st) + 2 * H, g_ = g; }
    template <int H>
    __device__ __forceinline__ void operands(const int t, half8_t (&b)[1]) {
        const int blk = t >> 1, w0 = (34 * blk) / 4;  // block blk starts at this dword (blk even) or two bytes into it
        const uint32_t *v = p_ + w0 + 4 * (t & 1) + 2 * g_;
        if (t % 2 == 0) ds[blk % 2] = f16_bits_to_f32((blk & 1 ? p_[w0] >> 16 : p_[w0]) & 0xFFFFu);
        if (blk & 1) b[0] = q8_operand(v[1], v[2]);
        else b[0] = q8_operand(__builtin_amdgcn_alignbit(v[1], v[0], 16), __builtin_amdgcn_alignbit(v[2], v[1], 16));
    }
    __device__ __forceinline__ half8_t sums(int) const { return half8_t{0, 0, 0, 0, 0, 0, 0, 0}; }
    __device__ __forceinline__ float scale(int t) const { return tile_scale(ds[(t >> 1) % 2]); }
};

template <int FMT>
struct KwQ23 {  // FMT 2: Q3_K, 3: Q2_K
    static constexpr int kBytes = Block16<FMT>::kBytes, kUnitHalves = 2, kPieces = FMT == 3 ? 6 : 7, kSums = 2, kTiles = 1, kFlush = 16;
    // Q2_K: scales, four of quants, bytes 68..83 (d, dmin in the last dword); Q3_K: two of hmask, four of quants, bytes 94..109
    static __device__ __forceinline__ uint32_t piece_off(int p) {
        return FMT == 3 ? (p < 5 ? 16u * (uint32_t)p : 68u) : (p < 6 ? 16u * (uint32_t)p : 94u);
    }
    static __device__ __forceinline__ uint32_t half_delta(int) { return 0; }
    static __device__ __forceinline__ int slot(int p, int) { return p; }
    uint32_t qd[4], hm[4];
    half2_t sc2[4], off2[4];
    half8_t br[FMT == 3 ? 2 : 1];  // Q2_K's mins
    half2_t dk;                     // Q3_K: d
    float d;
    template <int H>
    __device__ __forceinline__ void load(const uint4 *st, int, const int g) {
        const uint4 qv = st[(FMT == 3 ? 1 : 2) + 2 * H + g];
        qd[0] = qv.x, qd[1] = qv.y, qd[2] = qv.z, qd[3] = qv.w;
        uint32_t hdr[4], dbits;
        if (FMT == 3) {
            const uint4 sc = st[0], dd = st[5];
            hdr[0] = sc.x, hdr[1] = sc.y, hdr[2] = sc.z, hdr[3] = sc.w;
            dbits = dd.w;  // d | dmin << 16
        } else {
            const uint4 m = st[g], sd = st[6];
            hm[0] = m.x, hm[1] = m.y, hm[2] = m.z, hm[3] = m.w;  // hmask bytes 16 g ..
            // the twelve scale bytes as three dwords (they start two bytes into the piece), d behind them
            hdr[0] = __builtin_amdgcn_alignbit(sd.y, sd.x, 16), hdr[1] = __builtin_amdgcn_alignbit(sd.z, sd.y, 16);
            hdr[2] = __builtin_amdgcn_alignbit(sd.w, sd.z, 16), hdr[3] = 0;
            dbits = sd.w >> 16;
        }
        d = f16_bits_to_f32(dbits & 0xFFFFu);
        // scales (Q2_K: and what a sub-block subtracts per unit of its activation sum) of sub-blocks 8 H + 4 sp + 2 lh + g, index 2 sp + lh
        const uint32_t pick = g ? 0x04030401u : 0x04020400u;  // bytes g and g + 2
        const half2_t m1024 = {(_Float16)-1024.0f, (_Float16)-1024.0f};
        if constexpr (FMT == 2) dk = f16_twice(dbits);
#pragma unroll
        for (int sp = 0; sp < 2; sp++) {
            half2_t sc;
            if constexpr (FMT == 3) {
                sc = byte_pair(hdr[2 * H + sp] & 0x0F0F0F0Fu, pick);
                br[sp] = heads_and_tails(byte_pair((hdr[2 * H + sp] >> 4) & 0x0F0F0F0Fu, pick), -f16_twice(dbits >> 16));
            } else {
                sc = byte_pair(((hdr[sp] >> (4 * H)) & 0x0F0F0F0Fu) | (((hdr[2] >> (2 * (2 * H + sp))) & 0x03030303u) << 4), pick, -1056.0f);
            }
            sc2[2 * sp] = half2_t{sc[0], sc[0]}, sc2[2 * sp + 1] = half2_t{sc[1], sc[1]};
            off2[2 * sp] = sc2[2 * sp] * m1024, off2[2 * sp + 1] = sc2[2 * sp + 1] * m1024;  // exact: |sc| <= 32
        }
        if (FMT == 2) {
#pragma unroll
            for (int i = 0; i < 4; i++) hm[i] >>= 4 * H;
        }
    }
    template <int H>
    __device__ __forceinline__ void operands(const int t, half8_t (&b)[1]) {
        const int dw = t >> 1, sp = t & 1;
        uint32_t lo = (qd[dw] >> (4 * sp)) & 0x03030303u, hi = (qd[dw] >> (4 * sp + 2)) & 0x03030303u;
        if (FMT == 2) {
            const uint32_t m = hm[dw] >> (2 * sp);
            lo |= (m & 0x01010101u) << 2, hi |= (m & 0x02020202u) << 1;
        }
        const half2_t r0 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, lo, 0x04010400u)), sc2[2 * sp], off2[2 * sp]);
        const half2_t r1 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, lo, 0x04030402u)), sc2[2 * sp], off2[2 * sp]);
        const half2_t r2 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, hi, 0x04010400u)), sc2[2 * sp + 1], off2[2 * sp + 1]);
        const half2_t r3 = __builtin_elementwise_fma(__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, hi, 0x04030402u)), sc2[2 * sp + 1], off2[2 * sp + 1]);
        b[0] = half8_t{r0[0], r0[1], r1[0], r1[1], r2[0], r2[1], r3[0], r3[1]};
    }
    // (Q3_K subtracts 4 d sc: made from the scales where it is used.  Held over the half it took the 64 x 64 tile past 256 registers
    // and one of them to scratch memory)
    __device__ __forceinline__ half8_t sums(int i) const {
        if constexpr (FMT == 3) return br[i];
        else return heads_and_tails(half2_t{sc2[2 * i][0], sc2[2 * i + 1][0]} * half2_t{(_Float16)-4.0f, (_Float16)-4.0f}, dk);
    }
    __device__ __forceinline__ float scale(int) const { return d; }
};

// ------------------------------------------------------------------------------------------------
constexpr int kKwWaves = 8, kMostSplits = 4;  // (as the plan makes them)
// Forms of the kernel: without a K split, with one, and two weights of which one has tiles of four waves and the other of eight.  (One kernel for
// all: 0.1 us a call without a split, and up to 2 % of calls with short rows.)
constexpr int kPlain = 0, kSplit = 1, kMixed = 2;
// Bits beside kHasSecond: the tiles of the first, of the second weight have four waves of the workgroup's eight; they go two to a workgroup (see launch_kw);
// `outer` counts the blocks of activation rows
constexpr int kFirstOfFour = 2, kSecondOfFour = 4, kByTwos = 8, kByM = 16;
// A wave's accumulators lie in LDS as the 64 lanes' 16-byte slots (four rows of one column), lane l at tile_slot(l): a thread that
// reads four neighbouring columns back and one that writes its slot meet 64 different banks with the 15 beside them.
constexpr int kTileRun = 76;
__device__ __forceinline__ int tile_slot(const int l) { return 20 * (l & 3) + (l >> 2); }

template <class F, int MB, int NR>
struct Kw {
    static constexpr int kItems = 32 * NR * F::kPieces, kCopies = (kItems + 63) / 64;  // 16-byte pieces of a unit, whole-wave copies
    static constexpr int kSteps = 8 + F::kSums;                                        // k-steps and sum steps of a half
    // k-steps of activation fragments in flight: a divisor of the steps of a super-block
    static constexpr int kDepth = F::kSums == 1 ? 6 : F::kSums == 2 ? (MB * NR == 4 ? 4 : 5) : (MB * NR == 4 ? 2 : 4);
    static constexpr int kTile = MB * NR * 4 * kTileRun;                               // 16-byte slots of a wave's fp32 tile
    static_assert((2 * kSteps) % kDepth == 0, "the ring's slots are picked at compile time");
    static_assert(kDepth <= kSteps, "a unit's copies must be older than the fragments in flight when it is used");
};

template <class F, int MB, int NR>
struct KwCopy {  // a wave's copies of one unit
    uint32_t off[Kw<F, MB, NR>::kCopies];
    uint32_t by64 = 0, by32 = 0;  // bit j: copy j of this lane moves by 64, by 32 bytes for the second half (Q8_0: all by 128)
    template <int H>
    __device__ __forceinline__ void issue(const __amdgpu_buffer_rsrc_t r, const uint32_t sb_off, uint4 *dst, const int lane) const {
        using K = Kw<F, MB, NR>;
#pragma unroll
        for (int j = 0; j < K::kCopies; j++)
            if (64 * j + 64 <= K::kItems || 64 * j + lane < K::kItems) {
                uint32_t o = off[j];
                if (H && F::kFlush > 2) {
                    uint32_t a = by64, b = by32;
                    asm("" : "+v"(a), "+v"(b));  // (made anew for each unit: kept sums would be a second set of offsets in registers)
                    o += ((a >> j & 1u) << 6) + ((b >> j & 1u) << 5);
                }
                buf16(r, o, H && F::kFlush == 2 ? sb_off + 128u : sb_off, dst + 64 * j);
            }
    }
};

// Half H of a super-block.  cur: the staged unit; nxt: where the copies of the next unit go (half HN of the super-block at
// sb_next of every row); xa: the items of the k-step whose fragments are requested next; jump: from the end of this super-block's
// items to the wave's next ones.
template <class F, int MB, int NR, int H, bool NEXT>
__device__ __forceinline__ void kw_half(const uint4 *__restrict__ cur, uint4 *__restrict__ nxt, const __amdgpu_buffer_rsrc_t r, const uint32_t sb_next,
                                        const KwCopy<F, MB, NR> &C, const uint8_t *__restrict__ &xa, const uint32_t step, const size_t jump, const uint32_t a_off,
                                        half8_t (&af)[Kw<F, MB, NR>::kDepth][MB], const int lane, float16_t (&acc)[NR][MB], float16_t (&part)[NR][MB]) {
    using K = Kw<F, MB, NR>;
    const int col = lane & 31, g = lane >> 5;
    constexpr bool kNewUnit = F::kUnitHalves == 1 || H == 0;
    if (kNewUnit) wait_vm<K::kDepth * MB>();  // what is newer than this unit's copies is in the ring of fragments
    F op[NR];
#pragma unroll
    for (int rg = 0; rg < NR; rg++) op[rg].template load<H>(cur + (32 * rg + col) * F::kPieces, 32 * rg + col, g);
    if (kNewUnit && NEXT) {
        __builtin_amdgcn_sched_barrier(0);
        C.template issue<F::kUnitHalves == 1 && H == 0 ? 1 : 0>(r, sb_next, nxt, lane);
    }
    half8_t b[NR][F::kTiles];
#pragma unroll
    for (int rg = 0; rg < NR; rg++) op[rg].template operands<H>(0, b[rg]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < K::kSteps; s++) {
        const int slot = (H * K::kSteps + s) % K::kDepth;
        half8_t bn[NR][F::kTiles];
        if (s + 1 < K::kSteps) {
#pragma unroll
            for (int rg = 0; rg < NR; rg++) {
                if (s + 1 < 8) op[rg].template operands<H>(s + 1, bn[rg]);
                else bn[rg][0] = op[rg].sums(s + 1 - 8);
            }
        }
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int rg = 0; rg < NR; rg++) {
                const half8_t a = af[slot][i];
                if (s >= 8) {
                    acc[rg][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b[rg][0], acc[rg][i], 0, 0, 0);
                } else {
#pragma unroll
                    for (int tl = 0; tl < F::kTiles; tl++) {
                        if ((8 * H + s) % F::kFlush == 0 && tl == 0) {  // the first product behind a flush starts from zero
                            float16_t z;
#pragma unroll
                            for (int e = 0; e < 16; e++) z[e] = 0.0f;
                            part[rg][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b[rg][tl], z, 0, 0, 0);
                        } else {
                            part[rg][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b[rg][tl], part[rg][i], 0, 0, 0);
                        }
                    }
                }
            }
        // the slot takes the fragments of kDepth steps on (past the last step: items of another wave, or the slack behind them)
        if (H == 1 && s == K::kSteps - K::kDepth) xa += jump;
#pragma unroll
        for (int i = 0; i < MB; i++) af[slot][i] = *reinterpret_cast<const half8_t *>(at(xa, a_off) + 512 * i);
        xa += step;
        if (s + 1 < 8) {  // issue order: a matrix instruction, then the vector instructions that fit behind it
#pragma unroll
            for (int e = 0; e < MB * NR * F::kTiles; e++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, F::kTiles == 2 ? (16 + MB - 1) / MB : (11 + MB - 1) / MB, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (s < 8 && (8 * H + s + 1) % F::kFlush == 0) {
#pragma unroll
            for (int rg = 0; rg < NR; rg++) {
                const float d = op[rg].scale(s);
#pragma unroll
                for (int i = 0; i < MB; i++)
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[rg][i][e] = __builtin_fmaf(d, part[rg][i][e], acc[rg][i][e]);
                if (F::kFlush < 16)  // (added here and not where the sums are next used: the partial sums would stay in registers until then)
#pragma unroll
                    for (int i = 0; i < MB; i++) asm volatile("" : "+v"(acc[rg][i]));
            }
        }
#pragma unroll
        for (int rg = 0; rg < NR; rg++)
#pragma unroll
            for (int tl = 0; tl < F::kTiles; tl++) b[rg][tl] = bn[rg][tl];
    }
}

// Partial sums go from one workgroup to another inside a launch: stores and loads that every die sees (relaxed, agent scope), so that
// no cache has to be written back or emptied for them.  (A release and an acquire in their place, a write-back of the die's whole L2 for
// each workgroup, made a call 2 to 11 us longer: Q6_K 4096 x 14336 at 27 rows 26.8 -> 36.0.)
__device__ __forceinline__ void put_shared(float *to, const float v) { __hip_atomic_store(to, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float get_shared(const float *from) { return __hip_atomic_load(from, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Adds the waves' tiles in wave order and stores the sums.  Run (rg, block i, quarter q) of a tile: lane l = 32 g + c left rows 8 q + 4 g
// .. + 3 of block i and column c of row group rg at tile_slot(l).  A thread takes COLS neighbouring columns of four rows, as many
// as leave every thread something to do: with four a row of the result leaves in 8 or 16 bytes a lane, with one in 2 or 4.
// (One column a thread throughout, stores of 2 bytes a lane: a workgroup of four waves and a 64 x 64 tile took 2.9 us from its loop's end to
// its last store, 1.5 now; 14336 x 4096 M = 64 with four waves 23.4 -> 22.3 us a call, Q8_0 4999 x 3584 M = 203 34.3 -> 32.9.)
template <int TILE, int MB, int NR, int COLS, int WAVES, bool SHARED>
__device__ __forceinline__ void add_tiles(const float4_t *red, const float *rs, const int tid, const int threads, const int nwaves, const int m0,
                                          const int n0, const int M, const int Mp, const int N, const int z, const int ybf16, void *__restrict__ yg, float *__restrict__ partial) {
    constexpr int kPer = 32 / COLS;  // threads of a row
    for (int u = tid; u < MB * NR * 8 * kPer; u += threads) {
        const int j = u % kPer, g = u / kPer & 1, rg = u / (2 * kPer) % NR, q = u / (2 * kPer * NR) & 3, i = u / (8 * kPer * NR);
        const int n = n0 + 32 * rg + COLS * j, ml = 32 * i + 8 * q + 4 * g, m = m0 + ml;
        const float4_t *src = red + ((rg * MB + i) * 4 + q) * kTileRun + tile_slot(32 * g + COLS * j);
        float4_t t[WAVES][COLS];  // (all asked for at once)
#pragma unroll
        for (int w = 0; w < WAVES; w++)
#pragma unroll
            for (int c = 0; c < COLS; c++) t[w][c] = src[(w < nwaves ? w : 0) * TILE + 20 * c];
        const float4_t scale = partial ? float4_t{1.0f, 1.0f, 1.0f, 1.0f} : *reinterpret_cast<const float4_t *>(rs + ml);
#pragma unroll
        for (int c = 0; c < COLS; c++) {
#pragma unroll
            for (int w = 1; w < WAVES; w++)
                if (w < nwaves) t[0][c] += t[w][c];
            t[0][c] *= scale;
        }
        const bool bf = !partial && ybf16;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (m + e >= M) break;
            float *to = partial ? partial + ((size_t)z * Mp + m + e) * N + n : reinterpret_cast<float *>(yg) + (size_t)(m + e) * N + n;
            uint16_t *to16 = reinterpret_cast<uint16_t *>(yg) + (size_t)(m + e) * N + n;
            if (SHARED) {
#pragma unroll
                for (int c = 0; c < COLS; c++)
                    if (n + c < N) put_shared(to + c, t[0][c][e]);
            } else if (COLS > 1 && n + COLS <= N) {
                if (bf) {
                    RowPiece<uint32_t, 2, COLS / 2> v;
#pragma unroll
                    for (int c = 0; c < COLS / 2; c++) v.v[c] = bf16_rne_bits(t[0][2 * c][e]) | bf16_rne_bits(t[0][2 * c + (COLS > 1 ? 1 : 0)][e]) << 16;
                    *reinterpret_cast<RowPiece<uint32_t, 2, COLS / 2> *>(to16) = v;
                } else {
                    RowPiece<float, 4, COLS> v;
#pragma unroll
                    for (int c = 0; c < COLS; c++) v.v[c] = t[0][c][e];
                    *reinterpret_cast<RowPiece<float, 4, COLS> *>(to) = v;
                }
            } else {
#pragma unroll
                for (int c = 0; c < COLS; c++) {
                    if (n + c >= N) break;
                    if (bf) to16[c] = (uint16_t)bf16_rne_bits(t[0][c][e]);
                    else to[c] = t[0][c][e];
                }
            }
        }
    }
}

// The splits of K of a tile, each of which has left its partial sums: the workgroup that comes last adds them in split order, as k_rw_reduce
// does, whose launch it saves: us of a call at 27 rows with that launch / so, Q4_K 4096 x 14336 19.6 / 18.6, 2560 x 9728 14.7 / 13.9, Q6_K 25.4 /
// 24.4, 17.9 / 17.1, Q8_0 24.0 / 23.2; four splits of 64 x 32 tiles 1 to 2 %.  (Who is last does not change the result.  Nobody waits for
// anybody: `arrived` counts, and the pre-pass has cleared it.)  The counter is relaxed, too, and no release by the language's rules. What orders the
// sums is the instruction set: a store at agent scope writes through to where every die sees it (sc1), s_waitcnt vmcnt(0) returns when
// it has arrived there, the barrier holds the count back until all waves are that far, and the loads behind it (sc1) pass by the die's own copies.
template <int MB, int NR>
__device__ __forceinline__ void join_splits(uint32_t *arrived, const int splits, const int m0, const int n0, const int M, const int Mp, const int N,
                                            const float *__restrict__ rowscale, const int ybf16, void *__restrict__ yg, const float *partial) {
    __shared__ uint32_t before;
    wait_vm<0>();  // this wave's partial sums have arrived where every die sees them; behind the barrier, everyone's
    __syncthreads();
    if (threadIdx.x == 0) before = __hip_atomic_fetch_add(arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (before + 1 != (uint32_t)splits) return;
    constexpr int kAtATime = MB * NR == 1 ? 2 : 8;  // outputs a thread asks for together: a trip to memory each otherwise
    const size_t plane = (size_t)Mp * N;
    for (int u0 = (int)threadIdx.x; u0 < 1024 * MB * NR; u0 += kAtATime * (int)blockDim.x) {
        float t[kAtATime][kMostSplits], rs[kAtATime];
#pragma unroll
        for (int e = 0; e < kAtATime; e++) {
            const int u = u0 + e * (int)blockDim.x, m = m0 + u / (32 * NR), n = n0 + u % (32 * NR);
            const bool in = u < 1024 * MB * NR && m < M && n < N;
            const float *src = partial + (in ? (size_t)m * N + n : 0);
            rs[e] = rowscale[in ? m : 0];
#pragma unroll
            for (int z = 0; z < kMostSplits; z++) t[e][z] = get_shared(src + (z < splits ? z : 0) * plane);
        }
#pragma unroll
        for (int e = 0; e < kAtATime; e++) {
            const int u = u0 + e * (int)blockDim.x, m = m0 + u / (32 * NR), n = n0 + u % (32 * NR);
            if (u >= 1024 * MB * NR || m >= M || n >= N) continue;
            float v = t[e][0];
#pragma unroll
            for (int z = 1; z < kMostSplits; z++)
                if (z < splits) v += t[e][z];
            v *= rs[e];
            if (ybf16) reinterpret_cast<uint16_t *>(yg)[(size_t)m * N + n] = (uint16_t)bf16_rne_bits(v);
            else reinterpret_cast<float *>(yg)[(size_t)m * N + n] = v;
        }
    }
}

// With a K split there is no second weight, and `arrived` has a cleared counter a tile, or is NULL where k_rw_reduce adds the splits.
// grid (8, inner x splits of K, outer / 8), up to eight waves; split z has super-blocks [z * chunk, min(spr, (z + 1) * chunk)).
// Workgroups eight apart are on one die: `outer` counts the tiles of the larger operand (by_m: the blocks of activation rows,
// otherwise the tiles of weight rows), so each die's cache holds an eighth of that one and all of the other (M = 2048, 1024 x 4096 Q4_K with the activations, 19 MB, read by every die: 60.6 us; by an eighth each: 39.1).
// The first 64 bytes of arguments arrive with the wave. The others, and the number and size of the workgroups behind them, are fetched from one piece of 128
// bytes: with 18 bytes past it a call took 0.2 to 0.6 us longer (Q2_K 1326 x 768 M = 63 7.18 -> 7.39, on another machine Q6_K 430 x 512 M = 418 8.2 -> 8.9).
static_assert(64 + 16 + sizeof(pmh::GemmSecond) + 18 <= 128, "arguments in one piece");
template <class F, int MB, int NR, int FORM>
__global__ __launch_bounds__(64 * kKwWaves) void k_qgemm_kw(const uint8_t *__restrict__ W, const uint4 *__restrict__ xs,
                                                             const float *__restrict__ rowscale, void *__restrict__ yg, int M, int Mp, int N,
                                                             int spr, int chunk, int inner, int outer, int flags,
                                                             float *partial, uint32_t *arrived, const pmh::GemmSecond second) {
    using K = Kw<F, MB, NR>;
    constexpr bool SPLIT = FORM == kSplit, MIXED = FORM == kMixed;
    extern __shared__ uint4 smem[];
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), block_waves = (int)(blockDim.x >> 6);
    const int out = (int)blockIdx.z * 8 + (int)blockIdx.x, z = (int)blockIdx.y / inner, in = (int)blockIdx.y - z * inner;
    if (out >= outer) return;  // (the whole workgroup)
    const bool by_m = flags & kByM;
    const int ybf16 = MIXED ? flags & 1 : flags & 7;  // (as a condition, & 1, it gave the tail of the other forms up to 100 instructions more)
    int nt = by_m ? in : out, nwaves = block_waves, tile_wave = wave, which = 0, tile_threads = (int)blockDim.x;
    if (!SPLIT) {
        const bool of_four = MIXED && (flags & (nt >= second.first ? kSecondOfFour : kFirstOfFour)), by_twos = of_four && (flags & kByTwos);
        take_weight(second, flags, nt, W, yg, N);
        if (MIXED) {
            nwaves = of_four ? 4 : spr < nwaves ? spr : nwaves;
            if (by_twos) {
                tile_threads = 256, which = wave >> 2, tile_wave = wave & 3, nt = 2 * nt + which;
                if (nt * (32 * NR) >= N) nt--, M = 0;  // (an odd last tile has none beside it: once more, and not stored)
            }
        }
        partial = nullptr;
    }
    const int m0 = (by_m ? out : in) * (32 * MB);
    const int n0 = nt * (32 * NR);
    // wave w takes every nwaves'th super-block of the split from the w'th on: what the workgroup reads at a time lies side by side
    const int own = (spr < (z + 1) * chunk ? spr : (z + 1) * chunk) - z * chunk - tile_wave;
    const bool idle = own < 1;  // the last split is the shortest: a wave left without work multiplies one super-block for nothing
    const int sb0 = idle ? 0 : z * chunk + tile_wave, cnt = idle ? 1 : (own + nwaves - 1) / nwaves;
    const uint32_t row_bytes = (uint32_t)spr * F::kBytes;
    KwCopy<F, MB, NR> C;
#pragma unroll
    for (int j = 0; j < K::kCopies; j++) {
        int idx = lane + 64 * j;
        idx = idx < K::kItems ? idx : K::kItems - 1;
        const int row = idx / F::kPieces, p = F::slot(idx % F::kPieces, row);  // (the swizzle is its own inverse)
        int n = n0 + row;
        n = n < N ? n : N - 1;  // rows past the last repeat it
        C.off[j] = (uint32_t)(n - n0) * row_bytes + F::piece_off(p);
        C.by64 |= (F::half_delta(p) >> 6 & 1u) << j, C.by32 |= (F::half_delta(p) >> 5 & 1u) << j;
    }
    uint4 *st0 = smem + wave * (2 * K::kItems), *st1 = st0 + K::kItems;
    uint32_t sb_off = (uint32_t)sb0 * F::kBytes;
    const size_t left = (size_t)(N - n0) * row_bytes;
    const __amdgpu_buffer_rsrc_t r =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(W + (size_t)n0 * row_bytes), 0, (int)(left < 0xFFFFFFF0u ? left : 0xFFFFFFF0u), 0x00027000);
    const uint32_t step = 32u * (uint32_t)Mp, a_off = (uint32_t)(g * Mp + m0 + col) * 16u;
    const uint8_t *xa = reinterpret_cast<const uint8_t *>(xs) + (size_t)(sb0 * 2 * K::kSteps) * step;
    // (beside a weight of eight waves a tile of four may have four more in its workgroup, which wait and store)
    const bool works = !MIXED || tile_wave < nwaves;
    float rs_mine = 0.0f;
    float16_t acc[NR][MB], part[NR][MB];
    if (works) {
        C.template issue<0>(r, sb_off, st0, lane);
        __builtin_amdgcn_sched_barrier(0);
        half8_t af[Kw<F, MB, NR>::kDepth][MB];
#pragma unroll
        for (int s = 0; s < K::kDepth; s++) {
#pragma unroll
            for (int i = 0; i < MB; i++) af[s][i] = *reinterpret_cast<const half8_t *>(at(xa, a_off) + 512 * i);
            xa += step;
        }
        __builtin_amdgcn_sched_barrier(0);
        rs_mine = lane < 32 * MB ? rowscale[m0 + lane] : 0.0f;
#pragma unroll
        for (int rg = 0; rg < NR; rg++)
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int e = 0; e < 16; e++) acc[rg][i][e] = 0.0f, part[rg][i][e] = 0.0f;
        const size_t jump = (size_t)(nwaves - 1) * (2 * K::kSteps) * step;  // (past 4 GiB from 2.2 million activation rows on)
        for (int s = 0; s + 1 < cnt; s++) {
            if (F::kUnitHalves == 1) {
                kw_half<F, MB, NR, 0, true>(st0, st1, r, sb_off, C, xa, step, jump, a_off, af, lane, acc, part);
                sb_off += (uint32_t)nwaves * F::kBytes;
                kw_half<F, MB, NR, 1, true>(st1, st0, r, sb_off, C, xa, step, jump, a_off, af, lane, acc, part);
            } else {
                sb_off += (uint32_t)nwaves * F::kBytes;
                kw_half<F, MB, NR, 0, true>(st0, st1, r, sb_off, C, xa, step, jump, a_off, af, lane, acc, part);
                kw_half<F, MB, NR, 1, true>(st0, st1, r, sb_off, C, xa, step, jump, a_off, af, lane, acc, part);
                uint4 *t = st0;
                st0 = st1, st1 = t;
            }
        }
        kw_half<F, MB, NR, 0, F::kUnitHalves == 1>(st0, st1, r, sb_off, C, xa, step, 0, a_off, af, lane, acc, part);
        kw_half<F, MB, NR, 1, false>(F::kUnitHalves == 1 ? st1 : st0, st1, r, sb_off, C, xa, step, 0, a_off, af, lane, acc, part);
    }
    wait_vm<0>();
    __syncthreads();
    float4_t *red = reinterpret_cast<float4_t *>(smem);
    float *rs = reinterpret_cast<float *>(smem) + (size_t)block_waves * K::kTile * 4 + 32 * MB * which;
    if (works) {
#pragma unroll
        for (int rg = 0; rg < NR; rg++)
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int q = 0; q < 4; q++)
                    red[wave * K::kTile + ((rg * MB + i) * 4 + q) * kTileRun + tile_slot(lane)] =
                        idle ? float4_t{0.0f, 0.0f, 0.0f, 0.0f}
                             : float4_t{acc[rg][i][4 * q], acc[rg][i][4 * q + 1], acc[rg][i][4 * q + 2], acc[rg][i][4 * q + 3]};
    }
    if (tile_wave == 0 && lane < 32 * MB) rs[lane] = rs_mine;
    __syncthreads();
    if (MIXED) red += 4 * which * K::kTile;
    const int tile_tid = MIXED ? tid - 256 * which : (int)threadIdx.x, threads = MIXED ? tile_threads : (int)blockDim.x;
    constexpr bool kJoins = SPLIT && pmh::joins_splits(MB, NR);
    if (nwaves > 4) add_tiles<K::kTile, MB, NR, (MB * NR == 4 ? 2 : 1), kKwWaves, kJoins>(red, rs, tile_tid, threads, nwaves, m0, n0, M, Mp, N, z, ybf16, yg, partial);
    else add_tiles<K::kTile, MB, NR, MB * NR, 4, kJoins>(red, rs, tile_tid, threads, nwaves, m0, n0, M, Mp, N, z, ybf16, yg, partial);
    if constexpr (kJoins) {
        if (arrived) join_splits<MB, NR>(arrived + out * inner + in, (int)gridDim.y / inner, m0, n0, M, Mp, N, rowscale, ybf16, yg, partial);
    }
}

}  // namespace

namespace pmh {

template <class F, int MB, int NR>
static hipError_t launch_kw(const GemmPlan &p, const uint8_t *w, const uint4 *xs, const float *rowscale, void *y, bool y_bf16, int64_t m, int64_t n, int spr,
                            float *partial, uint32_t *arrived, GemmSecond second, int second_nw, hipStream_t s) {
    using K = Kw<F, MB, NR>;
    auto waves_of = [&](int nw) { return p.chunk < nw ? p.chunk : nw; };
    const int w0 = waves_of(p.nw), w1 = second.n > 0 ? waves_of(second_nw) : w0;
    // Two weights, tiles of eight waves (or what a short row has of them) and of four: workgroups of eight for both, so that either result
    // is the sum that it is alone.
    const bool mixed = w0 != w1;
    const int nwaves = mixed ? kKwWaves : w0;
    auto kern = p.splits > 1 ? k_qgemm_kw<F, MB, NR, kSplit> : mixed ? k_qgemm_kw<F, MB, NR, kMixed> : k_qgemm_kw<F, MB, NR, kPlain>;
    const size_t stage = (size_t)nwaves * 2 * K::kItems * 16, red = (size_t)nwaves * K::kTile * 16 + (mixed ? 2 : 1) * 32 * MB * 4, lds = stage > red ? stage : red;
    static_assert((size_t)kKwWaves * 2 * K::kItems * 16 <= 160 * 1024 && (size_t)kKwWaves * K::kTile * 16 + 2 * 32 * MB * 4 <= 160 * 1024, "LDS");
    if (lds > 64 * 1024) {
        hipError_t a = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (a != hipSuccess) return a;
    }
    const int t0 = (int)((n + 32 * NR - 1) / (32 * NR)), t1 = (second.n + 32 * NR - 1) / (32 * NR), mblocks = (int)((m + 32 * MB - 1) / (32 * MB));
    const bool by_m = kw_by_m(mblocks, t0 + t1, MB, NR, F::kBytes);
    // Tiles of four go two to a workgroup where that is fewer rounds of the busiest die's compute units.
    // Otherwise a workgroup each, whose other four waves wait: a machine that is not full has more of it at work (us, by twos / alone: Q8_0
    // 4096 and 2048 x 4096 M = 96 30.6 / 23.4, Q4_K 4096 and 1024 x 4096 M = 100 24.1 / 17.6).
    const bool by_twos = mixed && kw_mixed(mblocks, w0 == 4 ? t0 : t1, w0 == 4 ? t1 : t0, by_m, MB, NR).by_twos;
    const int of_four = !mixed ? 0 : (w0 == 4 ? kFirstOfFour : kSecondOfFour) | (by_twos ? kByTwos : 0);
    second.first = by_twos && w0 == 4 ? (t0 + 1) / 2 : t0;
    const int tiles = second.first + (by_twos && w1 == 4 ? (t1 + 1) / 2 : t1);  // (or pairs of them)
    const int inner = by_m ? tiles : mblocks, outer = by_m ? mblocks : tiles;
    const dim3 grid(8, (unsigned)(inner * p.splits), (unsigned)((outer + 7) / 8));
    hipLaunchKernelGGL(kern, grid, dim3(64 * nwaves), lds, s, w, xs, rowscale, y, (int)m, p.mp, (int)n, spr, p.chunk, inner, outer,
                       (y_bf16 ? 1 : 0) | (by_m ? kByM : 0) | (second.n > 0 ? kHasSecond | of_four : 0), p.splits > 1 ? partial : nullptr, arrived, second);
    return hipGetLastError();
}

template <class F>
static hipError_t launch_kw_tile(const GemmPlan &p, const uint8_t *w, const uint4 *xs, const float *rowscale, void *y, bool y_bf16, int64_t m, int64_t n,
                                 int spr, float *partial, uint32_t *arrived, GemmSecond second, int second_nw, hipStream_t s) {
    if (p.mb == 1 && p.nr == 1) return launch_kw<F, 1, 1>(p, w, xs, rowscale, y, y_bf16, m, n, spr, partial, arrived, second, second_nw, s);
    if (p.mb == 1) return launch_kw<F, 1, 2>(p, w, xs, rowscale, y, y_bf16, m, n, spr, partial, arrived, second, second_nw, s);
    if (p.nr == 1) return launch_kw<F, 2, 1>(p, w, xs, rowscale, y, y_bf16, m, n, spr, partial, arrived, second, second_nw, s);
    return launch_kw<F, 2, 2>(p, w, xs, rowscale, y, y_bf16, m, n, spr, partial, arrived, second, second_nw, s);
}

hipError_t launch_qgemm_kw(uint32_t type, const GemmPlan &p, const uint8_t *w, const void *xs, const float *rowscale, void *y, bool y_bf16, int64_t m,
                           int64_t n, int spr, uint32_t order, float *partial, uint32_t *arrived, const GemmSecond &second, int second_nw, hipStream_t s) {
    const uint4 *x4 = reinterpret_cast<const uint4 *>(xs);
    const bool ref = order == kOrderRef;
    auto go = [&](auto format) { return launch_kw_tile<decltype(format)>(p, w, x4, rowscale, y, y_bf16, m, n, spr, partial, arrived, second, second_nw, s); };
    switch (type) {
    case kTypeQ4K: return ref ? go(KwQ45<0, 0>{}) : go(KwQ45<1, 0>{});
    case kTypeQ5K: return ref ? go(KwQ45<0, 1>{}) : go(KwQ45<1, 1>{});
    case kTypeQ6K: return go(KwQ6{});
    case kTypeQ8_0: return go(KwQ8{});
    case kTypeQ3K: return go(KwQ23<2>{});
    case kTypeQ2K: return go(KwQ23<3>{});
    default: return hipErrorInvalidValue;
    }
}

}  // namespace pmh
