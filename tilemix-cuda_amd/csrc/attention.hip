// Routed INT8/FP16 fused attention for gfx950 (MI355X).
//
// Replaces fused_fp16_attention + launch_fused_fp16_attention of the reference
// (src/tilemix.cu:51-220, 238-278). Design (not a translation):
//
//  * A 256-thread workgroup (4 wave64s) owns 128 query rows of one head - one
//    Q quantization block - and streams the keys in 64-key tiles, one K
//    quantization block each, so q_scale is constant per workgroup and
//    k_scale per tile.
//  * Each wave owns 32 query rows (two 16-row routing cells tall) and works
//    on 32x32 MFMA blocks. Scores are computed transposed, S^T = K Q^T, with
//    v_mfma_f32_32x32x16_f16 (FP16 cells) or v_mfma_i32_32x32x32_i8 (INT8
//    cells, exact int32 dots), one block per 32 keys. In that layout lane
//    (q, h) = (lane % 32, lane / 32) holds 16 keys of query row q, so a row's
//    online-softmax state lives in lanes q and q + 32 and its maximum needs
//    one cross-lane step. A 32x32 MFMA does the work of two 16x16 ones but
//    holds the wave's instruction issue about as long as one, which leaves
//    the SIMD free for the other wave's (or this wave's) VALU work.
//  * The probabilities stay in registers and feed O^T += V^T P^T on
//    v_mfma_f32_32x32x16_f16: the accumulator elements of 8 consecutive
//    score slots are exactly the P^T operand of one 16-key step, and the V^T
//    operand is read from the row-major V tile in LDS with
//    ds_read_b64_tr_b16, which transposes 16-bit elements across each
//    16-lane group (key order inside a step permuted identically on both
//    operands). Row sums add exactly the fp16 probabilities P.V uses
//    (v_dot2_f32_f16 against ones); the two lanes of a row are summed once,
//    at the end.
//  * K, K8 and V tiles move HBM -> LDS with buffer_load ... lds (no VGPR
//    staging): per-lane offsets into the LDS rows (unpadded with rotated
//    16-byte chunks: all K8 rows, K / V rows of 128 or 256 bytes) are
//    computed once, each tile only changes a scalar offset, and rows past
//    the end of the head read as zero. Every wave issues the same number of
//    loads per buffer (spare slots read out of range into a 1 KiB landing
//    area), so the issue code has no branches. V has two buffers, K and K8
//    one each: the next tile's K, K8 and V are all fetched after the tile's
//    second barrier, while softmax and P.V run, so no tile load is issued
//    among the score MFMAs; two barriers per tile. At d = 128, 56 KiB of tile
//    buffers per workgroup.
//  * Each SIMD runs one wave of each of the CU's two workgroups. A tile is an
//    MFMA phase (P.V, barrier, next scores) and a VALU phase (softmax). A
//    wave's issue priority is low in the first half of each phase and high
//    in the second, so of two waves in the same phase the one further along
//    wins arbitration and leaves it first: this pushes the pair apart, one
//    on the matrix core while the other runs exponentials.
//  * A 32-key MFMA block is one routing cell wide and two cells (the wave's
//    two 16-row halves) tall. The branch is taken on wave-uniform route
//    masks; a wave whose cells mix routes computes both score kinds and
//    selects per lane.
//  * The optional in-kernel Q quantization reproduces quantize_tilemix_qk's
//    bytes exactly: the workgroup's 128 rows are exactly one Q block. The
//    bytes reach the INT8 operand layout through a lane swap between the
//    two halves of the wave, not through LDS.

#include "attention_common.h"
#include "attention_rules.h"
#include "tilemix_capi.h"

#include <atomic>
#include <cmath>
#include <cstring>
#include <mutex>
#include <type_traits>

namespace tilemix {
namespace {

constexpr int kThreadsPerGroup = 256;
constexpr int kWavesPerGroup = kThreadsPerGroup / kWave;
constexpr int kRowsPerWave = 32;

template <int DC>
struct Layout {
    static constexpr int kDP = 32 * DC;            // padded head dim, fp16 path
    static constexpr int kD8C = (DC + 1) / 2;      // 64-feature chunks, int8 path
    static constexpr int kDP8 = 64 * kD8C;
    // K / V rows hold 2 * kDP bytes. Rows of 256 bytes (d > 96) and 128 bytes
    // (32 < d <= 64) are unpadded, with 16-byte chunk c of row r at chunk
    // position (c + rot(r)) mod (chunks per row), so that the fragment reads
    // are free of LDS bank conflicts with no pad bytes to move (rot below).
    // Other rows are padded by 16 (K) or 32 (V) bytes. K8 rows are 128 bytes
    // (d > 64) or 64 bytes, rotated the same way.
    static constexpr int kRowBytes = kDP * 2;
    static constexpr bool kRotate = kRowBytes == 256 || kRowBytes == 128;
    static constexpr bool kRotate8 = kDP8 == 128 || kDP8 == 64;
    static constexpr int kKStride = kRotate ? kRowBytes : kRowBytes + 16;
    static constexpr int kVStride = kRotate ? kRowBytes : kRowBytes + 32;
    static constexpr int kK8Stride = kRotate8 ? kDP8 : kDP8 + 16;
    static constexpr int kKBytes = kTileKeys * kKStride;
    static constexpr int kVBytes = kTileKeys * kVStride;
    static constexpr int kK8Bytes = kTileKeys * kK8Stride;
    // One buffer_load ... lds per wave moves 1 KiB (64 lanes x 16 bytes).
    static constexpr int kKLoads = kKBytes / 1024;
    static constexpr int kVLoads = kVBytes / 1024;
    static constexpr int kK8Loads = kK8Bytes / 1024;
    static constexpr int kKPerWave = (kKLoads + kWavesPerGroup - 1) / kWavesPerGroup;
    static constexpr int kVPerWave = (kVLoads + kWavesPerGroup - 1) / kWavesPerGroup;
    static constexpr int kK8PerWave = (kK8Loads + kWavesPerGroup - 1) / kWavesPerGroup;
    // K, V buffer 0, K8, V buffer 1.
    static constexpr int kV1Offset = kVBytes + kK8Bytes;  // V buffer 1 - V buffer 0
    static constexpr int kSmemBytes = kKBytes + kVBytes + kK8Bytes + kVBytes;
    static_assert(kKBytes % 1024 == 0 && kVBytes % 1024 == 0 && kK8Bytes % 1024 == 0,
                  "tiles are whole wave loads");
    // Chunk rotation of a rotated row of kChunks 16-byte chunks. Key rows
    // (K, K8) are read as 32 consecutive rows x one chunk per half-wave: the
    // rows that share one 256-byte sweep of the banks share a rotation, and
    // consecutive sweeps step it by one chunk (measured on 64-byte K8 rows:
    // 13 % of LDS-active cycles in bank conflicts with a rotation that steps
    // every two rows, 0.9 % with this one). Value rows are read by
    // ds_read_b64_tr_b16 in 4-row x 16-feature blocks.
    template <int kChunks, bool kKey>
    __device__ static int rot(int row) {
        static_assert(kChunks == 16 || kChunks == 8 || kChunks == 4, "rotated rows are 256, 128 or 64 bytes");
        if constexpr (kKey)
            return kChunks == 16 ? row & 15 : kChunks == 8 ? (row >> 1) & 7 : (row >> 2) & 3;
        else
            return kChunks == 16 ? (2 * row) & 15 : kChunks == 8 ? row & 6 : 2 * ((row >> 2) & 1);
    }
    // Offset of byte `byte` of row `row` in a rotated tile.
    template <int kChunks, bool kKey>
    __device__ static int rotated(int row, int byte) {
        return row * 16 * kChunks + ((((byte >> 4) + rot<kChunks, kKey>(row)) & (kChunks - 1)) << 4) + (byte & 15);
    }
    // Global offset that DMA lane `lane` of 1 KiB piece w fetches for a
    // rotated tile (kOutOfRange past the row's bytes): the inverse of rotated.
    template <int kChunks, bool kKey>
    __device__ static int rotated_lane(int w, int lane, int row_bytes, int global_row_bytes) {
        const int landing = 1024 * w + 16 * lane;
        const int row = landing / (16 * kChunks);
        const int column = ((((landing >> 4) & (kChunks - 1)) - rot<kChunks, kKey>(row)) & (kChunks - 1)) << 4;
        return column < row_bytes ? row * global_row_bytes + column : kOutOfRange;
    }
    // Offset of byte `byte` (< 2 * kDP, or < kDP8 for K8) of row `row` in the
    // K / V / K8 tile.
    __device__ static int k_at(int row, int byte) {
        if constexpr (kRotate) return rotated<kRowBytes / 16, true>(row, byte);
        else return row * kKStride + byte;
    }
    __device__ static int v_at(int row, int byte) {
        if constexpr (kRotate) return rotated<kRowBytes / 16, false>(row, byte);
        else return row * kVStride + byte;
    }
    __device__ static int k8_at(int row, int byte) {
        if constexpr (kRotate8) return rotated<kDP8 / 16, true>(row, byte);
        else return row * kK8Stride + byte;
    }
    // Global offset that DMA lane `lane` of 1 KiB piece w fetches.
    template <bool kKey>
    __device__ static int kv_lane_offset(int w, int lane, int stride, int row_bytes, int global_row_bytes) {
        if constexpr (kRotate) return rotated_lane<kRowBytes / 16, kKey>(w, lane, row_bytes, global_row_bytes);
        else return lane_offset(w, lane, stride, row_bytes, global_row_bytes);
    }
    __device__ static int k8_lane_offset(int w, int lane, int row_bytes) {
        if constexpr (kRotate8) return rotated_lane<kDP8 / 16, true>(w, lane, row_bytes, row_bytes);
        else return lane_offset(w, lane, kK8Stride, row_bytes, row_bytes);
    }
};

typedef float float16v __attribute__((ext_vector_type(16)));
typedef int int16v __attribute__((ext_vector_type(16)));

// Online-softmax state of the query row a lane owns (row lane & 31 of the
// wave's 32; lanes l and l ^ 32 hold the same row, each for half of every
// 32-key block), scores in the log2 domain, m raised lazily (kLazyRescale).
template <int kOB>
struct RowState {
    // O^T accumulators: o[fb][j] is output row R = 8 (j / 4) + 4 h + j % 4
    // (h = lane / 32) of feature block fb, i.e. feature 16 fb + R for R < 16
    // and kDP / 2 + 16 fb + R - 16 above (the two 16-row halves of a block
    // sit kDP / 2 features apart, which keeps the transposed V reads free of
    // bank conflicts).
    float16v o[kOB];
    float lsum;       // this lane's part of the row sum of P (the fp16 values P.V uses)
    float m;
};

// Maximum of the 16 values of a 32x32 accumulator block, 8 v_max3.
[[maybe_unused]] __device__ __forceinline__ float block_max16(const float16v& x) {
    const float a = max3(x[0], x[1], x[2]), b = max3(x[3], x[4], x[5]), e = max3(x[6], x[7], x[8]);
    const float f = max3(x[9], x[10], x[11]), g = max3(x[12], x[13], x[14]);
    return max3(max3(a, b, e), max3(f, g, x[15]), x[15]);
}

// x[kb][j] holds the score of the lane's row against key 32 kb + 8 (j / 4) +
// 4 h + j % 4; c is the per-tile log2-domain factor (>= 0; explicit scores
// pass c = 1). ph[ks] / pl[ks] receive the fp16 probabilities of keys
// 16 ks + {4h .. 4h + 3, 8 + 4h .. 8 + 4h + 3}: the B operand (P^T) of the
// 32x32x16 P.V MFMA for key step ks.
template <int kOB, bool kPrecise, bool kPriority = true>
__device__ __forceinline__ void softmax_tile(RowState<kOB>& st, const float16v (&x)[2], float c,
                                             half8 (&ph)[4], half8 (&pl)[4]) {
    const float tile = max3(block_max16(x[0]), block_max16(x[1]), block_max16(x[1])) * c;  // c >= 0
    // The row's maximum exceeds m + kLazyRescale exactly when one of its two
    // lanes' own maxima does.
    if (__any(tile > st.m + kLazyRescale)) {
        float a = tile, b = tile;
        permlane32_swap(a, b);
        const float m_new = fmaxf(st.m, max3(a, b, b));
        // Rows with no visible key yet keep m = -inf (their sums are still 0).
        const float alpha = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(st.m - m_new);
        st.m = m_new;
#pragma unroll
        for (int fb = 0; fb < kOB; ++fb) st.o[fb] *= alpha;
        st.lsum *= alpha;
    }
    // m == -inf only while every score seen, this tile included, is masked.
    const float neg_m = st.m == -INFINITY ? 0.0f : -st.m;
    const half2v ones{1.0f16, 1.0f16};
    float part[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const int kb = ks >> 1, base = 8 * (ks & 1);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float v = __builtin_amdgcn_exp2f(__builtin_fmaf(x[kb][base + e], c, neg_m));
            const _Float16 hv = static_cast<_Float16>(v);
            ph[ks][e] = hv;
            if constexpr (kPrecise) pl[ks][e] = static_cast<_Float16>(v - static_cast<float>(hv));
        }
        // Row sums of exactly the fp16 values the P.V MFMAs use.
        float sum = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            sum = __builtin_amdgcn_fdot2(half2v{ph[ks][e], ph[ks][e + 1]}, ones, sum, false);
            if constexpr (kPrecise) sum = __builtin_amdgcn_fdot2(half2v{pl[ks][e], pl[ks][e + 1]}, ones, sum, false);
        }
        part[ks] = sum;
        if (kPriority && ks == 1) set_priority<2>();  // second half of the VALU phase
    }
    st.lsum += (part[0] + part[1]) + (part[2] + part[3]);
}

// load_to_lds with M0 = lds_address + kOffset, the add issued inside the asm
// so that the compiler keeps one scalar address per buffer, not one per slot.
template <int kOffset>
__device__ __forceinline__ void load_to_lds_at(int4v rsrc, unsigned lds_address, int voffset, int soffset) {
    if constexpr (kOffset == 0) {
        load_to_lds(rsrc, lds_address, voffset, soffset);
    } else {
        asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                     :
                     : "s"(lds_address), "v"(voffset), "s"(rsrc), "s"(soffset), "i"(kOffset)
                     : "memory", "scc");
    }
}

// The 1 KiB pieces one wave moves of a tile buffer that splits evenly over
// the workgroup's four waves: slot t lands 4 KiB past slot t - 1 (pieces
// wave, wave + 4, ...), so all slots share the first one's LDS address.
template <int t, int kSlots>
__device__ __forceinline__ void load_slots_from(int4v rsrc, unsigned first, const int (&voffset)[kSlots], int soffset) {
    if constexpr (t < kSlots) {
        load_to_lds_at<4096 * t>(rsrc, first, voffset[t], soffset);
        load_slots_from<t + 1, kSlots>(rsrc, first, voffset, soffset);
    }
}
template <int kSlots>
__device__ __forceinline__ void load_slots(int4v rsrc, unsigned first, const int (&voffset)[kSlots], int soffset) {
    load_slots_from<0, kSlots>(rsrc, first, voffset, soffset);
}

// The pieces one of eight waves moves of a tile buffer kBase bytes past the
// wave's first LDS address: slot t lands 8 KiB past slot t - 1. `base` bytes
// are added to the lanes' offsets, so the range check covers the whole address.
template <int kBase, int t, int kSlots>
__device__ __forceinline__ void load_slots_at(int4v rsrc, unsigned first, const int (&voffset)[kSlots], int base) {
    if constexpr (t < kSlots) {
        load_to_lds_at<kBase + 8192 * t>(rsrc, first, voffset[t] + base, 0);
        load_slots_at<kBase, t + 1, kSlots>(rsrc, first, voffset, base);
    }
}

// fp32 rows of 128 or 64 features (O, or a split's partial rows) leave the
// kernels without dot export through LDS. From registers, each store
// instruction writes 16 bytes to each of 32 rows, i.e. 32 partial cache lines,
// and those lines, held in the XCD's L2 until written back, evict K / V tiles.
// Staged, each store writes 8 rows x 128 bytes (full cache lines) with a
// non-temporal hint, so the rows bypass the L2. Each wave stages its 32 rows
// (qw .. qw + 31 of M) in kOB passes of 32 features through its own region of
// kStageBytes, which no other wave or load uses. out / out_row: the head's
// first row and the distance between rows, in floats; every value is
// multiplied by factor.
constexpr int kStageBytes = 32 * 128;
template <int kOB>
__device__ __forceinline__ void store_staged(const RowState<kOB>& st, unsigned char* region, float* out,
                                             std::int64_t out_row, float factor, int qw, int M) {
    constexpr int kRowBytes = 128;  // 32 features per pass
    constexpr int kPasses = kOB;
    constexpr int kPassesPerHalf = kPasses / 2;  // passes over the first half of the features
    // The lane's number, counted afresh here: the stage addresses depend on it
    // only, and kept or computed before the key loop they would hold registers
    // through it.
    int none = 0;
    asm volatile("" : "+v"(none));
    const int me = static_cast<int>(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, static_cast<unsigned>(none))));
    const int my_q = me & 31, my_h = me >> 5;
    const int c = me & 7, sub = me >> 3;  // read side: chunk c of row sub of each 8-row piece
#pragma unroll
    for (int pass = 0; pass < kPasses; ++pass) {
        // Features 32 pass .. 32 pass + 31: slots
        // r4 = 2 (pass / kPassesPerHalf) + r of blocks
        // fb = 2 (pass % kPassesPerHalf) + b hold features
        // 32 pass + 16 b + 8 r + 4 h (+ 0..3) of row q, i.e. 16-byte
        // chunk 4 b + 2 r + h of the pass, stored rotated by the row.
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const int r4 = 2 * (pass / kPassesPerHalf) + r, fb = 2 * (pass % kPassesPerHalf) + b;
                const float4v value{st.o[fb][4 * r4], st.o[fb][4 * r4 + 1], st.o[fb][4 * r4 + 2], st.o[fb][4 * r4 + 3]};
                const int chunk = 4 * b + 2 * r + my_h;
                *reinterpret_cast<float4v*>(region + my_q * kRowBytes + (((chunk + my_q) & 7) << 4)) = value * factor;
            }
        // Piece i: rows 8 i .. 8 i + 7 of the wave, 8 lanes per row. Every
        // read is issued before any store (the reads stay in the wave's
        // region; only the stores depend on the row).
        float4v piece[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int local = 8 * i + sub;
            piece[i] = *reinterpret_cast<const float4v*>(region + local * kRowBytes + (((c + local) & 7) << 4));
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(piece[i]));  // keep the reads here
        float* const first = out + static_cast<std::int64_t>(qw + sub) * out_row + 32 * pass + 4 * c;
        const std::int64_t piece_step = 8 * out_row;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (qw + 8 * i + sub < M)
                __builtin_nontemporal_store(piece[i], reinterpret_cast<float4v*>(first + i * piece_step));
    }
}

// A wave's 32 query rows in registers. qf: B operand of the 32x32x16 QK^T
// MFMA, lane (q, h) holding features 16c + 8h .. 16c + 8h + 7 of its row for
// chunk c. With INT8 operands also q8f, the B operand of the INT8 MFMA (lane
// (q, h): features 32m + 16h .. 32m + 16h + 15 for chunk m), and q_scale:
// quantized here (p.fuse_q_quant) or read from Q8. `group_bits` (shared, one
// entry per wave of the workgroup, `waves` of them): the maxima of the waves;
// those of this wave's Q block start at entry `block_first`. Every wave of the
// workgroup calls it. writer: this workgroup writes Q8 / q_scales where asked.
template <int DC, int kPiece>
__device__ __forceinline__ void prepare_q(const AttnParams& p, std::int64_t head, int qblock, int row, int lane,
                                          unsigned* group_bits, int waves, int wave, int block_first, bool writer,
                                          half8 (&qf)[2 * DC], int4v (&q8f)[2 * Layout<DC>::kD8C], float& q_scale) {
    using L = Layout<DC>;
    constexpr int kQC = 2 * DC;
    constexpr int kQ8C = 2 * L::kD8C;
    constexpr bool kVector = kPiece >= 8;
    const int M = p.M, d = p.d;
    const int h = lane >> 5;
    const std::uint16_t* Qh = p.Q + head * p.q_stride;
    {
#pragma unroll
        for (int c = 0; c < kQC; ++c) {
            const int feature = 16 * c + 8 * h;
            if constexpr (kVector) {
                qf[c] = (row < M && feature < d)
                    ? *reinterpret_cast<const half8*>(Qh + static_cast<std::int64_t>(row) * p.q_row + feature)
                    : half8{};
            } else if constexpr (kPiece == 4) {
                uint4v words{0u, 0u, 0u, 0u};
#pragma unroll
                for (int w = 0; w < 4; ++w)
                    if (row < M && feature + 2 * w < d)
                        words[w] = *reinterpret_cast<const std::uint32_t*>(Qh + static_cast<std::int64_t>(row) * p.q_row + feature + 2 * w);
                qf[c] = __builtin_bit_cast(half8, words);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    qf[c][e] = (row < M && feature + e < d)
                        ? __builtin_bit_cast(_Float16, Qh[static_cast<std::int64_t>(row) * p.q_row + feature + e])
                        : static_cast<_Float16>(0.0f);
            }
        }
    }

    if (p.int8_operands) {
        if (p.fuse_q_quant) {
            // Four waves' rows are exactly one 128-row Q block. Its
            // maximum |x| as fp16 bit patterns: unsigned order is float order
            // for them, NaN patterns (> 0x7c00) sorting above +inf.
            unsigned top = 0;
#pragma unroll
            for (int c = 0; c < kQC; ++c) {
                const uint4v words = __builtin_bit_cast(uint4v, qf[c]);
#pragma unroll
                for (int w = 0; w < 4; ++w) top = max_u16x2(top, words[w] & 0x7fff7fffu);
            }
            unsigned bits = wave_max_bits(max(top & 0xffffu, top >> 16));
            if (lane == 0) group_bits[wave] = bits;
            __syncthreads();
            const unsigned* const block_bits = group_bits + block_first;
            bits = max(max(block_bits[0], block_bits[1]), max(block_bits[2], block_bits[3]));
            unsigned any = bits;
            if (waves > 4)
                for (int w = 0; w < waves; ++w) any = max(any, group_bits[w]);
            if (any > 0x7c00u) {
                // A NaN in the workgroup: the maximum skips NaNs, as fmaxf does.
                unsigned clean = 0;
#pragma unroll
                for (int c = 0; c < kQC; ++c)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        // The element is copied out first: __builtin_bit_cast
                        // applied to a vector element expression reads
                        // element 0 under this compiler.
                        const _Float16 x = qf[c][e];
                        const unsigned hb = __builtin_bit_cast(std::uint16_t, x) & 0x7fffu;
                        clean = hb <= 0x7c00u ? max(clean, hb) : clean;
                    }
                clean = wave_max_bits(clean);
                __syncthreads();
                if (lane == 0) group_bits[wave] = clean;
                __syncthreads();
                bits = max(max(block_bits[0], block_bits[1]), max(block_bits[2], block_bits[3]));
            }
            const float scale = block_scale(half_bits_to_float(static_cast<std::uint16_t>(bits)));
            const float recip = 1.0f / scale;
            const _Float16 stored = static_cast<_Float16>(scale);
            q_scale = static_cast<float>(stored);
            if (writer && p.q_scales_out && wave == block_first && lane == 0)
                p.q_scales_out[head * p.q_blocks + qblock] = __builtin_bit_cast(std::uint16_t, stored);
            {
                // Bytes of fp16 chunk c (features 16c + 8h .. + 7 of the row).
                uint2v packed[L::kDP8 / 16];
#pragma unroll
                for (int c = 0; c < L::kDP8 / 16; ++c) {
                    packed[c] = uint2v{0u, 0u};
                    if (c < kQC && scale > 0.0f) {
                        const uint4v words = __builtin_bit_cast(uint4v, qf[c < kQC ? c : 0]);
                        int v[8];
#pragma unroll
                        for (int w = 0; w < 4; ++w) {
                            v[2 * w] = quantize_half<0>(words[w], scale, recip);
                            v[2 * w + 1] = quantize_half<1>(words[w], scale, recip);
                        }
                        packed[c][0] = pack_bytes(v[0], v[1], v[2], v[3]);
                        packed[c][1] = pack_bytes(v[4], v[5], v[6], v[7]);
                    }
                    const int feature = 16 * c + 8 * h;
                    if (p.q8_out && writer && row < M && feature < d) {
                        std::int8_t* dst = p.q8_out + head * static_cast<std::int64_t>(M) * d +
                                           static_cast<std::int64_t>(row) * d + feature;
                        if constexpr (kVector) {
                            *reinterpret_cast<uint2v*>(dst) = packed[c];
                        } else {
                            for (int e = 0; e < 8 && feature + e < d; ++e)
                                dst[e] = static_cast<std::int8_t>(packed[c][e / 4] >> (8 * (e % 4)));
                        }
                    }
                }
                // INT8 chunk m = fp16 chunks 2m (features 32m .. 32m + 15)
                // and 2m + 1 (32m + 16 .. 32m + 31). Lanes h = 0 keep their
                // bytes of chunk 2m and take lane (q, 1)'s; lanes h = 1 keep
                // their bytes of chunk 2m + 1 and take lane (q, 0)'s: one
                // v_permlane32_swap per dword.
#pragma unroll
                for (int m = 0; m < kQ8C; ++m) {
                    const uint2v keep = h ? packed[2 * m + 1] : packed[2 * m];
                    const uint2v send = h ? packed[2 * m] : packed[2 * m + 1];
                    std::uint32_t got[2];
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        const std::uint32_t word = send[k];  // copied out before the bit cast, see above
                        float a = __builtin_bit_cast(float, word), b = a;
                        permlane32_swap(a, b);  // a: lane (q, 0)'s dword, b: lane (q, 1)'s
                        got[k] = __builtin_bit_cast(std::uint32_t, h ? a : b);
                    }
                    q8f[m] = h ? int4v{static_cast<int>(got[0]), static_cast<int>(got[1]), static_cast<int>(keep[0]),
                                       static_cast<int>(keep[1])}
                               : int4v{static_cast<int>(keep[0]), static_cast<int>(keep[1]), static_cast<int>(got[0]),
                                       static_cast<int>(got[1])};
                }
            }
        } else {
            // Q8 rows already come in the operand layout: 16 bytes per lane
            // and chunk, read straight into q8f.
            q_scale = half_bits_to_float(p.q_scales[head * p.q_blocks + qblock]);
            const std::int8_t* Q8h = p.Q8 + head * static_cast<std::int64_t>(M) * d;
#pragma unroll
            for (int m = 0; m < kQ8C; ++m) {
                const int feature = 32 * m + 16 * h;
                int4v chunk;
                if constexpr (kPiece == 16) {
                    chunk = (row < M && feature < d)
                        ? *reinterpret_cast<const int4v*>(Q8h + static_cast<std::int64_t>(row) * d + feature)
                        : int4v{0, 0, 0, 0};
                } else if constexpr (kPiece != 0) {
                    chunk = int4v{0, 0, 0, 0};
#pragma unroll
                    for (int w = 0; w < 4; ++w)
                        if (row < M && feature + 4 * w < d)
                            chunk[w] = *reinterpret_cast<const int*>(Q8h + static_cast<std::int64_t>(row) * d + feature + 4 * w);
                } else {
                    unsigned char bytes[16];
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        bytes[e] = (row < M && feature + e < d)
                            ? static_cast<unsigned char>(Q8h[static_cast<std::int64_t>(row) * d + feature + e])
                            : 0;
                    chunk = __builtin_bit_cast(int4v, bytes);
                }
                q8f[m] = chunk;
            }
        }
    }
}

// kPiece: what rows allow (access_piece). 16: tiles move by LDS DMA in 16-byte
// pieces. 8 (d a multiple of 8 only): K and V the same way, and K8 rows, which
// start on 8 bytes, in 16-byte pieces from dword-aligned addresses; a row's
// last piece may carry the next row's first bytes, which meet zeros of Q8. 4:
// K and V rows too; what a K row's last piece carries past d is masked when it
// is read (V's reaches only features past d of O). A tile of which a piece would
// end past the head comes in by dwords instead (load_tile_dwords). 0: single
// elements.
// kRange: what a workgroup covers of its 128-row block's key tiles. kWhole: all
// of them. kSplit: one range (AttnParams::splits), whose partial row state it
// writes. kInTurn: all ranges of a split call one after the other, each with a
// row state of its own, merged as split_combine_kernel merges them: the split
// call's bits without a workspace, for a stream that is being captured. It
// holds a second O in LDS, so one workgroup per CU; a call that is split has no
// more. Reading and writing that O takes 1.1 to 1.5 us a range: captured, 8
// heads x 512 x 8192 x 128 take 197 us (kWhole, whose sums have another order,
// 174), 4 x 2048 x 128 causal 56 (47), 12 x 1003 x 72 causal precise 38 (36).
enum class KeyRange { kWhole, kSplit, kInTurn };
template <int DC, int kPiece, bool kPrecise, bool kDots, KeyRange kRange>
__global__ __launch_bounds__(kThreadsPerGroup, kGroupsPerCU) void attention_kernel(const AttnParams p) {
    constexpr bool kSplit = kRange == KeyRange::kSplit, kInTurn = kRange == KeyRange::kInTurn;
    using L = Layout<DC>;
    constexpr int kDP = L::kDP;
    constexpr int kOB = DC;               // 32-feature output blocks
    constexpr int kQC = kDP / 16;         // 16-feature Q / K chunks (fp16 MFMA k-steps)
    constexpr int kQ8C = L::kDP8 / 32;    // 32-feature Q8 / K8 chunks (int8 MFMA k-steps)
    constexpr bool kVector = kPiece >= 8;  // 16-byte pieces of fp16 rows, whole-vector stores
    __shared__ __attribute__((aligned(16))) unsigned char smem[L::kSmemBytes];
    __shared__ unsigned group_bits[kWavesPerGroup];
    // Landing area of the spare DMA slots (written with zeros, never read).
    __shared__ __attribute__((aligned(16))) unsigned char lds_spare[1024];
    // kInTurn: the merged O. Dynamic (kMergedBytes), as with a size that it knows
    // the compiler allocates registers for one workgroup per CU and keeps the
    // accumulators in AGPRs, copied to and fro: 273 us for the first call above.
    extern __shared__ float4v lds_merged[];
    unsigned char* const lds_k = smem;
    unsigned char* const lds_v = smem + L::kKBytes;
    unsigned char* const lds_k8 = smem + L::kKBytes + L::kVBytes;
    // LDS byte addresses of the tile buffers (M0 of the tile DMA), converted once.
    const unsigned lds_k_address = lds_address_of(smem);
    const unsigned lds_v_address = lds_k_address + L::kKBytes;
    const unsigned lds_k8_address = lds_v_address + L::kVBytes;

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15;
    const int q = lane & 31;  // the lane's query row within the wave (and its MFMA column)
    const int h = lane >> 5;  // which half of each 32-key / 16-feature block the lane holds

    int head32, qblock;
    int item = blockIdx.x, split = 0;
    if constexpr (kSplit) {
        item = blockIdx.x / p.splits;
        split = blockIdx.x - item * p.splits;
    }
    map_block(item, p.heads, p.q_blocks, p.causal != 0, head32, qblock);
    const std::int64_t head = head32;
    const int q0 = qblock * kRowsPerGroup;
    const int qw = q0 + wave * kRowsPerWave;
    const int M = p.M, N = p.N, d = p.d;
    const std::int64_t part = kSplit ? (head * p.splits + split) * M : 0;  // this split's first partial row
    if constexpr (kSplit && !kDots) {
        // A range that lies past the block's causal diagonal: no key, no O.
        if (p.causal && split * p.split_tiles * kTileKeys > q0 + kRowsPerGroup - 1) {
            if (tid < kRowsPerGroup && q0 + tid < M)
                *reinterpret_cast<float2v*>(p.part_ml + 2 * (part + q0 + tid)) = float2v{-INFINITY, kNoPart};
            return;
        }
    }

    const std::uint16_t* Kh = p.K + head * p.k_stride;
    const std::uint16_t* Vh = p.V + head * p.v_stride;
    const std::int8_t* K8h = p.K8 + head * static_cast<std::int64_t>(N) * d;
    unsigned char* const Oh = static_cast<unsigned char*>(p.O) + head * p.o_stride * (p.o_dtype == TILEMIX_DTYPE_F32 ? 4 : 2);

    // ---------------------------------------------------------------- Q
    half8 qf[kQC];
    int4v q8f[kQ8C];
    float q_scale = 0.0f;
    prepare_q<DC, kPiece>(p, head, qblock, qw + q, lane, group_bits, kWavesPerGroup, wave, 0, split == 0, qf, q8f, q_scale);

    // Key tiles are visited first to last, or last to first in a reversed
    // round (AttnParams::reverse_slots; the online softmax takes the tiles in
    // any order).
    const int step = (kRange == KeyRange::kWhole && reversed_round(blockIdx.x, p.reverse_slots)) ? -1 : 1;

    // ------------------------------------------------------ routing masks
    // One pass decodes four tiles: lane 16t + c decodes cell c (row c / 2,
    // key half c % 2) of tile jb + t from the route / skip word it keeps for
    // its query tile; the word is reloaded only when the tile's group moves
    // to another 64-group block. The two 64-bit ballots hold the four tiles'
    // wave-uniform masks, bit 16t + 2r + h <-> tile jb + t, cell (r, h). The
    // pass starts at the tile asked for (jb = j) when the walk goes forward,
    // and ends at it (jb = j - 3) when it goes backward; tiles before the
    // first read as skipped.
    const int qt0 = q0 / 16;
    const int my_qt = qt0 + ((lane & 15) >> 1);
    const bool my_row_valid = my_qt < p.q_tiles16;
    const std::int64_t my_word_base =
        head * p.words_per_head + static_cast<std::int64_t>(my_qt) * p.words_per_row;
    std::int64_t cached_block = -1;
    std::uint64_t cached_route = 0, cached_skip = 0;
    std::uint64_t batch_int8 = 0, batch_skip = 0;
    int batch_first = -4;
    auto tile_masks = [&](int j, std::uint32_t& int8_mask, std::uint32_t& skip_mask) {
        if (static_cast<unsigned>(j - batch_first) >= 4u) {
            batch_first = step < 0 ? j - 3 : j;
            const int kt = 2 * (batch_first + (lane >> 4)) + (lane & 1);
            bool skip = true, int8 = false;
            if (my_row_valid && kt >= 0 && kt < p.key_tiles32) {
                const unsigned group = p.group_shift >= 0 ? static_cast<unsigned>(kt) >> p.group_shift
                                                          : static_cast<unsigned>(kt) / static_cast<unsigned>(p.key_tiles_per_group);
                const std::int64_t block = group >> 6;
                if (block != cached_block) {
                    cached_block = block;
                    cached_route = p.route_words ? p.route_words[my_word_base + block] : 0ull;
                    cached_skip = p.skip_words ? p.skip_words[my_word_base + block] : 0ull;
                }
                const unsigned bit = static_cast<unsigned>(group & 63);
                skip = (cached_skip >> bit) & 1u;
                int8 = !skip && ((cached_route >> bit) & 1u);
            }
            batch_int8 = __ballot(int8);
            batch_skip = __ballot(skip);
        }
        const int shift = 16 * (j - batch_first);
        int8_mask = static_cast<std::uint32_t>(batch_int8 >> shift) & 0xffffu;
        skip_mask = static_cast<std::uint32_t>(batch_skip >> shift) & 0xffffu;
    };

    // ------------------------------------------------------ tile movement
    // Buffer ranges end after the last row's d elements; row strides apart.
    const std::int64_t k_bytes = (static_cast<std::int64_t>(N - 1) * p.k_row + d) * 2;
    const std::int64_t v_bytes = (static_cast<std::int64_t>(N - 1) * p.v_row + d) * 2;
    const int4v rsrc_k = make_rsrc(Kh, static_cast<int>(k_bytes));
    const int4v rsrc_v = make_rsrc(Vh, static_cast<int>(v_bytes));
    const int4v rsrc_k8 = make_rsrc(p.int8_operands ? K8h : p.K8,
                                    static_cast<int>(p.int8_operands ? static_cast<std::int64_t>(N) * d : 0));
    const int k_row_bytes = static_cast<int>(p.k_row * 2), v_row_bytes = static_cast<int>(p.v_row * 2);
    // Each wave issues the same number of DMAs per tile buffer, so the issue
    // code has no branches: slot t of a wave moves 1 KiB piece wave + 4t, and
    // a slot past the buffer's last piece reads out of range (zeros, no
    // memory traffic) into lds_spare.
    const unsigned lds_spare_address = lds_address_of(lds_spare);
    int off_k[L::kKPerWave], off_v[L::kVPerWave], off_k8[L::kK8PerWave];
    unsigned dst_k[L::kKPerWave], dst_v[L::kVPerWave], dst_k8[L::kK8PerWave];
    if constexpr (kPiece != 0) {
#pragma unroll
        for (int t = 0; t < L::kKPerWave; ++t) {
            const int w = wave + kWavesPerGroup * t;
            off_k[t] = w < L::kKLoads ? L::template kv_lane_offset<true>(w, lane, L::kKStride, 2 * d, k_row_bytes) : kOutOfRange;
            dst_k[t] = w < L::kKLoads ? lds_k_address + 1024 * w : lds_spare_address;
        }
#pragma unroll
        for (int t = 0; t < L::kVPerWave; ++t) {
            const int w = wave + kWavesPerGroup * t;
            off_v[t] = w < L::kVLoads ? L::template kv_lane_offset<false>(w, lane, L::kVStride, 2 * d, v_row_bytes) : kOutOfRange;
            dst_v[t] = w < L::kVLoads ? lds_v_address + 1024 * w : lds_spare_address;
        }
#pragma unroll
        for (int t = 0; t < L::kK8PerWave; ++t) {
            const int w = wave + kWavesPerGroup * t;
            off_k8[t] = w < L::kK8Loads ? L::k8_lane_offset(w, lane, d) : kOutOfRange;
            dst_k8[t] = w < L::kK8Loads ? lds_k8_address + 1024 * w : lds_spare_address;
        }
    }
    // Tile DMA of one buffer: every slot of this wave from resource r at
    // scalar offset soffset. A tile that runs past the last key (the head's
    // last tile when N % 64 != 0) is issued through a view starting at the
    // tile (rsrc_from), so that its rows past N fail the range check.
    auto k_slots = [&](int4v r, int soffset) {
        if constexpr (L::kKLoads % kWavesPerGroup == 0) {
            load_slots(r, dst_k[0], off_k, soffset);
        } else {
#pragma unroll
            for (int t = 0; t < L::kKPerWave; ++t) load_to_lds(r, dst_k[t], off_k[t], soffset);
        }
    };
    auto k8_slots = [&](int4v r, int soffset) {
        if constexpr (L::kK8Loads % kWavesPerGroup == 0) {
            load_slots(r, dst_k8[0], off_k8, soffset);
        } else {
#pragma unroll
            for (int t = 0; t < L::kK8PerWave; ++t) load_to_lds(r, dst_k8[t], off_k8[t], soffset);
        }
    };
    // V into buffer `buffer` (0 or 1); spare slots keep their landing area.
    auto v_slots = [&](int4v r, int soffset, int buffer) {
        const unsigned shift = buffer ? static_cast<unsigned>(L::kV1Offset) : 0u;
        if constexpr (L::kVLoads % kWavesPerGroup == 0) {
            load_slots(r, dst_v[0] + shift, off_v, soffset);
        } else {
#pragma unroll
            for (int t = 0; t < L::kVPerWave; ++t)
                load_to_lds(r, dst_v[t] == lds_spare_address ? dst_v[t] : dst_v[t] + shift, off_v[t], soffset);
        }
    };
    // A tile whose rows are not whole 16-byte pieces and of which a piece would
    // end past the head (that of the head's last row, and for K8 rows of four
    // bytes that of up to three rows before it): dwords through registers,
    // zeros past d and N. at(row, byte): the LDS position.
    auto load_tile_dwords = [&](unsigned char* tile, const unsigned char* head_rows, std::int64_t row_bytes, int k0,
                                int valid_bytes, int padded_bytes, auto&& at) {
        const int per_row = padded_bytes / 4;
        for (int e = tid; e < kTileKeys * per_row; e += kThreadsPerGroup) {
            const int row = e / per_row, byte = 4 * (e % per_row);
            *reinterpret_cast<std::uint32_t*>(tile + at(row, byte)) =
                (k0 + row < N && byte < valid_bytes)
                    ? *reinterpret_cast<const std::uint32_t*>(head_rows + (k0 + row) * row_bytes + byte)
                    : 0u;
        }
    };
    // K (FP16 cells) and K8 (INT8 cells) of tile j.
    auto issue_k = [&](int j, bool need16, bool need8) {
        const int k0 = j * kTileKeys;
        if constexpr (kPiece != 0) {
            const bool tail = k0 + kTileKeys > N;
            const bool last = k0 + kTileKeys >= N;  // holds the head's last row
            if (need16) {
                if (kPiece == 4 && last)
                    load_tile_dwords(lds_k, reinterpret_cast<const unsigned char*>(Kh), p.k_row * 2, k0, 2 * d, 2 * kDP,
                                     [](int row, int byte) { return L::k_at(row, byte); });
                else if (tail) k_slots(rsrc_from(rsrc_k, k0 * k_row_bytes), 0);
                else k_slots(rsrc_k, k0 * k_row_bytes);
            }
            if (need8) {
                if (kPiece != 16 && (last || (kPiece == 4 && k8_pieces_pass_end(k0, N, d))))
                    load_tile_dwords(lds_k8, reinterpret_cast<const unsigned char*>(K8h), d, k0, d, L::kDP8,
                                     [](int row, int byte) { return L::k8_at(row, byte); });
                else if (tail) k8_slots(rsrc_from(rsrc_k8, k0 * d), 0);
                else k8_slots(rsrc_k8, k0 * d);
            }
        } else {
            if (need16) {
                for (int e = tid; e < kTileKeys * kDP; e += kThreadsPerGroup) {
                    const int row = e / kDP, f = e % kDP, key = k0 + row;
                    *reinterpret_cast<std::uint16_t*>(lds_k + L::k_at(row, 2 * f)) =
                        (key < N && f < d) ? Kh[static_cast<std::int64_t>(key) * p.k_row + f] : 0;
                }
            }
            if (need8) {
                for (int e = tid; e < kTileKeys * L::kDP8; e += kThreadsPerGroup) {
                    const int row = e / L::kDP8, f = e % L::kDP8, key = k0 + row;
                    lds_k8[L::k8_at(row, f)] =
                        (key < N && f < d) ? static_cast<unsigned char>(K8h[static_cast<std::int64_t>(key) * d + f]) : 0;
                }
            }
        }
    };
    auto issue_v = [&](int j, int buffer) {
        const int k0 = j * kTileKeys;
        if constexpr (kPiece != 0) {
            if (kPiece == 4 && k0 + kTileKeys >= N)
                load_tile_dwords(lds_v + (buffer ? L::kV1Offset : 0), reinterpret_cast<const unsigned char*>(Vh),
                                 p.v_row * 2, k0, 2 * d, 2 * kDP, [](int row, int byte) { return L::v_at(row, byte); });
            else if (k0 + kTileKeys > N) v_slots(rsrc_from(rsrc_v, k0 * v_row_bytes), 0, buffer);
            else v_slots(rsrc_v, k0 * v_row_bytes, buffer);
        } else {
            unsigned char* const dst = lds_v + (buffer ? L::kV1Offset : 0);
            for (int e = tid; e < kTileKeys * kDP; e += kThreadsPerGroup) {
                const int row = e / kDP, f = e % kDP, key = k0 + row;
                *reinterpret_cast<std::uint16_t*>(dst + L::v_at(row, 2 * f)) =
                    (key < N && f < d) ? Vh[static_cast<std::int64_t>(key) * p.v_row + f] : 0;
            }
        }
    };
    // Own loads complete (vmcnt 0), then the workgroup barrier.
    auto tile_barrier = [&]() {
        __builtin_amdgcn_s_waitcnt(0x0f70);
        __syncthreads();
    };

    // Per-lane LDS offsets of the K fragment (feature chunk dc, key block 0)
    // and V^T fragment (feature block fb, key step 0) reads; key blocks and
    // steps add whole rows (multiples of 16, which keep the chunk rotation).
    // K / K8 fragments: lane (q, h) reads key q of the key block, 16 bytes
    // at feature chunk c. V^T fragments (ds_read_b64_tr_b16): the 16-lane
    // group (fh, h) = ((lane / 16) & 1, lane / 32) reads keys 4h .. 4h + 3
    // (then 8 + 4h ..) x features 16 fb + fh kDP / 2 .. + 15, lane i
    // receiving feature 16 fb + fh kDP / 2 + i (output row 16 fh + i).
    int k_lane[kQC], v_lane[kOB], k8_lane[kQ8C];
#pragma unroll
    for (int m = 0; m < kQ8C; ++m) k8_lane[m] = L::k8_at(q, 32 * m + 16 * h);
#pragma unroll
    for (int c = 0; c < kQC; ++c) k_lane[c] = L::k_at(q, 32 * c + 16 * h);
#pragma unroll
    for (int fb = 0; fb < kOB; ++fb)
        v_lane[fb] = L::v_at(4 * h + (i >> 2), 2 * (16 * fb + (kDP / 2) * ((lane >> 4) & 1) + 4 * (i & 3)));
    // ---------------------------------------------------------- key loop
    RowState<kOB> st;
#pragma unroll
    for (int fb = 0; fb < kOB; ++fb) st.o[fb] = float16v{};
    st.lsum = 0.0f;
    st.m = -INFINITY;
    // kInTurn: the merge of the ranges before the current one, which ends
    // before tile turn_end, and how many ranges have not been merged. Its O lies
    // in LDS, each thread's values its own.
    float merged_m = -INFINITY, merged_l = 0.0f;
    int turn_end = p.split_tiles, turns = p.splits;
    if constexpr (kInTurn)
        for (int x = 0; x < 4 * kOB; ++x) lds_merged[x * kThreadsPerGroup + tid] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
    auto end_turn = [&]() {
        float a = st.lsum, b = st.lsum;
        permlane32_swap(a, b);
        const PartWeights w = merge_part(merged_m, merged_l, st.m, a + b);
        float4v* const mine = lds_merged + tid;
#pragma unroll
        for (int fb = 0; fb < kOB; fb += kOB % 2 ? 1 : 2) {
            constexpr int kBatch = kOB % 2 ? 4 : 8;
            float4v sum[kBatch];
#pragma unroll
            for (int x = 0; x < kBatch; ++x) sum[x] = mine[(4 * fb + x) * kThreadsPerGroup];
            asm volatile("" ::: "memory");  // reads first: they wait once a batch
#pragma unroll
            for (int x = 0; x < kBatch; ++x) {
                const float16v& o = st.o[fb + x / 4];
                const int e = 4 * (x % 4);
                mine[(4 * fb + x) * kThreadsPerGroup] = merged(sum[x], float4v{o[e], o[e + 1], o[e + 2], o[e + 3]}, w);
            }
        }
#pragma unroll
        for (int fb = 0; fb < kOB; ++fb) st.o[fb] = float16v{};
        st.lsum = 0.0f;
        st.m = -INFINITY;
        turn_end += p.split_tiles;
        --turns;
    };
    const bool positive_scale = p.score_scale >= 0.0f;

    const int key_tiles64 = (N - 1) / kTileKeys + 1;
    int tiles = key_tiles64;
    if (p.causal) tiles = min(tiles, (q0 + kRowsPerGroup - 1) / kTileKeys + 1);
    // A split workgroup covers its own range of key tiles.
    const int tile_begin = kSplit ? split * p.split_tiles : 0;
    if constexpr (kSplit) tiles = max(tile_begin, min(tiles, tile_begin + p.split_tiles));
    const std::int64_t trace_base = head * static_cast<std::int64_t>(p.q_tiles16) * p.key_tiles32;
    auto write_trace = [&](int j, std::uint32_t int8_mask, std::uint32_t skip_mask) {
        if (wave == 0 && lane < 16) {
            const int qt = qt0 + (lane >> 1), kt = 2 * j + (lane & 1);
            if (qt < p.q_tiles16 && kt < p.key_tiles32)
                p.trace[trace_base + static_cast<std::int64_t>(qt) * p.key_tiles32 + kt] =
                    static_cast<std::uint8_t>(((skip_mask >> lane) & 1u) ? 2u : ((int8_mask >> lane) & 1u));
        }
    };
    auto needs16 = [](std::uint32_t int8_mask, std::uint32_t skip_mask) {
        return ((~int8_mask & ~skip_mask) & 0xffffu) != 0;
    };

    // The loop visits tiles tile_begin .. tiles - 1 in the order of `step`;
    // in_walk(j) says whether j is still inside that range. The walk starts
    // at one end (tiles >= tile_begin: N >= 1, and a split's range is
    // clamped) and moves by one tile, so it reaches tile_end exactly.
    const int tile_end = step > 0 ? tiles : tile_begin - 1;
    auto in_walk = [&](int j) { return j != tile_end; };
    // Tiles whose 16 cells are all skipped are stepped over: next_tile(j)
    // returns the first tile from j on (in the walk's order) with a visible
    // cell, or the first tile past the range, with that tile's masks,
    // writing the routing trace of the tiles it passes.
    std::uint32_t cur_int8 = 0, cur_skip = 0;
    auto next_tile = [&](int j) {
        for (; in_walk(j); j += step) {
            tile_masks(j, cur_int8, cur_skip);
            if (kDots && p.trace) write_trace(j, cur_int8, cur_skip);
            if (cur_skip != 0xffffu) break;
        }
        return j;
    };
    // Tile j's V sits in buffer v_buffer. The loads of the next visible tile
    // (K, K8, and V into the other buffer) are issued after the tile's second
    // barrier: by then every wave has finished its scores (the K and K8
    // buffers are free) and the previous tile's P.V (its V buffer is free).
    int j = next_tile(step > 0 ? tile_begin : tiles - 1);
    int v_buffer = 0;
    if (in_walk(j)) {
        issue_k(j, needs16(cur_int8, cur_skip), cur_int8 != 0);
        issue_v(j, v_buffer);
    }

    // One iteration per visible tile. A wave with no visible key in the tile
    // (rows above a causal diagonal, or all its cells skipped) takes part in
    // the tile's loads and barriers only: its probabilities would all be 0,
    // so the softmax and P.V would leave m, l and O unchanged.
    while (in_walk(j)) {
        if constexpr (kInTurn)
            while (j >= turn_end) end_turn();
        const int k0 = j * kTileKeys;
        const std::uint32_t int8_mask = cur_int8, skip_mask = cur_skip;
        tile_barrier();  // K_j, V_j landed; every wave finished P.V of the previous tile
        set_priority<2>();  // second half of the MFMA phase (P.V, then these scores)

        const unsigned wave_int8 = (int8_mask >> (4 * wave)) & 0xfu;
        const unsigned wave_skip = (skip_mask >> (4 * wave)) & 0xfu;
        const bool active = qw < M && wave_skip != 0xfu && !(p.causal && k0 > qw + kRowsPerWave - 1);
        // Tiles needing no element mask and a non-negative scale use the fast
        // path: raw MFMA results go straight into the exponent FMA.
        const bool masked = k0 + kTileKeys > N || (p.causal && k0 + kTileKeys - 1 > qw);
        const bool fast = positive_scale && !masked;

        float16v s[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int e = 0; e < 16; ++e) s[kb][e] = -INFINITY;
        float c = 1.0f;
        if (active) {
            float k_factor = 0.0f;  // q_scale * k_scale * score_scale * log2(e)
            if (wave_int8) {
                const float k_scale = half_bits_to_float(load_uniform_u16(p.k_scales + head * p.k_blocks + j));
                k_factor = ((q_scale * k_scale) * p.score_scale) * kLog2e;
            }
            // ---- scores S^T[kb]: lane (q, h) holds row q against keys 32 kb + 8 (e / 4) + 4 h + e % 4
            auto fp16_scores = [&]() {
                // Feature chunk outermost (two independent accumulator
                // chains), K fragments read two chunks ahead.
                s[0] = float16v{};
                s[1] = float16v{};
                half8 kf[3][2];
                auto load_c = [&](int cc, half8 (&dst)[2]) {
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb) {
                        dst[kb] = *reinterpret_cast<const half8*>(lds_k + 32 * L::kKStride * kb + k_lane[cc]);
                        if constexpr (kPiece == 4) {  // features past d belong to the next row
                            uint4v words = __builtin_bit_cast(uint4v, dst[kb]);
#pragma unroll
                            for (int w = 0; w < 4; ++w)
                                if (16 * cc + 8 * h + 2 * w >= d) words[w] = 0u;
                            dst[kb] = __builtin_bit_cast(half8, words);
                        }
                    }
                };
                load_c(0, kf[0]);
                load_c(1, kf[1]);
#pragma unroll
                for (int cc = 0; cc < kQC; ++cc) {
                    if (cc + 2 < kQC) load_c(cc + 2, kf[(cc + 2) % 3]);
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb)
                        s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[cc % 3][kb], qf[cc], s[kb], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            // Exact int32 dots of both key blocks.
            auto int8_scores = [&](int16v (&acc)[2]) {
                acc[0] = int16v{};
                acc[1] = int16v{};
                int4v kf8[2][2];
                auto load_m = [&](int m, int4v (&dst)[2]) {
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb)
                        dst[kb] = *reinterpret_cast<const int4v*>(lds_k8 + 32 * L::kK8Stride * kb + k8_lane[m]);
                };
                load_m(0, kf8[0]);
#pragma unroll
                for (int m = 0; m < kQ8C; ++m) {
                    if (m + 1 < kQ8C) load_m(m + 1, kf8[(m + 1) & 1]);
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb)
                        acc[kb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf8[m & 1][kb], q8f[m], acc[kb], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            // Raw int32 dots of key block kb (verification output).
            auto store_dots = [&](int kb, const int16v& acc) {
                const int query = qw + q;
                std::int32_t* row = p.dots + head * static_cast<std::int64_t>(M) * N +
                                    static_cast<std::int64_t>(query) * N;
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const int key = k0 + 32 * kb + 8 * (e >> 2) + 4 * h + (e & 3);
                    if (query < M && key < N && !(p.causal && key > query)) row[key] = acc[e];
                }
            };
            const int qh = q >> 4;  // the lane's 16-row routing cell of the wave
            if (wave_skip == 0 && wave_int8 == 0) {
                fp16_scores();
                c = p.score_log2;
            } else if (wave_skip == 0 && wave_int8 == 0xfu) {
                int16v acc[2];
                int8_scores(acc);
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    if (kDots && p.dots) store_dots(kb, acc[kb]);
#pragma unroll
                    for (int e = 0; e < 16; ++e) s[kb][e] = static_cast<float>(acc[kb][e]);
                }
                c = k_factor;
            } else {
                // Mixed routes inside the wave: both score kinds where present,
                // explicitly scaled, then selected per lane (cell bit 2 qh + kb).
                const unsigned wave_fp16 = ~(wave_int8 | wave_skip) & 0xfu;
                if (wave_fp16) {
                    fp16_scores();
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb) s[kb] *= p.score_log2;
                } else {
                    s[0] = float16v{};
                    s[1] = float16v{};
                }
                if (wave_int8) {
                    int16v acc[2];
                    int8_scores(acc);
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb) {
                        const bool cell_int8 = (wave_int8 >> (2 * qh + kb)) & 1u;
                        if (kDots && p.dots && cell_int8) store_dots(kb, acc[kb]);
#pragma unroll
                        for (int e = 0; e < 16; ++e)
                            s[kb][e] = cell_int8 ? static_cast<float>(acc[kb][e]) * k_factor : s[kb][e];
                    }
                }
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
                    if ((wave_skip >> (2 * qh + kb)) & 1u)
#pragma unroll
                        for (int e = 0; e < 16; ++e) s[kb][e] = -INFINITY;
                c = 1.0f;
            }
            if (!fast && c != 1.0f) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) s[kb] *= c;
                c = 1.0f;
            }
            // ---- element masks: key tail and causal diagonal (explicit scores)
            if (masked) {
                const int query = qw + q;
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        const int key = k0 + 32 * kb + 8 * (e >> 2) + 4 * h + (e & 3);
                        if (key >= N || (p.causal && key > query)) s[kb][e] = -INFINITY;
                    }
            }
        }


        tile_barrier();  // every wave finished reading K_j (and P.V of the previous tile)
        set_priority<0>();  // first half of the VALU phase
        const int j_next = next_tile(j + step);
        if (in_walk(j_next)) {
            issue_k(j_next, needs16(cur_int8, cur_skip), cur_int8 != 0);
            issue_v(j_next, v_buffer ^ 1);
        }

        // ---- online softmax, then O^T += V^T P^T
        if (active) {
            half8 ph[4], pl[4];
            softmax_tile<kOB, kPrecise>(st, s, c, ph, pl);
            {
                // V^T fragment of step t = (key step t / kOB, feature block
                // t % kOB), read kAhead steps before its MFMA.
                auto v_frag = [&](int t) {
                    const unsigned char* v_lo = lds_v + (v_buffer ? L::kV1Offset : 0) + 16 * L::kVStride * (t / kOB) + v_lane[t % kOB];
                    return concat(read_tr16(v_lo), read_tr16(v_lo + 8 * L::kVStride));
                };
                constexpr int kSteps = 4 * kOB;
                constexpr int kAhead = 3;
                set_priority<0>();  // first half of the MFMA phase
                half8 vf[kAhead + 1];
#pragma unroll
                for (int t = 0; t < kAhead; ++t)
                    if (t < kSteps) vf[t] = v_frag(t);
#pragma unroll
                for (int t = 0; t < kSteps; ++t) {
                    if (t + kAhead < kSteps) vf[(t + kAhead) % (kAhead + 1)] = v_frag(t + kAhead);
                    const int ks = t / kOB, fb = t % kOB;
                    st.o[fb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[t % (kAhead + 1)], ph[ks], st.o[fb], 0, 0, 0);
                    if constexpr (kPrecise)
                        st.o[fb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[t % (kAhead + 1)], pl[ks], st.o[fb], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        j = j_next;
        v_buffer ^= 1;
    }

    if constexpr (kInTurn) {
        // Ranges without a visible tile too: each is a part of the merge.
        while (turns > 0) end_turn();
#pragma unroll
        for (int x = 0; x < 4 * kOB; ++x) {
            const float4v value = lds_merged[x * kThreadsPerGroup + tid];
#pragma unroll
            for (int e = 0; e < 4; ++e) st.o[x / 4][4 * (x % 4) + e] = value[e];
        }
    }

    // Routing trace of tiles a causal workgroup never visits (of its range, the
    // last one's to the end).
    if (kDots && p.trace && p.causal) {
        const int range_end = kSplit && split + 1 < p.splits ? min(key_tiles64, tile_begin + p.split_tiles) : key_tiles64;
        for (int j = tiles; j < range_end; ++j) {
            std::uint32_t int8_mask = 0, skip_mask = 0;
            tile_masks(j, int8_mask, skip_mask);
            write_trace(j, int8_mask, skip_mask);
        }
    }

    // Staged stores (store_staged): the regions are the K tile buffer (both 4
    // KiB regions of it at d = 64, all four at d = 128) and at d = 64 the V
    // buffer the last tile did not use: every wave has passed the last tile's
    // second barrier, so no wave reads them any more and no load targets them.
    constexpr bool kStaged = kPiece == 16 && !kDots && (kDP == 128 || kDP == 64);
    unsigned char* stage = lds_k + wave * kStageBytes;
    if constexpr (kStaged && kDP == 64) {
        static_assert(L::kKBytes >= 2 * kStageBytes && L::kVBytes >= 2 * kStageBytes, "stage regions fit K and V");
        if (wave >= 2) stage = lds_v + (v_buffer ? L::kV1Offset : 0) + (wave - 2) * kStageBytes;
    } else if constexpr (kStaged) {
        static_assert(L::kKBytes >= kWavesPerGroup * kStageBytes, "stage regions fit the K buffer");
    }
    // ---------------------------------------------------------- epilogue
    if constexpr (kSplit) {
        // This split's unnormalised rows and their (m, l), for the combine.
        float a = st.lsum, b = st.lsum;
        permlane32_swap(a, b);
        const int row = qw + q;
        if constexpr (kStaged) {
            if (d == kDP) {
                store_staged<kOB>(st, stage, p.part_o + part * d, d, 1.0f, qw, M);
                if (row < M && h == 0) {
                    float* const ml = p.part_ml + 2 * (part + row);
                    ml[0] = st.m;
                    ml[1] = a + b;
                }
                return;
            }
        }
        if (row < M) {
            unsigned char* const part_rows = reinterpret_cast<unsigned char*>(p.part_o + part * d);
            const std::int64_t row_offset = static_cast<std::int64_t>(row) * d;
#pragma unroll
            for (int fb = 0; fb < kOB; ++fb)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    const int feature = (r4 < 2 ? 0 : kDP / 2 - 16) + 16 * fb + 8 * r4 + 4 * h;
                    const float4v value{st.o[fb][4 * r4], st.o[fb][4 * r4 + 1], st.o[fb][4 * r4 + 2], st.o[fb][4 * r4 + 3]};
                    store_output(part_rows, TILEMIX_DTYPE_F32, row_offset + feature, value, d - feature, kPiece != 0);
                }
            if (h == 0) {
                float* const ml = p.part_ml + 2 * (part + row);
                ml[0] = st.m;
                ml[1] = a + b;
            }
        }
    } else {
        float a = st.lsum, b = st.lsum;
        permlane32_swap(a, b);  // the row's other half, held by lane ^ 32
        const float l = kInTurn ? merged_l : a + b;
        const float inverse = l > 0.0f ? 1.0f / l : 0.0f;
        const int row = qw + q;
        if constexpr (kStaged) {
            if (p.o_dtype == TILEMIX_DTYPE_F32 && d == kDP) {
                store_staged<kOB>(st, stage, reinterpret_cast<float*>(Oh), p.o_row, inverse, qw, M);
                return;
            }
        }
        if (row < M) {
            const std::int64_t row_offset = static_cast<std::int64_t>(row) * p.o_row;
#pragma unroll
            for (int fb = 0; fb < kOB; ++fb)
#pragma unroll
                for (int r4 = 0; r4 < 4; ++r4) {
                    // Output row R = 8 r4 + 4 h (+ 0..3) of block fb is feature
                    // 16 fb + R (R < 16) or kDP / 2 + 16 fb + R - 16.
                    const int feature = (r4 < 2 ? 0 : kDP / 2 - 16) + 16 * fb + 8 * r4 + 4 * h;
                    const float4v value{st.o[fb][4 * r4], st.o[fb][4 * r4 + 1], st.o[fb][4 * r4 + 2], st.o[fb][4 * r4 + 3]};
                    store_output(Oh, p.o_dtype, row_offset + feature, value * inverse, d - feature, kVector || p.o_vector);
                }
        }
    }
}

// ------------------------------------------------------------- wide kernel
//
// The same rows, arithmetic and tile order as attention_kernel, for launches
// with enough row blocks: one workgroup of eight waves per CU owns 256 query
// rows (two Q quantization blocks), so each K / K8 / V tile is loaded into LDS
// once for 256 rows instead of 128, and its two halves (waves 0-3 and 4-7, one
// wave of each on every SIMD) run half a tile apart. A tile is two slots
// between barriers of the whole workgroup:
//   matrix slot  P.V of the previous tile, then this tile's scores;
//   vector slot  routes, masks and softmax of this tile.
// The second half enters one barrier later, so in every slot one wave of each
// SIMD has the matrix core while the other runs exponentials. Tile buffers are
// all double: K (i + 1) and V (i) of walk position i are fetched from the slot
// in which the first half starts position i (the slot before, the second half
// finished the tiles that were there) and waited for two slots later:
//   slot         2i              2i + 1
//   first half   P.V i-1, QK i   softmax i
//   second half  softmax i-1     P.V i-1, QK i
//   loads        issue K i+1, V i; all waves wait for them at the end of 2i+1
// Everything a wave has to know of a tile is decided once, before the walk:
// the visited tiles of the workgroup, in walking order, with the wave's cells
// as one word each (Entry). Tile offsets go into the lanes' offsets, which the
// buffer range check covers, so a tail tile is loaded like any other, and the
// walk is unrolled twice so that buffers are constants: a tile's scalar work is
// a few instructions. (With the routes decoded in the walk, tail tiles through
// views of their own and buffers in variables, the slots' control alone took
// half of the kernel's time.)
// What bounds it, at 128 features, dense (32 heads x 8192: 1033 us, 1.06
// PFLOP/s; 1064 us with attention_kernel): about 1800 cycles a slot at 1.79 GHz
// under the power limit. Counted (GRBM_GUI_ACTIVE over the slots of a CU's
// rounds): 1690 cycles a slot for 32 heads x 16384 with three quarters INT8, MFMA
// busy 49 % of SIMD cycles; 1710 and 36 % for 32 x 8192 three-way; at 64 features
// 1850, prologue and epilogue included, and 24 % (64 x 2048). The matrix slot
// alone takes 1540 (1024 of them MFMAs; the LDS reads of V's transposed
// fragments, at half the rate of K's, take longer than the P.V MFMAs they feed),
// the vector slot alone 1500 (32 exponentials at 16 cycles, 110 other
// instructions): from copies of the kernel with the other slot's work left out.
// A slot ends in a barrier of all eight waves, so it takes as long as its slowest
// wave: what a wave saves on an INT8 or skipped cell is lost there unless all
// save it. Interleaving P.V with the
// scores MFMA by MFMA spilled 160 registers at 128 features and was 3 % slower
// at 64; three tile buffers of each were no faster.
constexpr int kWideThreads = 512;
#define TILEMIX_INLINE __attribute__((always_inline))  // lambdas the walk uses twice
constexpr int kWideWaves = kWideThreads / kWave;
constexpr int kWideRows = 256;

// A wave's view of one visited tile: cell bits (2 r + key half) in INT8 and
// SKIP, what any wave of the workgroup needs of it, how this wave scores it.
struct Entry {
    static constexpr unsigned kInt8 = 0xfu, kSkipShift = 4;
    static constexpr unsigned kNeeds16 = 1u << 8, kNeeds8 = 1u << 9, kVisited = 1u << 10;
    static constexpr unsigned kModeShift = 11;  // 2 bits
    static constexpr unsigned kFp16 = 0, kAllInt8 = 1, kMixed = 2, kIdle = 3;
    static constexpr unsigned kMasked = 1u << 13;  // holds keys that some row of the wave does not see
    static constexpr unsigned kTileShift = 16;
    static constexpr unsigned kEnd = kIdle << kModeShift;
};

template <int DC>
__global__ __launch_bounds__(kWideThreads, 1) void attention_wide_kernel(const AttnParams p) {
    using L = Layout<DC>;
    constexpr int kDP = L::kDP;
    constexpr int kOB = DC;
    constexpr int kQC = kDP / 16;
    constexpr int kQ8C = L::kDP8 / 32;
    static_assert(L::kRotate && L::kRotate8, "wide kernel: rotated rows");
    // K0 K1 | K8_0 K8_1 | V0 V1
    constexpr int kK8Base = 2 * L::kKBytes, kVBase = kK8Base + 2 * L::kK8Bytes;
    __shared__ __attribute__((aligned(16))) unsigned char smem[kVBase + 2 * L::kVBytes];
    __shared__ unsigned group_bits[kWideWaves];
    __shared__ unsigned entries[kWideWaves][kWideMaxTiles];

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool second = wave >= kWideWaves / 2;
    const int i = lane & 15;
    const int q = lane & 31;
    const int h = lane >> 5;
    const int blocks = (p.q_blocks + 1) / 2;
    int head32, block;
    map_block(blockIdx.x, p.heads, blocks, p.causal != 0, head32, block);
    const std::int64_t head = head32;
    const int q0 = block * kWideRows;
    const int qw = q0 + wave * kRowsPerWave;
    const int M = p.M, N = p.N, d = p.d;

    // ------------------------------------------------------ route table
    int tiles = (N - 1) / kTileKeys + 1;
    if (p.causal) tiles = min(tiles, (q0 + kWideRows - 1) / kTileKeys + 1);
    const bool reversed = reversed_round(blockIdx.x, p.reverse_slots);
    {
        const int qt = qw / 16;
        const std::int64_t words = head * p.words_per_head + static_cast<std::int64_t>(qt) * p.words_per_row;
        for (int x = lane; x < tiles; x += kWave) {
            const int tile = reversed ? tiles - 1 - x : x;
            unsigned int8 = 0, skip = 0;
#pragma unroll
            for (int cell = 0; cell < 4; ++cell) {
                const int r = cell >> 1, kt = 2 * tile + (cell & 1);
                bool is_skip = qt + r >= p.q_tiles16 || kt >= p.key_tiles32, is_int8 = false;
                if (!is_skip && (p.route_words || p.skip_words)) {
                    const unsigned group = p.group_shift >= 0 ? static_cast<unsigned>(kt) >> p.group_shift
                                                              : static_cast<unsigned>(kt) / static_cast<unsigned>(p.key_tiles_per_group);
                    const std::int64_t word = words + r * p.words_per_row + (group >> 6);
                    const unsigned bit = group & 63u;
                    is_skip = p.skip_words && ((p.skip_words[word] >> bit) & 1u);
                    is_int8 = !is_skip && p.route_words && ((p.route_words[word] >> bit) & 1u);
                }
                int8 |= static_cast<unsigned>(is_int8) << cell;
                skip |= static_cast<unsigned>(is_skip) << cell;
            }
            // No row of the wave, or none that sees a key of the tile.
            const int k0 = tile * kTileKeys;
            if (qw >= M || (p.causal && k0 > qw + kRowsPerWave - 1)) {
                int8 = 0;
                skip = 0xfu;
            }
            const bool masked = k0 + kTileKeys > N || (p.causal && k0 + kTileKeys - 1 > qw);
            const unsigned mode = skip == 0xfu ? Entry::kIdle
                                  : skip != 0  ? Entry::kMixed
                                  : int8 == 0  ? Entry::kFp16
                                               : (int8 == 0xfu ? Entry::kAllInt8 : Entry::kMixed);
            entries[wave][x] = int8 | (skip << Entry::kSkipShift) | (mode << Entry::kModeShift) |
                               (masked ? Entry::kMasked : 0u) | (static_cast<unsigned>(tile) << Entry::kTileShift);
        }
    }

    half8 qf[kQC];
    int4v q8f[kQ8C];
    float q_scale = 0.0f;
    const int qblock = min(2 * block + (second ? 1 : 0), p.q_blocks - 1);
    prepare_q<DC, 16>(p, head, qblock, qw + q, lane, group_bits, kWideWaves, wave, second ? kWideWaves / 2 : 0,
                      2 * block + (second ? 1 : 0) < p.q_blocks, qf, q8f, q_scale);

    // What any wave needs of a tile, and the visited tiles moved to the front
    // (in place: a wave's entry moves to its own or an earlier place; what the
    // other waves' words say is read before any word moves).
    int count = 0;
    for (int first = 0; first < tiles; first += kWave) {
        __syncthreads();
        const int x = first + lane;
        unsigned mine = Entry::kEnd, needs = 0;
        if (x < tiles) {
            mine = entries[wave][x];
#pragma unroll
            for (int w = 0; w < kWideWaves; ++w) {
                const unsigned word = entries[w][x], int8 = word & Entry::kInt8, skip = (word >> Entry::kSkipShift) & 0xfu;
                needs |= (skip != 0xfu ? Entry::kVisited : 0u) | (((~int8 & ~skip) & 0xfu) ? Entry::kNeeds16 : 0u) |
                         (int8 ? Entry::kNeeds8 : 0u);
            }
        }
        const std::uint64_t visited = __ballot(needs != 0);
        __syncthreads();
        if (needs)
            entries[wave][count + __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(visited >> 32),
                                                            __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(visited), 0u))] =
                mine | needs;
        count += __popcll(visited);
    }
    // Lane l of the window holds the entry at position window + l (kEnd past
    // the last) and its K block's scale.
    int window = 0;
    unsigned window_entry;
    float window_scale = 0.0f;
    auto load_window = [&]() TILEMIX_INLINE {
        const int at = window + lane;
        window_entry = at < count ? entries[wave][at] : Entry::kEnd;
        if (p.int8_operands && at < count)
            window_scale = half_bits_to_float(p.k_scales[head * p.k_blocks + (window_entry >> Entry::kTileShift)]);
    };
    struct Position {
        unsigned entry;
        float k_scale;
    };
    auto position = [&](int x) TILEMIX_INLINE {
        if (x - window >= kWave) {
            window += kWave;
            load_window();
        }
        return Position{static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(window_entry), x - window)),
                        __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, window_scale), x - window))};
    };

    // ------------------------------------------------------ tile movement
    const int4v rsrc_k = make_rsrc(p.K + head * p.k_stride, static_cast<int>((static_cast<std::int64_t>(N - 1) * p.k_row + d) * 2));
    const int4v rsrc_v = make_rsrc(p.V + head * p.v_stride, static_cast<int>((static_cast<std::int64_t>(N - 1) * p.v_row + d) * 2));
    const int4v rsrc_k8 = make_rsrc(p.K8 + (p.int8_operands ? head * static_cast<std::int64_t>(N) * d : 0),
                                    static_cast<int>(p.int8_operands ? static_cast<std::int64_t>(N) * d : 0));
    const int k_tile_bytes = static_cast<int>(p.k_row * 2 * kTileKeys), v_tile_bytes = static_cast<int>(p.v_row * 2 * kTileKeys);
    const int k8_tile_bytes = d * kTileKeys;
    constexpr int kKSlots = L::kKLoads / kWideWaves, kVSlots = L::kVLoads / kWideWaves;
    static_assert(L::kKLoads % kWideWaves == 0 && L::kVLoads % kWideWaves == 0 && L::kK8Loads <= kWideWaves,
                  "K and V split evenly over the waves, K8 is one piece at most");
    int off_k[kKSlots], off_v[kVSlots];
#pragma unroll
    for (int t = 0; t < kKSlots; ++t)
        off_k[t] = L::template kv_lane_offset<true>(wave + kWideWaves * t, lane, L::kKStride, 2 * d, static_cast<int>(p.k_row * 2));
#pragma unroll
    for (int t = 0; t < kVSlots; ++t)
        off_v[t] = L::template kv_lane_offset<false>(wave + kWideWaves * t, lane, L::kVStride, 2 * d, static_cast<int>(p.v_row * 2));
    const bool k8_mover = wave < L::kK8Loads;
    const int off_k8 = k8_mover ? L::k8_lane_offset(wave, lane, d) : kOutOfRange;
    // This wave's first piece of a tile, from the start of a buffer.
    const unsigned lds_wave = lds_address_of(smem) + 1024 * wave;
    auto issue_k = [&](unsigned entry, auto buffer) TILEMIX_INLINE {
        constexpr int b = decltype(buffer)::value;
        const int tile = static_cast<int>(entry >> Entry::kTileShift);
        if (entry & Entry::kNeeds16) load_slots_at<b * L::kKBytes, 0, kKSlots>(rsrc_k, lds_wave, off_k, tile * k_tile_bytes);
        if ((entry & Entry::kNeeds8) && k8_mover)
            load_to_lds_at<kK8Base + b * L::kK8Bytes>(rsrc_k8, lds_wave, off_k8 + tile * k8_tile_bytes, 0);
    };
    auto issue_v = [&](unsigned entry, auto buffer) TILEMIX_INLINE {
        constexpr int b = decltype(buffer)::value;
        if (entry & Entry::kVisited)
            load_slots_at<kVBase + b * L::kVBytes, 0, kVSlots>(rsrc_v, lds_wave, off_v,
                                                                static_cast<int>(entry >> Entry::kTileShift) * v_tile_bytes);
    };

    int k_lane[kQC], v_lane[kOB], k8_lane[kQ8C];
#pragma unroll
    for (int m = 0; m < kQ8C; ++m) k8_lane[m] = kK8Base + L::k8_at(q, 32 * m + 16 * h);
#pragma unroll
    for (int c = 0; c < kQC; ++c) k_lane[c] = L::k_at(q, 32 * c + 16 * h);
#pragma unroll
    for (int fb = 0; fb < kOB; ++fb)
        v_lane[fb] = kVBase + L::v_at(4 * h + (i >> 2), 2 * (16 * fb + (kDP / 2) * ((lane >> 4) & 1) + 4 * (i & 3)));

    RowState<kOB> st;
#pragma unroll
    for (int fb = 0; fb < kOB; ++fb) st.o[fb] = float16v{};
    st.lsum = 0.0f;
    st.m = -INFINITY;
    const unsigned explicit_scores = p.score_scale >= 0.0f ? 0u : 1u;
    float16v s[2];      // scores, or (INT8 tiles) the bits of their int32 dots, matrix slot -> vector slot
    half8 ph[4], unused[4];  // probabilities, vector slot -> next matrix slot
    bool pv_pending = false;

    // Exact int32 dots / fp16 scores of both key blocks.
    auto fp16_scores = [&](auto buffer, float16v (&x)[2]) TILEMIX_INLINE {
        constexpr int kAt = decltype(buffer)::value * L::kKBytes;
        x[0] = float16v{};
        x[1] = float16v{};
        half8 kf[3][2];
        auto load_c = [&](int cc, half8 (&dst)[2]) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
                dst[kb] = *reinterpret_cast<const half8*>(smem + kAt + 32 * L::kKStride * kb + k_lane[cc]);
        };
        load_c(0, kf[0]);
        load_c(1, kf[1]);
#pragma unroll
        for (int cc = 0; cc < kQC; ++cc) {
            if (cc + 2 < kQC) load_c(cc + 2, kf[(cc + 2) % 3]);
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
                x[kb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[cc % 3][kb], qf[cc], x[kb], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto int8_scores = [&](auto buffer, int16v (&acc)[2]) TILEMIX_INLINE {
        constexpr int kAt = decltype(buffer)::value * L::kK8Bytes;
        acc[0] = int16v{};
        acc[1] = int16v{};
        int4v kf8[2][2];
        auto load_m = [&](int m, int4v (&dst)[2]) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
                dst[kb] = *reinterpret_cast<const int4v*>(smem + kAt + 32 * L::kK8Stride * kb + k8_lane[m]);
        };
        load_m(0, kf8[0]);
#pragma unroll
        for (int m = 0; m < kQ8C; ++m) {
            if (m + 1 < kQ8C) load_m(m + 1, kf8[(m + 1) & 1]);
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
                acc[kb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf8[m & 1][kb], q8f[m], acc[kb], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto k_factor_of = [&](const Position& at) TILEMIX_INLINE { return ((q_scale * at.k_scale) * p.score_scale) * kLog2e; };

    // ------------------------------------------------------- matrix slot
    // P.V of the tile before, then the scores of position `at`; the read
    // offsets flip to the other buffers with each.
    auto probabilities_times_values = [&](auto buffer) TILEMIX_INLINE {
        constexpr int kAt = decltype(buffer)::value * L::kVBytes;
        if (!pv_pending) return;
        auto v_frag = [&](int t) TILEMIX_INLINE {
            const unsigned char* v_lo = smem + kAt + 16 * L::kVStride * (t / kOB) + v_lane[t % kOB];
            return concat(read_tr16(v_lo), read_tr16(v_lo + 8 * L::kVStride));
        };
        constexpr int kSteps = 4 * kOB;
        constexpr int kAhead = 3;
        half8 vf[kAhead + 1];
#pragma unroll
        for (int t = 0; t < kAhead; ++t)
            if (t < kSteps) vf[t] = v_frag(t);
#pragma unroll
        for (int t = 0; t < kSteps; ++t) {
            if (t + kAhead < kSteps) vf[(t + kAhead) % (kAhead + 1)] = v_frag(t + kAhead);
            const int ks = t / kOB, fb = t % kOB;
            st.o[fb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[t % (kAhead + 1)], ph[ks], st.o[fb], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto scores = [&](const Position& at, auto buffer) TILEMIX_INLINE {
        // The scores of the position before end here, on every path: on that of
        // an idle wave they would otherwise stay in registers through P.V.
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) asm volatile("" : "=v"(s[kb]));
        const unsigned mode = (at.entry >> Entry::kModeShift) & 3u;
        if (mode == Entry::kFp16) {
            fp16_scores(buffer, s);
        } else if (mode == Entry::kAllInt8) {
            int16v acc[2];
            int8_scores(buffer, acc);
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) s[kb] = __builtin_bit_cast(float16v, acc[kb]);
        } else if (mode == Entry::kMixed) {
            const unsigned int8 = at.entry & Entry::kInt8, skip = (at.entry >> Entry::kSkipShift) & 0xfu;
            // Both kinds where present, explicitly scaled, then
            // selected per lane (cell bit 2 (q / 16) + kb).
            const int qh = q >> 4;
            if (~(int8 | skip) & 0xfu) {
                fp16_scores(buffer, s);
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) s[kb] *= p.score_log2;
            } else {
                s[0] = float16v{};
                s[1] = float16v{};
            }
            if (int8) {
                const float k_factor = k_factor_of(at);
                int16v acc[2];
                int8_scores(buffer, acc);
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
                    const bool cell_int8 = (int8 >> (2 * qh + kb)) & 1u;
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        s[kb][e] = cell_int8 ? static_cast<float>(acc[kb][e]) * k_factor : s[kb][e];
                }
            }
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
                if ((skip >> (2 * qh + kb)) & 1u)
#pragma unroll
                    for (int e = 0; e < 16; ++e) s[kb][e] = -INFINITY;
        }
    };

    // ------------------------------------------------------- vector slot
    auto softmax = [&](const Position& at) TILEMIX_INLINE {
        const unsigned mode = (at.entry >> Entry::kModeShift) & 3u;
        pv_pending = mode != Entry::kIdle;
        // Likewise the probabilities.
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) asm volatile("" : "=v"(ph[ks]));
        if (!pv_pending) return;
        float c = p.score_log2;
        if (mode == Entry::kAllInt8) {
            c = k_factor_of(at);
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const int16v acc = __builtin_bit_cast(int16v, s[kb]);
#pragma unroll
                for (int e = 0; e < 16; ++e) s[kb][e] = static_cast<float>(acc[e]);
            }
        } else if (mode == Entry::kMixed) {
            c = 1.0f;
        }
        const unsigned masked = at.entry & Entry::kMasked;
        if (masked | explicit_scores) {
            if (c != 1.0f) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) s[kb] *= c;
                c = 1.0f;
            }
            if (masked) {
                // The last key this lane's row sees, counted from the tile's
                // first key of the lane.
                const int k0 = static_cast<int>(at.entry >> Entry::kTileShift) * kTileKeys;
                int seen = (p.causal ? min(N - 1, qw + q) : N - 1) - k0 - 4 * h;
                asm volatile("" : "+v"(seen));
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        if (32 * kb + 8 * (e >> 2) + (e & 3) > seen) s[kb][e] = -INFINITY;
            }
        }
        softmax_tile<kOB, false, false>(st, s, c, ph, unused);
    };
    // Slot ends: LDS reads done, then the workgroup barrier; with `loads` also
    // this wave's tile loads.
    auto slot_end = [&](bool loads) TILEMIX_INLINE {
        __builtin_amdgcn_sched_barrier(0);
        if (loads) wait_vmcnt<0>();
        lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };

    // ----------------------------------------------------------- the walk
    __syncthreads();
    load_window();
    using Zero = std::integral_constant<int, 0>;
    using One = std::integral_constant<int, 1>;
    Position now = position(0), next = position(1);
    issue_k(now.entry, Zero{});
    slot_end(true);
    if (second) {
        // Slot 0: the loads of the first half's slot 0, then its barrier.
        issue_k(next.entry, One{});
        issue_v(now.entry, Zero{});
        slot_end(false);
    }
    // Every wave walks `count` positions and passes 2 count + 1 slot ends here;
    // position x has its tiles in buffers x mod 2.
    int x = 0;
    auto walk_position = [&](auto own, auto other) TILEMIX_INLINE {
        if (!second) {
            issue_k(next.entry, other);
            issue_v(now.entry, own);
        }
        set_priority<1>();
        probabilities_times_values(other);
        scores(now, own);
        set_priority<0>();
        const Position after = position(x + 2);
        slot_end(second);
        if (second) {
            issue_k(after.entry, own);
            issue_v(next.entry, other);
        }
        softmax(now);
        slot_end(!second);
        now = next;
        next = after;
        ++x;
    };
    // Two positions a turn; an odd last one is followed by an idle one.
    while (x < count) {
        walk_position(Zero{}, One{});
        walk_position(One{}, Zero{});
    }
    probabilities_times_values(One{});
    if (!second) slot_end(false);

    // ---------------------------------------------------------- epilogue
    // What only the epilogue needs of the parameters is read again here (the
    // kernel's first argument), so that it holds no registers during the walk.
    const auto* late = (const __attribute__((address_space(4))) AttnParams*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(late));
    const int dtype = late->o_dtype;
    const std::int64_t o_row = late->o_row;
    float a = st.lsum, b = st.lsum;
    permlane32_swap(a, b);
    const float l = a + b;
    const float inverse = l > 0.0f ? 1.0f / l : 0.0f;
    const int row = qw + q;
    unsigned char* const Oh = static_cast<unsigned char*>(late->O) + head * late->o_stride * (dtype == TILEMIX_DTYPE_F32 ? 4 : 2);
    if (dtype == TILEMIX_DTYPE_F32 && d == kDP) {
        // Stage regions: nobody reads K or K8 any more; at 64 features the
        // second half also takes the V buffer that the last tile did not use.
        unsigned char* stage = smem + wave * kStageBytes;
        if constexpr (2 * L::kKBytes < kWideWaves * kStageBytes) {
            static_assert(2 * L::kKBytes >= 4 * kStageBytes && 2 * L::kK8Bytes >= 2 * kStageBytes &&
                              L::kVBytes >= 2 * kStageBytes, "stage regions fit K, K8 and V");
            if (wave >= 6) stage = smem + kVBase + (wave - 6) * kStageBytes;
        }
        store_staged<kOB>(st, stage, reinterpret_cast<float*>(Oh), o_row, inverse, qw, M);
        return;
    }
    if (row < M) {
        const std::int64_t row_offset = static_cast<std::int64_t>(row) * o_row;
#pragma unroll
        for (int fb = 0; fb < kOB; ++fb)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                const int feature = (r4 < 2 ? 0 : kDP / 2 - 16) + 16 * fb + 8 * r4 + 4 * h;
                const float4v value{st.o[fb][4 * r4], st.o[fb][4 * r4 + 1], st.o[fb][4 * r4 + 2], st.o[fb][4 * r4 + 3]};
                store_output(Oh, dtype, row_offset + feature, value * inverse, d - feature, true);
            }
    }
}

// O of a key-range split launch: each row's parts merged (merge_part), splits in
// order; those past a causal diagonal hold a state only (kNoPart). One thread
// per head, row and 4 features. Splits are taken kBatch at a time, every load of
// a batch issued before any use (one memory round trip per batch).
template <bool kVector>
__global__ __launch_bounds__(256) void split_combine_kernel(const AttnParams p) {
    constexpr int kBatch = 16;
    const int M = p.M, d = p.d, splits = p.splits;
    const int groups = (d + 3) / 4;
    const std::int64_t index = static_cast<std::int64_t>(blockIdx.x) * 256 + threadIdx.x;
    const std::int64_t head_row = index / groups;
    if (head_row >= static_cast<std::int64_t>(p.heads) * M) return;
    const std::int64_t head = head_row / M;
    const int row = static_cast<int>(head_row - head * M);
    const int f0 = 4 * static_cast<int>(index - head_row * groups);
    const float2v* const ml = reinterpret_cast<const float2v*>(p.part_ml);
    float m = -INFINITY, l = 0.0f;
    float4v acc{0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = 0; s0 < splits; s0 += kBatch) {
        float2v state[kBatch];
        float4v value[kBatch];
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
            const std::int64_t r = (head * splits + (s0 + b < splits ? s0 + b : s0)) * M + row;
            state[b] = ml[r];
            const float* src = p.part_o + r * d + f0;
            if constexpr (kVector) {
                value[b] = *reinterpret_cast<const float4v*>(src);
            } else {
                for (int e = 0; e < 4; ++e) value[b][e] = f0 + e < d ? src[e] : 0.0f;
            }
        }
        merge_batch<kBatch, false>(
            m, l, splits - s0,
            [&](int b) TILEMIX_INLINE { return state[b][1] != kNoPart ? state[b] : float2v{-INFINITY, 0.0f}; },
            [&](int b, PartWeights w) TILEMIX_INLINE {
                acc = merged(acc, state[b][1] != kNoPart ? value[b] : float4v{0.0f, 0.0f, 0.0f, 0.0f}, w);
            });
    }
    const float inverse = l > 0.0f ? 1.0f / l : 0.0f;
    unsigned char* const Oh = static_cast<unsigned char*>(p.O) + head * p.o_stride * (p.o_dtype == TILEMIX_DTYPE_F32 ? 4 : 2);
    store_output(Oh, p.o_dtype, static_cast<std::int64_t>(row) * p.o_row + f0, acc * inverse, d - f0, p.o_vector != 0);
}

template <int DC, int kPiece, bool kDots, KeyRange kRange>
hipError_t launch_variant(const AttnParams& p, bool precise, hipStream_t stream) {
    const unsigned blocks = static_cast<unsigned>(p.q_blocks) * static_cast<unsigned>(p.heads) *
                            static_cast<unsigned>(kRange == KeyRange::kSplit ? p.splits : 1);
    constexpr unsigned kMergedBytes = kRange == KeyRange::kInTurn ? 4 * DC * kThreadsPerGroup * sizeof(float4v) : 0;
    if (precise)
        attention_kernel<DC, kPiece, true, kDots, kRange><<<blocks, kThreadsPerGroup, kMergedBytes, stream>>>(p);
    else
        attention_kernel<DC, kPiece, false, kDots, kRange><<<blocks, kThreadsPerGroup, kMergedBytes, stream>>>(p);
    return hipGetLastError();
}

// A split call without a workspace takes its ranges in turn.
template <int DC, int kPiece, bool kDots>
hipError_t launch_vp(const AttnParams& p, bool precise, hipStream_t stream) {
    if (p.splits <= 1) return launch_variant<DC, kPiece, kDots, KeyRange::kWhole>(p, precise, stream);
    return p.part_o ? launch_variant<DC, kPiece, kDots, KeyRange::kSplit>(p, precise, stream)
                    : launch_variant<DC, kPiece, kDots, KeyRange::kInTurn>(p, precise, stream);
}

template <int DC>
hipError_t launch_wide(AttnParams p, hipStream_t stream) {
    const unsigned blocks = static_cast<unsigned>((p.q_blocks + 1) / 2) * static_cast<unsigned>(p.heads);
    p.reverse_slots /= 2;  // half as many workgroups, of twice the rows, per XCD
    attention_wide_kernel<DC><<<blocks, kWideThreads, 0, stream>>>(p);
    return hipGetLastError();
}

}  // namespace

// Verification outputs (dots, trace) take the 16-byte or the element kernel.
// Each head-dimension class DC is compiled in a unit of its own (TILEMIX_DC,
// set by the build), in parallel; the unit without it holds the host side.
template <int DC>
hipError_t launch_dc(const AttnParams& p, int piece, bool precise, bool wide, hipStream_t stream) {
    if (p.dots != nullptr || p.trace != nullptr)
        return piece == 16 ? launch_vp<DC, 16, true>(p, precise, stream) : launch_vp<DC, 0, true>(p, precise, stream);
    if constexpr (DC == 2 || DC == 4)
        if (wide) return launch_wide<DC>(p, stream);
    switch (piece) {
        case 16: return launch_vp<DC, 16, false>(p, precise, stream);
        case 8: return launch_vp<DC, 8, false>(p, precise, stream);
        case 4: return launch_vp<DC, 4, false>(p, precise, stream);
        default: return launch_vp<DC, 0, false>(p, precise, stream);
    }
}

#ifdef TILEMIX_DC
template hipError_t launch_dc<TILEMIX_DC>(const AttnParams&, int, bool, bool, hipStream_t);
}  // namespace tilemix
#else
extern template hipError_t launch_dc<1>(const AttnParams&, int, bool, bool, hipStream_t);
extern template hipError_t launch_dc<2>(const AttnParams&, int, bool, bool, hipStream_t);
extern template hipError_t launch_dc<3>(const AttnParams&, int, bool, bool, hipStream_t);
extern template hipError_t launch_dc<4>(const AttnParams&, int, bool, bool, hipStream_t);

namespace {

std::size_t words_per_row(int N, int group) {
    const std::size_t key_tiles = (static_cast<std::size_t>(N) - 1) / kCellKeys + 1;
    const std::size_t groups = (key_tiles - 1) / static_cast<std::size_t>(group) + 1;
    return (groups - 1) / 64 + 1;
}

std::size_t word_count(int M, int N, int group) {
    if (M <= 0 || N <= 0 || group <= 0) return 0;
    return ((static_cast<std::size_t>(M) - 1) / kCellRows + 1) * words_per_row(N, group);
}

// gfx950 check, cached per device (the reference queries device properties
// on every call, src/tilemix.cu:254-260), with the device's compute-unit
// count (0 when the device is not cached).
constexpr int kMaxDevices = 64;

hipError_t check_device(int* compute_units = nullptr) {
    static std::atomic<int> verdict[kMaxDevices];  // 0 unknown, 1 supported, 2 unsupported
    static std::atomic<int> units[kMaxDevices];
    int device = 0;
    hipError_t status = hipGetDevice(&device);
    if (status != hipSuccess) return status;
    const bool cached = device >= 0 && device < kMaxDevices;
    if (compute_units) *compute_units = 0;
    if (cached) {
        const int known = verdict[device].load(std::memory_order_relaxed);
        if (known == 2) return hipErrorNotSupported;
        if (known == 1) {
            if (compute_units) *compute_units = units[device].load(std::memory_order_relaxed);
            return hipSuccess;
        }
    }
    hipDeviceProp_t properties{};
    status = hipGetDeviceProperties(&properties, device);
    if (status != hipSuccess) return status;
    const bool supported = std::strncmp(properties.gcnArchName, "gfx950", 6) == 0;
    if (cached) {
        units[device].store(properties.multiProcessorCount, std::memory_order_relaxed);
        verdict[device].store(supported ? 1 : 2, std::memory_order_relaxed);
        if (compute_units) *compute_units = properties.multiProcessorCount;
    }
    return supported ? hipSuccess : hipErrorNotSupported;
}

// `units`: the device's compute units (check_device).
hipError_t launch_attention(AttnParams p, int units, bool precise, hipStream_t stream) {
    if (static_cast<long long>(p.q_blocks) * p.heads > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    // Non-causal heads in the per-XCD head-major order whose query blocks
    // outnumber an XCD's workgroup slots stream K / V once per round of
    // slots; alternate rounds walk the keys in opposite directions.
    const int xcd_slots = units / kXcds * kGroupsPerCU;
    p.reverse_slots = (!p.causal && p.splits <= 1 && p.heads % kXcds == 0 && xcd_slots > 0 && p.q_blocks > xcd_slots)
                          ? xcd_slots : 0;
    // DMA paths address a head's K / V with 32-bit buffer offsets; longer
    // heads take the element-wise path. The 16-byte store forms need aligned
    // rows of O (and 8-byte ones of Q8); without them the dword form, which
    // picks its stores at run time, takes the call. Measured (12 heads x 1003
    // x 72, causal, precise P.V): 300 us with elements, 42.6 with pieces; d = 100
    // 347 and 68.7.
    const std::int64_t k_range = (static_cast<std::int64_t>(p.N - 1) * p.k_row + p.d) * 2;
    const std::int64_t v_range = (static_cast<std::int64_t>(p.N - 1) * p.v_row + p.d) * 2;
    int piece = k_range < (std::int64_t{1} << 31) && v_range < (std::int64_t{1} << 31) ? access_piece(p) : 0;
    if (piece >= 8 && !(p.o_vector && (!p.q8_out || aligned(p.q8_out, 8)))) piece = 4;
    const int dc = (p.d + 31) / 32;
    const bool wide = piece == 16 && (dc == 2 || dc == 4) && !precise && p.splits <= 1 && !p.dots && !p.trace && wide_pays(p, units);
    switch (dc) {
        case 1: return launch_dc<1>(p, piece, precise, wide, stream);
        case 2: return launch_dc<2>(p, piece, precise, wide, stream);
        case 3: return launch_dc<3>(p, piece, precise, wide, stream);
        default: return launch_dc<4>(p, piece, precise, wide, stream);
    }
}

}  // namespace
}  // namespace tilemix

// Workspaces of the key-range splits (partial O rows and row states of every
// split) and the arrival counters of the decode kernel. kWorkspaces copies per
// GPU, held until the process ends; the library allocates nothing. A stream's
// calls use the copy that its last call used; another stream takes the one that
// was used least recently. Calls that use the same copy are ordered through its
// event (each waits for the previous one's last kernel, whatever its stream), so
// concurrent streams never share a copy at once, and up to kWorkspaces of them
// do not wait for one another (with one copy, a split call waited for all that
// any stream had queued before its last one). Calls made while their stream is
// being captured into a graph use none.
static constexpr int kWorkspaces = 4;  // as many as hardware queues, HIP's default
static constexpr std::size_t kSplitScratchFloats = std::size_t{8} << 20;  // 32 MiB each
static constexpr std::size_t kSplitArrivals = 1024;
static __device__ __align__(256) float split_scratch[kWorkspaces * kSplitScratchFloats];
static __device__ unsigned split_arrivals[kWorkspaces * kSplitArrivals];  // zero between launches

namespace tilemix {
namespace {

// A split covers at least `tiles` key tiles, and a call whose longest row block
// has fewer than `longest` is not split: the split's fixed cost (partial rows,
// the combine launch, the ordering event) is about that of a few tiles'
// walk. Measured per call, per-head API (M = 4096, d = 128): at N = 256 the
// plain launch is 23 % faster than two splits; at N = 512 four 2-tile splits
// are 14 % faster than two 4-tile ones, and the reference demo (16 tiles) 7 %
// with 8 splits than with 4; from N = 4096 on the slot count limits the splits.
// Batched calls are split where split_pays says so.
// Unsplit | splits of at least 2, 4, 8 tiles (us): 4 heads x 512 x 512 x 64
// 16.1 | 18.7, 19.8, -; 4 x 2048 causal x 128 46.5 | 26.1, 26.0, 28.2; 16 x
// 128 x 4096 x 128 80.4 | 32.3, 28.7, 31.6; 8 x 512 x 8192 x 128 168.6 | 36.4,
// 35.1, 35.0.
// in_turn: a call without a workspace takes the ranges in turn, for the split
// call's bits, which batched calls keep under capture; the per-head call, which
// never promised them, takes the faster unsplit launch there (captured, 4096 x
// 4096 x 128 116 us against 135, 1000 x 1003 x 128 37.7 against 46.7).
struct SplitRule {
    int tiles;
    int longest;
    bool weigh;
    bool in_turn;
};
constexpr SplitRule kSplitHead{2, 8, false, false};
constexpr SplitRule kSplitBatch{4, 16, true, true};

// Whether a split saves more than it costs, from the calls measured above and
// below. A lone workgroup of a CU walks a tile in about 0.5 + d / 160 us (half
// as much again with precise P.V, a quarter with routes and no skipped tiles),
// two walk 9 % slower each; a split costs 4.5 us for the second kernel and the
// event, and 0.75 us per MB of partial rows, written and read. Unsplit and
// split, both sides of the line (us): 4 heads x 1024 x 64 20.3, 15.3; 12 x 1003
// causal x 72 precise 42.6, 31.2; 8 x 2048 causal x 128 52.9, 49.4; 4 x 4096
// causal x 128 87.5, 56.0 | 32 x 1024 x 64 21.2, 34.8; 16 x 2048 x 64 37.2,
// 45.9; 16 x 1024 causal x 128 26.6, 34.7; 200 x 64 x 1500 x 64 three-way
// 40.7, 42.1.
bool split_pays(const AttnParams& p, bool precise, std::int64_t longest, std::int64_t split_tiles) {
    const std::int64_t splits = (longest + split_tiles - 1) / split_tiles;
    const double tile_us = (0.5 + p.d / 160.0) * (precise ? 1.5 : 1.0) * (p.route_words && !p.skip_words ? 1.25 : 1.0);
    const double saved_us = (longest - 1.09 * split_tiles) * tile_us;
    const double partial_mb = 4e-6 * static_cast<double>(splits) * p.heads * p.M * (p.d + 2);
    return saved_us > 1.05 * (4.5 + 0.75 * partial_mb);
}

struct Workspace {
    hipEvent_t done = nullptr;
    bool recorded = false;
    hipStream_t stream = nullptr;  // of the last call
    std::uint64_t used = 0;        // that call's number
};

struct SplitDevice {
    float* scratch = nullptr;
    unsigned* arrivals = nullptr;
    Workspace workspaces[kWorkspaces];
    std::uint64_t calls = 0;
};

// The stream's own workspace, else the least recently used one. (A handle may
// name another stream than it did, so every call waits for the event.)
int choose_workspace(const SplitDevice& device, hipStream_t stream) {
    int oldest = 0;
    for (int i = 0; i < kWorkspaces; ++i) {
        if (device.workspaces[i].recorded && device.workspaces[i].stream == stream) return i;
        if (device.workspaces[i].used < device.workspaces[oldest].used) oldest = i;
    }
    return oldest;
}

std::mutex& split_lock() {
    static std::mutex lock;
    return lock;
}

SplitDevice* split_devices() {
    static SplitDevice devices[kMaxDevices];
    return devices;
}

// Key tiles of one split of a launch whose workgroups would fill less than
// half of the device's slots: as few as spread all tiles over one wave of
// workgroups, at least the rule's, and enough that the partial rows fit in the
// workspace (0 = no split).
int choose_split_tiles(const AttnParams& p, bool precise, int compute_units, const SplitRule& rule) {
    const std::int64_t resident = static_cast<std::int64_t>(compute_units) * kGroupsPerCU;
    const std::int64_t items = static_cast<std::int64_t>(p.heads) * p.q_blocks;
    if (compute_units <= 0 || 2 * items > resident) return 0;
    const std::int64_t tiles = (p.N - 1) / kTileKeys + 1;
    std::int64_t longest = tiles, total = items * tiles;
    if (p.causal) {
        constexpr int kTilesPerBlock = kRowsPerGroup / kTileKeys;
        longest = std::min<std::int64_t>(tiles, static_cast<std::int64_t>(kTilesPerBlock) * p.q_blocks);
        total = 0;
        for (int block = 0; block < p.q_blocks; ++block) total += std::min<std::int64_t>(tiles, (block + 1) * kTilesPerBlock);
        total *= p.heads;
    }
    if (longest < rule.longest) return 0;
    std::int64_t split_tiles;
    if (p.causal) {
        split_tiles = std::max<std::int64_t>((total + resident - 1) / resident, rule.tiles);
    } else {
        const std::int64_t splits = std::max<std::int64_t>(std::min(resident / items, tiles / rule.tiles), 1);
        split_tiles = (tiles + splits - 1) / splits;
    }
    const std::size_t row_floats = static_cast<std::size_t>(p.heads) * p.M * (p.d + 2);
    while (split_tiles < longest && (longest + split_tiles - 1) / split_tiles * row_floats > kSplitScratchFloats) ++split_tiles;
    if (split_tiles >= longest || (rule.weigh && !split_pays(p, precise, longest, split_tiles))) return 0;
    return static_cast<int>(split_tiles);
}

// The current device's number when a call on `stream` may use the workspace
// there, -1 when it may not (the stream is being captured, or the device is
// beyond the table).
int workspace_device(hipStream_t stream) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) return -1;
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return -1;
    return device;
}

// Calls launch(scratch, arrivals), which enqueues kernels on `stream` that use
// one workspace of `device` (the current one), ordered after that workspace's
// previous call and before its next one.
template <typename Launch>
hipError_t with_workspace(int device, hipStream_t stream, Launch&& launch) {
    std::lock_guard<std::mutex> guard(split_lock());
    SplitDevice& state = split_devices()[device];
    hipError_t status = hipSuccess;
    const int chosen = choose_workspace(state, stream);
    Workspace& workspace = state.workspaces[chosen];
    if (!state.scratch || !state.arrivals || !workspace.done) {
        // First split call on this device or workspace: another thread may be capturing a
        // graph in global mode, which would reject these runtime calls (they
        // enqueue no work), so this thread's capture mode is relaxed around
        // them and then restored.
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        status = hipThreadExchangeStreamCaptureMode(&mode);
        if (status != hipSuccess) return status;
        void* address = nullptr;
        if (!state.scratch) {
            status = hipGetSymbolAddress(&address, HIP_SYMBOL(split_scratch));
            if (status == hipSuccess) state.scratch = static_cast<float*>(address);
        }
        if (status == hipSuccess && !state.arrivals) {
            status = hipGetSymbolAddress(&address, HIP_SYMBOL(split_arrivals));
            if (status == hipSuccess) state.arrivals = static_cast<unsigned*>(address);
        }
        if (status == hipSuccess && !workspace.done)
            status = hipEventCreateWithFlags(&workspace.done, hipEventDisableTiming | hipEventDisableSystemFence);
        const hipError_t restored = hipThreadExchangeStreamCaptureMode(&mode);
        if (status != hipSuccess) return status;
        if (restored != hipSuccess) return restored;
    }
    if (workspace.recorded) {
        status = hipStreamWaitEvent(stream, workspace.done, 0);
        if (status != hipSuccess) return status;
    }
    status = launch(state.scratch + chosen * kSplitScratchFloats, state.arrivals + chosen * kSplitArrivals);
    if (status != hipSuccess) return status;
    status = hipEventRecord(workspace.done, stream);
    if (status != hipSuccess) return status;
    workspace.recorded = true;
    workspace.stream = stream;
    workspace.used = ++state.calls;
    return hipSuccess;
}

// launch_attention, with the key range split over several workgroups per
// 128-row block when choose_split_tiles says so: the attention kernel writes
// each split's partial rows to the workspace, split_combine_kernel merges them
// into O, both on `stream`. Where the workspace is not to be used, one workgroup
// takes a block's ranges in turn, to the same bits, or all its keys at once
// (SplitRule::in_turn).
hipError_t launch_attention_split(AttnParams p, int units, bool precise, const SplitRule& rule, hipStream_t stream) {
    const int split_tiles = choose_split_tiles(p, precise, units, rule);
    const int device = split_tiles > 0 ? workspace_device(stream) : -1;
    if (device < 0 && (split_tiles == 0 || !rule.in_turn)) return launch_attention(p, units, precise, stream);
    int tiles = (p.N - 1) / kTileKeys + 1;
    if (p.causal) tiles = std::min(tiles, p.q_blocks * (kRowsPerGroup / kTileKeys));
    p.split_tiles = split_tiles;
    p.splits = (tiles + split_tiles - 1) / split_tiles;
    if (device < 0) return launch_attention(p, units, precise, stream);  // the ranges in turn
    return with_workspace(device, stream, [&](float* scratch, unsigned*) {
        p.part_o = scratch;
        p.part_ml = scratch + static_cast<std::size_t>(p.heads) * p.splits * p.M * p.d;
        const hipError_t status = launch_attention(p, units, precise, stream);
        if (status != hipSuccess) return status;
        const std::int64_t threads = static_cast<std::int64_t>(p.heads) * p.M * ((p.d + 3) / 4);
        const unsigned blocks = static_cast<unsigned>((threads + 255) / 256);
        if (p.d % 4 == 0)
            split_combine_kernel<true><<<blocks, 256, 0, stream>>>(p);
        else
            split_combine_kernel<false><<<blocks, 256, 0, stream>>>(p);
        return hipGetLastError();
    });
}

// Whether the decode kernel (decode.hip) takes the call: one 16-row cell of
// queries per head, no causal mask (whose query i sees keys up to i only), and
// rows that 32-bit buffer offsets reach, up to a step past the last one. At 16
// rows and below the prefill kernel has query rows for half of one wave of its
// four. Measured against it, 128 features: 4 heads x 64 keys 9.5 us either
// way; 32 x 1024 30.1 -> 12.7 us; 32 x 16384 428 -> 54 us. Verification
// outputs do not change the choice, so they never change O.
bool decode_ok(const AttnParams& p, int units) {
    constexpr std::int64_t kReach = std::int64_t{1} << 30;  // halves
    return p.M <= kMaxDecodeRows && !p.causal && p.q_row * kMaxDecodeRows < kReach &&
           (p.N + std::int64_t{64}) * p.k_row < kReach && (p.N + std::int64_t{64}) * p.v_row < kReach &&
           decode_worthwhile(p, units);
}

hipError_t launch_decode_split(AttnParams p, int units, bool precise, hipStream_t stream) {
    const int splits = plan_decode(p, units, kSplitScratchFloats, kSplitArrivals);
    const int device = splits > 1 ? workspace_device(stream) : -1;
    if (device < 0) return launch_decode(p, splits, precise, stream);  // the ranges in turn
    return with_workspace(device, stream, [&](float* scratch, unsigned* arrivals) {
        p.part_o = scratch;
        p.arrivals = arrivals;
        return launch_decode(p, splits, precise, stream);
    });
}

// The kernel that takes the call.
hipError_t launch_call(const AttnParams& p, bool precise, const SplitRule& rule, hipStream_t stream) {
    int units = 0;
    const hipError_t found = check_device(&units);
    if (found != hipSuccess) return found;
    return decode_ok(p, units) ? launch_decode_split(p, units, precise, stream)
                               : launch_attention_split(p, units, precise, rule, stream);
}

// O takes whole vector stores: 16-byte fp32 or 8-byte 16-bit pieces of rows.
int o_vector(const AttnParams& p) {
    return p.d % 4 == 0 && aligned(p.O, 16) && p.o_stride % 4 == 0 && p.o_row % 4 == 0;
}

AttnParams base_params(const std::uint16_t* Q, const std::uint16_t* K, const std::uint16_t* V, float* O,
                       int heads, int M, int N, int d, float score_scale, int group) {
    AttnParams p{};
    p.Q = Q;
    p.K = K;
    p.V = V;
    p.O = O;
    p.heads = heads;
    p.M = M;
    p.N = N;
    p.d = d;
    p.key_tiles_per_group = group;
    p.group_shift = (group & (group - 1)) == 0 ? __builtin_ctz(static_cast<unsigned>(group)) : -1;
    p.q_tiles16 = (M - 1) / kCellRows + 1;
    p.key_tiles32 = (N - 1) / kCellKeys + 1;
    p.q_blocks = (M - 1) / kQBlockRows + 1;
    p.k_blocks = (N - 1) / kKBlockRows + 1;
    p.words_per_row = static_cast<std::int64_t>(words_per_row(N, group));
    p.words_per_head = static_cast<std::int64_t>(word_count(M, N, group));
    p.score_scale = score_scale;
    p.score_log2 = score_scale * kLog2e;
    p.q_stride = static_cast<std::int64_t>(M) * d;
    p.k_stride = static_cast<std::int64_t>(N) * d;
    p.v_stride = static_cast<std::int64_t>(N) * d;
    p.o_stride = static_cast<std::int64_t>(M) * d;
    p.q_row = p.k_row = p.v_row = p.o_row = d;
    p.o_dtype = TILEMIX_DTYPE_F32;
    return p;
}

}  // namespace
}  // namespace tilemix

extern "C" int tilemix_attention(const std::uint16_t* Q, const std::uint16_t* K, const std::uint16_t* V,
                                 float* O, int M, int N, int d, float score_scale, void* stream,
                                 const std::uint64_t* route_words, std::size_t route_word_count,
                                 int key_tiles_per_group, std::uint8_t* decoded_bits,
                                 const std::int8_t* Q8, const std::int8_t* K8,
                                 const std::uint16_t* q_scales, const std::uint16_t* k_scales,
                                 std::int32_t* score_dots) {
    using namespace tilemix;
    // Validation order and codes of src/tilemix.cu:242-253; every argument
    // error returns before the first HIP runtime call.
    if (!Q || !K || !V || !O || M <= 0 || N <= 0 || d <= 0 || !std::isfinite(score_scale) ||
        key_tiles_per_group <= 0 || (!route_words && route_word_count != 0))
        return hipErrorInvalidValue;
    if (d > kMaxHeadDim) return hipErrorNotSupported;
    if (route_words && route_word_count < word_count(M, N, key_tiles_per_group)) return hipErrorInvalidValue;
    const bool has_quantized = Q8 && K8 && q_scales && k_scales;
    const bool any_quantized = Q8 || K8 || q_scales || k_scales || score_dots;
    if ((any_quantized && !has_quantized) || (route_words && !has_quantized)) return hipErrorInvalidValue;

    AttnParams p = base_params(Q, K, V, O, 1, M, N, d, score_scale, key_tiles_per_group);
    p.route_words = route_words;
    p.trace = decoded_bits;
    p.dots = route_words ? score_dots : nullptr;  // only INT8 cells write dots
    p.int8_operands = route_words != nullptr;
    p.Q8 = Q8;
    p.K8 = K8;
    p.q_scales = q_scales;
    p.k_scales = k_scales;
    // The per-head API keeps the reference's fp32-level accuracy (its own test
    // suite checks 1e-5 + 1e-4|x| against fp64), so P.V runs in split precision.
    // A head too small to fill the device has its key range split.
    p.o_vector = o_vector(p);
    return launch_call(p, /*precise=*/true, kSplitHead, static_cast<hipStream_t>(stream));
}

extern "C" int tilemix_attention_batched(const TileMixBatchedArgs* args, void* stream) {
    using namespace tilemix;
    if (!args) return hipErrorInvalidValue;
    const TileMixBatchedArgs& a = *args;
    const int group = a.key_tiles_per_group;
    if (!a.Q || !a.K || !a.V || !a.O || a.heads <= 0 || a.M <= 0 || a.N <= 0 || a.d <= 0 ||
        !std::isfinite(a.score_scale) || group <= 0)
        return hipErrorInvalidValue;
    if (a.d > kMaxHeadDim) return hipErrorNotSupported;
    if (a.o_dtype < TILEMIX_DTYPE_F32 || a.o_dtype > TILEMIX_DTYPE_BF16) return hipErrorInvalidValue;
    const std::int64_t q_row = a.q_row_stride ? a.q_row_stride : a.d;
    const std::int64_t k_row = a.k_row_stride ? a.k_row_stride : a.d;
    const std::int64_t v_row = a.v_row_stride ? a.v_row_stride : a.d;
    const std::int64_t o_row = a.o_row_stride ? a.o_row_stride : a.d;
    if (!strided_heads_ok(a.heads, a.M, a.d, a.q_head_stride, q_row) ||
        !strided_heads_ok(a.heads, a.M, a.d, a.o_head_stride, o_row) ||
        !strided_heads_ok(a.heads, a.N, a.d, a.k_head_stride, k_row) ||
        !strided_heads_ok(a.heads, a.N, a.d, a.v_head_stride, v_row))
        return hipErrorInvalidValue;
    const bool int8 = a.route_words != nullptr;
    if (a.quantize < 0 || a.quantize > 2) return hipErrorInvalidValue;
    if (int8) {
        if (!a.K8 || !a.k_scales) return hipErrorInvalidValue;
        if (!a.quantize && (!a.Q8 || !a.q_scales)) return hipErrorInvalidValue;
        if (a.quantize && (!a.Q8) != (!a.q_scales)) return hipErrorInvalidValue;
    } else if (a.score_dots) {
        return hipErrorInvalidValue;
    }
    // Every check precedes the first launch: an error return leaves all
    // outputs (K8 / k_scales of the pre-pass included) untouched.
    if (static_cast<long long>((a.M - 1) / kQBlockRows + 1) * a.heads > 0x7fffffffLL)
        return hipErrorInvalidConfiguration;
    if (a.quantize == 1 && int8) {
        const QuantSide none = make_quant_side(nullptr, nullptr, nullptr, 0, 1, kQBlockRows, a.d);
        const QuantSide k = make_quant_side(a.K, a.K8, a.k_scales, a.k_head_stride, a.N, kKBlockRows, k_row);
        const hipError_t status = check_device();
        if (status != hipSuccess) return status;
        const hipError_t quant = launch_quantize(none, k, a.heads, a.d, static_cast<hipStream_t>(stream));
        if (quant != hipSuccess) return quant;
    }
    AttnParams p = base_params(a.Q, a.K, a.V, a.O, a.heads, a.M, a.N, a.d, a.score_scale, group);
    p.q_stride = a.q_head_stride;
    p.k_stride = a.k_head_stride;
    p.v_stride = a.v_head_stride;
    p.o_stride = a.o_head_stride;
    if (a.heads == 1) {
        p.q_stride = static_cast<std::int64_t>(a.M) * a.d;
        p.o_stride = p.q_stride;
        p.k_stride = static_cast<std::int64_t>(a.N) * a.d;
        p.v_stride = p.k_stride;
    }
    p.q_row = q_row;
    p.k_row = k_row;
    p.v_row = v_row;
    p.o_row = o_row;
    p.o_dtype = a.o_dtype;
    p.causal = a.causal != 0;
    p.route_words = a.route_words;
    p.skip_words = a.skip_words;
    p.trace = a.decoded_bits;
    p.dots = a.score_dots;
    p.int8_operands = int8;
    p.fuse_q_quant = int8 && a.quantize;
    p.Q8 = a.Q8;
    p.K8 = a.K8;
    p.q_scales = a.q_scales;
    p.k_scales = a.k_scales;
    if (p.fuse_q_quant) {
        p.q8_out = a.Q8;
        p.q_scales_out = a.q_scales;
    }
    p.o_vector = o_vector(p);
    return launch_call(p, a.precise != 0, kSplitBatch, static_cast<hipStream_t>(stream));
}

extern "C" std::size_t tilemix_routing_words_per_row_c(int N, int key_tiles_per_group) {
    if (N <= 0 || key_tiles_per_group <= 0) return 0;
    return tilemix::words_per_row(N, key_tiles_per_group);
}

extern "C" std::size_t tilemix_routing_word_count_c(int M, int N, int key_tiles_per_group) {
    return tilemix::word_count(M, N, key_tiles_per_group);
}

extern "C" std::size_t tilemix_shared_bytes_c(int d, int quantized) {
    if (d <= 0 || d > tilemix::kMaxHeadDim) return 0;
    const std::size_t padded = static_cast<std::size_t>((d + 15) / 16) * 16;
    return 2 * padded * (16 + 2 * 32) + 4 * 16 * 32 + (quantized ? (16 + 32) * padded : 0);
}

extern "C" const char* tilemix_version(void) { return "tilemix-hip 0.1 gfx950"; }
#endif  // TILEMIX_DC
