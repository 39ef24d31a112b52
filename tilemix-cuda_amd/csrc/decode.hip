// Routed INT8/FP16 attention of a few query rows per head (M <= 16) over a
// long key range for gfx950: the decode side of tilemix_attention_batched and
// tilemix_attention.
//
// What bounds it is memory: every key and value row is used by at most 16
// query rows, so the pass is one read of V and of each key tile in the form
// its cell is routed to. The prefill kernel (attention.hip) walks the keys of
// a head with one workgroup of which one wave of four has query rows, one
// tile in flight; here
//
//  * the key range is split over enough workgroups to fill the device
//    (plan_decode) and, inside a workgroup, over its waves, 32 keys
//    (one routing cell: M <= 16 rows are one cell tall) per wave and step;
//  * a wave reads its keys and values straight into registers - no LDS, no
//    barrier - and asks for the next step's 8 to 16 KiB before it computes one.
//    As compiled, little of that stays in flight: above 64 features a part of
//    the step's keys is kept in scratch memory (80 bytes a lane), and every
//    variant waits for most of the loads just issued before the current step's
//    MFMAs, so what hides the latency is the CU's other waves;
//  * scores are S^T = K Q^T with v_mfma_f32_16x16x32_f16 or
//    v_mfma_i32_16x16x64_i8 on 16 keys x 16 query rows. Lane (r, g) =
//    (lane % 16, lane / 16) holds features 64 m + 16 g .. + 15 of key r as two
//    16-byte fp16 pieces or one 16-byte int8 piece, and the same features of
//    query row r, so Q is quantized in its own lanes;
//  * O^T += V^T P^T with v_mfma_f32_16x16x32_f16. The accumulators of the two
//    16-key score blocks are the P^T operand as they are: slot e of group g is
//    key 16 (e / 4) + 4 g + e % 4 of the step. Lane (r, g) reads features
//    kFpl r .. kFpl r + kFpl - 1 of those eight keys (16 lanes read a whole
//    value row) and v_perm_b32 pairs up the keys of one feature: kFpl MFMAs,
//    the f-th over features kFpl row + f;
//  * the waves' row states meet in LDS; the splits' rows go to the
//    library's workspace and the workgroup that arrives last at a head merges
//    them, so a pass is one launch.
//
// Arithmetic is the prefill kernel's: fp32 scores in the log2 domain, fp16
// probabilities (precise: hi + lo), row sums of exactly those.
//
// Measured (MI355X, 32 heads x 4 rows x 16384 keys x 128, half the key tiles
// INT8, 235 MB read): 430 us per call with the prefill kernel, 54 to 55 us here
// (4.3 TB/s; a large copy reaches 5.2).

#include "attention_common.h"
#include "tilemix_capi.h"

#include <algorithm>
#include <type_traits>

namespace tilemix {
namespace {

constexpr int kStepKeys = 32;  // keys of one wave step: one routing cell

constexpr int kNonTemporal = 2;  // nt in a buffer instruction's aux operand

typedef __amdgpu_buffer_rsrc_t Rsrc;

__device__ __forceinline__ Rsrc buffer(const void* base, std::int64_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), kBufferFlags);
}

// kHalves consecutive fp16 values from byte `offset` (row start + 2 feature)
// of a row, `valid` of them inside the row (may be <= 0), the others zero, in
// pieces of kPiece bytes: 16 or 8 whole vectors (feature and d multiples of
// kHalves), 4 pairs, 0 single values. Offsets past the buffer read as zero.
template <int kHalves, int kPiece, int kAux = 0>
__device__ __forceinline__ uint4v load_halves(Rsrc r, unsigned offset, int valid) {
    constexpr unsigned kOut = 0x80000000u;
    uint4v out{0u, 0u, 0u, 0u};
    if constexpr (kPiece >= 8) {
        const unsigned at = valid > 0 ? offset : kOut;
        if constexpr (kHalves == 8) {
            out = __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, kAux);
        } else {
            const uint2v two = __builtin_amdgcn_raw_buffer_load_b64(r, at, 0, kAux);
            out[0] = two[0];
            out[1] = two[1];
        }
    } else if constexpr (kPiece == 4) {
#pragma unroll
        for (int j = 0; j < kHalves / 2; ++j)
            out[j] = __builtin_amdgcn_raw_buffer_load_b32(r, 2 * j < valid ? offset + 4 * j : kOut, 0, 0);
    } else {
#pragma unroll
        for (int j = 0; j < kHalves / 2; ++j) {
            const unsigned lo = __builtin_amdgcn_raw_buffer_load_b16(r, 2 * j < valid ? offset + 4 * j : kOut, 0, 0);
            const unsigned hi =
                __builtin_amdgcn_raw_buffer_load_b16(r, 2 * j + 1 < valid ? offset + 4 * j + 2 : kOut, 0, 0);
            out[j] = lo | (hi << 16);
        }
    }
    return out;
}

// 16 int8 values from byte `offset` of a row, `valid` of them inside the row.
template <int kPiece, int kAux = 0>
__device__ __forceinline__ uint4v load_bytes(Rsrc r, unsigned offset, int valid) {
    constexpr unsigned kOut = 0x80000000u;
    uint4v out{0u, 0u, 0u, 0u};
    if constexpr (kPiece == 16) {
        out = __builtin_amdgcn_raw_buffer_load_b128(r, valid > 0 ? offset : kOut, 0, kAux);
    } else if constexpr (kPiece >= 4) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            out[j] = __builtin_amdgcn_raw_buffer_load_b32(r, 4 * j < valid ? offset + 4 * j : kOut, 0, 0);
    } else {
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const unsigned byte = __builtin_amdgcn_raw_buffer_load_b8(r, j < valid ? offset + j : kOut, 0, 0);
            out[j / 4] |= (byte & 0xffu) << (8 * (j % 4));
        }
    }
    return out;
}

// Maximum / sum over the four lanes r, r + 16, r + 32, r + 48, in each of them.
__device__ __forceinline__ void permlane16_swap(float& a, float& b) {
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
}
__device__ __forceinline__ float groups_max(float x) {
    float a = x, b = x;
    permlane16_swap(a, b);
    a = fmaxf(a, b);
    b = a;
    permlane32_swap(a, b);
    return fmaxf(a, b);
}
__device__ __forceinline__ float groups_sum(float x) {
    float a = x, b = x;
    permlane16_swap(a, b);
    a = a + b;
    b = a;
    permlane32_swap(a, b);
    return a + b;
}

// The keys (fp16 or int8) and values of one wave step, as loaded.
template <int kBlocks>
struct StepData {
    uint4v k[2][2 * kBlocks];  // fp16: piece c of key block b; int8: block m of key block b in k[b][m]
    uint4v v[8];               // slot e: kFpl halves of one value row
    std::uint16_t k_scale;
};

// kBlocks: 64-feature blocks (1: d <= 64, 2: d <= 128). kPiece: bytes of a
// contiguous load (load_halves). kWaves: waves of a workgroup. kStream: keys
// and values are loaded with a non-temporal hint. kInTurn: the workgroup takes
// all of its head's ranges one after the other and merges them as the last of
// several workgroups does: a split call's bits without a workspace, for a
// stream that is being captured.
template <int kBlocks, int kPiece, bool kPrecise, int kWaves, bool kStream, bool kInTurn>
__global__ __launch_bounds__(kWaves * kWave, 8 / kWaves) void decode_kernel(const AttnParams p) {
    constexpr int kDP = 64 * kBlocks;
    constexpr int kFpl = 4 * kBlocks;  // value features per lane
    constexpr int kPieces = 2 * kBlocks;
    constexpr int kAux = kStream ? kNonTemporal : 0;
    __shared__ __attribute__((aligned(16))) float lds_o[kWaves][16][kDP];
    __shared__ float lds_ml[kWaves][16][2];
    __shared__ int lds_last;

    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15;  // key of a score block (A operand), query row (B operand and results)
    const int g = lane >> 4;
    const int head32 = kInTurn ? blockIdx.x : blockIdx.x / p.splits;
    const int first_split = kInTurn ? 0 : blockIdx.x - head32 * p.splits;
    const std::int64_t head = head32;
    const int M = p.M, N = p.N, d = p.d;

    const int q_row_bytes = static_cast<int>(p.q_row * 2);
    const int k_row_bytes = static_cast<int>(p.k_row * 2), v_row_bytes = static_cast<int>(p.v_row * 2);
    const Rsrc rq = buffer(p.Q + head * p.q_stride, (static_cast<std::int64_t>(M - 1) * p.q_row + d) * 2);
    const Rsrc rk = buffer(p.K + head * p.k_stride, (static_cast<std::int64_t>(N - 1) * p.k_row + d) * 2);
    const Rsrc rv = buffer(p.V + head * p.v_stride, (static_cast<std::int64_t>(N - 1) * p.v_row + d) * 2);
    const std::int64_t k8_bytes = static_cast<std::int64_t>(N) * d;
    const Rsrc rk8 = buffer(p.int8_operands ? p.K8 + head * k8_bytes : nullptr, p.int8_operands ? k8_bytes : 0);

    // Per-lane offsets of the first step's pieces; a step adds whole rows.
    unsigned k_at[kPieces], k8_at[kBlocks];
    int k_valid[kPieces], k8_valid[kBlocks];
#pragma unroll
    for (int c = 0; c < kPieces; ++c) {
        const int feature = 64 * (c / 2) + 16 * g + 8 * (c % 2);
        k_at[c] = static_cast<unsigned>(r * k_row_bytes + 2 * feature);
        k_valid[c] = d - feature;
    }
#pragma unroll
    for (int m = 0; m < kBlocks; ++m) {
        k8_at[m] = static_cast<unsigned>(r * d + 64 * m + 16 * g);
        k8_valid[m] = d - (64 * m + 16 * g);
    }
    const unsigned v_at = static_cast<unsigned>(4 * g * v_row_bytes + 2 * kFpl * r);
    const int v_valid = d - kFpl * r;
    const std::uint16_t* const k_scales = p.k_scales + head * p.k_blocks;

    // ------------------------------------------------------------ routes
    // All query rows lie in one 16-row tile: one route / skip bit per step.
    const bool routed = p.route_words != nullptr || p.skip_words != nullptr;
    const std::int64_t word_base = head * p.words_per_head;
    int cached_block = -1;
    std::uint64_t route_word = 0, skip_word = 0;
    auto uniform = [](std::uint64_t x) {
        const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(x));
        const unsigned hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(x >> 32));
        return (static_cast<std::uint64_t>(hi) << 32) | lo;
    };
    auto code_of = [&](int step) -> int {
        if (!routed) return TILEMIX_ROUTE_FP16;
        const unsigned group = p.group_shift >= 0 ? static_cast<unsigned>(step) >> p.group_shift
                                                  : static_cast<unsigned>(step) / static_cast<unsigned>(p.key_tiles_per_group);
        const int block = static_cast<int>(group >> 6);
        if (block != cached_block) {
            cached_block = block;
            route_word = p.route_words ? uniform(p.route_words[word_base + block]) : 0ull;
            skip_word = p.skip_words ? uniform(p.skip_words[word_base + block]) : 0ull;
        }
        const unsigned bit = group & 63u;
        if ((skip_word >> bit) & 1u) return TILEMIX_ROUTE_SKIP;
        return ((route_word >> bit) & 1u) ? TILEMIX_ROUTE_INT8 : TILEMIX_ROUTE_FP16;
    };
    // One range of steps, up to the merge of the workgroup's waves: the state and
    // O of each thread's row of it.
    float4v acc[kBlocks];
    float row_m, row_l;
    auto take_range = [&](int split) __attribute__((always_inline)) {
        // This workgroup's steps, dealt to its waves in turn. Every step is passed
        // once by one wave, which writes its routing trace.
        const int step_end = min((N - 1) / kStepKeys + 1, (split + 1) * p.split_tiles);
        int code = TILEMIX_ROUTE_FP16;
        auto next_step = [&](int step) {
            for (; step < step_end; step += kWaves) {
                code = code_of(step);
                if (p.trace && lane == 0) p.trace[head * p.key_tiles32 + step] = static_cast<std::uint8_t>(code);
                if (code != TILEMIX_ROUTE_SKIP) break;
            }
            return step;
        };
        auto load_step = [&](StepData<kBlocks>& data, int step, int route) {
            const unsigned k0 = static_cast<unsigned>(step * kStepKeys);
            if (route == TILEMIX_ROUTE_INT8) {
                data.k_scale = k_scales[step >> 1];
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int m = 0; m < kBlocks; ++m)
                        data.k[b][m] = load_bytes<kPiece, kAux>(rk8, (k0 + 16 * b) * d + k8_at[m], k8_valid[m]);
            } else {
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int c = 0; c < kPieces; ++c)
                        data.k[b][c] = load_halves<8, kPiece, kAux>(rk, (k0 + 16 * b) * k_row_bytes + k_at[c], k_valid[c]);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e)
                data.v[e] = load_halves<kFpl, kPiece, kAux>(rv, (k0 + 16 * (e / 4) + e % 4) * v_row_bytes + v_at, v_valid);
        };

        // The first step is fetched before Q is touched.
        StepData<kBlocks> even, odd;
        int step = next_step(split * p.split_tiles + wave);
        int step_code = code;
        if (step < step_end) load_step(even, step, step_code);

        // ------------------------------------------------------------ Q
        half8 qf[kPieces];
#pragma unroll
        for (int c = 0; c < kPieces; ++c) {
            const int feature = 64 * (c / 2) + 16 * g + 8 * (c % 2);
            const unsigned at = r < M ? static_cast<unsigned>(r * q_row_bytes + 2 * feature) : 0x80000000u;
            qf[c] = __builtin_bit_cast(half8, load_halves<8, kPiece>(rq, at, r < M ? d - feature : 0));
        }
        int4v q8f[kBlocks];
        float q_scale = 0.0f;
        if (p.int8_operands) {
            if (p.fuse_q_quant) {
                // The head's M <= 16 rows are its one Q block, all in this wave:
                // the quantizer's maximum (integer order of the sign-cleared fp16
                // bits, NaNs passed over) and bytes.
                unsigned top = 0;
#pragma unroll
                for (int c = 0; c < kPieces; ++c) {
                    const uint4v words = __builtin_bit_cast(uint4v, qf[c]);
#pragma unroll
                    for (int w = 0; w < 4; ++w) top = max_u16x2(top, words[w] & 0x7fff7fffu);
                }
                unsigned bits = wave_max_bits(max(top & 0xffffu, top >> 16));
                if (bits > 0x7c00u) {
                    unsigned clean = 0;
#pragma unroll
                    for (int c = 0; c < kPieces; ++c) {
                        const uint4v words = __builtin_bit_cast(uint4v, qf[c]);
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            const unsigned hb = (words[e / 2] >> (16 * (e % 2))) & 0x7fffu;
                            clean = hb <= 0x7c00u ? max(clean, hb) : clean;
                        }
                    }
                    bits = wave_max_bits(clean);
                }
                const float scale = block_scale(half_bits_to_float(static_cast<std::uint16_t>(bits)));
                const float recip = 1.0f / scale;
                const _Float16 stored = static_cast<_Float16>(scale);
                q_scale = static_cast<float>(stored);
                const bool writer = split == 0 && wave == 0;
                if (writer && lane == 0 && p.q_scales_out) p.q_scales_out[head] = __builtin_bit_cast(std::uint16_t, stored);
#pragma unroll
                for (int m = 0; m < kBlocks; ++m) {
#pragma unroll
                    for (int half = 0; half < 2; ++half) {
                        const uint4v words = __builtin_bit_cast(uint4v, qf[2 * m + half]);
                        int b[8] = {};
                        if (scale > 0.0f) {
#pragma unroll
                            for (int w = 0; w < 4; ++w) {
                                b[2 * w] = quantize_half<0>(words[w], scale, recip);
                                b[2 * w + 1] = quantize_half<1>(words[w], scale, recip);
                            }
                        }
                        q8f[m][2 * half] = static_cast<int>(pack_bytes(b[0], b[1], b[2], b[3]));
                        q8f[m][2 * half + 1] = static_cast<int>(pack_bytes(b[4], b[5], b[6], b[7]));
                    }
                    if (writer && p.q8_out && r < M) {
                        const int feature = 64 * m + 16 * g;
                        std::int8_t* const dst = p.q8_out + (head * M + r) * d + feature;
                        for (int e = 0; e < 16 && feature + e < d; ++e)
                            dst[e] = static_cast<std::int8_t>(q8f[m][e / 4] >> (8 * (e % 4)));
                    }
                }
            } else {
                q_scale = half_bits_to_float(p.q_scales[head]);
                const Rsrc rq8 = buffer(p.Q8 + head * M * d, static_cast<std::int64_t>(M) * d);
#pragma unroll
                for (int m = 0; m < kBlocks; ++m) {
                    const int feature = 64 * m + 16 * g;
                    q8f[m] = __builtin_bit_cast(
                        int4v, load_bytes<kPiece>(rq8, static_cast<unsigned>(r * d + feature), r < M ? d - feature : 0));
                }
            }
        }

        // ------------------------------------------------------------ keys
        float4v o[kFpl];  // o[f][i]: query row r, feature kFpl (4 g + i) + f
#pragma unroll
        for (int f = 0; f < kFpl; ++f) o[f] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
        float row_max = -INFINITY, row_sum = 0.0f;  // row_sum: this lane's part
        const bool positive_scale = p.score_scale >= 0.0f;

        auto compute = [&](const StepData<kBlocks>& data, int at, int route) {
            const int k0 = at * kStepKeys;
            float4v s[2];  // s[b][i]: row r against key k0 + 16 b + 4 g + i
            float c;       // log2-domain factor
            if (route == TILEMIX_ROUTE_INT8) {
                c = ((q_scale * half_bits_to_float(data.k_scale)) * p.score_scale) * kLog2e;
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    int4v acc{0, 0, 0, 0};
#pragma unroll
                    for (int m = 0; m < kBlocks; ++m)
                        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(int4v, data.k[b][m]), q8f[m], acc, 0, 0, 0);
                    if (p.dots && r < M) {  // raw int32 dots (verification output)
                        std::int32_t* const row = p.dots + (head * M + r) * static_cast<std::int64_t>(N);
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            if (k0 + 16 * b + 4 * g + i < N) row[k0 + 16 * b + 4 * g + i] = acc[i];
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) s[b][i] = static_cast<float>(acc[i]);
                }
            } else {
                c = p.score_log2;
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    s[b] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int m = 0; m < kPieces; ++m)
                        s[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, data.k[b][m]), qf[m], s[b], 0, 0, 0);
                }
            }
            const bool tail = k0 + kStepKeys > N;
            if (tail || !positive_scale) {  // explicit scores
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        s[b][i] *= c;
                        if (k0 + 16 * b + 4 * g + i >= N) s[b][i] = -INFINITY;
                    }
                c = 1.0f;
            }
            const float top = max3(max3(s[0][0], s[0][1], s[0][2]), max3(s[0][3], s[1][0], s[1][1]),
                                   max3(s[1][2], s[1][3], s[1][3])) * c;  // c >= 0
            if (__any(top > row_max + kLazyRescale)) {
                const float m_new = fmaxf(row_max, groups_max(top));
                const float alpha = m_new == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(row_max - m_new);
                row_max = m_new;
#pragma unroll
                for (int f = 0; f < kFpl; ++f) o[f] *= alpha;
                row_sum *= alpha;
            }
            const float neg_m = row_max == -INFINITY ? 0.0f : -row_max;
            half8 ph, pl;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float v = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e / 4][e % 4], c, neg_m));
                const _Float16 hv = static_cast<_Float16>(v);
                ph[e] = hv;
                if constexpr (kPrecise) pl[e] = static_cast<_Float16>(v - static_cast<float>(hv));
            }
            const half2v ones{1.0f16, 1.0f16};
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                row_sum = __builtin_amdgcn_fdot2(half2v{ph[e], ph[e + 1]}, ones, row_sum, false);
                if constexpr (kPrecise) row_sum = __builtin_amdgcn_fdot2(half2v{pl[e], pl[e + 1]}, ones, row_sum, false);
            }
#pragma unroll
            for (int f = 0; f < kFpl; ++f) {
                // Keys of slots 2t, 2t + 1 for feature f of this lane's kFpl.
                constexpr unsigned kLow = 0x05040100u, kHigh = 0x07060302u;
                uint4v a;
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    a[t] = __builtin_amdgcn_perm(data.v[2 * t + 1][f / 2], data.v[2 * t][f / 2], f % 2 ? kHigh : kLow);
                o[f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), ph, o[f], 0, 0, 0);
                if constexpr (kPrecise)
                    o[f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), pl, o[f], 0, 0, 0);
            }
        };

        // Two steps per iteration, each fetching the other's data before it
        // computes its own; every wave leaves when its steps run out.
        while (step < step_end) {
            const int second = next_step(step + kWaves);
            const int second_code = code;
            if (second < step_end) load_step(odd, second, second_code);
            compute(even, step, step_code);
            if (second >= step_end) break;
            step = next_step(second + kWaves);
            step_code = code;
            if (step < step_end) load_step(even, step, step_code);
            compute(odd, second, second_code);
        }

        // ------------------------------------------------------- merge of waves
        const float l_row = groups_sum(row_sum);
        if (g == 0) {
            lds_ml[wave][r][0] = row_max;
            lds_ml[wave][r][1] = l_row;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int f = 0; f < kFpl; f += 4)
                *reinterpret_cast<float4v*>(&lds_o[wave][r][kFpl * (4 * g + i) + f]) =
                    float4v{o[f][i], o[f + 1][i], o[f + 2][i], o[f + 3][i]};
        __syncthreads();

        const int row = min(tid >> 4, 15), f0 = kFpl * (tid & 15);
        row_m = -INFINITY;
        row_l = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) row_m = fmaxf(row_m, lds_ml[w][row][0]);
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) acc[b] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float m_w = lds_ml[w][row][0];
            const float weight = m_w == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_w - row_m);
            row_l += weight * lds_ml[w][row][1];
#pragma unroll
            for (int b = 0; b < kBlocks; ++b) acc[b] += weight * *reinterpret_cast<const float4v*>(&lds_o[w][row][f0 + 4 * b]);
        }
    };
    if constexpr (kInTurn) {
        float4v sum[kBlocks] = {};
        float m = -INFINITY, l = 0.0f;
        for (int split = 0; split < p.splits; ++split) {
            take_range(split);
            const PartWeights w = merge_part(m, l, row_m, row_l);
#pragma unroll
            for (int b = 0; b < kBlocks; ++b) sum[b] = merged(sum[b], acc[b], w);
            __syncthreads();  // lds_o and lds_ml are read: the next range may write them
        }
        row_l = l;
#pragma unroll
        for (int b = 0; b < kBlocks; ++b) acc[b] = sum[b];
    } else {
        take_range(first_split);
    }

    // Thread (row, f0) of the merges: kFpl features of one row; rows past M - 1
    // (threads of the upper waves among them) only arrive.
    const int row = min(tid >> 4, 15), f0 = kFpl * (tid & 15);
    const bool mine = (tid >> 4) < M;
    // ------------------------------------------------------ merge of splits
    if (!kInTurn && p.splits > 1) {
        const int split = first_split;
        // part_o [heads][splits][M][kDP], part_ml [heads][splits][M][2]; both
        // within the workspace, so byte offsets fit 32 bits.
        const int parts = p.heads * p.splits * M;
        const Rsrc ro = shared_rows(p.part_o, static_cast<std::int64_t>(parts) * kDP);
        const Rsrc rml = shared_rows(p.part_ml, static_cast<std::int64_t>(parts) * 2);
        if (mine) {
            const int part = (head32 * p.splits + split) * M + row;
#pragma unroll
            for (int b = 0; b < kBlocks; ++b)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4v, acc[b]), ro, (part * kDP + f0 + 4 * b) * 4,
                                                       0, kDeviceScope);
            if (f0 == 0)
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(uint2v, float2v{row_m, row_l}), rml, part * 8, 0,
                                                      kDeviceScope);
        }
        if (!last_arrival(p.arrivals + head, p.splits, &lds_last)) return;
        if (mine) {
            const int first = head32 * p.splits * M + row;
            row_m = -INFINITY;
            row_l = 0.0f;
#pragma unroll
            for (int b = 0; b < kBlocks; ++b) acc[b] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
            // Batches of splits, every load of a batch issued before any use.
            auto merge_parts = [&](auto batch) __attribute__((always_inline)) {
                constexpr int kBatch = decltype(batch)::value;
                for (int s0 = 0; s0 < p.splits; s0 += kBatch) {
                    float2v state[kBatch];
                    float4v value[kBatch][kBlocks];
#pragma unroll
                    for (int u = 0; u < kBatch; ++u) {
                        const int from = first + min(s0 + u, p.splits - 1) * M;
                        state[u] = __builtin_bit_cast(float2v, __builtin_amdgcn_raw_buffer_load_b64(rml, from * 8, 0, kDeviceScope));
#pragma unroll
                        for (int b = 0; b < kBlocks; ++b)
                            value[u][b] = __builtin_bit_cast(
                                float4v, __builtin_amdgcn_raw_buffer_load_b128(ro, (from * kDP + f0 + 4 * b) * 4, 0, kDeviceScope));
                    }
                    merge_batch<kBatch, true>(
                        row_m, row_l, p.splits - s0, [&](int u) __attribute__((always_inline)) { return state[u]; },
                        [&](int u, PartWeights w) __attribute__((always_inline)) {
#pragma unroll
                            for (int b = 0; b < kBlocks; ++b) acc[b] = merged(acc[b], value[u][b], w);
                        });
                }
            };
            if (p.splits <= 8)
                merge_parts(std::integral_constant<int, 8>{});
            else
                merge_parts(std::integral_constant<int, 16>{});
        }
    }
    if (mine) {
        const float inverse = row_l > 0.0f ? 1.0f / row_l : 0.0f;
        unsigned char* const Oh = static_cast<unsigned char*>(p.O) + head * p.o_stride * (p.o_dtype == TILEMIX_DTYPE_F32 ? 4 : 2);
        const std::int64_t at = static_cast<std::int64_t>(row) * p.o_row + f0;
#pragma unroll
        for (int b = 0; b < kBlocks; ++b)
            store_output(Oh, p.o_dtype, at + 4 * b, acc[b] * inverse, d - f0 - 4 * b, p.o_vector != 0);
    }
}

// Keys and values of more than this many bytes do not stay in the 256 MiB
// Infinity Cache until the next call: they are read with a non-temporal hint,
// and long walks by four waves per CU. Measured (three calls' buffers in turn,
// 128 features, eight waves without the hint, with it, four waves with it):
// 32 heads x 16384, half INT8 61.9, 55.3, 53.9 us | 32 x 32768 dense 132, 118,
// 107 us | 100 x 3000, 47 steps per workgroup -, 31.9, 36.9 us; but 32 x 4096
// (58 MB) 20.9, 22.2 us.
constexpr std::int64_t kStreamBytes = std::int64_t{128} << 20;
constexpr int kLongWalk = 64;  // steps of a workgroup

// Calls of this many heads fill the device several times over unsplit: two
// workgroups of four waves per CU, whose beginnings and ends overlap (2000
// heads x 512 keys x 64: 60.9 us with eight waves, 46.7 with four). Below,
// eight waves share a head's keys (200 heads x 4096 x 64: 33.9 us, with four
// 36.7).
constexpr int kManyHeads = 512;

// A split call without a workspace takes its ranges in turn.
template <int kBlocks, int kPiece, bool kPrecise, int kWaves, bool kStream>
void launch_decode_kernel(const AttnParams& p, hipStream_t stream) {
    const unsigned heads = static_cast<unsigned>(p.heads);
    if (p.splits > 1 && !p.part_o)
        decode_kernel<kBlocks, kPiece, kPrecise, kWaves, false, true><<<heads, kWaves * kWave, 0, stream>>>(p);
    else
        decode_kernel<kBlocks, kPiece, kPrecise, kWaves, kStream, false>
            <<<heads * static_cast<unsigned>(p.splits), kWaves * kWave, 0, stream>>>(p);
}

// The number of waves, which orders a row's sums as the split does, depends on
// sizes and the device's compute units (through split_tiles) only: never on
// alignment or routes, nor on whether the stream is being captured.
template <int kBlocks, int kPiece, bool kPrecise>
void launch_decode_variant(const AttnParams& p, hipStream_t stream) {
    const bool large = static_cast<std::int64_t>(p.heads) * p.N * p.d * 4 > kStreamBytes;
    const bool four = p.heads >= kManyHeads || (large && p.split_tiles >= kLongWalk);
    constexpr bool kStream = kPiece == 16;
    if (four)
        large ? launch_decode_kernel<kBlocks, kPiece, kPrecise, 4, kStream>(p, stream)
              : launch_decode_kernel<kBlocks, kPiece, kPrecise, 4, false>(p, stream);
    else
        large ? launch_decode_kernel<kBlocks, kPiece, kPrecise, 8, kStream>(p, stream)
              : launch_decode_kernel<kBlocks, kPiece, kPrecise, 8, false>(p, stream);
}

template <int kBlocks, int kPiece>
void launch_decode_piece(const AttnParams& p, bool precise, hipStream_t stream) {
    precise ? launch_decode_variant<kBlocks, kPiece, true>(p, stream) : launch_decode_variant<kBlocks, kPiece, false>(p, stream);
}

template <int kBlocks>
void launch_decode_blocks(const AttnParams& p, bool precise, hipStream_t stream) {
    switch (access_piece(p)) {
        case 16: return launch_decode_piece<kBlocks, 16>(p, precise, stream);
        case 8: return launch_decode_piece<kBlocks, 8>(p, precise, stream);
        case 4: return launch_decode_piece<kBlocks, 4>(p, precise, stream);
        default: return launch_decode_piece<kBlocks, 0>(p, precise, stream);
    }
}

}  // namespace

// A workgroup covers at least this many steps, one for each of its waves (32
// heads x 1024 keys x 128: 14.7 us per call with 8, 16.9 with 16).
constexpr int kMinDecodeSteps = 8;

int plan_decode(const AttnParams& p, int compute_units, std::size_t scratch_floats, std::size_t max_arrivals) {
    const int steps = (p.N - 1) / kStepKeys + 1;
    const std::size_t row_floats = 64 * static_cast<std::size_t>((p.d + 63) / 64) + 2;
    // One workgroup per CU: more splits of a head cost its last workgroup more
    // to merge than they gain (8 heads x 16384 x 128: 26 us at 256 workgroups,
    // 42 at 512).
    if (compute_units <= 0 || static_cast<std::size_t>(p.heads) > max_arrivals) return 1;
    std::int64_t splits = std::min<std::int64_t>(compute_units / p.heads, steps / kMinDecodeSteps);
    splits = std::min<std::int64_t>(splits, scratch_floats / (row_floats * p.heads * p.M));
    if (splits <= 1) return 1;
    const int per_split = static_cast<int>((steps + splits - 1) / splits);
    return (steps + per_split - 1) / per_split;
}

hipError_t launch_decode(AttnParams p, int splits, bool precise, hipStream_t stream) {
    const int steps = (p.N - 1) / kStepKeys + 1;
    p.splits = splits;
    p.split_tiles = (steps + splits - 1) / splits;
    if (splits > 1) p.part_ml = p.part_o + static_cast<std::size_t>(p.heads) * splits * p.M * (64 * ((p.d + 63) / 64));
    p.d <= 64 ? launch_decode_blocks<1>(p, precise, stream) : launch_decode_blocks<2>(p, precise, stream);
    return hipGetLastError();
}

}  // namespace tilemix
