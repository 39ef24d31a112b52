// Block INT8 quantizer for TileMix on gfx950.
//
// Replaces quantize_tilemix_qk / quantize_blocks<BlockRows> of the reference
// (src/tilemix.cu:16-49, 223-236). One 256-thread workgroup owns one
// quantization block (128 Q rows or 64 K rows x d features). Because rows are
// contiguous, a block is one contiguous span of rows*d halves: the piece paths
// read it once with 16-byte or 8-byte loads into registers (at most 64 halves
// per thread), reduce the absmax across the workgroup and quantize from
// registers, so HBM sees exactly one read of the input and one write of the
// int8 output. The absmax runs on packed fp16 pairs (magnitudes by clearing the
// sign bits) and the per-element quotient uses the block's reciprocal with an
// exact correction step instead of a division (quantize_value_recip).

#include "tilemix_device.h"
#include "tilemix_launch.h"

#include <algorithm>

namespace tilemix {
namespace {

constexpr int kQuantThreads = 256;
constexpr int kQuantMaxElements = 128 * 128;  // of a block: 64 per thread
constexpr int kLineHalves = 64;  // fp16 values of a 128-byte cache line

template <int kPiece>
struct PieceTypes;  // kPiece fp16 values in, kPiece bytes out
template <>
struct PieceTypes<8> {
    typedef uint4v Halves;
    typedef uint2v Bytes;
};
template <>
struct PieceTypes<4> {
    typedef uint2v Halves;
    typedef std::uint32_t Bytes;
};

// kPiece: elements a load takes, 0 for the element-wise form. Pieces of 8 are
// 16-byte loads of rows that are whole and 16-byte aligned in them; pieces of
// 4, 8-byte loads, take the other rows that are multiples of 4 elements and
// 8-byte aligned (d = 100, 36, or d = 128 at a row stride of 132). HBM bound:
// 64 heads x 4096 x 100 in pieces of 4 31.4 us (157 MB, 5.0 TB/s), element by
// element 131.1 us; in pieces of 8 x 128 37.9 us (201 MB, 5.3 TB/s).
// kContiguous: rows are d elements apart, so a block is one span of
// rows * d halves; otherwise piece c of the block is piece c % (d / kPiece) of
// row c / (d / kPiece). kPieces: pieces held per thread, enough for the larger
// block of the launch (4 of 8 for 64 x 128 K blocks, 8 for 128 x 128 Q).
// heads_first: the grid is [heads, blocks] instead of [blocks, heads].
template <int kPiece, bool kContiguous, int kPieces>
__global__ __launch_bounds__(kQuantThreads) void quantize_blocks_kernel(QuantSide q, QuantSide k, int d,
                                                                            bool heads_first) {
    __shared__ float partial[kQuantThreads / kWave];
    __shared__ unsigned partial_bits[kQuantThreads / kWave];
    const int at_block = static_cast<int>(heads_first ? blockIdx.y : blockIdx.x);
    const bool is_q = at_block < q.blocks;
    const QuantSide side = is_q ? q : k;
    const int block = is_q ? at_block : at_block - q.blocks;
    const std::int64_t head = heads_first ? blockIdx.x : blockIdx.y;
    const int first = block * side.block_rows;
    const int last = min(side.rows, first + side.block_rows);
    const int count = (last - first) * d;
    const std::uint16_t* in = side.x + head * side.in_head_stride + static_cast<std::int64_t>(first) * side.in_row_stride;
    const std::int64_t row_stride = side.in_row_stride;
    std::int8_t* out = side.x8 + head * static_cast<std::int64_t>(side.rows) * d +
                       static_cast<std::int64_t>(first) * d;
    const int t = threadIdx.x;

    float absmax = 0.0f;
    constexpr int kWords = kPiece ? kPiece / 2 : 1;  // 32-bit words of a piece
    using Types = PieceTypes<kPiece ? kPiece : 8>;
    typename Types::Halves piece[kPieces];
    const int pieces = kPiece ? count / (kPiece ? kPiece : 1) : 0;
    if constexpr (kPiece > 0) {
        // Pieces past the block's end load its last piece again (in-block
        // values, which leave the maximum unchanged; they are not stored).
        const int per_row = d / kPiece;
#pragma unroll
        for (int c = 0; c < kPieces; ++c) {
            const int index = t + c * kQuantThreads;
            const int at = index < pieces ? index : pieces - 1;
            const std::uint16_t* source;
            if constexpr (kContiguous) {
                source = in + kPiece * at;
            } else {
                source = in + (at / per_row) * row_stride + kPiece * (at % per_row);
            }
            piece[c] = *reinterpret_cast<const typename Types::Halves*>(source);
        }
        // |x| as fp16 bit patterns: unsigned order is float order for them,
        // NaN patterns (> 0x7c00) sorting above +inf.
        unsigned top = 0;
#pragma unroll
        for (int c = 0; c < kPieces; ++c)
#pragma unroll
            for (int w = 0; w < kWords; ++w) top = max_u16x2(top, piece[c][w] & 0x7fff7fffu);
        unsigned bits = wave_max_bits(max(top & 0xffffu, top >> 16));
        if ((t & (kWave - 1)) == 0) partial_bits[t / kWave] = bits;
        __syncthreads();
        bits = max(max(partial_bits[0], partial_bits[1]), max(partial_bits[2], partial_bits[3]));
        if (bits > 0x7c00u) {
            // A NaN in the block: the maximum skips NaNs, as fmaxf does.
            unsigned clean = 0;
#pragma unroll
            for (int c = 0; c < kPieces; ++c)
#pragma unroll
                for (int e = 0; e < kPiece; ++e) {
                    const unsigned h = (piece[c][e / 2] >> (16 * (e % 2))) & 0x7fffu;
                    clean = h <= 0x7c00u ? max(clean, h) : clean;
                }
            clean = wave_max_bits(clean);
            __syncthreads();
            if ((t & (kWave - 1)) == 0) partial_bits[t / kWave] = clean;
            __syncthreads();
            bits = max(max(partial_bits[0], partial_bits[1]), max(partial_bits[2], partial_bits[3]));
        }
        absmax = half_bits_to_float(static_cast<std::uint16_t>(bits));
    } else {
        for (int index = t; index < count; index += kQuantThreads)
            absmax = fmaxf(absmax, fabsf(half_bits_to_float(in[(index / d) * row_stride + index % d])));
        absmax = wave_max(absmax);
        if ((t & (kWave - 1)) == 0) partial[t / kWave] = absmax;
        __syncthreads();
        absmax = fmaxf(fmaxf(partial[0], partial[1]), fmaxf(partial[2], partial[3]));
    }
    const float scale = block_scale(absmax);
    const float recip = 1.0f / scale;  // used only when scale > 0
    if (t == 0) side.scales[head * side.blocks + block] = float_to_half_bits(scale);

    if constexpr (kPiece > 0) {
        if (scale > 0.0f) {
#pragma unroll
            for (int c = 0; c < kPieces; ++c) {
                const int index = t + c * kQuantThreads;
                if (index < pieces) {
                    int v[kPiece];
#pragma unroll
                    for (int e = 0; e < kPiece; e += 2) {
                        v[e] = quantize_half<0>(piece[c][e / 2], scale, recip);
                        v[e + 1] = quantize_half<1>(piece[c][e / 2], scale, recip);
                    }
                    typename Types::Bytes packed;
                    if constexpr (kPiece == 8) {
                        packed[0] = pack_bytes(v[0], v[1], v[2], v[3]);
                        packed[1] = pack_bytes(v[4], v[5], v[6], v[7]);
                    } else {
                        packed = pack_bytes(v[0], v[1], v[2], v[3]);
                    }
                    reinterpret_cast<typename Types::Bytes*>(out)[index] = packed;
                }
            }
        } else {
#pragma unroll
            for (int c = 0; c < kPieces; ++c) {
                const int index = t + c * kQuantThreads;
                if (index < pieces) reinterpret_cast<typename Types::Bytes*>(out)[index] = typename Types::Bytes{};
            }
        }
    } else {
        for (int index = t; index < count; index += kQuantThreads)
            out[index] = static_cast<std::int8_t>(
                quantize_value_recip(half_bits_to_float(in[(index / d) * row_stride + index % d]), scale, recip));
    }
}

bool aligned(const void* pointer, std::size_t bytes) {
    return (reinterpret_cast<std::uintptr_t>(pointer) % bytes) == 0;
}

// Whether the rows of a side move in pieces of `piece` elements: rows that are
// whole in them, at addresses that are multiples of a piece. With d % piece ==
// 0 every block's bytes start at a multiple of `piece` too.
bool takes_pieces(const QuantSide& side, int d, int piece) {
    return side.blocks == 0 || (d % piece == 0 && aligned(side.x, 2 * piece) && aligned(side.x8, piece) &&
                                side.in_head_stride % piece == 0 && side.in_row_stride % piece == 0);
}

template <int kPiece, int kPieces>
void launch_pieces(bool contiguous, bool heads_first, dim3 grid, hipStream_t stream, const QuantSide& q,
                   const QuantSide& k, int d) {
    if (contiguous)
        quantize_blocks_kernel<kPiece, true, kPieces><<<grid, kQuantThreads, 0, stream>>>(q, k, d, heads_first);
    else
        quantize_blocks_kernel<kPiece, false, kPieces><<<grid, kQuantThreads, 0, stream>>>(q, k, d, heads_first);
}

}  // namespace

hipError_t launch_quantize(const QuantSide& q, const QuantSide& k, int heads, int d,
                           hipStream_t stream) {
    const int blocks = q.blocks + k.blocks;
    if (blocks == 0) return hipSuccess;
    if (heads > 65535) return hipErrorInvalidConfiguration;
    bool contiguous = true;
    bool heads_first = d % kLineHalves == 0 && blocks <= 65535;
    int most_rows = 0;  // of a block of the launch
    for (const QuantSide* side : {&q, &k}) {
        if (side->blocks == 0) continue;
        contiguous = contiguous && side->in_row_stride == d;
        heads_first = heads_first && side->in_head_stride < side->in_row_stride &&
                      side->in_head_stride % kLineHalves == 0;
        most_rows = std::max(most_rows, side->block_rows);
    }
    // Workgroups that run together read memory that lies together: the blocks of
    // a head in turn, or where rows hold all heads ([rows, heads, d]) the heads
    // of a block: 64 heads x 4096 x 128 46.5 -> 41.1 us, 8 x 16384 x 128 20.1 ->
    // 19.7, 64 x 4096 x 64 20.9 both ways. Heads that share cache lines keep the
    // first order: 32 x 4096 x 100 17.3 us against 19.4.
    const dim3 grid(static_cast<unsigned>(heads_first ? heads : blocks),
                    static_cast<unsigned>(heads_first ? blocks : heads));
    // Registers for half of the largest block where that is enough.
    const bool small = most_rows * d <= kQuantMaxElements / 2;
    if (takes_pieces(q, d, 8) && takes_pieces(k, d, 8)) {
        if (small)
            launch_pieces<8, kQuantMaxElements / 2 / 8 / kQuantThreads>(contiguous, heads_first, grid, stream, q, k, d);
        else
            launch_pieces<8, kQuantMaxElements / 8 / kQuantThreads>(contiguous, heads_first, grid, stream, q, k, d);
    } else if (takes_pieces(q, d, 4) && takes_pieces(k, d, 4)) {
        if (small)
            launch_pieces<4, kQuantMaxElements / 2 / 4 / kQuantThreads>(contiguous, heads_first, grid, stream, q, k, d);
        else
            launch_pieces<4, kQuantMaxElements / 4 / kQuantThreads>(contiguous, heads_first, grid, stream, q, k, d);
    } else {
        quantize_blocks_kernel<0, false, 1><<<grid, kQuantThreads, 0, stream>>>(q, k, d, heads_first);
    }
    return hipGetLastError();
}

QuantSide make_quant_side(const std::uint16_t* x, std::int8_t* x8, std::uint16_t* scales,
                          std::int64_t head_stride, int rows, int block_rows, std::int64_t row_stride) {
    QuantSide side{};
    side.x = x;
    side.x8 = x8;
    side.scales = scales;
    side.in_head_stride = head_stride;
    side.in_row_stride = row_stride;
    side.rows = rows;
    side.block_rows = block_rows;
    side.blocks = x ? (rows - 1) / block_rows + 1 : 0;
    return side;
}

}  // namespace tilemix

extern "C" int tilemix_quantize_qk(const std::uint16_t* Q, const std::uint16_t* K, std::int8_t* Q8,
                                   std::int8_t* K8, std::uint16_t* q_scales, std::uint16_t* k_scales,
                                   int M, int N, int d, void* stream) {
    // Validation order of src/tilemix.cu:227-230.
    if (!Q || !K || !Q8 || !K8 || !q_scales || !k_scales || M <= 0 || N <= 0 || d <= 0)
        return hipErrorInvalidValue;
    if (d > tilemix::kMaxHeadDim) return hipErrorNotSupported;
    const auto q = tilemix::make_quant_side(Q, Q8, q_scales, 0, M, tilemix::kQBlockRows, d);
    const auto k = tilemix::make_quant_side(K, K8, k_scales, 0, N, tilemix::kKBlockRows, d);
    return tilemix::launch_quantize(q, k, 1, d, static_cast<hipStream_t>(stream));
}

extern "C" int tilemix_quantize_qk_strided(const std::uint16_t* Q, const std::uint16_t* K,
                                           std::int8_t* Q8, std::int8_t* K8,
                                           std::uint16_t* q_scales, std::uint16_t* k_scales,
                                           int heads, int M, int N, int d,
                                           std::int64_t q_head_stride, std::int64_t k_head_stride,
                                           std::int64_t q_row_stride, std::int64_t k_row_stride,
                                           void* stream) {
    const bool q_side = Q || Q8 || q_scales;
    const bool k_side = K || K8 || k_scales;
    if ((q_side && (!Q || !Q8 || !q_scales)) || (k_side && (!K || !K8 || !k_scales)) ||
        (!q_side && !k_side) || heads <= 0 || d <= 0 || (q_side && M <= 0) || (k_side && N <= 0))
        return hipErrorInvalidValue;
    const std::int64_t q_row = q_row_stride ? q_row_stride : d;
    const std::int64_t k_row = k_row_stride ? k_row_stride : d;
    if ((q_side && !tilemix::strided_heads_ok(heads, M, d, q_head_stride, q_row)) ||
        (k_side && !tilemix::strided_heads_ok(heads, N, d, k_head_stride, k_row)))
        return hipErrorInvalidValue;
    if (d > tilemix::kMaxHeadDim) return hipErrorNotSupported;
    const auto q = tilemix::make_quant_side(q_side ? Q : nullptr, Q8, q_scales, q_head_stride,
                                            q_side ? M : 1, tilemix::kQBlockRows, q_row);
    const auto k = tilemix::make_quant_side(k_side ? K : nullptr, K8, k_scales, k_head_stride,
                                            k_side ? N : 1, tilemix::kKBlockRows, k_row);
    return tilemix::launch_quantize(q, k, heads, d, static_cast<hipStream_t>(stream));
}

extern "C" int tilemix_quantize_qk_batched(const std::uint16_t* Q, const std::uint16_t* K,
                                           std::int8_t* Q8, std::int8_t* K8,
                                           std::uint16_t* q_scales, std::uint16_t* k_scales,
                                           int heads, int M, int N, int d,
                                           std::int64_t q_head_stride, std::int64_t k_head_stride,
                                           void* stream) {
    return tilemix_quantize_qk_strided(Q, K, Q8, K8, q_scales, k_scales, heads, M, N, d, q_head_stride,
                                       k_head_stride, 0, 0, stream);
}
