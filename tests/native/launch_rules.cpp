// Host-only program over the rules that the launches of the HIP library follow
// (csrc/attention_common.h, csrc/attention_rules.h): the edges of the addressing,
// restated here from single bytes, and calls on both sides of the dispatch rules
// for a device of 256 compute units. Prints one line per failure; exit status 1 if there was one.

#include "attention_common.h"
#include "attention_rules.h"

#include <cstdio>

namespace {

int failures = 0;

// A K8 row's last 16-byte piece, for every row that a whole tile moves in
// pieces: its end lies inside the head's N * d bytes.
void k8_pieces_stay_inside_the_head() {
    using namespace tilemix;
    for (int d = 4; d <= 128; d += 4) {
        for (int N = 1; N <= 4 * kTileKeys; ++N) {
            for (int k0 = 0; k0 < N; k0 += kTileKeys) {
                bool passes = false;
                for (int row = k0; row < k0 + kTileKeys && row < N; ++row)
                    for (int piece = 0; piece < d; piece += 16) passes = passes || row * d + piece + 16 > N * d;
                if (passes != k8_pieces_pass_end(k0, N, d)) {
                    std::printf("k8_pieces_pass_end(%d, %d, %d) is not %d\n", k0, N, d, passes);
                    ++failures;
                }
                // What the kernel assumed before: only the tile with the head's last row can.
                if (passes && k0 + kTileKeys < N && d != 4) {
                    std::printf("d = %d, N = %d: tile %d passes the end too\n", d, N, k0 / kTileKeys);
                    ++failures;
                }
            }
        }
    }
}

tilemix::AttnParams call(int heads, int M, int N, int d, bool causal) {
    tilemix::AttnParams p{};
    p.heads = heads;
    p.M = M;
    p.N = N;
    p.d = d;
    p.causal = causal;
    p.q_blocks = (M - 1) / tilemix::kRowsPerGroup + 1;
    return p;
}

// The 256-row kernel: never for heads of one 128-row block, never in more
// rounds of workgroups than the 128-row kernel's, never for a causal walk of
// fewer than 32 tiles (64 at 64 features) however many keys there are; and the
// measured calls on both sides of the line.
void wide_kernel_rule() {
    using namespace tilemix;
    constexpr int kUnits = 256;
    auto expect = [](int heads, int M, int N, int d, bool causal, bool wide) {
        if (wide_pays(call(heads, M, N, d, causal), kUnits) == wide) return;
        std::printf("wide_pays(%d heads x %d x %d x %d, causal %d) is not %d\n", heads, M, N, d, causal, wide);
        ++failures;
    };
    for (int heads = 1; heads <= 2048; ++heads)
        for (int M : {1, 16, 64, 128, 129, 256, 300, 384, 640, 1152}) {
            const bool wide = wide_pays(call(heads, M, 4096, 128, false), kUnits);
            const int blocks = (M + 127) / 128;
            const int wide_rounds = (heads * ((blocks + 1) / 2) + kUnits - 1) / kUnits;
            const int rounds = (heads * blocks + 2 * kUnits - 1) / (2 * kUnits);
            if (wide && (blocks == 1 || wide_rounds > rounds)) expect(heads, M, 4096, 128, false, false);
            if (M < 1920) expect(heads, M, 8192, 128, true, false);
        }
    expect(64, 2048, 2048, 64, false, true);
    expect(32, 16384, 16384, 128, false, true);
    expect(64, 4096, 4096, 128, true, true);
    expect(64, 4096, 2048, 128, true, true);
    expect(256, 300, 4096, 128, false, true);
    expect(256, 129, 4096, 128, false, true);
    expect(512, 384, 4096, 128, false, false);
    expect(16, 2048, 2048, 64, false, false);
    expect(48, 3000, 3000, 128, false, false);
    expect(64, 1024, 1024, 128, false, false);
    expect(16, 4096, 4096, 128, true, false);
    expect(64, 4096, 4096, 64, true, true);
    expect(128, 2048, 2048, 64, true, false);
    expect(128, 2048, 2048, 128, true, true);
    // A causal call with skipped tiles keeps the 128-row kernel up to 64 features.
    const std::uint64_t words = 0;
    for (int d : {40, 64, 112, 128}) {
        AttnParams p = call(64, 4096, 4096, d, true);
        p.skip_words = &words;
        if (wide_pays(p, kUnits) != (d > 64)) {
            std::printf("wide_pays(causal with skipped tiles, d %d) is not %d\n", d, d > 64);
            ++failures;
        }
    }
}

// The decode kernel: up to one head per CU, and beyond that for rows of at most
// 128 bytes or rows that only single elements can read.
void decode_rule() {
    using namespace tilemix;
    auto expect = [](int heads, int d, std::int64_t k_row, bool decode) {
        AttnParams p = call(heads, 4, 2048, d, false);
        p.q_row = p.v_row = d;
        p.k_row = k_row;
        p.q_stride = 4 * d;
        p.k_stride = 2048 * k_row;
        p.v_stride = 2048 * d;
        if (decode_worthwhile(p, 256) == decode) return;
        std::printf("decode_worthwhile(%d heads, d %d, row %d) is not %d\n", heads, d, static_cast<int>(k_row), decode);
        ++failures;
    };
    for (int d : {128, 112, 100, 72}) {
        expect(1, d, d, true);
        expect(256, d, d, true);
        expect(257, d, d, false);
        expect(511, d, d, false);
        expect(2000, d, d, false);
        expect(300, d, d + 2, false);
        expect(300, d, d + 1, true);
    }
    for (int d : {64, 40, 33}) expect(300, d, d, true);
    for (int d : {65, 102}) expect(1000, d, d, true);
}

}  // namespace

int main() {
    wide_kernel_rule();
    decode_rule();
    k8_pieces_stay_inside_the_head();
    if (failures == 0) std::printf("launch rules OK\n");
    return failures != 0;
}
