// Host-only program over the rules that the launches of the HIP library follow
// (csrc/attention_common.h): the edges of the addressing, restated here from
// single bytes. Prints one line per failure; exit status 1 if there was one.

#include "attention_common.h"

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

}  // namespace

int main() {
    k8_pieces_stay_inside_the_head();
    if (failures == 0) std::printf("launch rules OK\n");
    return failures != 0;
}
