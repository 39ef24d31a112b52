#pragma once
// Which kernel takes an attention call: rules on its sizes and the device's
// compute units, host code only (tests/native/launch_rules.cpp runs them on
// the CPU).

#include "attention_common.h"

#include <algorithm>
#include <cstdint>

namespace tilemix {

inline constexpr int kRowsPerGroup = 128;  // rows of a prefill workgroup: one Q quantization block
#ifndef TILEMIX_GROUPS_PER_CU
#define TILEMIX_GROUPS_PER_CU 2
#endif
// Workgroups per CU that attention_kernel's register allocation is sized for (launch bound).
inline constexpr int kGroupsPerCU = TILEMIX_GROUPS_PER_CU;
inline constexpr int kWideMaxTiles = 1024;  // key tiles that attention_wide_kernel's table holds

// Whether the wide kernel is the faster one for a launch that it can take
// (whole 16-byte pieces, head dimensions 33 .. 64 and 97 .. 128, fast P.V, no
// split, no verification outputs). It halves the tile loads and keeps the
// matrix cores and exponentials of a CU's two halves apart, but has one
// workgroup per CU, whose prologue and epilogue nothing overlaps: it needs long
// walks (a causal one ends at the head's last row), heads of more than one
// 128-row block, and whole rounds of workgroups, no more of them than the
// 128-row kernel takes (an odd block's empty half costs a round where the
// 128-row kernel fills that place with another block). Rows of a reversed round
// keep the direction that the 128-row kernel gives them (even number of row
// blocks).
// 128-row kernel | wide kernel (us), 64 features: 64 heads x 2048 101.3 | 96.9;
// 32 x 2048 routed 53.3 | 51.1; 64 x 4096 causal 180.3 | 175.9; 16 x 2048 37.5 |
// 39.6; 64 x 1024 25.8 | 26.2. 128 features: 32 x 16384 routed 3551 | 3363; 32 x
// 8192 three-way 787 | 755; 32 x 8192 dense 1064 | 1033, causal 530 | 517; 64 x
// 4096 causal dense 288.4 | 284.5, routed in a band with the K quantizer 311.1 |
// 310.8 on one box and 306.2 | 300.9 on another; 16 x 4096 causal 106.3 | 108.2; 48 x 3000 (2.25
// rounds) 258.4 | 263.5; 64 x 1024 46.8 | 48.0; 16 x 2048 48.6 | 53.5. Precise
// P.V, whose matrix slot is twice as long: 32 x 4096 causal 203.8 | 207.2.
// Rows x 4096 keys x 128 features: 256 heads x 129 136.7 | 128.5; 256 x 300 247.8
// | 224.3 (1.5 rounds against two); 512 x 384 446.5 | 498.1 (three against four).
// One block a head: 512 x 128 187.4 | 225.4, 252 x 128 127 | 144, 256 x 128 125 |
// 114, 256 x 64 x 2048 routed 59.8 | 71.8, 232 x 128 x 3000 x 64 59.0 | 63.1, 256
// x 128 x 2048 x 64 39.5 | 35.7: no rule on sizes alone separates them. Causal
// walks of 16 tiles, 256 x 1024 x 64 over 4096 keys: 65.7 | 73.0; of 32, 128 x
// 2048 x 64 routed 111.3 | 114.7, x 128 173 | 167. Causal with skipped tiles
// (three-way), which its waves wait for one another over: 64 x 4096 x 64 172.4 |
// 176.8, 128 x 2048 x 64 102.8 | 110.6, x 128 157.6 | 157.9.
inline bool wide_pays(const AttnParams& p, int compute_units) {
    const int long_walk = p.causal && p.d <= 64 ? 64 : 32;  // key tiles
    const int tiles = (p.N - 1) / kTileKeys + 1;
    const int walk = p.causal ? std::min<std::int64_t>(tiles, std::int64_t{kRowsPerGroup / kTileKeys} * p.q_blocks) : tiles;
    if (compute_units <= 0 || walk < long_walk || tiles > kWideMaxTiles) return false;
    if (p.q_blocks < 2 || (p.reverse_slots > 0 && p.q_blocks % 2 != 0)) return false;
    const std::int64_t workgroups = static_cast<std::int64_t>(p.heads) * ((p.q_blocks + 1) / 2);
    if (p.causal) return workgroups >= 2 * static_cast<std::int64_t>(compute_units) && !(p.skip_words && p.d <= 64);
    // Whole rounds: at most a tenth of the last one empty.
    const std::int64_t rounds = (workgroups + compute_units - 1) / compute_units;
    const std::int64_t slots = std::int64_t{kGroupsPerCU} * compute_units;
    const std::int64_t narrow_rounds = (static_cast<std::int64_t>(p.heads) * p.q_blocks + slots - 1) / slots;
    return rounds <= narrow_rounds && 10 * workgroups >= 9 * rounds * compute_units;
}

// Whether the decode kernel is the faster one for a call that it can take. It
// has one workgroup of eight waves per CU (four from 512 heads on), so past one
// head per CU a second round begins; with rows of more than 128 bytes the
// prefill kernel, whose tile loads take whole KiB by each wave and which runs
// two heads per CU, is then the faster one if they move in pieces at all.
// Decode | prefill (us, 4 rows a head): 256 heads x 2048 x 128 56.7 | 72.5; 260
// 78.9 | 70.3; 300 82.4 | 72.3, half INT8 75.6 | 72.7; 480 111 | 91, half INT8 96 |
// 82; 480 x 8192 424 | 342; 300 x 2048 x 100 130 | 90; 1000 x 1024 x 72 76 | 67;
// rows at 4-byte addresses, 300 x 2048 x 128 188 | 100. Up to 64 features: 300 x
// 2048 x 64 36.9 | 50.5, 1000 81 | 106; element by element: 300 x 1000 x 102 151 |
// 370.
inline bool decode_worthwhile(const AttnParams& p, int compute_units) {
    return compute_units <= 0 || p.heads <= compute_units || p.d <= 64 || access_piece(p) == 0;
}

}  // namespace tilemix
