// Which form of the streaming MoE GEMM a launch takes: host arithmetic on sizes alone.
#pragma once
#include <cmath>
#include <cstdint>

namespace dlb {

// Up to this many rows per expert, on average over the routed slots, the streaming kernel runs tiles of 16 rows.
constexpr int kSmallMeanRows = 7;

// Sizes of one grouped GEMM.  (Not the routing, which the host does not know: where a rule needs the experts or the row
// tiles that have rows, it takes them for a routing that spreads the tokens evenly.)
struct MoeLaunch {
  bool gated;
  int64_t slots, tokens, topk, experts, local;  // routed slots; experts: all, and those whose weights are here
  int64_t columns, row_bytes;                   // output columns (gated: I), bytes per row of the reduction
  int64_t cus;
  bool mean_up_to(int64_t rows) const { return slots <= rows * experts; }  // rows per expert, on average
  // experts that can have a row at most, and how many of them do
  int64_t most_experts() const { return slots < local ? slots : local; }
  double hit_experts() const {
    const double miss = topk < experts ? 1.0 - (double)topk / (double)experts : 0.0;
    return (double)local * (1.0 - std::pow(miss, (double)tokens));
  }
};

// 16 bit, side by side.  down: tiles of up to 128 rows, which store whole rows, take over from those of 32 at once
// (64-row tiles / 128-row ones, in both layouts alike: 128 experts of 2048 x 768, 28 rows 219.4 / 211.7 us; 64 of 3072 x
// 2048, 28 rows 411 / 390; 64 of 4096 x 1024, 28 rows 275.5 / 270.7; 64 of 2048 x 1408 188.9 / 188.3; 21 rows 183.9 /
// 183.6; 32-row ones there 199 / 185).  gate_up, which writes half as much: 64-row tiles, with two chunks of activations
// on their way, up to 36 rows (64-row / 128-row: 64 of 2048 x 1408, 28 rows 188.3 / 191.2, 37 rows 194.1 / 195.8, 43 rows
// 197.9 / 197.6; 64 of 1024 x 1408, 28 rows 105.6 / 109.9; 128 of 1536 x 512, 28 rows 120.6 / 122.2; 128 of 2048 x 768,
// 36 rows 217.3 / 216.3; 64 of 3072 x 2048, 28 rows 390.2 / 390.1, 37 rows 402.9 / 397.8).
// A launch of few column tiles (few experts, or a rank's share of them) is bound by the CUs that it leaves idle, and by
// those that get one workgroup more than the others.  Where four waves side by side give more workgroups than every other
// CU but fewer than one each, splitting K gives most CUs two of half the size, which is no less for the busiest, and the
// partial sums on top (layer, split / side by side: 16 experts of 2176 x 1536, 192 and 144 tiles, 25 rows 83.0 / 78.0 us,
// 50 rows, then of 128, 90.3 / 82.5; 32 of 2048 x 768, 192 and 256, 37 rows 76.2 / 69.0; but gate_up of 8 of 4096 x 2048,
// 128 tiles, 25 rows 78.7 / 91.1, and of 8 of 4096 x 4096, 256 tiles, 141.4 / 150.6).  The down GEMM's tall tiles, which
// store whole rows, pay up to twice as many (32 of 2816 x 704, 352 tiles, 22 rows 95.4 / 85.9; gate_up, 384 tiles, 128 of
// 1792 x 384, 40 rows 116.9 / 122.3).
// With fewer tiles the shape is the first in this order that has a workgroup for somewhat more than every other CU: 128
// rows, 64 side by side, 64 with K split in two, 32, 16 with K split in four, which has to fit the CUs once.  us of a
// layer with gate_up in each:
//                                                     128    64   64/2  32/2  16/4
//   8 of 2816 x 896, 4 of them here (28 tiles)  15 rows                 37.0  29.8
//                                               32             42.6  40.6  37.4
//                                               63      68.8  65.5  49.7  45.5  45.6
//                                              125      79.9  68.6  53.2  48.8  64.7
//   8 of 2048 x 1024 (64 tiles)                 32             39.7  38.7  44.1
//                                               64      61.1  56.2  46.0  53.0  59.6
//                                              128      71.3  60.2  62.4  66.9  83.6
//   16 of 2048 x 1408, 8 here (88 tiles)       125      79.9  68.9  72.7  88.8
//   16 of 1024 x 512, 4 here (16 tiles)         25             27.8  26.6  23.2
//                                               75      39.4  38.1  32.8  30.2  30.1
// (4000 tokens through the last, 1000 rows: 133 workgroups of 128 rows 53.8 us, 258 of 64, one CU with two, 58.8.)
// Three more things count (us of a layer with one GEMM in each shape, other weights at each step).
// Above 52 rows, gate_up, 62 to 84 rows, with K split in two: half of the experts have a second tile of 64 rows, and where
// some CUs get two such workgroups that way and none gets two of 32 rows side by side, those are faster (128 / 64 / 64 in
// two / 32 side by side: 16 experts of 3840 x 640, 66 rows 86.9 / 84.0 / 85.7 / 79.8; 16 of 1280 x 1408, 8 of them here, 72
// rows 60.3 / 56.4 / 60.3 / 54.1; but 8 of 2048 x 2816, 4 here, 72 rows 87.0 / 81.5 / 86.9 / 90.2).
// down, up to 76 rows, where 64-row tiles would have one for most CUs: few experts have a second one, and a tall tile reads
// the weights once (128 / 64 rows, 53 - 76 rows per expert: K from 1280 on 0.975 on average, of 768 and less 1.00; 78 - 120
// rows 1.01 - 1.06; 16 of 1792 x 1280, 68 rows 65.5 / 73.5; but 16 of 3584 x 2688, 8 here, 75 rows 114.6 / 113.7).
// 35 to 44 rows, where 32-row tiles have second ones and 64-row ones do not: 64 in two from 0.55 of the CUs on (64 / 32 in
// two: 16 of 1024 x 1280, 8 here, 42 rows 41.0 / 44.7; down, 16 of 1280 x 1792, 36 rows 55.5 / 60.6; but 30 rows 48.0 / 46.8,
// 48 rows 62.0 / 57.3 and 84.9 / 81.8).
// Of 900 GEMMs (7 to 330 rows, few column tiles, half of them where the three apply) four are more than 1 % slower than
// without them, one of them 11 %, 2.1 % and 1.3 % less on average where they apply (gate_up, down).
struct StreamShape { int cw, nt; };  // (four waves, cw of them side by side; rows 16 nt)
inline StreamShape stream_shape_16bit(const MoeLaunch& p) {
  const int64_t wave_columns = p.gated ? 32 : 64, experts = p.most_experts(), cus = p.cus;
  const auto column_tiles = [&](int cw) { return (p.columns + cw * wave_columns - 1) / (cw * wave_columns) * experts; };
  const int64_t tiles = column_tiles(4);
  // Workgroups with rows: on average an expert's last row tile is half full, and an expert of
  // up to three quarters of a tile seldom has a second one.
  const auto blocks = [&](int cw, int nt) {
    const double full = (double)p.slots / ((double)p.experts * 16 * nt);
    return (double)column_tiles(cw) * (full <= 0.75 ? 1.0 : full + 0.5);
  };
  const bool one_round = 2 * tiles > cus && 10 * tiles <= 9 * cus, beside = tiles >= 2 * cus;
  if (p.mean_up_to(kSmallMeanRows)) return {beside ? 4 : 1, 1};
  if (one_round || beside) {
    if (p.mean_up_to(19)) return {4, 2};
    return {4, p.gated && p.mean_up_to(36) ? 4 : 8};
  }
  if (!p.mean_up_to(52) && (2 * tiles >= cus || blocks(4, 4) > cus)) return {4, 8};
  if (!p.mean_up_to(22)) {
    if (!p.gated && tiles > cus / 2) return {4, 8};
    if (!p.mean_up_to(52)) {
      const bool tall = blocks(4, 4) >= 0.55 * cus;
      if (p.gated && !p.mean_up_to(62) && p.mean_up_to(84) && blocks(2, 4) > 0.95 * cus && blocks(4, 2) <= 0.95 * cus)
        return {4, 2};
      if (tall) return {4, !p.gated && p.row_bytes >= 2560 && p.mean_up_to(76) ? 8 : 4};
    }
    if (blocks(2, 4) >= (!p.mean_up_to(34) && p.mean_up_to(44) ? 0.55 : 0.65) * cus) return {2, 4};
  }
  if (blocks(2, 2) >= 0.55 * cus || blocks(1, 1) > 1.1 * cus) return {2, 2};
  return {1, 1};
}

// fp8, up to kSmallMeanRows rows per expert: where the activations and the intermediate are quantised.
//   kInSteps    activations by every wave in every step of its main loop, the intermediate by gate_up's epilogue, whose
//               column tiles are whole quantisation groups
//   kAhead      activations once per workgroup before its main loop
//   kHandedOver ... and gate_up leaves the intermediate in fp32, which the down GEMM quantises in that way: gate_up's
//               tiles have 32 columns then
// What counts is how many of gate_up's 128-column tiles have rows.  With fewer than every other CU one, the shorter tiles
// use the CUs that these leave idle.  With more, up to one for each, nothing helps; and with up to 1.4 for each, some
// CUs have twice the weights of others and short tiles even that out, if rows are long enough that their start does
// not cost more.  (Short rows, fewer than 0.45 of the CUs: 16 experts of 1152 x 1664, 4 per token, 3 tokens (120) 20.2 / 20.7 /
// 21.9; 64 of 1152 x 256, 8 per token, 18 tokens (116) 22.8 / 23.1 / 25.0; 16 of 1408 x 896, 24 tokens (112) 0.95 of
// kInSteps.)  us a layer, 64 experts of 2048 x 1408, 6 per token: 1 token (66 tiles) 28.6 / 27.0 / 25.3, 2 (126)
// 33.9 / 32.4 / 31.5, 4 (230) 44.1 / 44.9 / 46.2, 8 (386) 63.5 / 60.7 / 65.7; 128 of 1152 x 512, 8 per token: 10 tokens
// (243) 34.3 / 34.5 / 40.9, 14 (305) 43.9 / 41.3 / 43.8, 23 (396) 48.3 / 45.9 / 51.8; 64 of 4096 x 1024, 8 per token:
// 6 tokens (282) 100.6 / 99.3 / 88.6, 8 (336) 103.9 / 103.2 / 95.9, 16 (452) 125.8 / 124.4 / 126.4; 32 of 1536 x 1280, 4
// per token: 8 tokens (210) 34.4 / 34.1 / 38.1, 12 (255) 44.5 / 42.4 / 42.3; 64 of 1536 x 768, 8 per token, one half of
// 128: 16 tokens (247) 38.8 / 39.0 / 44.5.  Of 694 sizes in both weight layouts the choice is up to 1.5 % above kInSteps,
// 10 % below it on average and 0.7 % above the best.  (Counting the tiles that could have rows at most: up to 22 %.)
enum class FewRows { kInSteps, kAhead, kHandedOver };
inline FewRows fp8_few_rows(const MoeLaunch& up) {
  if (up.row_bytes > 4096) return FewRows::kInSteps;  // (rows in fp8 have to fit LDS)
  const int64_t groups = (up.columns + 127) / 128;
  const double busy = (double)groups * up.hit_experts(), cus = (double)up.cus;
  const bool long_rows = up.row_bytes >= 1536;
  if (up.columns <= 4096) {
    const bool idle = busy <= (long_rows ? 0.48 : 0.45) * cus || (long_rows && 2 * groups * up.most_experts() <= up.cus);
    const bool uneven = long_rows && busy >= 0.98 * cus && busy <= 1.4 * cus && 2 * up.slots <= 3 * up.experts;
    if (idle || uneven) return FewRows::kHandedOver;
  }
  // (64 experts of 2048 x 1408, 64 tokens, six rows: 98.4 / 98.9; 8 of 4096 x 4096, 20 tokens, 256 tiles: 76.4 / 80.5)
  return busy >= cus && 2 * up.slots <= 5 * up.experts ? FewRows::kAhead : FewRows::kInSteps;
}

}  // namespace dlb
