// Which form of the streaming MoE GEMM a launch takes: host arithmetic on sizes alone.
#pragma once
#include <cmath>
#include <cstdint>

namespace dlb {

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

// fp8, up to kSmallMeanRows rows per expert: where the activations and the intermediate are quantised.
//   kInSteps    activations by every wave in every step of its main loop, the intermediate by gate_up's epilogue, whose
//               column tiles are whole quantisation groups
//   kAhead      activations once per workgroup before its main loop
//   kHandedOver ... and gate_up leaves the intermediate in fp32, which the down GEMM quantises in that way: gate_up's
//               tiles have 32 columns then
// What counts is how many of gate_up's 128-column tiles have rows.  With fewer than every other CU one, the shorter tiles
// use the CUs that these leave idle.  With more, up to one for each, nothing helps; and with up to 1.4 for each, some
// CUs have twice the weights of others and short tiles even that out, if rows are long enough that their start does
// not cost more.  us a layer, 64 experts of 2048 x 1408, 6 per token: 1 token (66 tiles) 28.6 / 27.0 / 25.3, 2 (126)
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
    const bool idle = busy <= 0.48 * cus || (long_rows && 2 * groups * up.most_experts() <= up.cus);
    const bool uneven = long_rows && busy >= 0.98 * cus && busy <= 1.4 * cus && 2 * up.slots <= 3 * up.experts;
    if (idle || uneven) return FewRows::kHandedOver;
  }
  // (64 experts of 2048 x 1408, 64 tokens, six rows: 98.4 / 98.9; 8 of 4096 x 4096, 20 tokens, 256 tiles: 76.4 / 80.5)
  return busy >= cus && 2 * up.slots <= 5 * up.experts ? FewRows::kAhead : FewRows::kInSteps;
}

}  // namespace dlb
