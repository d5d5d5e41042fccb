// How a prefill launch is cut, where it follows from sizes alone: host arithmetic.
#pragma once
#include <cstdint>

namespace dlb {

// Do the heads of a KV group share workgroups (SHARE kernels)?  Then 32-query blocks of all of them fill the workgroups,
// whose waves see the same keys; but where every workgroup finds a place at once, those that finish early help their
// neighbours when each has one head, and lose that.  So from 1.35 rounds of workgroups on, packed, and 0.95 over
// histories, whose unequal lengths leave more to even out.  Counted are the workgroups that have rows (the tokens / 128, and
// half a row tile per sequence), not those that would have if all sequences were as long as the longest.  A CU holds
// one with more than 128 dims (128 KB of LDS), two with more than 64, four with up to 64, of which histories leave three
// (140 registers).  tokens 0: not known; the other sequences count as 0.6 of the longest.
// us, a head each / shared: 32 heads (8 kv) of 128, 8 x 512 - 4096 tokens 284 / 275, 16 x up to 700 (3.6 rounds) 55 / 51;
// 28 (4), 8 x 300 - 1000 over 2000 110 / 99; 28 (4) of 256, 8 x 1024 (7.4) 215 / 201, 64 (8) of 256, 16 x up to 660 (10.7)
// 202 / 169.  One long prompt among fifteen of 60 - 250: 8 (1) of 128, 4000 (0.9) 63.2 / 64.7, 2000 and 1500 (0.8) 35.2 /
// 36.8; 16 (4) of 128, 4000 (1.8) 82.8 / 82.8; 28 (4), 4000 (3.1) 133.5 / 128.6.
// Over histories, where new tokens per sequence differ too (less than 0.85 of the longest on average), the order in which
// workgroups find places decides by more than sharing gives, and it has to be 2.1 rounds, or three as if all were as
// long as the longest (and 1.3 with more than 128 dims: 16 (4) of 256, 1000 tokens among fifteen of up to 60, 1.2 rounds,
// 215 / 236): 32 (8) of 128, 8 x 300 - 600 over up to 4096, each step on other caches, ten batches of 1.9 - 2.1
// rounds 0.91 - 1.03 (197 / 202, 189 / 191, 240 / 222); 18 of up to 106 over up to 440 (1.1) 29.0 / 30.9; but 8 x 512 over
// up to 4096 (2.0) 222 / 219, and none of 90 batches of equal lengths more than 0.3 % slower.
// 480 random batches over histories: 2.7 % less than a head each on average, one of them more than 1 % slower (1.8 %).
inline bool heads_share_workgroups(bool paged, int D, int64_t B, int64_t heads, int64_t max_len, int64_t tokens, int64_t cus) {
  const double longest = (double)((max_len + 127) / 128), all = longest * (double)B;
  double tiles = tokens > 0 ? (double)tokens / 128.0 + 0.5 * (double)B : longest * (0.4 + 0.6 * (double)B);
  if (tiles > all) tiles = all;
  const int64_t per_cu = D > 128 ? 1 : D > 64 ? 2 : paged ? 3 : 4;
  const double round = (double)(cus * per_cu) / (double)heads;  // (of row tiles)
  if (!paged) return tiles > 1.35 * round;
  const bool alike = (double)tokens >= 0.85 * (double)B * (double)max_len;
  if (alike) return tiles > 0.95 * round;
  return tiles > (D > 128 ? 1.3 : 0.95) * round && (tiles > 2.1 * round || all > 3.0 * round);
}

}  // namespace dlb
