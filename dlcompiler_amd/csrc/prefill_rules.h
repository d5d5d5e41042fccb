// How a prefill launch is cut, where it follows from sizes alone: host arithmetic.
#pragma once
#include <cstdint>

namespace dlb {

// Do the heads of a KV group share workgroups (SHARE kernels)?  Then 32-query blocks of all of them fill the workgroups,
// whose waves see the same keys; but where every workgroup finds a place at once, those that finish early help their
// neighbours when each has one head, and lose that.  So from 1.35 rounds of workgroups on, packed, and 0.95 (1.3 with more
// than 128 dims) over histories, whose unequal lengths leave more to even out.  Counted are the workgroups that have
// rows (the tokens / 128, and half a row tile per sequence), not those that would have if all sequences were as long
// as the longest.  A CU holds one with more than 128 dims (128 KB of LDS), two with more than 64, four with up to 64, of
// which histories leave three (140 registers).  tokens 0: not known; the other sequences count as 0.6 of the longest.
// us, a head each / shared: 32 heads (8 kv) of 128, 8 x 512 - 4096 tokens 284 / 275, 16 x up to 700 (3.6 rounds) 55 / 51;
// 28 (4), 8 x 300 - 1000 over 2000 110 / 99; 28 (4) of 256, 8 x 1024 (7.4) 215 / 201, 64 (8) of 256, 16 x up to 660 (10.7)
// 202 / 169.  One long prompt among fifteen of 60 - 250: 8 (1) of 128, 4000 (0.9) 63.2 / 64.7, 2000 and 1500 (0.8) 35.2 /
// 36.8; 16 (4) of 128, 4000 (1.8) 82.8 / 82.8; 28 (4), 4000 (3.1) 133.5 / 128.6.  1000 tokens among fifteen of up to 60,
// over histories: 32 (8) of 64 (0.8) 78.8 / 86.4, 16 (4) of 256 (1.2) 215 / 236.  420 random batches, packed and paged, 64
// to 256 dims: 2.4 % less on average, two slower by more than 1 %, 1.5 at most; counted by the longest 1.4 %, five and 5 %.
inline bool heads_share_workgroups(bool paged, int D, int64_t B, int64_t heads, int64_t max_len, int64_t tokens, int64_t cus) {
  const double longest = (double)((max_len + 127) / 128), all = longest * (double)B;
  double tiles = tokens > 0 ? (double)tokens / 128.0 + 0.5 * (double)B : longest * (0.4 + 0.6 * (double)B);
  if (tiles > all) tiles = all;
  const int64_t per_cu = D > 128 ? 1 : D > 64 ? 2 : paged ? 3 : 4;
  const double rounds = !paged ? 1.35 : D > 128 ? 1.3 : 0.95;
  return (double)heads * tiles > rounds * (double)(cus * per_cu);
}

}  // namespace dlb
