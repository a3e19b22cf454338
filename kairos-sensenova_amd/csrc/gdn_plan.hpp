// How many parts the fixed-length K = 256 forward runs in.  Plain C++.
#pragma once

#include <stdint.h>

namespace kgdn {

struct PipePlan {
  int parts;
  double growth;              // each part's length over the one's before it
};

// nt chunks of each of seq_heads (sequence, head) pairs whose recurrence takes vtiles workgroups of a CU each.
// A part boundary costs the caller's stream about 16 us of waits, and what it hides is the prepare of the later
// parts (about 0.05 us per (chunk, head) on all CUs), so short calls run in one part.  So do calls whose
// recurrence leaves the prepare no room: less than a quarter of the CUs, or with more workgroups than CUs
// less than three tenths over its rounds.  Measured in us at V = 512 (256 CUs), one part / two / four growing
// by 1.4:
//   20 heads: 25 chunks 99 and four 188; 64 225 / 238 / 294; 128 434 / 434 / 475; 256 849 / 795 / 808; 512 1667 / 1543
//   / 1499; 24: 512 1767 / 1725 / 1710; 28: 128 490 / 509 / 563, 256 955 / 963 / 1012; 32: 256 1031 / 1058 / 1106;
//   36: 256 1624 / 1535 / 1522; 40: 128 860 / 826 / 852, 512 3456 / 3217 / 3083; 48: 256 1821 / 1982 / 2048;
//   60: 128 997 / 1126 / 1201, 256 1994 / 2207 / 2327; 80: 128 1396 / 1477 / 1531.
// Where the recurrence takes at most half of the CUs the later prepares run on the others several times faster
// than it walks, so the first part can be small: two parts growing by 3 (10 heads, 128 chunks 379 in one part,
// 372; 512 1443, 1353, four by 1.4 1371; 5 heads, 512 chunks 1347, 1306, 1343; V = 256, 20 heads, 64
// chunks 204, 223, 128 chunks 450, 431), as long as the second part's prepare, three times the first's chunks at
// 0.05 us a (chunk, head) on all CUs (0.08 with `conv`, where it convolves too) ends within about twice the first
// part's recurrence of 2.3 us a chunk (V = 256, 32 heads, 512 chunks 1795, by 1.4 in four 1649; with the
// convolution 16 heads, 375 chunks 1399, 1296, 188 chunks 756, in two by 1.4 704).  With one or two value
// tiles a head little of what prepare wrote is read ahead of the steps, and four parts by 1.4 keep more of it in
// the last cache (V = 64, 5 heads, 512 chunks: one part 1699, two by 3 1657, four 1459; 10 heads, 256 chunks
// 980 / 938 / 833; V = 128, 20 heads, 128 chunks 538 / 494 / 474; with 1280 items one part is best, 20
// heads of 64 chunks 196 / 210 / 229); two below 64 chunks a value tile (V = 128, 40 heads, 64 chunks 346 in
// one, two by 1.4 330, four 353).
// `norm`: the gated norm runs by parts too, the last part's after everything else, so a smaller last part pays
// earlier (20 heads, with the norm: 188 chunks 748 in two parts, 743 in four; 256 989 / 963; 375 1436 / 1381; two
// sequences of 128 979 / 993).
constexpr PipePlan wide_pipe_plan(int64_t nt, int64_t seq_heads, int64_t vtiles, int64_t cus, bool norm, bool conv) {
  const int64_t items = nt * seq_heads, units = seq_heads * vtiles, slots = (units + cus - 1) / cus * cus;
  if (units <= cus ? 4 * (cus - units) < cus : 10 * (slots - units) < 3 * slots) return {1, 1.0};
  if (2 * units <= cus) {
    if (vtiles <= 2 && items >= 2048) return {nt >= 64 * vtiles ? 4 : 2, 1.4};
    const int two = items >= 1280 && nt >= 128 ? 2 : 1;
    if (3 * seq_heads * (conv ? 8 : 5) * cus < 2 * 230 * (cus - units)) return {two, 3.0};
    return {items >= (norm || conv ? 3584 : 8192) ? 4 : two, 1.4};
  }
  return {items >= (norm && units <= cus ? 4096 : 8192) ? 4 : items >= 3072 ? 2 : 1, 1.4};
}

}  // namespace kgdn
