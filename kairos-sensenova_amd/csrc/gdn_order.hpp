// Which (sequence, head, column slice) a workgroup takes, in the kernels whose slices of a head read the
// same operands.  Host and device, without HIP headers.
#pragma once

namespace kgdn {

constexpr int kXcds = 8;          // workgroup b runs on XCD b % 8; workgroups start in order of b

struct WgUnit {
  int seq, head, slice;
  bool ok;                        // false: a workgroup without work (the grid is rounded up)
};

constexpr int div_up(int a, int b) { return (a + b - 1) / b; }

// Whole heads to an XCD: head u = seq H + head runs on XCD u % 8, its slices one after another.  Its
// operands then come into one L2 once, each sequence is spread over all XCDs, and so are the sequences of
// a batch of few heads.
// Otherwise the slices of each sequence are laid over the XCDs in equal runs, successive sequences from
// successive XCDs on; a head may then lie on two XCDs.
constexpr int unit_grid(int n_seqs, int H, int slices, bool whole) {
  return whole ? kXcds * div_up(n_seqs * H, kXcds) * slices : kXcds * n_seqs * div_up(H * slices, kXcds);
}

constexpr WgUnit unit_of(unsigned block, unsigned n_seqs, unsigned H, unsigned slices, bool whole) {
  const unsigned xcd = block % kXcds, j = block / kXcds;
  if (whole) {
    const unsigned u = j / slices * kXcds + xcd, seq = u / H;
    return {(int)seq, (int)(u - seq * H), (int)(j % slices), seq < n_seqs};
  }
  const unsigned run = (H * slices + kXcds - 1) / kXcds, seq = j / run;
  const unsigned i = (xcd + seq) % kXcds * run + (j - seq * run), head = i / slices;
  return {(int)seq, (int)head, (int)(i - head * slices), head < H};
}

// For kernels of one workgroup per CU: whole heads from two sequences on, unless they need more rounds of an
// XCD's CUs than equal runs (two sequences of 21 heads of 12 slices on 256 CUs: 72 workgroups on some
// XCDs, 64 in runs).  K = 256 forward, us: 8 sequences of 128 chunks with 5 heads 872 in runs, 778 whole; 4
// of 128 with 10 heads 804 / 784; 20 of 31 with one head 134 / 109.
// `beside`: another kernel fills the CUs that this one leaves, and should find as many on every XCD: equal runs
// where heads that 8 does not divide take more than half of the CUs (20 heads of 512 chunks: one sequence 1491 in
// runs, 1587 whole; two sequences of 10 1481 / 1548.  Without it one and two of 64 chunks 207 / 209 and 216 / 207).
constexpr bool whole_heads(int n_seqs, int H, int slices, int cus, bool beside) {
  const int heads = n_seqs * H, per = cus >= kXcds ? cus / kXcds : 1;
  if (n_seqs == 1 || (beside && heads % kXcds != 0 && heads * slices <= cus && 2 * heads * slices > cus)) return false;
  return div_up(div_up(heads, kXcds) * slices, per) <= div_up(n_seqs * div_up(H * slices, kXcds), per);
}

}  // namespace kgdn
