// LDS layouts that permute their elements against bank conflicts, as plain constexpr index functions (host and
// device): the kernels address LDS through them, and a host test counts the conflicts of every access.
//
// What the counts assume, measured with SQ_LDS_BANK_CONFLICT / SQ_LDS_IDX_ACTIVE on probes of each width: 4-byte
// accesses are served per half-wave from 32 banks of 4 bytes, 16-byte accesses per 16 lanes from 64.
#pragma once

namespace kdn {

// The fp32 state kernel's LDS copy of one K fragment (16 tokens x 32 features, 64 slots of eight floats), written as
// fragments and read back as K^T operands.  The word of token 4g + e, feature 4q + i + 16 half: a slot holds four
// features and those sixteen further on; its halves change places for odd g.
//   written (kf32_write): lane l the token l & 15 and the features of q = l >> 4, 16 bytes a half: of the 16 lanes of one
//     q, e is on bank bits 3-4, g & 1 on bit 2 and g >> 1 on bit 5, so that they take the 64 banks once;
//   read (kf32_read): lane l the feature l & 15 of token 4 (l >> 4) + e, 4 bytes: of a half-wave (g >> 1 fixed), i is on
//     bits 0-1, g & 1 on bit 2 and q on bits 3-4, 32 banks once.
// (With g >> 1 deciding the halves and g & 1 on bit 5, the reads' lanes of g and g ^ 1 met on one bank: 43.7 % of the
// kernel's busy LDS cycles.)
constexpr int kf32_word(int g, int e, int q, int half) {
  return 8 * ((q ^ e) + 4 * (g >> 1) + 8 * (e + 4 * (g & 1))) + 4 * (half ^ (g & 1));
}
constexpr int kf32_write(int lane, int half) { return kf32_word((lane & 15) >> 2, lane & 3, lane >> 4, half); }
constexpr int kf32_read(int lane, int e, int half) { return kf32_word(lane >> 4, e, (lane & 15) >> 2, half) + (lane & 3); }

// A and T of the 64 x 64 unit-lower inverse in 16 x 16 blocks (unit_lower_inverse_blocked).
//
// A by columns, the rows of a column in sixteen groups of four, the groups XORed with a permutation of the column's low four
// bits c3 c2 c1 c0 (c0 to bit 3, c2 to bit 2, c3 to bit 1, c1 to bit 0).
//   4-byte accesses of A[16i + m][16k + 4g + kb] (lane (g, m); the column walk's reads, and the stores of a tile held
//     with its rows over the lanes): m & 3 on bank bits 0-1, m >> 2 (XORed) on bits 2-3 and (i ^ g) & 1 on bit 4, which
//     differs over a half-wave's two g; of i and kb only i & 1 and kb >> 1 meet a lane's bits, so that four lane
//     addresses serve all of a walk's reads;
//   16-byte accesses of rows 4s .. 4s + 3 of sixteen consecutive columns (the stores of a tile held with its columns over
//     the lanes): sixteen groups;
//   16-byte reads of rows 16b + 4p .. + 3 of one column by the lanes p (the substitution): four groups, each broadcast.
// (In four rows of residue p = row & 3 a column, the stores by columns were four 4-byte ones that met four ways on a bank:
// prep8_kernel's conflicts 6.7 % of its busy LDS cycles.  4.1 % with this; 2.7 % with the column's bits unpermuted, where
// a walk takes twelve lane addresses and the kernel 0.5 us more in a call of 520 chunks, 34.75 for 34.2: the rest is pairs
// of the walk's reads that the compiler merges, whose two words lie on one bank and are counted, at no cost in time.)
constexpr int a_word(int row, int col) {
  const int f = (col >> 1 & 1) | (col >> 3 & 1) << 1 | (col >> 2 & 1) << 2 | (col & 1) << 3;
  return col * 64 + 4 * ((row >> 2) ^ f) + (row & 3);
}

// T by rows, the 16-byte groups of a row's columns XORed with h(r) = 4 (a ^ p) + a, a = (r >> 2) & 3, p = r & 3, so that
// each of these falls on distinct banks: 4-byte accesses of rows 4a + 0..3 (a fixed; accumulator tiles) or of rows
// 4·0..3 + p (p fixed; the substitution's stores) at columns of one 16-column block per instruction (h >> 2 differs over
// p for fixed a and over a for fixed p), and 16-byte reads of four consecutive columns of 16 consecutive rows (h is a
// bijection on a 16-row block).
constexpr int t_swizzle(int r, int c) {
  const int a = (r >> 2) & 3, p = r & 3;
  return c ^ (16 * (a ^ p)) ^ (4 * a);
}

}  // namespace kdn
