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

}  // namespace kdn
