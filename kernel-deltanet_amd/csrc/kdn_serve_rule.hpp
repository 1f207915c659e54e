// Where a serving step from a slot map runs its decodes, as a plain function of the step's sizes (a host test checks it).
#pragma once
#include <cstdint>

namespace kdn {

// Whether the decodes of a step with an auxiliary stream run on it beside the prefill's last launches, rather than before
// the prefill on the caller's stream.  The second stream costs two events, 15 to 40 us of the host's time, and saves the
// decode's, which goes by the bytes of the states it streams (5.5 TB/s, read and written): 128 KB a state at d_v = 64.
//   Above 1024 tokens: beside, as in the step with host offsets; the host is done long before the GPU.
//   Distinct runs have distinct slots, so at most min(tokens, slots) sequences decode, and a step of more tokens than
// slots holds a prefill (or padding) for sure.  There it pays from 64 MB of states on; us a step, waited for / queued,
// on one stream and beside (bf16, d_v = 64; decodes x heads + prefill):
//     9 x 16 + 300     103 / 76     106 / 66        64 x 16 + 300    140 / 114    129 / 91
//     128 x 4 + 300    102 / 76     101 / 60        224 x 16 + 300   256 / 229    252 / 210
//   A step of as many tokens as slots, or fewer, is most often decodes alone, which the events only delay: 16 x 16
// 49 / 28 on one stream, 81 / 55 on two; 128 x 16 139 / 112 and 158 / 116.  From 512 MB on they no longer show where steps
// are queued (512 x 16 413 / 385 and 430 / 381), and a prefill among the tokens gains 20 us.
constexpr bool slot_decode_beside(int64_t tokens, int64_t slots, int64_t H, int D, int d_v) {
  if (tokens > 1024) return true;
  const int64_t bytes = (tokens < slots ? tokens : slots) * H * D * d_v * 4;
  return bytes >= (tokens > slots ? (int64_t)64 << 20 : (int64_t)512 << 20);
}

}  // namespace kdn
