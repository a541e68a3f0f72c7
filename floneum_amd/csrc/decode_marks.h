// The marks by which the workgroups of a split-KV decode unit see each other's arrivals (fused_merge_tail in attn_decode.hip).
//
// They lie in the call's own workspace, which nothing clears: before the launch their words hold whatever another call, of any shape,
// left there, partial results among it.  A mark is 64 bits wide, of which all but the XCC id are compared, so such a word is taken for a
// mark with a probability of 2^-60; and the tags of a device handle's calls differ for 2^52 of them.
#pragma once
#include <cstdint>

namespace fhip {

// tag (52 bits) | XCC id of the workgroup (4) | arrivals (8)
constexpr uint64_t MARK_XCC = 0xf00, MARK_TAG = ~(uint64_t)0xfff;

// The tag of the nth call: consecutive numbers are spread over all bits (by an odd factor, one to one), for they are also compared with
// other handles' and with plain numbers.  n % 2^52 == 0 has no tag (0).
constexpr uint64_t mark_tag(uint64_t n) { return (n * 0x9e3779b97f4a7c15ull) << 12; }
constexpr uint64_t mark_of(uint64_t tag, uint32_t xcc, uint32_t arrivals) { return tag | (uint64_t)xcc << 8 | arrivals; }
constexpr uint32_t mark_arrivals(uint64_t word) { return (uint32_t)word & 255u; }
constexpr bool mark_is_of(uint64_t word, uint64_t tag) { return (word & MARK_TAG) == tag; }                       // with any count
constexpr bool mark_is(uint64_t word, uint64_t tag, uint32_t arrivals) { return (word & ~MARK_XCC) == (tag | arrivals); }
constexpr bool mark_same_xcc(uint64_t word, uint32_t xcc) { return (word & MARK_XCC) == (uint64_t)xcc << 8; }

}  // namespace fhip
