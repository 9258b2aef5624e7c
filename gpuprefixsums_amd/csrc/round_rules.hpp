// Host rules of the one-round scans (device_common.hpp): which calls may run
// them. Plain C++, so that they can be tested without a device.
#pragma once

#include <stdint.h>

namespace gps {

// Polls of a status window before a wave computes a missing tile's aggregate
// itself: tens of microseconds, far beyond what a workgroup that has started
// needs. Fewer cost time where a launch has more tiles than run at once:
// 12,345,677 elements 17.8 us so, 48 after 4 polls.
constexpr uint32_t kRoundPatience = 64;

// A CSDL handle's spin limit, 4 unless given, says nothing but on one that
// asks for the tile schedule: there limits below 4 let a wave sum sooner, after
// 4^(spin_limit - 1) polls (at 1 after the first, which tests use). The limit
// that a handle reports makes another handle with the same patience.
constexpr uint32_t round_patience(bool tile_schedule, uint32_t spin_limit) {
    return tile_schedule && spin_limit < 4u ? 1u << (2u * (spin_limit - 1u)) : kRoundPatience;
}

inline bool ranges_overlap(const void* a, uint64_t a_bytes, const void* b, uint64_t b_bytes) {
    const uint64_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
    return x < y + b_bytes && y < x + a_bytes;
}

// A wave of a one-round scan may sum a tile in its workgroup's place, so a
// workgroup may store while an earlier one has not loaded its tile yet: only
// buffers that are the same or apart are safe. The ticketed kernels store a
// tile after every earlier one has been loaded, which also serves an output
// that begins before the input and overlaps it.
inline bool round_buffers(const void* in, uint64_t in_bytes, const void* out, uint64_t out_bytes) {
    return !ranges_overlap(in, in_bytes, out, out_bytes) || (in == out && in_bytes == out_bytes);
}

// Carry words likewise (null: none): the last tile may end, and write the
// carry-out, before tile 0 or a wave that sums tile 0 in its place has read
// the carry-in, and any tile may store before that.
inline bool round_carries(const uint32_t* carry_in, const uint32_t* carry_out, const void* in, const void* out,
                          uint64_t bytes) {
    if (carry_in && (carry_in == carry_out || ranges_overlap(carry_in, 4, out, bytes))) return false;
    return !carry_out || !(ranges_overlap(carry_out, 4, in, bytes) || ranges_overlap(carry_out, 4, out, bytes));
}

}  // namespace gps
