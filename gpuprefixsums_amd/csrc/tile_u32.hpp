// Register-tile routines for the uint32 scans (per-thread uint4 vectors,
// wave-striped so every load/store instruction moves 1 KiB contiguous).
//
// Reference counterparts: GPUPrefixSumsCUDA/ScanCommon.cuh:12-135
// (Scan{In,Ex}clusive{Full,Partial}, Propagate{Full,Partial}).
//
// Tile geometry for BLOCK threads and VEC uint4 per thread:
//   element of (wave w, vector k, lane l, component c) =
//       tile * TILE + w * (256 * VEC) + k * 256 + l * 4 + c
// so wave w owns a contiguous run of 256*VEC elements, scanned in order k,
// then lane, then component.
#pragma once

#include "device_common.hpp"

namespace gps {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int BLOCK, int VEC>
struct TileCfg {
    static_assert(BLOCK % 64 == 0 && BLOCK <= 1024, "BLOCK must be whole waves");
    static constexpr uint32_t kWaves = BLOCK / 64;
    static constexpr uint32_t kItems = VEC * 4;
    static constexpr uint32_t kTile = BLOCK * kItems;
    static constexpr uint32_t kWaveElems = 64 * kItems;
};

// Element offset of this thread's first vector inside its tile.
template <int VEC>
__device__ __forceinline__ uint32_t thread_offset() {
    return (threadIdx.x / kWave) * (256u * VEC) + lane_id() * 4u;
}

// Tile input and output. Buffers are only element-aligned (a slice x[1:] is an
// ordinary input) and n is any number, so:
//   - vectors are moved as dwordx4 from any 4-byte address, which gfx950 does
//     at full rate (a wave's 1 KiB then spans nine 128-byte lines, not eight);
//   - a partial tile is a raw buffer that ends at n: its loads return zero and
//     its stores do nothing for each dword past the end. Stores go through the
//     buffer always, so they need no second path; full tiles load through
//     plain addresses (buffer loads took 341.5 us for the 2^28 scan, plain
//     ones 340.0).
// Four guarded 4-byte accesses per vector, each a quarter of a line's bytes,
// took twice as long where a whole scan ran on them, and one partial tile of
// them at the end held up aligned scans too: 12,345,677 elements one element
// into a buffer 45.7 -> 21.0 us, the same aligned 26.3 -> 20.3 us; 2^28
// elements off by one 653 -> 343 us.
typedef u32x4 u32x4_any __attribute__((aligned(4)));

// base and bytes are the same in every lane (the resource is scalar).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t raw_buffer(const void* base, uint32_t bytes) {
    const uint64_t p = reinterpret_cast<uint64_t>(base);
    // The builtin returns int: the casts keep a low word of 2^31 or more from
    // extending its sign over the high one.
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)p);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(p >> 32));
    const uint64_t u = (uint64_t)hi << 32 | lo;
    return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(u), 0, __builtin_amdgcn_readfirstlane(bytes),
                                             0x00020000);
}
constexpr int kNontemporal = 2;  // buffer cache policy: nt

// Valid elements of the tile that starts at `start` (uniform).
__device__ __forceinline__ uint32_t tile_valid(uint64_t start, uint64_t n, uint32_t tile_elems) {
    const uint64_t left = n - start;
    return left < tile_elems ? (uint32_t)left : tile_elems;
}

// Inputs up to a quarter of the 256 MiB Infinity Cache are loaded with the
// ordinary policy, so that what is there is used and stays; larger ones stream
// past it. Nontemporal / ordinary loads, one input again and again: 2^20
// elements 6.1 / 5.3 us, 2^24 25.2 / 22.7, 2^25 48.4 / 40.5, 2^28 340 / 348;
// three inputs in turn: 2^24 25.4 / 22.8, 2^25 48.8 / 48.7, 2^26 89.8 / 91.0.
// So from 2^25 on it pays only for a caller that scans the same large input
// again, and costs 1-5% otherwise. (Ordinary stores are slower at every size:
// the output pushes the input out.)
constexpr uint64_t kCachedBytes = 64ull << 20;

// LEAN: no address registers for the streaming path (buffer loads there too).
template <int VEC, bool LEAN = false>
__device__ __forceinline__ void load_tile(u32x4 (&d)[VEC], const uint32_t* in, uint64_t start, uint64_t n,
                                          uint32_t tile_elems) {
    const uint32_t valid = tile_valid(start, n, tile_elems), at = thread_offset<VEC>();
    const bool stream = 4u * n > kCachedBytes;
    if (LEAN && stream) {
        const __amdgpu_buffer_rsrc_t r = raw_buffer(in + start, 4u * valid);
#pragma unroll
        for (int k = 0; k < VEC; ++k)
            d[k] = __builtin_amdgcn_raw_buffer_load_b128(r, 4u * at + k * 1024u, 0, kNontemporal);
    } else if (stream && valid == tile_elems) {
        const u32x4_any* v = reinterpret_cast<const u32x4_any*>(in + start + at);
#pragma unroll
        for (int k = 0; k < VEC; ++k) d[k] = __builtin_nontemporal_load(v + k * 64);
    } else {
        const __amdgpu_buffer_rsrc_t r = raw_buffer(in + start, 4u * valid);
#pragma unroll
        for (int k = 0; k < VEC; ++k) d[k] = __builtin_amdgcn_raw_buffer_load_b128(r, 4u * at + k * 1024u, 0, 0);
    }
}

// `add`: a uint32, or a u32x4 for the struct scan.
template <int VEC, class Add>
__device__ __forceinline__ void store_tile(uint32_t* out, const u32x4 (&d)[VEC], Add add, uint64_t start, uint64_t n,
                                           uint32_t tile_elems) {
    const uint32_t valid = tile_valid(start, n, tile_elems), at = 4u * thread_offset<VEC>();
    const __amdgpu_buffer_rsrc_t r = raw_buffer(out + start, 4u * valid);
#pragma unroll
    for (int k = 0; k < VEC; ++k)
        __builtin_amdgcn_raw_buffer_store_b128(d[k] + add, r, at + k * 1024u, 0, kNontemporal);
}

// Scans the wave's run in registers. On return d holds, per element, the
// inclusive (INCL) or exclusive scan of the wave's run; returns the run total
// (uniform). Per vector: serial scan of the 4 components, DPP scan of the
// lane totals, and a running carry kept uniform via readlane.
template <int VEC, bool INCL>
__device__ __forceinline__ uint32_t wave_scan_run(u32x4 (&d)[VEC]) {
    uint32_t carry = 0;
#pragma unroll
    for (int k = 0; k < VEC; ++k) {
        u32x4 v = d[k];
        v.y += v.x;
        v.z += v.y;
        v.w += v.z;
        const uint32_t t = v.w;
        const uint32_t s = wave_incl_scan(t);
        const uint32_t add = carry + (s - t);
        if (INCL) {
            d[k] = v + add;
        } else {
            d[k] = (u32x4){add, v.x + add, v.y + add, v.z + add};
        }
        carry += readlane(s, 63);
    }
    return carry;
}

// Plain sum of the thread's vectors (fallback and reduce passes).
template <int VEC>
__device__ __forceinline__ uint32_t thread_sum(const u32x4 (&d)[VEC]) {
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < VEC; ++k) s += d[k].x + d[k].y + d[k].z + d[k].w;
    return s;
}

// Exclusive prefix of this wave inside the tile, and the tile total, from the
// per-wave totals in LDS (after a barrier).
// Lane j loads wave j's total and the wave scans them with DPP, so each
// thread needs one LDS read and two registers whatever the block size.
template <int WAVES>
__device__ __forceinline__ void combine_waves(const uint32_t* s_wave, uint32_t wave, uint32_t& wave_prefix,
                                              uint32_t& tile_total) {
    const uint32_t lane = lane_id();
    const uint32_t v = lane < (uint32_t)WAVES ? s_wave[lane] : 0u;
    const uint32_t s = wave_incl_scan(v);
    wave_prefix = __builtin_amdgcn_readlane(s - v, wave);
    tile_total = readlane(s, WAVES - 1);
}

}  // namespace gps
