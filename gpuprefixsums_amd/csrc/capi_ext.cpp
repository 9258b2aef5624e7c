// C ABI of the scan forms beside the plain uint32 scan: batched segmented
// scan (one launch, graph-capturable) and its per-segment-launch baseline.
#include <hip/hip_runtime.h>

#include <new>

#include "handle.hpp"

using gps::fail;
using gps::hip_fail;

namespace {

// The persistent segmented kernel unless the handle asks for one workgroup
// per tile. A default handle runs it above 2^23 elements (100 / 16000 segments,
// against one workgroup per tile at 1024 x 8: 9,000,000 17.8 / 19.7 against
// 21.6 / 24.0 us, 2^23 16.9 / 17.8 against 13.9 / 15.7, 5,000,000 12.5 / 13.2
// against 10.9 / 12.4; with three inputs in turn 2^23 17.5 / 18.4 against 16.3 / 17.8).
bool seg_persistent(const gps_handle* h, uint64_t n) {
    if (h->size_adaptive) return n > (1ull << 23);
    return h->schedule != GPS_SCHEDULE_TILE;
}

// Segmented kernels use the handle's tile shape when it is one of theirs,
// otherwise 1024 threads x 8 uint4 (32768-element tiles). A default handle
// picks the shape from n: 1024 x 2 up to 9 * 2^18 elements (100 / 16000
// segments: 1,500,000 6.3 / 8.0 us against 7.1 / 8.7 for 1024 x 4, 3,000,000 8.6 /
// 10.9 against 7.5 / 9.6), 1024 x 4 up to 2^22 (there 9.1 / 11.2 against
// 10.7 / 12.7 for 1024 x 8; 6,000,000 1024 x 8), 1024 x 8 above.
gps::TileShape seg_shape(const gps_handle* h, uint64_t n) {
    if (h->size_adaptive)
        return n <= (9ull << 18) ? gps::TileShape{1024, 2} : n <= (1ull << 22) ? gps::TileShape{1024, 4}
                                                                              : gps::TileShape{1024, 8};
    return gps::seg_shape_supported(h->shape, seg_persistent(h, n)) ? h->shape : gps::TileShape{1024, 8};
}

// FP kernels likewise: the handle's shape when it is an FP shape, else
// 1024 x 4. A default handle picks from n (sweep timings and back-to-back
// launches on MI355X): one FP scan uses 256 x 4 up to 2^19 elements (2^18 + 1
// pairs: 5.2 against 5.9 us for 1024 x 4; 2^20: 7.7 against 6.8), 1024 x 4 up
// to 2^22 and 1024 x 8 above. The segmented FP kernel uses 256 x 4 below 2^20,
// for pairs 512 x 4 up to 9 * 2^18, and 1024 x 4 above: the pair kernel's runs
// are walked through LDS twice, and until the chip is full smaller workgroups start and end that
// earlier (FP32 pairs, 100 / 100000 segments: 700,000 elements 6.4 / 7.6 us at
// 256 x 4, 6.7 / 7.8 at 512 x 4; 2,000,000 7.6 / 8.6 at 512 x 4, 8.8 / 10.1 at
// 1024 x 4; 2,500,000 9.0 / 10.2 at 512 x 4, 8.6 / 10.4 at 1024 x 4).
gps::TileShape fp_shape(const gps_handle* h, uint64_t n, bool segmented, int compensated) {
    if (h->size_adaptive) {
        if (segmented)
            return n < (1ull << 20) ? gps::TileShape{256, 4}
                   : n <= (9ull << 18) && compensated == gps::kFpPair ? gps::kSegFpMid
                                                                      : gps::TileShape{1024, 4};
        return n <= (1ull << 19) ? gps::TileShape{256, 4} : n <= (1ull << 22) ? gps::TileShape{1024, 4}
                                                                               : gps::TileShape{1024, 8};
    }
    return gps::fp_shape_supported(h->shape) ? h->shape : gps::TileShape{1024, 4};
}

int check_seg(gps_handle* h, const void* in, const void* out, const void* offsets, uint64_t n) {
    if (!h) return fail(GPS_ERR_INVALID, "null handle");
    if (int rc_ = gps::check_device(h)) return rc_;
    if (h->algo != GPS_ALGO_CSDL) return fail(GPS_ERR_UNSUPPORTED, "segmented scans need a CSDL handle");
    if (n && (!in || !out)) return fail(GPS_ERR_INVALID, "null data pointer");
    if (!offsets) return fail(GPS_ERR_INVALID, "null offsets");
    if (n > h->max_n)
        return fail(GPS_ERR_TOO_LARGE, "n=%llu exceeds handle max_n=%llu", (unsigned long long)n,
                    (unsigned long long)h->max_n);
    if ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 3u)
        return fail(GPS_ERR_INVALID, "uint32 buffers must be 4-byte aligned");
    if (reinterpret_cast<uintptr_t>(offsets) & 7u) return fail(GPS_ERR_INVALID, "offsets must be 8-byte aligned");
    return GPS_OK;
}

int enqueue_segmented(gps_handle* h, const uint32_t* in, uint32_t* out, const uint64_t* offsets,
                      uint64_t num_segments, uint64_t n, bool inclusive, hipStream_t s) {
    if (n == 0) return GPS_OK;
    HIP_TRY(gps::before_epoch_launch(h, s));
    HIP_TRY(gps::launch_segscan_u32(seg_shape(h, n), inclusive, seg_persistent(h, n), h->round_patience, in, out, offsets,
                                    num_segments, n, h->status, h->ticket, h->err, s));
    return GPS_OK;
}

}  // namespace

namespace {

// One FP scan with pair or plain carries runs the persistent kernel on a
// handle with the persistent schedule (the CSDL default). A default handle
// picks it for pairs above 2^23 elements, against one workgroup per tile, both
// at 1024 x 8: FP32 2^23 15.4 against 13.0 us, 9,000,000 16.6 against 20.3;
// BF16 14.1 against 12.8 and 14.8 against 19.7. (Between 5 and 7 million FP32
// it is up to 8% faster, BF16 slower.) For plain carries above 2^24: at
// 10,000,000 it is 6% faster, but one workgroup per tile adds the aggregates
// before a tile in fewer roundings (relative error 2.3e-7 against 2.5e-7).
bool fp_persistent(const gps_handle* h, uint64_t n, int compensated) {
    if (h->size_adaptive) return n > (compensated == gps::kFpPair ? 1ull << 23 : 1ull << 24);
    return h->schedule == GPS_SCHEDULE_PERSISTENT;
}

int scan_fp(gps_handle* h, const void* in, float* out, uint64_t n, bool bf16, int compensated, void* stream) {
    if (!h) return fail(GPS_ERR_INVALID, "null handle");
    if (int rc_ = gps::check_device(h)) return rc_;
    if (h->algo != GPS_ALGO_CSDL) return fail(GPS_ERR_UNSUPPORTED, "floating-point scans need a CSDL handle");
    if (n && (!in || !out)) return fail(GPS_ERR_INVALID, "null data pointer");
    if (n > h->max_n)
        return fail(GPS_ERR_TOO_LARGE, "n=%llu exceeds handle max_n=%llu", (unsigned long long)n,
                    (unsigned long long)h->max_n);
    if (compensated < gps::kFpPlain || compensated > gps::kFpPair)
        return fail(GPS_ERR_INVALID, "compensated must be 0 (plain) or 1 (two-float pairs)");
    const uintptr_t ia = reinterpret_cast<uintptr_t>(in), oa = reinterpret_cast<uintptr_t>(out);
    if ((ia & (bf16 ? 1u : 3u)) || (oa & 3u)) return fail(GPS_ERR_INVALID, "misaligned buffer");
    if (n == 0) return GPS_OK;
    const gps::TileShape s = fp_shape(h, n, false, compensated);
    hipStream_t st = static_cast<hipStream_t>(stream);
    HIP_TRY(gps::before_epoch_launch(h, st));
    HIP_TRY(gps::launch_scan_fp(s, bf16, compensated, fp_persistent(h, n, compensated), h->round_patience, in, out, n,
                                h->status, h->ticket, h->err, st));
    return GPS_OK;
}

// The segmented FP scan runs its persistent kernel on a handle with the
// persistent schedule. A default handle runs it, at 1024 x 8, above 2^22
// elements (4096 log-normal segments of 50.9 M elements: FP32 pairs 0.1021
// against 0.1145 ms for one workgroup per tile at 1024 x 4, plain 0.0804
// against 0.1030 ms, BF16 pairs 0.0999 against 0.1032 ms).
bool segfp_persistent(const gps_handle* h, uint64_t n) {
    if (h->size_adaptive) return n > (1ull << 22);
    return h->schedule == GPS_SCHEDULE_PERSISTENT;
}

int segscan_fp(gps_handle* h, const void* in, float* out, const uint64_t* offsets, uint64_t num_segments,
               uint64_t n, bool bf16, int compensated, void* stream) {
    if (!h) return fail(GPS_ERR_INVALID, "null handle");
    if (int rc_ = gps::check_device(h)) return rc_;
    if (h->algo != GPS_ALGO_CSDL) return fail(GPS_ERR_UNSUPPORTED, "floating-point scans need a CSDL handle");
    if (n && (!in || !out)) return fail(GPS_ERR_INVALID, "null data pointer");
    if (!offsets) return fail(GPS_ERR_INVALID, "null offsets");
    if (n > h->max_n)
        return fail(GPS_ERR_TOO_LARGE, "n=%llu exceeds handle max_n=%llu", (unsigned long long)n,
                    (unsigned long long)h->max_n);
    const uintptr_t ia = reinterpret_cast<uintptr_t>(in), oa = reinterpret_cast<uintptr_t>(out);
    if ((ia & (bf16 ? 1u : 3u)) || (oa & 3u)) return fail(GPS_ERR_INVALID, "misaligned buffer");
    if (reinterpret_cast<uintptr_t>(offsets) & 7u) return fail(GPS_ERR_INVALID, "offsets must be 8-byte aligned");
    if (compensated < gps::kFpPlain || compensated > gps::kFpPair)
        return fail(GPS_ERR_INVALID, "compensated must be 0 (plain) or 1 (two-float pairs)");
    if (n == 0) return GPS_OK;
    const bool persistent = segfp_persistent(h, n);
    const gps::TileShape s = persistent && h->size_adaptive ? gps::TileShape{1024, 8} : fp_shape(h, n, true, compensated);
    hipStream_t st = static_cast<hipStream_t>(stream);
    HIP_TRY(gps::before_epoch_launch(h, st));
    HIP_TRY(gps::launch_segscan_fp(s, bf16, compensated != 0, persistent, h->round_patience, in, out, offsets,
                                   num_segments, n, h->status, h->ticket, h->err, st));
    return GPS_OK;
}

int scan_u32x4(gps_handle* h, const uint32_t* in, uint32_t* out, uint64_t n, bool inclusive, void* stream) {
    if (!h) return fail(GPS_ERR_INVALID, "null handle");
    if (int rc_ = gps::check_device(h)) return rc_;
    if (h->algo != GPS_ALGO_CSDL) return fail(GPS_ERR_UNSUPPORTED, "struct scans need a CSDL handle");
    if (n && (!in || !out)) return fail(GPS_ERR_INVALID, "null data pointer");
    if (n > h->max_n)
        return fail(GPS_ERR_TOO_LARGE, "n=%llu exceeds handle max_n=%llu", (unsigned long long)n,
                    (unsigned long long)h->max_n);
    if ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15u)
        return fail(GPS_ERR_INVALID, "uint4 struct buffers must be 16-byte aligned");
    if (n == 0) return GPS_OK;
    gps::TileShape s = gps::v4_shape_supported(h->shape) ? h->shape : gps::TileShape{1024, 8};
    bool persistent = h->schedule != GPS_SCHEDULE_TILE;
    if (h->size_adaptive) {
        // As for the plain scan, measured on MI355X: one workgroup per tile
        // below 2^22 structs (3,000,000: 21.4 against 21.3 us for the persistent
        // kernel, 2,000,000 12.4 against 14.8), 1024 x 4 up to 2^20 (1,000,003:
        // 8.5 against 9.3 us for 1024 x 8; 2,000,000 15.9 against 12.4).
        if (n <= (1ull << 20)) {
            s = {1024, 4};
            persistent = false;
        } else if (n < (1ull << 22)) {
            s = {1024, 8};
            persistent = false;
        }
    }
    const uint64_t tile = (uint64_t)s.block * s.vec;
    if ((n + tile - 1) / tile > h->max_tiles) return fail(GPS_ERR_TOO_LARGE, "not enough status slots");
    hipStream_t st = static_cast<hipStream_t>(stream);
    HIP_TRY(gps::before_epoch_launch(h, st));
    HIP_TRY(gps::launch_csdl_u32x4(s, inclusive, persistent, h->round_patience, in, out, n, h->status, h->ticket,
                                   h->err, st));
    return GPS_OK;
}

}  // namespace

// The graph, and the launch that is its one node.
struct gps_graph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    int device = 0;
    gps::TileShape shape{};
    bool inclusive = false, persistent = false;
    uint32_t patience = 0;
    const uint32_t* in = nullptr;
    uint32_t* out = nullptr;
    const uint64_t* offsets = nullptr;
    uint64_t num_segments = 0, n = 0;
    uint64_t *status = nullptr, *ticket = nullptr;
    uint32_t* err = nullptr;

    hipError_t launch(hipStream_t s) const {
        if (n == 0) return hipSuccess;
        return gps::launch_segscan_u32(shape, inclusive, persistent, patience, in, out, offsets, num_segments, n, status,
                                       ticket, err, s);
    }
};

extern "C" {

int gps_segmented_scan_u32(gps_handle* h, const uint32_t* d_in, uint32_t* d_out, const uint64_t* d_offsets,
                           uint64_t num_segments, uint64_t n, int inclusive, void* stream) {
    int rc = check_seg(h, d_in, d_out, d_offsets, n);
    if (rc) return rc;
    return enqueue_segmented(h, d_in, d_out, d_offsets, num_segments, n, inclusive != 0,
                             static_cast<hipStream_t>(stream));
}

int gps_segmented_scan_u32_per_segment(gps_handle* h, const uint32_t* d_in, uint32_t* d_out,
                                       const uint64_t* h_offsets, uint64_t num_segments, int inclusive,
                                       void* stream) {
    if (!h) return fail(GPS_ERR_INVALID, "null handle");
    if (int rc_ = gps::check_device(h)) return rc_;
    if (!h_offsets) return fail(GPS_ERR_INVALID, "null offsets");
    for (uint64_t s = 0; s < num_segments; ++s) {
        const uint64_t a = h_offsets[s], b = h_offsets[s + 1];
        if (b < a) return fail(GPS_ERR_INVALID, "offsets must be non-decreasing (segment %llu)", (unsigned long long)s);
        if (b == a) continue;
        const int rc = inclusive ? gps_inclusive_scan_u32(h, d_in + a, d_out + a, b - a, stream)
                                 : gps_exclusive_scan_u32(h, d_in + a, d_out + a, b - a, stream);
        if (rc) return rc;
    }
    return GPS_OK;
}

int gps_segmented_graph_create(gps_handle* h, const uint32_t* d_in, uint32_t* d_out, const uint64_t* d_offsets,
                               uint64_t num_segments, uint64_t n, int inclusive, gps_graph** out) {
    if (!out) return fail(GPS_ERR_INVALID, "null output pointer");
    *out = nullptr;
    int rc = check_seg(h, d_in, d_out, d_offsets, n);
    if (rc) return rc;
    HIP_TRY(gps::prepare_segscan_u32(seg_shape(h, n), inclusive != 0, seg_persistent(h, n)));
    hipStream_t s = nullptr;
    HIP_TRY(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    gps_graph* g = new (std::nothrow) gps_graph();
    if (!g) {
        (void)hipStreamDestroy(s);
        return fail(GPS_ERR_INVALID, "out of host memory");
    }
    g->device = h->device;
    g->shape = seg_shape(h, n);
    g->inclusive = inclusive != 0;
    g->persistent = seg_persistent(h, n);
    g->patience = h->round_patience;
    g->in = d_in;
    g->out = d_out;
    g->offsets = d_offsets;
    g->num_segments = num_segments;
    g->n = n;
    g->status = h->status;
    g->ticket = h->ticket;
    g->err = h->err;
    hipError_t e = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
    if (e == hipSuccess) {
        // No re-arm check inside a capture: a graph node must not depend on
        // the host-side launch count (gps_reset re-arms explicitly).
        rc = g->launch(s) == hipSuccess ? GPS_OK : GPS_ERR_HIP;
        hipGraph_t graph = nullptr;
        e = hipStreamEndCapture(s, &graph);
        g->graph = graph;
        if (rc != GPS_OK && e == hipSuccess) e = hipErrorLaunchFailure;
    }
    if (e == hipSuccess) e = hipGraphInstantiate(&g->exec, g->graph, nullptr, nullptr, 0);
    (void)hipStreamDestroy(s);
    if (e != hipSuccess) {
        if (g->exec) (void)hipGraphExecDestroy(g->exec);
        if (g->graph) (void)hipGraphDestroy(g->graph);
        delete g;
        return hip_fail(e, "segmented graph capture");
    }
    *out = g;
    return GPS_OK;
}

int gps_inclusive_scan_f32(gps_handle* h, const float* d_in, float* d_out, uint64_t n, int compensated,
                           void* stream) {
    return scan_fp(h, d_in, d_out, n, false, compensated, stream);
}

int gps_inclusive_scan_bf16_f32(gps_handle* h, const uint16_t* d_in, float* d_out, uint64_t n, int compensated,
                                void* stream) {
    return scan_fp(h, d_in, d_out, n, true, compensated, stream);
}

int gps_segmented_scan_f32(gps_handle* h, const float* d_in, float* d_out, const uint64_t* d_offsets,
                           uint64_t num_segments, uint64_t n, int compensated, void* stream) {
    return segscan_fp(h, d_in, d_out, d_offsets, num_segments, n, false, compensated, stream);
}

int gps_segmented_scan_bf16_f32(gps_handle* h, const uint16_t* d_in, float* d_out, const uint64_t* d_offsets,
                                uint64_t num_segments, uint64_t n, int compensated, void* stream) {
    return segscan_fp(h, d_in, d_out, d_offsets, num_segments, n, true, compensated, stream);
}

int gps_survey_segment_u32(int alg, uint32_t* segment) {
    if (!segment) return fail(GPS_ERR_INVALID, "null argument");
    const uint32_t s = gps::survey_segment(alg);
    if (!s) return fail(GPS_ERR_INVALID, "unknown survey network %d", alg);
    *segment = s;
    return GPS_OK;
}

int gps_survey_scan_u32(int alg, const uint32_t* d_in, uint32_t* d_out, uint64_t n, int inclusive, void* stream) {
    const uint32_t seg = gps::survey_segment(alg);
    if (!seg) return fail(GPS_ERR_INVALID, "unknown survey network %d", alg);
    if (n % seg) return fail(GPS_ERR_INVALID, "n=%llu is not a multiple of the segment (%u)", (unsigned long long)n, seg);
    if (n == 0) return GPS_OK;
    if (!d_in || !d_out) return fail(GPS_ERR_INVALID, "null data pointer");
    const uintptr_t mask = alg == gps::kSurveyTileRegisters ? 15u : 3u;
    if ((reinterpret_cast<uintptr_t>(d_in) | reinterpret_cast<uintptr_t>(d_out)) & mask)
        return fail(GPS_ERR_INVALID, "buffers must be %u-byte aligned", (unsigned)mask + 1u);
    HIP_TRY(gps::launch_survey_u32(alg, inclusive != 0, d_in, d_out, n, static_cast<hipStream_t>(stream)));
    return GPS_OK;
}

int gps_estimate_occupancy(gps_handle* h, const uint32_t* d_in, uint32_t* d_out, uint64_t n, int struct_scan,
                           void* stream, uint32_t* measured, uint32_t* resident) {
    if (!h || !measured || !resident) return fail(GPS_ERR_INVALID, "null argument");
    if (int rc_ = gps::check_device(h)) return rc_;
    if (h->algo != GPS_ALGO_CSDL) return fail(GPS_ERR_UNSUPPORTED, "the occupancy estimate needs a CSDL handle");
    if (!d_in || !d_out) return fail(GPS_ERR_INVALID, "null data pointer");
    if (n == 0) return fail(GPS_ERR_INVALID, "n must be positive");
    if (n > h->max_n)
        return fail(GPS_ERR_TOO_LARGE, "n=%llu exceeds handle max_n=%llu", (unsigned long long)n,
                    (unsigned long long)h->max_n);
    const uintptr_t mask = struct_scan ? 15u : 3u;
    if ((reinterpret_cast<uintptr_t>(d_in) | reinterpret_cast<uintptr_t>(d_out)) & mask)
        return fail(GPS_ERR_INVALID, struct_scan ? "uint4 struct buffers must be 16-byte aligned"
                                                 : "uint32 buffers must be 4-byte aligned");
    hipStream_t st = static_cast<hipStream_t>(stream);
    unsigned long long* count = h->counters + gps::kCounterOccupancy;
    HIP_TRY(hipMemsetAsync(count, 0, sizeof(unsigned long long), st));
    HIP_TRY(gps::before_epoch_launch(h, st));
    if (struct_scan) {
        const gps::TileShape s = gps::v4_shape_supported(h->shape) ? h->shape : gps::TileShape{1024, 8};
        *resident = gps::v4_resident_workgroups(s, true);
        HIP_TRY(gps::launch_csdl_u32x4(s, true, true, h->round_patience, d_in, d_out, n, h->status, h->ticket, h->err,
                                       st, count, true));
    } else {
        gps::ScanParams p{};
        const uint64_t tile = h->shape.tile();
        p.in = d_in;
        p.out = d_out;
        p.n = n;
        p.num_tiles = (uint32_t)((n + tile - 1) / tile);
        p.status = h->status;
        p.ticket = h->ticket;
        p.err = h->err;
        p.occupancy = count;
        *resident = gps::pp_resident_workgroups(h->shape, true);
        HIP_TRY(gps::launch_csdl_pp_u32(h->shape, true, p, st, true));
    }
    unsigned long long c = 0;
    HIP_TRY(hipMemcpyAsync(&c, count, sizeof c, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    *measured = (uint32_t)c;
    return GPS_OK;
}

int gps_inclusive_scan_u32x4(gps_handle* h, const uint32_t* d_in, uint32_t* d_out, uint64_t n, void* stream) {
    return scan_u32x4(h, d_in, d_out, n, true, stream);
}

int gps_exclusive_scan_u32x4(gps_handle* h, const uint32_t* d_in, uint32_t* d_out, uint64_t n, void* stream) {
    return scan_u32x4(h, d_in, d_out, n, false, stream);
}

int gps_inclusive_scan_fp_per_segment(gps_handle* h, const void* d_in, float* d_out, const uint64_t* h_offsets,
                                      uint64_t num_segments, int bf16, int compensated, void* stream) {
    if (!h || !h_offsets) return fail(GPS_ERR_INVALID, "null argument");
    const size_t esize = bf16 ? 2 : 4;
    for (uint64_t s = 0; s < num_segments; ++s) {
        const uint64_t a = h_offsets[s], b = h_offsets[s + 1];
        if (b < a) return fail(GPS_ERR_INVALID, "offsets must be non-decreasing (segment %llu)", (unsigned long long)s);
        if (b == a) continue;
        const void* in = static_cast<const char*>(d_in) + a * esize;
        const int rc = scan_fp(h, in, d_out + a, b - a, bf16 != 0, compensated, stream);
        if (rc) return rc;
    }
    return GPS_OK;
}

// A replay of one kernel is that kernel's launch: 3.1 us of the host against
// 14 for hipGraphLaunch, whose packets also put 4 us between kernels (50.9 M
// elements 75.6 against 79.7 us a replay). A stream that is being captured
// records it, where hipGraphLaunch reports success and records nothing. The
// graph is launched where another device is current than its own, or an error
// of an earlier HIP call is pending, which the launch would return as its own;
// into a capture such a replay is refused.
int gps_graph_launch(gps_graph* g, void* stream) {
    if (!g || !g->exec) return fail(GPS_ERR_INVALID, "null graph");
    const hipStream_t s = static_cast<hipStream_t>(stream);
    int device = -1;
    if (hipPeekAtLastError() == hipSuccess && hipGetDevice(&device) == hipSuccess && device == g->device) {
        HIP_TRY(g->launch(s));
        return GPS_OK;
    }
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (s && hipStreamIsCapturing(s, &capture) == hipSuccess && capture != hipStreamCaptureStatusNone)
        return fail(GPS_ERR_HIP, "a capture cannot record the replay: another device is current or an earlier HIP "
                                 "call's error is pending");
    HIP_TRY(hipGraphLaunch(g->exec, s));
    return GPS_OK;
}

int gps_graph_destroy(gps_graph* g) {
    if (!g) return fail(GPS_ERR_INVALID, "null graph");
    if (g->exec) (void)hipGraphExecDestroy(g->exec);
    if (g->graph) (void)hipGraphDestroy(g->graph);
    delete g;
    return GPS_OK;
}

}  // extern "C"
