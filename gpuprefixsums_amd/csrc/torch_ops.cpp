// The device kernels of torch.ops.gps.cumsum and segmented_cumsum for the
// ordinary call: a contiguous 1-D tensor on the current device, no gradient
// asked for, on a stream that has a handle. It allocates the output and
// launches; every other call, and every error, goes to the operator's Python
// implementation (torch_ops.py), which also defines the operators, makes the
// handles and enters them here.
//
// What bounds a small scan through the operator is the host: 16.7 us a call
// at 1021 elements when each went through the Python autograd wrapper, the
// Python body and ctypes, of which the launch itself is 3.2 us and the
// allocation 1.3 us; 4.6 us so.
#include <ATen/core/Tensor.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/core/grad_mode.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/library.h>

#include <map>
#include <mutex>
#include <utility>

#include "gps.h"

namespace {

struct Entry {
    gps_handle* handle;
    uint64_t max_n;
};

// The handle of a (device, stream), as torch_ops.py keeps it: entered once it
// exists, replaced by a larger one, never closed before the process ends.
struct Handles {
    std::mutex mutex;
    std::map<std::pair<int, hipStream_t>, Entry> entries;
};

Handles& handles() {
    static Handles* const h = new Handles;  // not destroyed: threads may still launch at exit
    return *h;
}

gps_handle* find_handle(int device, hipStream_t stream, uint64_t n) {
    Handles& h = handles();
    const std::lock_guard<std::mutex> lock(h.mutex);
    const auto at = h.entries.find({device, stream});
    return at == h.entries.end() || at->second.max_n < n ? nullptr : at->second.handle;
}

// The Python kernels are registered under alias keys; a backend without a
// kernel of its own has them in its dispatch table.
at::Tensor python_kernel(const c10::OperatorHandle& op, c10::DispatchKey other, c10::DispatchKeySet ks,
                         torch::jit::Stack stack) {
    op.getComputedKernelForDispatchKey(other).callBoxed(op, ks, &stack);
    return stack.back().toTensor();
}

struct Call {
    gps_handle* handle = nullptr;
    hipStream_t stream = nullptr;
    at::Tensor out;
    bool integer = false, bf16 = false;
};

// An ordinary call's handle, stream and output; false for any other call.
bool ordinary(const at::Tensor& x, bool inclusive, Call& c) {
    const auto type = x.scalar_type();
    c.integer = type == at::kInt || type == at::kUInt32;
    c.bf16 = type == at::kBFloat16;
    if (!c.integer && (!inclusive || !(c.bf16 || type == at::kFloat))) return false;
    const int device = x.get_device();
    if (x.dim() != 1 || x.numel() == 0 || !x.is_contiguous() || device != c10::hip::current_device()) return false;
    c.stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
    c.handle = find_handle(device, c.stream, (uint64_t)x.numel());
    if (!c.handle) return false;
    c.out = c.integer ? at::empty_like(x) : at::empty(x.sizes(), at::TensorOptions(x.device()).dtype(at::kFloat));
    return true;
}

const c10::TypedOperatorHandle<at::Tensor(const at::Tensor&, bool, bool)>& cumsum_op() {
    static const auto op = c10::Dispatcher::singleton()
                               .findSchemaOrThrow("gps::cumsum", "")
                               .typed<at::Tensor(const at::Tensor&, bool, bool)>();
    return op;
}

const c10::TypedOperatorHandle<at::Tensor(const at::Tensor&, const at::Tensor&, bool, bool)>& segmented_op() {
    static const auto op = c10::Dispatcher::singleton()
                               .findSchemaOrThrow("gps::segmented_cumsum", "")
                               .typed<at::Tensor(const at::Tensor&, const at::Tensor&, bool, bool)>();
    return op;
}

at::Tensor cumsum(c10::DispatchKeySet ks, const at::Tensor& x, bool inclusive, bool compensated) {
    Call c;
    if (ordinary(x, inclusive, c)) {
        const uint64_t n = (uint64_t)x.numel();
        const void* const in = x.const_data_ptr();
        void* const out = c.out.mutable_data_ptr();
        const int rc =
            c.integer ? gps_scan_u32(c.handle, static_cast<const uint32_t*>(in), static_cast<uint32_t*>(out), n,
                                     inclusive, c.stream)
            : c.bf16 ? gps_inclusive_scan_bf16_f32(c.handle, static_cast<const uint16_t*>(in),
                                                   static_cast<float*>(out), n, compensated, c.stream)
                     : gps_inclusive_scan_f32(c.handle, static_cast<const float*>(in), static_cast<float*>(out), n,
                                              compensated, c.stream);
        if (rc == GPS_OK) return std::move(c.out);
    }
    return python_kernel(cumsum_op(), c10::DispatchKey::XLA, ks, {x, inclusive, compensated});
}

at::Tensor segmented_cumsum(c10::DispatchKeySet ks, const at::Tensor& x, const at::Tensor& offsets, bool inclusive,
                            bool compensated) {
    Call c;
    if (offsets.scalar_type() == at::kLong && offsets.dim() == 1 && offsets.numel() > 0 && offsets.is_contiguous() &&
        offsets.device() == x.device() && ordinary(x, inclusive, c)) {
        const uint64_t n = (uint64_t)x.numel(), segments = (uint64_t)offsets.numel() - 1;
        const void* const in = x.const_data_ptr();
        void* const out = c.out.mutable_data_ptr();
        const uint64_t* const off = static_cast<const uint64_t*>(offsets.const_data_ptr());
        const int rc =
            c.integer ? gps_segmented_scan_u32(c.handle, static_cast<const uint32_t*>(in),
                                               static_cast<uint32_t*>(out), off, segments, n, inclusive, c.stream)
            : c.bf16 ? gps_segmented_scan_bf16_f32(c.handle, static_cast<const uint16_t*>(in),
                                                   static_cast<float*>(out), off, segments, n, compensated, c.stream)
                     : gps_segmented_scan_f32(c.handle, static_cast<const float*>(in), static_cast<float*>(out), off,
                                              segments, n, compensated, c.stream);
        if (rc == GPS_OK) return std::move(c.out);
    }
    return python_kernel(segmented_op(), c10::DispatchKey::XLA, ks, {x, offsets, inclusive, compensated});
}

// Without a gradient to record there is nothing to do here.
at::Tensor cumsum_autograd(c10::DispatchKeySet ks, const at::Tensor& x, bool inclusive, bool compensated) {
    if (at::GradMode::is_enabled() && x.requires_grad())
        return python_kernel(cumsum_op(), c10::DispatchKey::AutogradXLA, ks, {x, inclusive, compensated});
    const at::AutoDispatchBelowAutograd below;
    return cumsum_op().redispatch(ks & c10::after_autograd_keyset, x, inclusive, compensated);
}

at::Tensor segmented_autograd(c10::DispatchKeySet ks, const at::Tensor& x, const at::Tensor& offsets, bool inclusive,
                              bool compensated) {
    if (at::GradMode::is_enabled() && (x.requires_grad() || offsets.requires_grad()))
        return python_kernel(segmented_op(), c10::DispatchKey::AutogradXLA, ks, {x, offsets, inclusive, compensated});
    const at::AutoDispatchBelowAutograd below;
    return segmented_op().redispatch(ks & c10::after_autograd_keyset, x, offsets, inclusive, compensated);
}

}  // namespace

// ROCm tensors carry the CUDA dispatch keys.
TORCH_LIBRARY_IMPL(gps, CUDA, m) {
    m.impl("cumsum", TORCH_FN(cumsum));
    m.impl("segmented_cumsum", TORCH_FN(segmented_cumsum));
}

TORCH_LIBRARY_IMPL(gps, AutogradCUDA, m) {
    m.impl("cumsum", TORCH_FN(cumsum_autograd));
    m.impl("segmented_cumsum", TORCH_FN(segmented_autograd));
}

// Enters the handle of a (device, stream); the caller keeps it open until the
// process ends. Not entered (out of memory) means the Python implementation.
extern "C" void gps_torch_set_handle(int device, void* stream, gps_handle* handle, uint64_t max_n) noexcept {
    try {
        Handles& h = handles();
        const std::lock_guard<std::mutex> lock(h.mutex);
        h.entries[{device, static_cast<hipStream_t>(stream)}] = {handle, max_n};
    } catch (...) {
    }
}
