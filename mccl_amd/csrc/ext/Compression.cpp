#include "Compression.hpp"

#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <chrono>

#include "../../../include/mccl_hip.h"
#include <hip/hip_runtime_api.h>

#include "Errors.hpp"
#include "FP16Compression.hpp"
#include "HipKernels.hpp"
#include "Logging.hpp"
#include "TensorChecks.hpp"
#include "TopKCompression.hpp"

namespace mccl {

std::unique_ptr<Compressor> make_compressor(CompressionMode mode, double param) {
    switch (mode) {
        case CompressionMode::NONE: return nullptr;
        case CompressionMode::FP16: return std::make_unique<FP16Compressor>();
        case CompressionMode::TOPK: return std::make_unique<TopKCompressor>(param > 0 ? param : 0.01);
        default:
            throw MCCLError("Unknown compression mode: " + std::to_string(static_cast<int>(mode)));
    }
}

namespace {
void device_copy(void* dst, const void* src, size_t nbytes) {
    if (nbytes == 0) return;
    const hipError_t e = hipMemcpyAsync(dst, src, nbytes, hipMemcpyDeviceToDevice,
                                        c10::hip::getCurrentHIPStream().stream());
    MCCL_CHECK(e == hipSuccess, std::string("FP16 passthrough copy failed: ") + hipGetErrorString(e));
}
}  // namespace

// csrc/compression/FP16Compression.cpp:117-143
size_t FP16Compressor::compress(const void* src, size_t nbytes, void* dst, size_t dst_capacity,
                                at::ScalarType dtype, uint64_t /*stable_id*/) {
    if (dtype == at::kHalf) {
        MCCL_CHECK(dst_capacity >= nbytes, "FP16 compress: buffer too small");
        device_copy(dst, src, nbytes);
        return nbytes;
    }
    MCCL_CHECK(dtype == at::kFloat, "FP16 compression only supports float32 input");
    const size_t count = nbytes / sizeof(float);
    const size_t compressed_bytes = count * sizeof(uint16_t);
    MCCL_CHECK(dst_capacity >= compressed_bytes, "FP16 compress: buffer too small");
    throw_on_status(mccl_hip_cast_f32_to_f16(static_cast<const float*>(src), dst, count,
                                             c10::hip::getCurrentHIPStream().stream()),
                    "FP16 compress");
    MCCL_TRACE("FP16 compress: %zu -> %zu bytes", nbytes, compressed_bytes);
    return compressed_bytes;
}

// csrc/compression/FP16Compression.cpp:145-163
void FP16Compressor::decompress(const void* src, size_t compressed_size, void* dst, size_t nbytes,
                                at::ScalarType dtype) {
    if (dtype == at::kHalf) {
        MCCL_CHECK(compressed_size == nbytes, "FP16 decompress: size mismatch");
        device_copy(dst, src, nbytes);
        return;
    }
    MCCL_CHECK(dtype == at::kFloat, "FP16 decompression only supports float32 output");
    const size_t count = nbytes / sizeof(float);
    MCCL_CHECK(compressed_size == count * sizeof(uint16_t), "FP16 decompress: compressed size mismatch");
    throw_on_status(mccl_hip_cast_f16_to_f32(src, static_cast<float*>(dst), count,
                                             c10::hip::getCurrentHIPStream().stream()),
                    "FP16 decompress");
}

TopKCompressor::TopKCompressor(double k_ratio) : k_ratio_(k_ratio) {
    MCCL_CHECK(k_ratio > 0 && k_ratio <= 1.0, "k_ratio must be in (0, 1], got " + std::to_string(k_ratio));
}

TopKCompressor::~TopKCompressor() {
    if (end_) (void)hipEventDestroy(static_cast<hipEvent_t>(end_));
}

// The residual map keeps the reference's rules (csrc/compression/TopKCompression.cpp:57-67):
// a new id while 1024 ids are live clears the map; an id whose element count changed starts
// again from zeros.  Caller holds mu_.
at::Tensor& TopKCompressor::residual_for(uint64_t stable_id, size_t count) {
    const auto opts_f = at::TensorOptions().dtype(at::kFloat).device(at::kCUDA);
    auto it = error_buffers_.find(stable_id);
    if (it == error_buffers_.end() && error_buffers_.size() >= kMaxErrorBuffers) {
        MCCL_WARN("TopK: evicting all %zu error feedback buffers (unstable tensor identities?)",
                  error_buffers_.size());
        error_buffers_.clear();
        evictions_++;
        it = error_buffers_.end();
    }
    if (it != error_buffers_.end() && static_cast<size_t>(it->second.numel()) == count) return it->second;
    return error_buffers_[stable_id] = at::zeros({static_cast<int64_t>(count)}, opts_f);
}

namespace {
void wait_for_current_stream() {
    throw_on_status(mccl_hip_sync(c10::hip::getCurrentHIPStream().stream()), "TopK stream wait");
}
}  // namespace

// The word the compress launches report a give-up through (a block of a launch that waited too
// long for another block of it).  The launches are asynchronous, so the word is looked at by the
// calls that wait for the stream anyway: decompress() and check_compress_status().  It is device
// memory, which goes back to its allocator in stream order: launches may still be under way when the
// compressor goes (a pinned word would be another tensor's by then).  Caller holds mu_.
namespace {
constexpr int64_t kCountersAt = 64;  // words

bool capturing(void* stream) {
    hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
    if (!stream) return false;
    if (hipStreamIsCapturing(static_cast<hipStream_t>(stream), &s) == hipSuccess) return s != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;
}
}  // namespace

// The decompress launches' counters lie behind the word, so that a compressor's first call clears both at once.
at::Tensor TopKCompressor::zeroed_words() {
    void* const stream = c10::hip::getCurrentHIPStream().stream();
    counters_ = at::zeros({kCountersAt + MCCL_HIP_DONE_BYTES / 4}, at::TensorOptions().dtype(at::kInt).device(at::kCUDA));
    counters_stream_ = stream;
    counters_usable_ = !capturing(stream);  // else nothing has been cleared
    counters_seen_ = false;
    return counters_;
}

int* TopKCompressor::compress_status() {
    if (!words_.defined()) words_ = zeroed_words();
    compressed_ = true;
    return words_.data_ptr<int>();
}

// Counters for a decompress launch on `stream`; null when they belong to another GPU.  Until a launch has reported
// through them they are known to be zero only in the order of the stream that cleared them.
void* TopKCompressor::decompress_counters(void* stream) {
    if (!counters_.defined() || !counters_usable_ || (!counters_seen_ && stream != counters_stream_)) zeroed_words();
    return counters_.get_device() == c10::hip::current_device() ? counters_.data_ptr<int>() + kCountersAt : nullptr;
}

// `st`: what the word held when the current stream had been waited for.
void TopKCompressor::throw_if_compress_failed(int st) {
    if (st == 0) return;
    words_.narrow(0, 0, 1).zero_();
    if (st == MCCL_HIP_ERR_TIMEOUT)
        throw TimeoutError("TopK compress: a block gave up waiting for another block of its launch; "
                           "the payloads of that call are invalid");
    throw_on_status(st, "TopK compress");
}

void TopKCompressor::check_compress_status() {
    std::lock_guard<std::mutex> lock(mu_);
    if (!compressed_) return;
    throw_if_compress_failed(words_.select(0, 0).item<int>());
}

// One bucket on `stream`: csrc/compression/TopKCompression.cpp:38-120.  Caller holds mu_.
size_t TopKCompressor::compress_on(const void* src, size_t nbytes, void* dst, size_t dst_capacity,
                                   at::Tensor& residual, at::Tensor& workspace, void* stream) {
    const size_t count = nbytes / sizeof(float);
    const uint32_t k = mccl_hip_topk_k(count, k_ratio_);
    const size_t output_size = sizeof(uint32_t) + static_cast<size_t>(k) * 8;
    const uint64_t ws_bytes = mccl_hip_topk_workspace_bytes(count, count, k_ratio_);
    if (!workspace.defined() || static_cast<uint64_t>(workspace.numel()) < ws_bytes) {
        workspace = at::empty({static_cast<int64_t>(ws_bytes)},
                              at::TensorOptions().dtype(at::kByte).device(at::kCUDA));
    }
    // The payload's pairs start 4 bytes in; the stride only has to be a multiple of 4.
    const uint64_t stride = static_cast<uint64_t>(dst_capacity) & ~uint64_t(3);
    const int rc = mccl_hip_topk_compress(static_cast<const float*>(src), residual.data_ptr<float>(), count,
                                          count, k_ratio_, dst, stride, workspace.data_ptr(),
                                          static_cast<uint64_t>(workspace.numel()), compress_status(), stream);
    if (rc == MCCL_HIP_ERR_CAPACITY) throw MCCLError("TopK compress: buffer too small");
    throw_on_status(rc, "TopK compress");
    MCCL_TRACE("TopK compress: %zu elements -> %u values, output %zu bytes", count, k, output_size);
    return output_size;
}

size_t TopKCompressor::compress(const void* src, size_t nbytes, void* dst, size_t dst_capacity,
                                at::ScalarType dtype, uint64_t stable_id) {
    MCCL_CHECK(dtype == at::kFloat, "TopK compression currently supports float32 only");
    const size_t count = nbytes / sizeof(float);
    MCCL_CHECK(count > 0, "TopK compress: empty input");
    const uint32_t k = mccl_hip_topk_k(count, k_ratio_);
    MCCL_CHECK(dst_capacity >= sizeof(uint32_t) + static_cast<size_t>(k) * 8, "TopK compress: buffer too small");
    std::lock_guard<std::mutex> lock(mu_);
    metal_kernels_init();
    at::Tensor& residual = residual_for(stable_id, count);
    return compress_on(src, nbytes, dst, dst_capacity, residual, workspace_,
                       c10::hip::getCurrentHIPStream().stream());
}

std::vector<at::Tensor> TopKCompressor::compress_many(const std::vector<at::Tensor>& buckets,
                                                      const std::vector<uint64_t>& stable_ids) {
    MCCL_CHECK(buckets.size() == stable_ids.size(), "compress_many: one stable id per bucket");
    std::vector<at::Tensor> payloads;
    if (buckets.empty()) return payloads;
    std::lock_guard<std::mutex> lock(mu_);
    metal_kernels_init();
    std::vector<at::Tensor*> residuals;
    payloads.reserve(buckets.size());
    residuals.reserve(buckets.size());
    const bool watched = allocations_are_watched();
    for (size_t i = 0; i < buckets.size(); i++) {
        const at::Tensor& t = buckets[i];
        check_single_tensor(t);
        MCCL_CHECK(t.scalar_type() == at::kFloat, "TopK compression currently supports float32 only");
        MCCL_CHECK(t.numel() > 0, "TopK compress: empty input");
        for (size_t j = 0; j < i; j++)
            MCCL_CHECK(stable_ids[j] != stable_ids[i], "compress_many: the same stable id twice in one call");
        // (allocated at its size: a narrowed view of a larger buffer takes the host another 0.6 us per bucket)
        payloads.push_back(empty_beside(t, static_cast<int64_t>(compressed_size(static_cast<size_t>(t.numel()))), at::kByte, watched));
    }
    const uint64_t evictions = evictions_;
    for (size_t i = 0; i < buckets.size(); i++)
        residuals.push_back(&residual_for(stable_ids[i], static_cast<size_t>(buckets[i].numel())));
    // (when the 1025th id has cleared the map on the way, the references from before that dangle)
    for (size_t i = 0; i < buckets.size() && evictions != evictions_; i++) {
        auto it = error_buffers_.find(stable_ids[i]);
        MCCL_CHECK(it != error_buffers_.end() && it->second.numel() == buckets[i].numel(),
                   "compress_many: more distinct stable ids than the compressor holds residuals for");
        residuals[i] = &it->second;
    }
    // the list goes to the library in chunks of MCCL_HIP_TOPK_LIST_MAX buckets: one launch per chunk or a few (topk_route.h)
    const int device = buckets[0].get_device();
    void* stream = c10::hip::getCurrentHIPStream(device).stream();
    for (size_t first = 0; first < buckets.size(); first += MCCL_HIP_TOPK_LIST_MAX) {
        const size_t n = std::min<size_t>(MCCL_HIP_TOPK_LIST_MAX, buckets.size() - first);
        std::vector<const float*> grads(n);
        std::vector<float*> res(n);
        std::vector<uint64_t> counts(n), caps(n);
        std::vector<void*> wires(n);
        for (size_t i = 0; i < n; i++) {
            grads[i] = buckets[first + i].data_ptr<float>();
            res[i] = residuals[first + i]->data_ptr<float>();
            counts[i] = static_cast<uint64_t>(buckets[first + i].numel());
            wires[i] = payloads[first + i].data_ptr();
            caps[i] = static_cast<uint64_t>(payloads[first + i].numel());
        }
        const uint64_t need = mccl_hip_topk_list_workspace_bytes(counts.data(), static_cast<uint32_t>(n), k_ratio_);
        if (!list_workspace_.defined() || static_cast<uint64_t>(list_workspace_.numel()) < need)
            list_workspace_ = at::empty({static_cast<int64_t>(need)},
                                        at::TensorOptions().dtype(at::kByte).device(at::kCUDA));
        const int rc = mccl_hip_topk_compress_list(grads.data(), res.data(), counts.data(), wires.data(), caps.data(),
                                                   static_cast<uint32_t>(n), k_ratio_, list_workspace_.data_ptr(),
                                                   static_cast<uint64_t>(list_workspace_.numel()), compress_status(),
                                                   stream);
        if (rc == MCCL_HIP_ERR_CAPACITY) throw MCCLError("TopK compress: buffer too small");
        throw_on_status(rc, "TopK compress");
    }
    return payloads;
}

// Marks the end of the launch on its stream, which the host does while it would only poll.  A program that waits for the
// stream or the GPU right behind the call has such a marker put there, and waits for that one, unless one is there
// already.  Compress and decompress at 1 % with a wait for the GPU behind them, us, waiting for the stream / reporting /
// reporting with the marker: 2000 elements 24.8 / 29.0 / 23.0, 65,537 32.6 / 36.4 / 30.5, 6,553,600 56.8 / 61.7 / 55.7.
// Pass after pass, without a wait, 1000 elements 21.1 / 18.0 / 17 to 20 from process to process, 65,537 29.1 / 25.8 / 25.2 to 26.6.
void TopKCompressor::mark_end(void* stream) {
    if (end_ && end_device_ != counters_.get_device()) {
        (void)hipEventDestroy(static_cast<hipEvent_t>(end_));
        end_ = nullptr;
    }
    if (!end_) {
        hipEvent_t event = nullptr;
        if (hipEventCreateWithFlags(&event, hipEventDisableTiming) == hipSuccess) end_ = event;
        end_device_ = counters_.get_device();
    }
    // (nothing but time depends on it)
    if (!end_ || hipEventRecord(static_cast<hipEvent_t>(end_), static_cast<hipStream_t>(stream)) != hipSuccess) (void)hipGetLastError();
}

// Waits until the decompress launch `ticket` has reported in status_, and returns what it reported: that
// precedes the end of the launch.  A report that takes longer than half a millisecond - earlier work on the stream -
// is waited for through the stream, like any other launch.
int TopKCompressor::wait_for_ticket(uint32_t ticket) {
    const uint64_t* const word = reinterpret_cast<const uint64_t*>(status_.data_ptr<int>() + 2);
    uint64_t seen = 0;
    const auto reported = [&] { return (seen = __atomic_load_n(word, __ATOMIC_ACQUIRE)) >> 32 == ticket; };
    const auto start = std::chrono::steady_clock::now();
    for (uint32_t polls = 0; !reported(); polls++) {
#if defined(__x86_64__)
        __builtin_ia32_pause();
#endif
        if ((polls & 63) == 63 && std::chrono::steady_clock::now() - start > std::chrono::microseconds(500)) {
            counters_usable_ = false;  // should the launch not have ended well
            wait_for_current_stream();
            MCCL_CHECK(reported(), "TopK decompress: the launch ended without a result");
            counters_usable_ = true;
            break;
        }
    }
    counters_seen_ = true;
    return static_cast<int>(static_cast<uint32_t>(seen));
}

// csrc/compression/TopKCompression.cpp:122-152.  The reference validates while
// it scatters and throws; here the launch reports in pinned host memory as soon as its
// stores have arrived, and brings the compress status along: no copy, and no wait for the
// end of the launch (the call is synchronous, as the reference's is).  A payload that does
// not ascend, or that breaks a rule, is expanded (again) by the kernels that take pairs in
// any order.
void TopKCompressor::decompress(const void* src, size_t compressed_size, void* dst, size_t nbytes,
                                at::ScalarType dtype) {
    MCCL_CHECK(dtype == at::kFloat, "TopK decompression currently supports float32 only");
    const size_t count = nbytes / sizeof(float);
    std::lock_guard<std::mutex> lock(mu_);
    metal_kernels_init();
    // int32 0: of the kernels that report a status, 1: the compress status as they bring it; 2, 3: wait_for_ticket's word
    if (!status_.defined()) status_ = at::zeros({4}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
    int* const word = status_.data_ptr<int>();
    void* const stream = c10::hip::getCurrentHIPStream().stream();
    float* const dense = static_cast<float*>(dst);
    const int* const flag = compressed_ ? words_.data_ptr<int>() : nullptr;
    const auto launched = [&](int rc) {
        if (rc == MCCL_HIP_ERR_SIZE) throw MCCLError("TopK decompress: size mismatch");
        throw_on_status(rc, "TopK decompress");
    };
    auto expand = [&](auto launch) {
        word[0] = word[1] = 0;
        launched(launch());
        wait_for_current_stream();
        return *static_cast<const volatile int*>(word);
    };
    int st = MCCL_HIP_ERR_ORDER;
    if (count) {
        // (a stream that is being captured refuses the wait, as it always has; the counters serve one GPU)
        int rc = MCCL_HIP_ERR_CAPACITY;
        void* const counters = capturing(stream) ? nullptr : decompress_counters(stream);
        if (counters) {
            if (++ticket_ == 0) ++ticket_;
            rc = mccl_hip_topk_decompress_sorted_done(src, compressed_size, dense, count, flag, counters,
                                                      reinterpret_cast<uint64_t*>(word + 2), ticket_, stream);
        }
        if (rc != MCCL_HIP_ERR_CAPACITY) {
            launched(rc);
            mark_end(stream);
            st = wait_for_ticket(ticket_);
        } else {
            st = expand([&] {
                return mccl_hip_topk_decompress_sorted_flag(src, compressed_size, dense, count, word, flag, flag ? word + 1 : nullptr, stream);
            });
            if (st == 0) st = *static_cast<const volatile int*>(word + 1);
        }
        if (st != MCCL_HIP_ERR_ORDER && st != MCCL_HIP_ERR_SIZE && st != MCCL_HIP_ERR_INDEX) {
            throw_if_compress_failed(st);
            return;
        }
    }
    st = expand([&] { return mccl_hip_topk_decompress(src, compressed_size, dense, count, word, stream); });
    if (flag) throw_if_compress_failed(words_.select(0, 0).item<int>());
    if (st == MCCL_HIP_ERR_SIZE) throw MCCLError("TopK decompress: size mismatch");
    if (st == MCCL_HIP_ERR_INDEX) throw MCCLError("TopK decompress: index out of bounds");
}

size_t TopKCompressor::max_compressed_size(size_t nbytes) const {
    return static_cast<size_t>(mccl_hip_topk_max_compressed_size(nbytes, k_ratio_));
}

size_t TopKCompressor::compressed_size(size_t count) const {
    return sizeof(uint32_t) + static_cast<size_t>(mccl_hip_topk_k(count, k_ratio_)) * 8;
}

void TopKCompressor::reset_error_feedback() {
    std::lock_guard<std::mutex> lock(mu_);
    error_buffers_.clear();
    MCCL_DEBUG("TopK: all error feedback buffers reset");
}

void TopKCompressor::reset_error_feedback_for_tensor(uint64_t stable_id) {
    std::lock_guard<std::mutex> lock(mu_);
    auto it = error_buffers_.find(stable_id);
    if (it != error_buffers_.end()) it->second.zero_();
}

size_t TopKCompressor::error_feedback_buffer_count() const {
    std::lock_guard<std::mutex> lock(mu_);
    return error_buffers_.size();
}

at::Tensor TopKCompressor::error_feedback_buffer(uint64_t stable_id) const {
    std::lock_guard<std::mutex> lock(mu_);
    auto it = error_buffers_.find(stable_id);
    return it == error_buffers_.end() ? at::Tensor() : it->second;
}

}  // namespace mccl
