// Staged transfers (see host_stage.h). A copy call between pageable memory and the device costs 15 to 30 us
// before its first byte, and the scene state needed one per array and a status read besides; here a kernel
// moves a piece between device memory and the page-locked slot (and converts it), the caller waits once,
// and the pieces of a long transfer overlap with the host's own copies. us per pass, pageable copies ->
// staged: one frame of 125 tet vertices and its readback 280 -> 243, four of 205,379 3150 -> 2663, six of 24
// scenes set and read back 4400 -> 3350.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "errors.h"
#include "host_stage.h"

namespace gvbd {

namespace {

// n words; consecutive lanes take consecutive words, so that a wave's accesses to host memory are whole
// bursts
__global__ __launch_bounds__(256) void stage_words_kernel(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                          int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) dst[i] = src[i];
}

// 3 floats per element from float4s: n floats in all
__global__ __launch_bounds__(256) void stage_pack_kernel(const float* __restrict__ src, float* __restrict__ dst, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        dst[i] = src[i / 3 * 4 + i % 3];
}

// float4s (w = 0) from 3 floats per element: n elements
__global__ __launch_bounds__(256) void stage_unpack_kernel(const float* __restrict__ src, float4* __restrict__ dst,
                                                           int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        dst[i] = make_float4(src[3 * (int64_t)i], src[3 * (int64_t)i + 1], src[3 * (int64_t)i + 2], 0.f);
}

struct Piece {
    StagePart::Kind kind;
    char *host, *device;
    int count;
    size_t bytes;  // on the host side
};

void launch_piece(const Piece& p, char* slot, bool down, hipStream_t stream) {
    const int threads = p.kind == StagePart::VEC3 && down ? 3 * p.count : p.count;
    const dim3 grid(std::min((threads + 255) / 256, 1024));
    if (p.kind == StagePart::WORDS) {
        const char* src = down ? p.device : slot;
        char* dst = down ? slot : p.device;
        hipLaunchKernelGGL(stage_words_kernel, grid, dim3(256), 0, stream, (const uint32_t*)src, (uint32_t*)dst, p.count);
    } else if (down) {
        hipLaunchKernelGGL(stage_pack_kernel, grid, dim3(256), 0, stream, (const float*)p.device, (float*)slot,
                           3 * p.count);
    } else {
        hipLaunchKernelGGL(stage_unpack_kernel, grid, dim3(256), 0, stream, (const float*)slot, (float4*)p.device,
                           p.count);
    }
    hip_check(hipGetLastError(), "staged transfer");
}

}  // namespace

HostStage::~HostStage() {
    release();
    for (hipEvent_t e : done_)
        if (e) (void)hipEventDestroy(e);
}

void HostStage::release() {
    if (buf_) (void)hipHostFree(buf_);
    buf_ = nullptr;
}

void HostStage::usePageLocked(bool on) {
    std::lock_guard<std::mutex> lock(mutex_);
    pageLocked_ = on;
    if (!on) release();  // no transfer is under way
}

bool HostStage::allocated() {
    if (buf_) return true;
    for (hipEvent_t& e : done_)
        if (!e) hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "event create");
    if (hipHostMalloc((void**)&buf_, kSlots * kSlotBytes, hipHostMallocDefault) == hipSuccess) return true;
    (void)hipGetLastError();
    buf_ = nullptr;
    return false;
}

void HostStage::transfer(const std::vector<StagePart>& parts, bool down) {
    std::lock_guard<std::mutex> lock(mutex_);
    int current = 0;
    hip_check(hipGetDevice(&current), "hipGetDevice");
    if (current != device_) hip_check(hipSetDevice(device_), "hipSetDevice");
    if (pageLocked_ && allocated())
        staged(parts, down);
    else
        plain(parts, down);
    if (current != device_) hip_check(hipSetDevice(current), "hipSetDevice");
}

void HostStage::plain(const std::vector<StagePart>& parts, bool down) {
    std::vector<float4> wide;
    for (const StagePart& p : parts) {
        const bool vec = p.kind == StagePart::VEC3;
        float* host = (float*)p.host;
        if (vec) wide.resize(p.count);
        if (vec && !down)
            for (int64_t i = 0; i < p.count; ++i) wide[i] = make_float4(host[3 * i], host[3 * i + 1], host[3 * i + 2], 0.f);
        void* mem = vec ? (void*)wide.data() : p.host;
        const size_t bytes = (size_t)p.count * (vec ? sizeof(float4) : 4);
        if (bytes)
            hip_check(hipMemcpyAsync(down ? mem : p.device, down ? p.device : mem, bytes,
                                     down ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice, stream_),
                      "transfer");
        hip_check(hipStreamSynchronize(stream_), "transfer wait");
        if (vec && down)
            for (int64_t i = 0; i < p.count; ++i) std::memcpy(host + 3 * i, &wide[i], 3 * sizeof(float));
    }
    if (parts.empty()) hip_check(hipStreamSynchronize(stream_), "transfer wait");
}

void HostStage::staged(const std::vector<StagePart>& parts, bool down) {
    std::vector<Piece> pieces;
    for (const StagePart& p : parts) {
        const size_t hostSize = p.kind == StagePart::VEC3 ? 12 : 4, deviceSize = p.kind == StagePart::VEC3 ? 16 : 4;
        const int64_t most = (int64_t)(kSlotBytes / hostSize);
        for (int64_t b = 0; b < p.count; b += most) {
            const int n = (int)std::min(most, p.count - b);
            pieces.push_back({p.kind, (char*)p.host + hostSize * b, (char*)p.device + deviceSize * b, n, hostSize * n});
        }
    }
    const int n = (int)pieces.size();
    const auto slot = [&](int i) { return buf_ + kSlotBytes * (i % kSlots); };
    const bool once = n <= kSlots && !down;  // uploads that fit wait for all at the end
    if (down) {
        // few pieces: one wait; more: a piece's copy to the caller while the next ones come
        const bool single = n <= 2;
        for (int head = 0, tail = 0; tail < n; ++tail) {
            for (; head < n && head < tail + kSlots; ++head) {
                launch_piece(pieces[head], slot(head), true, stream_);
                if (!single) hip_check(hipEventRecord(done_[head % kSlots], stream_), "transfer record");
            }
            if (!single)
                hip_check(hipEventSynchronize(done_[tail % kSlots]), "transfer wait");
            else if (tail == 0)
                hip_check(hipStreamSynchronize(stream_), "transfer wait");
            std::memcpy(pieces[tail].host, slot(tail), pieces[tail].bytes);
        }
    } else {
        for (int i = 0; i < n; ++i) {
            if (i >= kSlots) hip_check(hipEventSynchronize(done_[i % kSlots]), "transfer wait");
            std::memcpy(slot(i), pieces[i].host, pieces[i].bytes);
            launch_piece(pieces[i], slot(i), false, stream_);
            if (!once) hip_check(hipEventRecord(done_[i % kSlots], stream_), "transfer record");
        }
    }
    // also for an empty transfer: the work queued before it is complete
    if (!down || n == 0) hip_check(hipStreamSynchronize(stream_), "transfer wait");
}

}  // namespace gvbd
