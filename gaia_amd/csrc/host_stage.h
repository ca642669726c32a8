// Transfers between caller's arrays and device arrays through page-locked memory that kernels read and
// write themselves.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <mutex>
#include <vector>

namespace gvbd {

// One array of a transfer: `count` elements. Kinds: plain 4-byte words, or 3 floats per element on the
// host and a float4 (w = 0) on the device.
struct StagePart {
    enum Kind { WORDS, VEC3 } kind;
    void* host;
    void* device;
    int64_t count;
};

// Page-locked staging memory of a context (4 MB, allocated at the first transfer). A transfer is
// ordered on the stream and complete when it returns; transfers of several threads take turns. Where the
// memory cannot be had, or with usePageLocked(false), transfers are plain copies of pageable memory.
class HostStage {
public:
    HostStage(int device, hipStream_t stream) : device_(device), stream_(stream) {}
    ~HostStage();
    HostStage(const HostStage&) = delete;
    HostStage& operator=(const HostStage&) = delete;

    void download(const std::vector<StagePart>& parts) { transfer(parts, true); }
    void upload(const std::vector<StagePart>& parts) { transfer(parts, false); }
    void usePageLocked(bool on);

private:
    static constexpr int kSlots = 8;
    static constexpr size_t kSlotBytes = ((size_t)512 << 10) / 48 * 48;  // whole float4s and whole elements
    void transfer(const std::vector<StagePart>& parts, bool down);
    bool allocated();
    void staged(const std::vector<StagePart>& parts, bool down);
    void plain(const std::vector<StagePart>& parts, bool down);
    void release();

    int device_;
    hipStream_t stream_;
    std::mutex mutex_;
    bool pageLocked_ = true;
    char* buf_ = nullptr;
    hipEvent_t done_[kSlots] = {};
};

}  // namespace gvbd
