// One device allocation cut into pieces, freed as one: an allocation takes about 50 us and a
// free, which waits for the device, 100 us, so a build's dozens of buffers cost more than
// their kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace wx {

class DeviceArena {
  public:
    DeviceArena() = default;
    ~DeviceArena() {
        if (base_) (void)hipFree(base_);
    }
    DeviceArena(const DeviceArena &) = delete;
    DeviceArena &operator=(const DeviceArena &) = delete;

    // Bytes a piece takes: pieces start at multiples of 256.
    static constexpr size_t piece(size_t bytes) { return (bytes + 255u) & ~size_t(255); }

    hipError_t allocate(size_t bytes) {
        const hipError_t e = hipMalloc(&base_, bytes ? bytes : 256u);
        if (e != hipSuccess) base_ = nullptr;
        return e;
    }
    // The next piece; the allocation is the sum of all pieces taken.
    template <typename T>
    T *take(size_t bytes) {
        char *p = static_cast<char *>(base_) + at_;
        at_ += piece(bytes);
        return reinterpret_cast<T *>(p);
    }

  private:
    void *base_ = nullptr;
    size_t at_ = 0;
};

}  // namespace wx
