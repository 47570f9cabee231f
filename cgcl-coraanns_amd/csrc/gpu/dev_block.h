// The device arrays of one call of the index-build tools, in one allocation: a hipMalloc or hipFree
// of 2 MiB or more costs 10 to 40 us, a hipFree beyond 64 MiB 300 us, and a call holds up to
// twenty arrays.
#pragma once

#include <hip/hip_runtime.h>

#include <stddef.h>

namespace cora {

class DevBlock {
  public:
    DevBlock() = default;
    ~DevBlock() { release(); }
    DevBlock(const DevBlock &) = delete;
    DevBlock &operator=(const DevBlock &) = delete;

    // p [n] is part of the block from alloc() to release(). At most kParts parts, all added before.
    template <class T>
    void add(T *&p, size_t n) {
        part_[parts_++] = {reinterpret_cast<void **>(&p), size_};
        size_ += (n * sizeof(T) + 255) / 256 * 256;
    }
    hipError_t alloc() {
        const hipError_t e = hipMalloc(&base_, size_ ? size_ : 1);
        if (e != hipSuccess) {
            base_ = nullptr;
            return e;
        }
        for (int i = 0; i < parts_; ++i)
            *part_[i].p = static_cast<char *>(base_) + part_[i].at;
        return hipSuccess;
    }
    void release() {
        if (base_)
            (void)hipFree(base_);
        base_ = nullptr;
    }

  private:
    static constexpr int kParts = 24;
    struct Part {
        void **p;
        size_t at;
    };
    Part part_[kParts] = {};
    int parts_ = 0;
    size_t size_ = 0;
    void *base_ = nullptr;
};

}  // namespace cora
