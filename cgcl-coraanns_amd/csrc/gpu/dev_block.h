// The device arrays of one call of the index-build tools, in one allocation: a hipMalloc or hipFree
// of 2 MiB or more costs 10 to 40 us, a hipFree beyond 64 MiB 300 us, and a call holds up to
// twenty arrays.
//
// A block of up to kKeepBytes is kept for a later call, at most kKeepBlocks of them a device, the
// larger ones where there are more; calls from several threads never hold the same one. They
// are freed where the device has no room for a call's own.
#pragma once

#include <hip/hip_runtime.h>

#include <stddef.h>

#include <mutex>

namespace cora {

constexpr size_t kKeepBytes = size_t{256} << 20;
constexpr int kKeepBlocks = 2;  // a call's arrays and its split operands
constexpr int kKeepDevices = 16;

// The idle blocks. Never destroyed: at the process's end the runtime may already be gone.
class DevBlockPool {
  public:
    struct Block {
        void *p = nullptr;
        size_t size = 0;
    };
    static DevBlockPool &get() {
        static DevBlockPool *pool = new DevBlockPool();
        return *pool;
    }
    // the smallest idle block of at least size bytes
    Block take(int device, size_t size) {
        if (device < 0 || device >= kKeepDevices)
            return {};
        std::lock_guard<std::mutex> lock(mu_);
        Block *best = nullptr;
        for (Block &b : idle_[device])
            if (b.p && b.size >= size && (!best || b.size < best->size))
                best = &b;
        Block out;
        if (best) {
            out = *best;
            *best = Block();
        }
        return out;
    }
    // what is left over, to be freed (p == nullptr: nothing)
    Block keep(int device, Block block) {
        if (device < 0 || device >= kKeepDevices || block.size > kKeepBytes)
            return block;
        std::lock_guard<std::mutex> lock(mu_);
        Block *least = &idle_[device][0];
        for (Block &b : idle_[device])
            if (b.size < least->size)
                least = &b;
        if (least->size >= block.size)
            return block;
        const Block out = *least;
        *least = block;
        return out;
    }

  private:
    std::mutex mu_;
    Block idle_[kKeepDevices][kKeepBlocks];
};

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
    // on the current device
    hipError_t alloc() {
        if (hipGetDevice(&device_) != hipSuccess)
            device_ = -1;
        const size_t size = size_ ? size_ : 1;
        block_ = DevBlockPool::get().take(device_, size);
        if (!block_.p) {
            hipError_t e = hipMalloc(&block_.p, size);
            while (e == hipErrorOutOfMemory) {
                const DevBlockPool::Block idle = DevBlockPool::get().take(device_, 0);
                if (!idle.p)
                    break;
                (void)hipGetLastError();
                (void)hipFree(idle.p);
                e = hipMalloc(&block_.p, size);
            }
            if (e != hipSuccess) {
                block_ = {};
                return e;
            }
            block_.size = size;
        }
        for (int i = 0; i < parts_; ++i)
            *part_[i].p = static_cast<char *>(block_.p) + part_[i].at;
        return hipSuccess;
    }

  private:
    void release() {
        if (!block_.p)
            return;
        // the call's work is on the null stream; after an error some of it may still be in flight
        if (hipStreamSynchronize(nullptr) == hipSuccess)
            block_ = DevBlockPool::get().keep(device_, block_);
        if (block_.p)
            (void)hipFree(block_.p);
        block_ = {};
    }

    static constexpr int kParts = 24;
    struct Part {
        void **p;
        size_t at;
    };
    Part part_[kParts] = {};
    int parts_ = 0;
    size_t size_ = 0;
    int device_ = -1;
    DevBlockPool::Block block_;
};

}  // namespace cora
