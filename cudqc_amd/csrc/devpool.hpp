// Device buffers kept between handles and calls. A search opens a handle, whose clique store
// alone is 2.25 GiB, and closes it at the end; handing that much memory back to the driver and
// taking it again costs some 70 ms a call once the driver has to clear pages (a search of a
// 1,000-vertex graph takes 2 to 4 ms otherwise). Freed buffers are held here instead, at most
// POOL_BYTES in all, and serve the next request of the same size on the same device. They
// hold no data anyone relies on. They go back to the driver when an allocation fails (it is then
// tried again) or the bound is met, oldest first. Safe with several threads; a buffer is
// released only after the stream that used it was waited for, so any stream may take it.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <mutex>
#include <vector>

namespace dqc {

class DevicePool {
public:
    static constexpr size_t POOL_BYTES = 4ull << 30;
    static DevicePool& get() {
        static DevicePool* pool = new DevicePool();  // (never destroyed: the runtime may be gone by then)
        return *pool;
    }
    // Requests are rounded up to an eighth of their power of two, so that graphs of about the
    // same size share buffers.
    static size_t rounded(size_t bytes) {
        if (bytes > POOL_BYTES) return bytes;
        size_t step = 256;
        while (step * 16 <= bytes) step <<= 1;
        return (bytes + step - 1) / step * step;
    }
    // A buffer of `bytes` on the current device.
    hipError_t take(void** p, size_t bytes) {
        bytes = rounded(bytes);
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        {
            std::lock_guard<std::mutex> lock(mu_);
            for (size_t i = held_.size(); i-- > 0;)
                if (held_[i].dev == dev && held_[i].bytes == bytes) {
                    *p = held_[i].p;
                    total_ -= bytes;
                    held_.erase(held_.begin() + (std::ptrdiff_t)i);
                    return hipSuccess;
                }
        }
        e = hipMalloc(p, bytes);
        if (e == hipSuccess) return e;
        (void)hipGetLastError();
        drop(dev);
        return hipMalloc(p, bytes);
    }
    // Takes back a buffer of take() on the current device; all work that used it is done.
    void give(void* p, size_t bytes) {
        bytes = rounded(bytes);
        int dev = 0;
        if (bytes > POOL_BYTES || hipGetDevice(&dev) != hipSuccess) {
            hipFree(p);
            return;
        }
        std::vector<Block> out;
        {
            std::lock_guard<std::mutex> lock(mu_);
            held_.push_back({dev, bytes, p});
            total_ += bytes;
            while (total_ > POOL_BYTES) {
                out.push_back(held_.front());
                total_ -= held_.front().bytes;
                held_.erase(held_.begin());
            }
        }
        for (const Block& b : out) hipFree(b.p);
    }

private:
    struct Block { int dev; size_t bytes; void* p; };
    void drop(int dev) {
        std::vector<Block> out;
        {
            std::lock_guard<std::mutex> lock(mu_);
            for (size_t i = held_.size(); i-- > 0;)
                if (held_[i].dev == dev) {
                    out.push_back(held_[i]);
                    total_ -= held_[i].bytes;
                    held_.erase(held_.begin() + (std::ptrdiff_t)i);
                }
        }
        for (const Block& b : out) hipFree(b.p);
    }
    std::mutex mu_;
    std::vector<Block> held_;
    size_t total_ = 0;
};

}  // namespace dqc
