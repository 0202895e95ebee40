// host_scratch.h — one device buffer and one small pinned buffer per device for
// the host-array entry points (the *_host functions): the device buffer grown to
// the largest call, the pinned one to at most kHostStageMax, both kept until the
// process ends, so a call does not pay hipMalloc / hipFree.  A call holds the
// device's mutex from its first copy in to its last copy out; those calls are
// synchronous, so the buffers are free again when the mutex is released.
#ifndef NAV24_HOST_SCRATCH_H
#define NAV24_HOST_SCRATCH_H

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstring>
#include <mutex>
#include <vector>

namespace navba {

struct HostScratch {
    std::mutex mu;
    void* p = nullptr;
    size_t cap = 0;
    char* pin = nullptr;
    size_t pin_cap = 0;
};

// Largest call that goes through the pinned buffer.  A copy between pageable
// memory and the device costs the host 18 us whatever its size up to some
// hundred KiB, one queued from pinned memory 3 us and its share of one wait at
// the end; a megabyte is copied into the buffer in about 100 us, the time of the
// copies that it saves.
constexpr size_t kHostStageMax = size_t(1) << 20;

inline HostScratch& host_scratch(int device) {
    static std::mutex g;
    static std::vector<HostScratch*> v;
    std::lock_guard<std::mutex> lk(g);
    if ((int)v.size() <= device) v.resize(device + 1, nullptr);
    if (!v[device]) v[device] = new HostScratch();
    return *v[device];
}

// At least `bytes` on the current device; the caller holds s.mu.  nullptr if
// the allocation fails.
inline void* host_scratch_get(HostScratch& s, size_t bytes) {
    if (s.cap < bytes) {
        if (s.p) (void)hipFree(s.p);
        s.p = nullptr;
        s.cap = 0;
        if (hipMalloc(&s.p, bytes) != hipSuccess) {
            s.p = nullptr;
            return nullptr;
        }
        s.cap = bytes;
    }
    return s.p;
}

// At least `bytes` of pinned memory, which kernels can address; the caller holds
// s.mu.  nullptr above kHostStageMax or if the allocation fails: the call then
// copies from and to the caller's arrays themselves.
inline char* host_stage_get(HostScratch& s, size_t bytes) {
    if (bytes > kHostStageMax) return nullptr;
    if (s.pin_cap < bytes) {
        size_t cap = size_t(1) << 16;
        while (cap < bytes) cap *= 2;
        if (s.pin) (void)hipHostFree(s.pin);
        s.pin = nullptr;
        s.pin_cap = 0;
        void* q = nullptr;
        if (hipHostMalloc(&q, cap) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        s.pin = (char*)q;
        s.pin_cap = cap;
    }
    return s.pin;
}

// The arrays of one host-array call on the null stream: inputs, scratch and
// outputs laid out in the device buffer, inputs first and outputs last, so that
// one copy brings the inputs in and one the outputs back.
//   HostCall c;  auto a = c.in(src, bytes);  auto t = c.tmp(bytes);  auto r = c.out(dst, bytes);
//   if (!c.begin(hs)) ...;  launch with c.ptr<T>(a), ...;  if (!c.finish()) ...
// in, then tmp, then out; the caller holds the scratch's mutex.  begin fails for
// a null array of some bytes, as a copy from or to it would.
class HostCall {
public:
    int in(const void* src, size_t bytes) {
        null_ = null_ || (!src && bytes > 0);
        return add(src, nullptr, bytes, &in_end_);
    }
    int tmp(size_t bytes) { return add(nullptr, nullptr, bytes, &out_beg_); }
    int out(void* dst, size_t bytes) {
        null_ = null_ || (!dst && bytes > 0);
        return add(nullptr, dst, bytes, nullptr);
    }

    bool begin(HostScratch& hs) {
        if (null_) return false;
        if (out_beg_ < in_end_) out_beg_ = in_end_;
        d_ = (char*)host_scratch_get(hs, total_);
        if (!d_) return false;
        const size_t out_bytes = total_ - out_beg_;
        pin_ = host_stage_get(hs, in_end_ + out_bytes);
        if (pin_) {
            for (int k = 0; k < n_; ++k)
                if (a_[k].src && a_[k].bytes > 0) std::memcpy(pin_ + a_[k].at, a_[k].src, a_[k].bytes);
            return in_end_ == 0 || hipMemcpyAsync(d_, pin_, in_end_, hipMemcpyHostToDevice, nullptr) == hipSuccess;
        }
        for (int k = 0; k < n_; ++k)
            if (a_[k].src && a_[k].bytes > 0 &&
                hipMemcpy(d_ + a_[k].at, a_[k].src, a_[k].bytes, hipMemcpyHostToDevice) != hipSuccess)
                return false;
        return true;
    }

    // Waits for the launches and copies the outputs to the caller's arrays.
    bool finish() {
        if (pin_) {
            char* stage = pin_ + in_end_;
            bool ok = total_ == out_beg_ ||
                      hipMemcpyAsync(stage, d_ + out_beg_, total_ - out_beg_, hipMemcpyDeviceToHost, nullptr) == hipSuccess;
            ok = hipStreamSynchronize(nullptr) == hipSuccess && ok;
            for (int k = 0; k < n_ && ok; ++k)
                if (a_[k].dst && a_[k].bytes > 0) std::memcpy(a_[k].dst, stage + (a_[k].at - out_beg_), a_[k].bytes);
            return ok;
        }
        for (int k = 0; k < n_; ++k)
            if (a_[k].dst && a_[k].bytes > 0 &&
                hipMemcpy(a_[k].dst, d_ + a_[k].at, a_[k].bytes, hipMemcpyDeviceToHost) != hipSuccess)
                return false;
        return true;
    }

    // After a failed launch: nothing of the call may still be using the buffers.
    void abandon() { (void)hipStreamSynchronize(nullptr); }

    template <class T>
    T* ptr(int k) const { return (T*)(d_ + a_[k].at); }

private:
    static constexpr int kMaxArrays = 12;
    struct Array {
        const void* src;
        void* dst;
        size_t at, bytes;
    };
    int add(const void* src, void* dst, size_t bytes, size_t* end) {
        a_[n_] = Array{src, dst, total_, bytes};
        total_ += (bytes + 255) & ~size_t(255);
        if (end) *end = total_;
        return n_++;
    }
    Array a_[kMaxArrays];
    int n_ = 0;
    bool null_ = false;
    size_t total_ = 0, in_end_ = 0, out_beg_ = 0;
    char* d_ = nullptr;
    char* pin_ = nullptr;
};

}  // namespace navba

#endif  // NAV24_HOST_SCRATCH_H
