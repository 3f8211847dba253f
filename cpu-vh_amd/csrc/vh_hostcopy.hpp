// Device-to-host copies through pinned memory that its owner keeps.
//
// A download used to copy to the caller's pageable memory and then the error
// word to a local variable, each a staged copy of the runtime with a wait of
// its own, and in the mixed form allocated and freed a device buffer for the
// widened values (a free waits for the whole device).  Here the field's
// chunks and the error word go to pinned memory on the owner's stream, with
// one wait for a field of one chunk; a longer field's chunks alternate between
// two halves, one filled while the other is handed to the caller.  An FP32
// field crosses as it is stored and is widened on the way out.
#pragma once
#include <hip/hip_runtime.h>
#include <xmmintrin.h>

#include <algorithm>
#include <cstring>
#include <mutex>

namespace vh {

class HostCopy {
  public:
    // Room for copies of at most largest doubles (longer ones go in chunks).
    hipError_t init(size_t largest) {
        half_ = std::min(MAX_HALF, std::max<size_t>(largest, 1));
        hipError_t r = hipHostMalloc((void **)&buf_, 2 * half_ * sizeof(double) + ERR_BYTES, hipHostMallocDefault);
        for (int k = 0; k < 2 && r == hipSuccess; ++k) r = hipEventCreateWithFlags(&full_[k], hipEventDisableTiming);
        return r;
    }
    void release() {
        if (buf_) (void)hipHostFree(buf_);
        buf_ = nullptr;
        for (auto &e : full_) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
    }
    // Whether p is memory the runtime knows (pinned, managed, device): a copy
    // there needs no staging, and the owners make it directly.
    static bool registered(const void *p) {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        return a.type != hipMemoryTypeUnregistered;
    }
    // Whether the error word is set once the stream's work has ended; waits.
    hipError_t status(const int *d_err, hipStream_t st, bool *err) {
        std::lock_guard<std::mutex> lock(mu_);
        hipError_t r = fetch_err(d_err, st);
        const hipError_t w = hipStreamSynchronize(st);
        if (r == hipSuccess) r = w;
        if (r == hipSuccess) *err = words()[0] != 0;
        return r;
    }
    // n doubles, and whether the error word is set; waits.
    hipError_t fetch(double *out, const double *src, size_t n, const int *d_err, hipStream_t st, bool *err) {
        return chunks(
            n, d_err, st, err,
            [&](double *b, size_t at, size_t len) {
                return hipMemcpyAsync(b, src + at, len * sizeof(double), hipMemcpyDeviceToHost, st);
            },
            [&](const double *b, size_t at, size_t len) { std::memcpy(out + at, b, len * sizeof(double)); });
    }
    // n values hi (+ lo where not null), widened, and whether the error word is set; waits.
    hipError_t fetch_widened(double *out, const float *hi, const float *lo, size_t n, const int *d_err, hipStream_t st,
                             bool *err) {
        return chunks(
            n, d_err, st, err,
            [&](double *b, size_t at, size_t len) {
                float *f = reinterpret_cast<float *>(b);
                hipError_t r = hipMemcpyAsync(f, hi + at, len * sizeof(float), hipMemcpyDeviceToHost, st);
                if (r == hipSuccess && lo)
                    r = hipMemcpyAsync(f + len, lo + at, len * sizeof(float), hipMemcpyDeviceToHost, st);
                return r;
            },
            [&](const double *b, size_t at, size_t len) {
                const float *h = reinterpret_cast<const float *>(b);
                widen(out + at, h, lo ? h + len : nullptr, len);
            });
    }
    // out = hi (+ lo where not null), whatever the calling thread's MXCSR says:
    // a thread that takes subnormals as zero (torch.set_flush_denormal, programs
    // built with -ffast-math) gets an FP32 field's subnormal values all the same.
    __attribute__((noinline)) static void widen(double *out, const float *hi, const float *lo, size_t n) {
        const unsigned mxcsr = _mm_getcsr();
        _mm_setcsr(mxcsr & ~0x8040u);  // neither denormals-are-zero nor flush-to-zero
        if (lo)
            for (size_t i = 0; i < n; ++i) out[i] = (double)hi[i] + (double)lo[i];
        else
            for (size_t i = 0; i < n; ++i) out[i] = (double)hi[i];
        _mm_setcsr(mxcsr);
    }

  private:
    static constexpr size_t MAX_HALF = size_t(1) << 17;  // doubles: 1 MiB, within a core's L2
    static constexpr size_t ERR_BYTES = 64;
    int *words() { return reinterpret_cast<int *>(buf_ + 2 * half_); }  // the three error words
    hipError_t fetch_err(const int *d_err, hipStream_t st) {
        return hipMemcpyAsync(words(), d_err, 3 * sizeof(int), hipMemcpyDeviceToHost, st);
    }
    template <class COPY, class TAKE>
    hipError_t chunks(size_t n, const int *d_err, hipStream_t st, bool *err, COPY &&copy, TAKE &&take) {
        std::lock_guard<std::mutex> lock(mu_);
        const size_t count = (n + half_ - 1) / half_;
        auto start = [&](size_t c) {
            hipError_t r = copy(buf_ + (c & 1) * half_, c * half_, std::min(half_, n - c * half_));
            if (r == hipSuccess && c + 1 == count) r = fetch_err(d_err, st);
            return r == hipSuccess ? hipEventRecord(full_[c & 1], st) : r;
        };
        hipError_t r = start(0);
        for (size_t c = 0; c < count && r == hipSuccess; ++c) {
            if (c + 1 < count) r = start(c + 1);
            if (r == hipSuccess) r = hipEventSynchronize(full_[c & 1]);
            if (r == hipSuccess) take(buf_ + (c & 1) * half_, c * half_, std::min(half_, n - c * half_));
        }
        if (r != hipSuccess) (void)hipStreamSynchronize(st);  // no copy still writes the buffer
        else *err = words()[0] != 0;
        return r;
    }
    std::mutex mu_;  // held from the first copy into the pinned memory to its last reading: threads take turns
    double *buf_ = nullptr;
    size_t half_ = 0;
    hipEvent_t full_[2] = {};
};

}  // namespace vh
