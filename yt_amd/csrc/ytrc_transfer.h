// ytrc_transfer.h -- images and fields between pageable host memory and the
// device, through pinned buffers, by several host threads.
//
// What bounds a transfer: PCIe moves about 45 GB/s each way; one host thread
// moves 5 to 10 GB/s, less where it is the first to touch the pages of the
// caller's array.  A 1024^2 image is 4 to 12 MB of float32 planes on the
// device and 32 MB of float64 pixels for the caller, so one thread's copy,
// conversion and page faults took 2.5 ms for it, six times the projection
// kernel.  Here a kernel moves the planes to pinned memory, a quarter of them
// at a time, and up to 8 threads convert what has arrived.  Uploads run the
// other way: the threads fill a pinned buffer while the copy engine takes the
// one before it.
#pragma once
#include <hip/hip_runtime.h>
#include <sched.h>
#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace {

// Copies pixels [first, first + count) of nch planes of npix floats to pinned
// memory, plane c to dst + c stride (dst and stride: multiples of 4 floats;
// a plane itself starts at any float).  PCIe bounds it: 8 MB take about 0.2
// ms.  No LDS and few registers, so it runs beside the persistent kernels.
__global__ __launch_bounds__(256) void k_planes_to_host(const float *__restrict__ planes, int64_t npix, int64_t first,
                                                        int64_t count, int nch, float *__restrict__ dst, int64_t stride)
{
    for (int c = 0; c < nch; c++) {
        const float *s = planes + (int64_t)c * npix + first;
        float *d = dst + (int64_t)c * stride;
        for (int64_t i = 4 * ((int64_t)blockIdx.x * 256 + threadIdx.x); i < count; i += 1024 * (int64_t)gridDim.x) {
            if (i + 4 <= count) {
                *(float4 *)(d + i) = make_float4(s[i], s[i + 1], s[i + 2], s[i + 3]);
            } else {
                for (int64_t k = i; k < count; k++) d[k] = s[k];
            }
        }
    }
}

// A few host threads that help one caller at a time with a job of
// independent pieces, started at its first large one.  A helper that wakes
// after the job is over goes back to sleep: the caller waits only for those
// that entered it.
class Helpers {
  public:
    ~Helpers()
    {
        {
            std::lock_guard<std::mutex> lk(m_);
            quit_ = true;
        }
        cv_.notify_all();
        for (auto &t : threads_) t.join();
    }

    // Runs fn on the calling thread and on up to `helpers` others, until all
    // have returned.
    template <class F>
    void run(int helpers, F &fn)
    {
        if (helpers > 0) start();
        const int n = std::min<int>(helpers, (int)threads_.size());
        if (n <= 0) {
            fn();
            return;
        }
        {
            std::lock_guard<std::mutex> lk(m_);
            job_ = [](void *f) { (*(F *)f)(); };
            arg_ = &fn;
            room_ = n;
        }
        for (int i = 0; i < n; i++) cv_.notify_one();
        fn();
        std::unique_lock<std::mutex> lk(m_);
        room_ = 0;
        done_.wait(lk, [&] { return inside_ == 0; });
    }

  private:
    void start()
    {
        if (started_) return;
        started_ = true;
        cpu_set_t set;
        const int cpus = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
        try {
            for (int i = 0; i < std::min(cpus, 8) - 1; i++) threads_.emplace_back([this] { loop(); });
        } catch (const std::exception &) {
            // fewer helpers than wanted
        }
    }

    void loop()
    {
        std::unique_lock<std::mutex> lk(m_);
        while (true) {
            cv_.wait(lk, [&] { return quit_ || room_ > 0; });
            if (quit_) return;
            room_--;
            inside_++;
            void (*job)(void *) = job_;
            void *arg = arg_;
            lk.unlock();
            job(arg);
            lk.lock();
            if (--inside_ == 0) done_.notify_one();
        }
    }

    std::mutex m_;
    std::condition_variable cv_, done_;
    std::vector<std::thread> threads_;
    void (*job_)(void *) = nullptr;
    void *arg_ = nullptr;
    int room_ = 0, inside_ = 0;
    bool quit_ = false, started_ = false;
};

// A context's pinned buffers and helper threads.  One transfer at a time:
// `mu` is held by each; callers that find it taken copy by themselves.
class Transfer {
  public:
    struct Piece {
        const char *src;
        size_t bytes;
    };

    std::mutex mu;

    hipError_t open()
    {
        hipError_t e = hipHostMalloc((void **)&pin_, BUF, hipHostMallocMapped);
        if (e == hipSuccess) e = hipHostGetDevicePointer((void **)&d_pin_, pin_, 0);
        for (auto &ev : taken_)
            if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        for (auto &ev : part_)
            if (e == hipSuccess) e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        return e;
    }

    ~Transfer()
    {
        for (auto &ev : taken_)
            if (ev) hipEventDestroy(ev);
        for (auto &ev : part_)
            if (ev) hipEventDestroy(ev);
        if (pin_) hipHostFree(pin_);
        // (a forked child has none of the threads: nothing to wait for)
        if (pid_ == getpid()) delete helpers_;
    }

    // Calls each(first pixel, count, planes, stride) for consecutive runs of
    // the nch planes of npix floats at `planes` on the device, on several
    // threads at once: plane c of the run is at planes + c stride.  The
    // planes are read in order of stream s.  out and px_bytes: where the
    // caller's pixels go and what one takes there.
    template <class F>
    hipError_t read(hipStream_t s, const float *planes, int64_t npix, int nch, const void *out, size_t px_bytes, F &&each)
    {
        const int64_t most = (int64_t)(BUF / sizeof(float)) / nch / 4 * 4;
        for (int h = 0; h < 2; h++) {
            const hipError_t e = settle(h);
            if (e != hipSuccess) return e;
        }
        for (int64_t first = 0; first < npix; first += most) {
            const int64_t count = std::min(most, npix - first);
            const int64_t stride = (count + 3) / 4 * 4;
            // (parts of 256 KB or more, so that a small image is one launch)
            const int64_t part = std::max<int64_t>((count / PARTS + 3) / 4 * 4, 65536 / nch / 4 * 4);
            const int np = (int)((count + part - 1) / part);
            for (int k = 0; k < np; k++) {
                const int64_t at = k * part, n = std::min(part, count - at);
                const unsigned grid = (unsigned)std::min<int64_t>(256, (n + 1023) / 1024);
                hipLaunchKernelGGL(k_planes_to_host, dim3(grid), dim3(256), 0, s, planes, npix, first + at, n, nch,
                                   (float *)d_pin_ + at, stride);
                hipError_t e = hipGetLastError();
                if (e == hipSuccess) e = hipEventRecord(part_[k], s);
                if (e != hipSuccess) {
                    hipStreamSynchronize(s);
                    return e;
                }
            }
            const hipError_t e = hipEventSynchronize(part_[0]);
            if (e != hipSuccess) return e;
            std::atomic<int> err{(int)hipSuccess};
            std::atomic<int> here{1};  // parts known to have arrived
            convert((const float *)pin_, stride, count, (const char *)out + (size_t)first * px_bytes, px_bytes,
                    [&](int64_t a, int n, const float *p, int64_t st) {
                        for (int k = here.load(std::memory_order_acquire); (int64_t)k * part < a + n; k++) {
                            const hipError_t ee = hipEventSynchronize(part_[k]);
                            if (ee != hipSuccess) {
                                err.store((int)ee);
                                return;
                            }
                            here.store(k + 1, std::memory_order_release);
                        }
                        each(first + a, n, p, st);
                    });
            if (err.load() != (int)hipSuccess) {
                hipStreamSynchronize(s);
                return (hipError_t)err.load();
            }
        }
        return hipSuccess;
    }

    // read() of planes of npix floats that are in host memory already; by the
    // calling thread alone where it does not hold `mu`.
    template <class F>
    void read_here(bool held, const float *planes, int64_t npix, const void *out, size_t px_bytes, F &&each)
    {
        convert(planes, npix, npix, (const char *)out, px_bytes, each, held);
    }

    // Copies the pieces, one after another, to dst on the device in order of
    // stream s.  The last copies may still be running when it returns, and
    // reading the caller's memory: it stays until the stream has been waited
    // for.
    //
    // One or two pieces of up to 3 MB in all are copied as they are: the
    // runtime's own staging takes 20 us less than filling a window does (one
    // piece of 0.4 / 0.9 / 2.1 / 3.5 MB, upload and free: 62 / 78 / 150 / 205
    // us, through windows 88 / 143 / 166 / 198), but 12 us more for each
    // further piece, for two of up to 64 KB (20^3: 70 us, 60) and for one of
    // 16 to 48 KB (59 us, 50).  So are all pieces where another call has the
    // windows.
    hipError_t write(hipStream_t s, const std::vector<Piece> &pieces, char *dst)
    {
        std::vector<size_t> start(pieces.size() + 1, 0);
        for (size_t i = 0; i < pieces.size(); i++) start[i + 1] = start[i] + pieces[i].bytes;
        const size_t total = start.back();
        const bool few = total < FEW_BYTES && (pieces.size() == 1 ? total < UNIT / 4 || total > UNIT * 3 / 4
                                                                  : pieces.size() == 2 && total > 2 * UNIT);
        std::unique_lock<std::mutex> lk(mu, std::defer_lock);
        if (few || !lk.try_lock()) {
            for (size_t i = 0; i < pieces.size(); i++) {
                const hipError_t e =
                    hipMemcpyAsync(dst + start[i], pieces[i].src, pieces[i].bytes, hipMemcpyHostToDevice, s);
                if (e != hipSuccess) {
                    hipStreamSynchronize(s);
                    return e;
                }
            }
            return hipSuccess;
        }
        // quarters of a small upload, so that the copy engine starts early
        const size_t window = std::min(HALF, std::max<size_t>((total / 4 + 4095) / 4096 * 4096, 256u << 10));
        int h = 0;
        for (size_t w = 0; w < total; w += window, h ^= 1) {
            const size_t bytes = std::min(window, total - w);
            hipError_t e = settle(h);
            if (e != hipSuccess) return e;
            char *to = pin_ + h * HALF;
            const int nunit = (int)((bytes + UNIT - 1) / UNIT);
            std::atomic<int> next{0};
            auto job = [&] {
                for (int u; (u = next.fetch_add(1, std::memory_order_relaxed)) < nunit;) {
                    size_t a = w + (size_t)u * UNIT;
                    const size_t b = w + std::min(bytes, (size_t)(u + 1) * UNIT);
                    size_t i = (size_t)(std::upper_bound(start.begin(), start.end(), a) - start.begin()) - 1;
                    while (a < b) {
                        const size_t n = std::min(b, start[i + 1]) - a;
                        memcpy(to + (a - w), pieces[i].src + (a - start[i]), n);
                        a += n;
                        i++;
                    }
                }
            };
            helpers_->run(nunit - 1, job);
            e = hipMemcpyAsync(dst + w, to, bytes, hipMemcpyHostToDevice, s);
            if (e == hipSuccess) e = hipEventRecord(taken_[h], s);
            if (e != hipSuccess) {
                hipStreamSynchronize(s);
                return e;
            }
            busy_[h] = true;
        }
        return hipSuccess;
    }

    // For read-backs of finished images: the null stream, whose hardware
    // queue no context's stream shares.  (On a third stream they waited for
    // whole persistent kernels: a burst of 16 images took 15.3 instead of
    // 12.5 ms.)
    static constexpr hipStream_t stream = nullptr;

  private:
    static constexpr size_t BUF = 12u << 20;  // three planes of 1024^2
    static constexpr size_t HALF = 4u << 20;   // an upload's windows: the buffer's first two thirds
    static constexpr size_t UNIT = 64u << 10;  // of an upload, per thread
    static constexpr size_t FEW_BYTES = 3u << 20;
    static constexpr int PARTS = 4;
    static constexpr size_t PAGE = 2u << 20;

    // Runs each over the pixels in units of one huge page of the caller's
    // array: threads that fault on one page at once each clear 2 MB for it
    // and all but one throw it away.  Small arrays have small pages.
    template <class F>
    void convert(const float *planes, int64_t stride, int64_t count, const char *out, size_t px_bytes, F &&each,
                 bool helped = true)
    {
        const size_t bytes = (size_t)count * px_bytes;
        const size_t page = bytes >= 2 * PAGE ? PAGE : PAGE / 8;
        // pixels before the first page boundary, and of a page
        const int64_t unit = (int64_t)(page / px_bytes);
        int64_t lead = (int64_t)((page - (uintptr_t)out % page) % page / px_bytes);
        if (lead == 0) lead = unit;
        const int nu = count <= lead ? 1 : 1 + (int)((count - lead + unit - 1) / unit);
        std::atomic<int> next{0};
        auto job = [&] {
            for (int u; (u = next.fetch_add(1, std::memory_order_relaxed)) < nu;) {
                const int64_t a = u == 0 ? 0 : lead + (u - 1) * unit;
                const int64_t b = std::min(count, lead + u * unit);
                each(a, (int)(b - a), planes + a, stride);
            }
        };
        if (helped)
            helpers_->run(nu - 1, job);
        else
            job();
    }

    // Waits until the copy engine has taken half h.
    hipError_t settle(int h)
    {
        if (!busy_[h]) return hipSuccess;
        busy_[h] = false;
        return hipEventSynchronize(taken_[h]);
    }

    char *pin_ = nullptr, *d_pin_ = nullptr;
    hipEvent_t taken_[2] = {nullptr, nullptr};
    bool busy_[2] = {false, false};
    hipEvent_t part_[PARTS + 1] = {};
    Helpers *helpers_ = new Helpers();
    const pid_t pid_ = getpid();
};

}  // namespace
