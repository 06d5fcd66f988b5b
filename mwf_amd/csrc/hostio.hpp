// hostio.hpp -- the host boundary: states, spectra and fields between a
// caller's arrays and device memory.
//
// The reference's (slot, m, n) planes and the device's rows [n][slot][ldM] are
// transposed on the device (k_planes_out, k_planes_in); the host only copies
// bytes, through pinned staging chunks that the DMA fills or empties while
// other chunks are copied by a few threads (a caller's fresh pages fault in on
// all of them).  A state of M6 2048^2 modes (369 MB) came back in 50 ms when one
// thread transposed it, and takes 9.4 ms.
#pragma once
#include <hip/hip_runtime.h>

#include <condition_variable>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "common.hpp"

constexpr int PLT = 64; // m values per tile

// rows [n][slots][ldM] -> re, im planes (slots, M, NN) column-major
template <typename CT>
__global__ __launch_bounds__(256) void k_planes_out(const CT* __restrict__ rows, int slots, int M, int ldM,
                                                    double* __restrict__ re, double* __restrict__ im)
{
    extern __shared__ unsigned char smem_raw[];
    CT* tile = reinterpret_cast<CT*>(smem_raw); // [slots][PLT + 1]
    const int m0 = blockIdx.x * PLT, n = blockIdx.y;
    const int w = M - m0 < PLT ? M - m0 : PLT;
    for (int i = threadIdx.x; i < slots * PLT; i += blockDim.x) {
        const int s = i / PLT, m = i % PLT;
        if (m < w) tile[s * (PLT + 1) + m] = rows[((size_t)n * slots + s) * ldM + m0 + m];
    }
    __syncthreads();
    const size_t o = ((size_t)n * M + m0) * slots;
    for (int i = threadIdx.x; i < slots * w; i += blockDim.x) {
        const CT v = tile[(i % slots) * (PLT + 1) + i / slots];
        re[o + i] = (double)v.x;
        im[o + i] = (double)v.y;
    }
}

// the reverse; the padding m in [M, ldM) of every row is cleared
template <typename CT>
__global__ __launch_bounds__(256) void k_planes_in(const double* __restrict__ re, const double* __restrict__ im, int slots,
                                                   int M, int ldM, CT* __restrict__ rows)
{
    using E = decltype(CT{}.x);
    extern __shared__ unsigned char smem_raw[];
    CT* tile = reinterpret_cast<CT*>(smem_raw); // [slots][PLT + 1]
    const int m0 = blockIdx.x * PLT, n = blockIdx.y;
    const int w = M - m0 < PLT ? M - m0 : PLT, wp = ldM - m0 < PLT ? ldM - m0 : PLT;
    const size_t o = ((size_t)n * M + m0) * slots;
    for (int i = threadIdx.x; i < slots * w; i += blockDim.x)
        tile[(i % slots) * (PLT + 1) + i / slots] = CT{(E)re[o + i], (E)im[o + i]};
    __syncthreads();
    for (int i = threadIdx.x; i < slots * PLT; i += blockDim.x) {
        const int s = i / PLT, m = i % PLT;
        if (m < wp) rows[((size_t)n * slots + s) * ldM + m0 + m] = m < w ? tile[s * (PLT + 1) + m] : CT{(E)0, (E)0};
    }
}

// words of 8 bytes between device memory and a pinned chunk
static __global__ __launch_bounds__(256) void k_words(const unsigned long long* __restrict__ src, unsigned long long* __restrict__ dst,
                                                      unsigned n)
{
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

// A few copy threads, shared by every handle of the process and gone with the
// last one.  run() is one user's at a time; another caller meanwhile does its
// own work alone.
class CopyPool {
public:
    static std::shared_ptr<CopyPool> get()
    {
        static std::mutex mu;
        static std::weak_ptr<CopyPool> live;
        std::lock_guard<std::mutex> l(mu);
        auto p = live.lock();
        if (!p) live = p = std::shared_ptr<CopyPool>(new CopyPool());
        return p;
    }
    ~CopyPool()
    {
        {
            std::lock_guard<std::mutex> l(mu_);
            stop_ = true;
        }
        cv_.notify_all();
        for (auto& t : th_) t.join();
    }
    // memcpy(dst, src, n) in slices on the pool's threads and the caller's
    void copy(void* dst, const void* src, size_t n)
    {
        constexpr size_t MIN = 256 << 10; // a slice worth a wake-up
        std::unique_lock<std::mutex> one(user_, std::try_to_lock);
        if (n < 2 * MIN || !one.owns_lock() || !start()) {
            std::memcpy(dst, src, n);
            return;
        }
        {
            std::lock_guard<std::mutex> l(mu_);
            dst_ = (char*)dst;
            src_ = (const char*)src;
            n_ = n;
            slice_ = std::max(MIN, ((n / (NT + 1) + 4095) / 4096) * 4096);
            next_ = 0;
            busy_ = 0;
            gen_++;
        }
        for (size_t i = slice_; i < n; i += slice_) cv_.notify_one();
        work();
        std::unique_lock<std::mutex> l(mu_);
        done_.wait(l, [&] { return busy_ == 0; });
    }

private:
    static constexpr int NT = 7;
    bool start()
    {
        if (!th_.empty()) return true;
        try {
            for (int i = 0; i < NT; i++) th_.emplace_back([this] { loop(); });
        } catch (...) { // no more threads: those that started will do
        }
        return !th_.empty();
    }
    void work()
    {
        for (;;) {
            size_t o, m;
            {
                std::lock_guard<std::mutex> l(mu_);
                if (next_ >= n_) return;
                o = next_;
                m = std::min(slice_, n_ - o);
                next_ += m;
                busy_++;
            }
            std::memcpy(dst_ + o, src_ + o, m);
            std::lock_guard<std::mutex> l(mu_);
            if (--busy_ == 0 && next_ >= n_) done_.notify_one();
        }
    }
    void loop()
    {
        unsigned long long seen = 0;
        for (;;) {
            {
                std::unique_lock<std::mutex> l(mu_);
                cv_.wait(l, [&] { return stop_ || gen_ != seen; });
                if (stop_) return;
                seen = gen_;
            }
            work();
        }
    }
    std::mutex user_, mu_;
    std::condition_variable cv_, done_;
    std::vector<std::thread> th_;
    char* dst_ = nullptr;
    const char* src_ = nullptr;
    size_t n_ = 0, slice_ = 0, next_ = 0;
    int busy_ = 0;
    unsigned long long gen_ = 0;
    bool stop_ = false;
};

// Pinned staging of one handle: chunks, each with the event of its last copy.
// Transfers of up to DIRECT bytes are read or written by kernels in the first chunk
// itself, over the bus: a DMA after a kernel costs some 10 us more than the kernel
// alone, and now and then 100 (get_state of M4 32^2 modes, 54 KB, 28 us and at times
// 132 with the DMA, 18 without; 64^2, 220 KB, 35 and 24; 128^2, 889 KB, 64 and 53;
// from 1.4 MB on the two are alike).  A transfer that fits one chunk is one copy and
// one wait; longer ones run through all the chunks.
struct HostStage {
    static constexpr size_t CHUNK = 8 << 20; // M6 2048^2 get_state: 4 MB chunks 14 ms, 8 and 16 MB 9.4
    static constexpr int NSLOT = 4;
    static constexpr size_t DIRECT = 1 << 20;
    char* buf = nullptr;
    size_t chunk = 0;
    int nslot = 0;
    hipEvent_t ev[NSLOT] = {};
    std::shared_ptr<CopyPool> pool;

    hipError_t init(size_t most) // the largest transfer the handle is likely to make
    {
        nslot = most > CHUNK ? NSLOT : 1;
        chunk = std::min(CHUNK, (most + 4095) / 4096 * 4096);
        pool = CopyPool::get();
        hipError_t e = hipHostMalloc((void**)&buf, chunk * nslot, hipHostMallocCoherent); // kernels access it too (DIRECT)
        for (int i = 0; i < nslot && e == hipSuccess; i++) e = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming);
        return e;
    }
    void release()
    {
        for (auto& v : ev)
            if (v) (void)hipEventDestroy(v);
        if (buf) (void)hipHostFree(buf);
        *this = HostStage{};
    }
    // a transfer that kernels make themselves, to or from the first chunk
    bool direct(size_t bytes) const { return bytes <= DIRECT && bytes <= chunk; }
    hipError_t words(hipStream_t st, const void* src, void* dst, size_t bytes)
    {
        const unsigned n = (unsigned)(bytes / 8);
        hipLaunchKernelGGL(k_words, dim3((n + 255) / 256), dim3(256), 0, st, (const unsigned long long*)src,
                           (unsigned long long*)dst, n);
        return hipGetLastError();
    }
    // the first chunk to or from the host's arrays
    hipError_t drain(hipStream_t st, size_t bytes, void* dst0, size_t n0, void* dst1)
    {
        const hipError_t e = hipStreamSynchronize(st);
        if (e != hipSuccess) return e;
        pool->copy(dst0, buf, n0);
        if (bytes > n0) pool->copy(dst1, buf + n0, bytes - n0);
        return e;
    }
    void fill(size_t bytes, const void* src0, size_t n0, const void* src1)
    {
        pool->copy(buf, src0, n0);
        if (bytes > n0) pool->copy(buf + n0, src1, bytes - n0);
    }
    // device -> host, complete on return; the source's first n0 bytes go to dst0, the rest to dst1
    hipError_t d2h(hipStream_t st, const void* src, size_t bytes, void* dst0, size_t n0, void* dst1)
    {
        if (direct(bytes)) {
            const hipError_t e = words(st, src, buf, bytes);
            return e != hipSuccess ? e : drain(st, bytes, dst0, n0, dst1);
        }
        const size_t nc = (bytes + chunk - 1) / chunk;
        auto len = [&](size_t c) { return std::min(chunk, bytes - c * chunk); };
        auto slot = [&](size_t c) { return buf + (c % nslot) * chunk; };
        auto issue = [&](size_t c) {
            hipError_t e = hipMemcpyAsync(slot(c), (const char*)src + c * chunk, len(c), hipMemcpyDeviceToHost, st);
            return e != hipSuccess || nc == 1 ? e : hipEventRecord(ev[c % nslot], st);
        };
        hipError_t e = hipSuccess;
        for (size_t c = 0; c < nc && c < (size_t)nslot && e == hipSuccess; c++) e = issue(c);
        for (size_t c = 0; c < nc && e == hipSuccess; c++) {
            if ((e = nc == 1 ? hipStreamSynchronize(st) : hipEventSynchronize(ev[c % nslot])) != hipSuccess) break;
            const size_t a = c * chunk, b = a + len(c), m = std::min(std::max(a, n0), b);
            if (m > a) pool->copy((char*)dst0 + a, slot(c), m - a);
            if (b > m) pool->copy((char*)dst1 + (m - n0), slot(c) + (m - a), b - m);
            if (c + nslot < nc) e = issue(c + nslot);
        }
        if (e != hipSuccess) (void)hipStreamSynchronize(st); // nothing may still write the chunks
        return e;
    }
    hipError_t d2h(hipStream_t st, void* dst, const void* src, size_t bytes) { return d2h(st, src, bytes, dst, bytes, nullptr); }
    // host -> device, the sources read on return; n0 bytes from src0, the rest from src1
    hipError_t h2d(hipStream_t st, void* dst, size_t bytes, const void* src0, size_t n0, const void* src1)
    {
        if (direct(bytes)) {
            fill(bytes, src0, n0, src1);
            const hipError_t e = words(st, buf, dst, bytes);
            return e != hipSuccess ? e : hipStreamSynchronize(st);
        }
        const size_t nc = (bytes + chunk - 1) / chunk;
        hipError_t e = hipSuccess;
        for (size_t c = 0; c < nc && e == hipSuccess; c++) {
            char* s = buf + (c % nslot) * chunk;
            const size_t a = c * chunk, b = std::min(a + chunk, bytes), m = std::min(std::max(a, n0), b);
            if (c >= (size_t)nslot && (e = hipEventSynchronize(ev[c % nslot])) != hipSuccess) break;
            if (m > a) pool->copy(s, (const char*)src0 + a, m - a);
            if (b > m) pool->copy(s + (m - a), (const char*)src1 + (m - n0), b - m);
            if ((e = hipMemcpyAsync((char*)dst + a, s, b - a, hipMemcpyHostToDevice, st)) != hipSuccess) break;
            if (nc > 1) e = hipEventRecord(ev[c % nslot], st);
        }
        const hipError_t w = hipStreamSynchronize(st); // the chunks are free for the next transfer
        return e != hipSuccess ? e : w;
    }
    hipError_t h2d(hipStream_t st, void* dst, const void* src, size_t bytes) { return h2d(st, dst, bytes, src, bytes, nullptr); }
};

// Planes of `slots` slots, both directions; scratch holds 2 NN M slots doubles.
template <typename CT>
inline hipError_t planes_d2h(HostStage& hs, hipStream_t st, const Geo& g, int slots, const CT* rows, double* scratch,
                             double* re, double* im)
{
    const size_t n = (size_t)g.NN * g.M * slots, bytes = 2 * sizeof(double) * n;
    const bool direct = hs.direct(bytes);
    double* pl = direct ? reinterpret_cast<double*>(hs.buf) : scratch;
    hipLaunchKernelGGL(k_planes_out<CT>, dim3((g.M + PLT - 1) / PLT, g.NN), dim3(256), slots * (PLT + 1) * sizeof(CT), st,
                       rows, slots, g.M, g.ldM, pl, pl + n);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return direct ? hs.drain(st, bytes, re, bytes / 2, im) : hs.d2h(st, scratch, bytes, re, bytes / 2, im);
}
template <typename CT>
inline hipError_t planes_h2d(HostStage& hs, hipStream_t st, const Geo& g, int slots, const double* re, const double* im,
                             double* scratch, CT* rows)
{
    const size_t n = (size_t)g.NN * g.M * slots, bytes = 2 * sizeof(double) * n;
    const bool direct = hs.direct(bytes);
    hipError_t e = hipSuccess;
    if (direct) hs.fill(bytes, re, bytes / 2, im);
    else e = hs.h2d(st, scratch, bytes, re, bytes / 2, im);
    if (e != hipSuccess) return e;
    const double* pl = direct ? reinterpret_cast<const double*>(hs.buf) : scratch;
    hipLaunchKernelGGL(k_planes_in<CT>, dim3((g.ldM + PLT - 1) / PLT, g.NN), dim3(256), slots * (PLT + 1) * sizeof(CT), st, pl,
                       pl + n, slots, g.M, g.ldM, rows);
    e = hipGetLastError();
    return e == hipSuccess && direct ? hipStreamSynchronize(st) : e; // the chunk is free for the next transfer
}
