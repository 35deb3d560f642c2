// Field transfer between the device's structure-of-arrays state (FP64 or FP32 planes) and
// the caller's node-major double arrays.
//
// Large fields go through a ring of pinned buffers: a kernel converts and transposes one
// chunk between the device planes and a buffer (it addresses the pinned memory itself, so
// there is no second device copy), while worker threads move the finished chunks between
// the buffers and the caller's memory.  What bounds it is the host side: one thread
// writing fresh pages of the caller's array and transposing there ran at 4 GB/s of doubles
// (256^3 U in 103 ms), so the copies run on several threads and the layout change on the
// GPU.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

#include "case.h"
#include "transfer.h"

namespace mplb {

namespace {

constexpr int kBuffers = 8;
constexpr size_t kBufBytes = size_t(2) << 20;
constexpr int kWorkers = 8;

// doubles [first, first + n) of the node-major array <-> planes [comps][N]
template <typename T>
__global__ void __launch_bounds__(256) k_pack(const T* __restrict__ planes, int64_t N, int comps, int64_t first,
                                              int n, double* __restrict__ out) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int64_t g = first + e, i = g / comps;
    out[e] = (double)planes[(g - i * comps) * N + i];
}

template <typename T>
__global__ void __launch_bounds__(256) k_unpack(T* __restrict__ planes, int64_t N, int comps, int64_t first, int n,
                                                const double* __restrict__ in) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int64_t g = first + e, i = g / comps;
    planes[(g - i * comps) * N + i] = (T)in[e];
}

}  // namespace

// The pinned ring of one case: allocated at its first large transfer, freed with the case.
struct HostStage {
    double* buf[kBuffers] = {nullptr};
    hipEvent_t ev[kBuffers] = {nullptr};
};

static int stage_fail(mplb_case* c, hipError_t e, const char* what) {
    c->err = std::string(what) + ": " + hipGetErrorString(e);
    return MPLB_E_HIP;
}

void stage_free(mplb_case* c) {
    if (!c->stage) return;
    for (int i = 0; i < kBuffers; i++) {
        if (c->stage->buf[i]) (void)hipHostFree(c->stage->buf[i]);
        if (c->stage->ev[i]) (void)hipEventDestroy(c->stage->ev[i]);
    }
    delete c->stage;
    c->stage = nullptr;
}

bool stage_wanted(mplb_case* c, int64_t N, int comps) {
    if ((size_t)N * comps * sizeof(double) < 2 * kBufBytes) return false;
    if (c->stage) return true;
    const DeviceScope device(c->opts.device);
    c->stage = new HostStage();
    hipError_t e = device.err;
    for (int i = 0; i < kBuffers && e == hipSuccess; i++) {
        e = hipHostMalloc((void**)&c->stage->buf[i], kBufBytes, hipHostMallocDefault);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&c->stage->ev[i], hipEventDisableTiming);
    }
    if (e == hipSuccess) return true;
    (void)hipGetLastError();        // (not an error of the next launch)
    stage_free(c);
    return false;
}

int stage_transfer(mplb_case* c, void* planes, int64_t N, int comps, double* host, bool to_device) {
    const DeviceScope device(c->opts.device);
    if (device.err != hipSuccess) return stage_fail(c, device.err, "field transfer");
    HostStage* s = c->stage;
    const int64_t total = N * comps, per = kBufBytes / sizeof(double);
    const int64_t chunks = (total + per - 1) / per;
    auto launch = [&](int64_t k) {
        const int64_t first = k * per;
        const int n = (int)std::min<int64_t>(per, total - first);
        const dim3 grid((unsigned)((n + 255) / 256));
        double* b = s->buf[k % kBuffers];
        if (c->scalar_bytes == 8) {
            if (to_device) k_unpack<double><<<grid, 256, 0, c->stream>>>((double*)planes, N, comps, first, n, b);
            else k_pack<double><<<grid, 256, 0, c->stream>>>((const double*)planes, N, comps, first, n, b);
        } else {
            if (to_device) k_unpack<float><<<grid, 256, 0, c->stream>>>((float*)planes, N, comps, first, n, b);
            else k_pack<float><<<grid, 256, 0, c->stream>>>((const float*)planes, N, comps, first, n, b);
        }
        return hipEventRecord(s->ev[k % kBuffers], c->stream);
    };
    auto copy = [&](int64_t k) {
        const int64_t first = k * per;
        const size_t bytes = sizeof(double) * (size_t)std::min<int64_t>(per, total - first);
        if (to_device) std::memcpy(s->buf[k % kBuffers], host + first, bytes);
        else std::memcpy(host + first, s->buf[k % kBuffers], bytes);
    };
    // Chunks pass through two stages in order: host copy -> kernel (to the device) or
    // kernel -> host copy (from it).  `ready` chunks may be copied, `copied` marks the
    // copies that are done.
    std::mutex mu;
    std::condition_variable cv;
    std::vector<char> copied((size_t)chunks, 0);
    int64_t ready = 0, next = 0;
    auto work = [&]() {
        for (;;) {
            int64_t k;
            {
                std::unique_lock<std::mutex> lk(mu);
                cv.wait(lk, [&] { return next >= chunks || next < ready; });
                if (next >= chunks) return;
                k = next++;
            }
            copy(k);
            {
                std::lock_guard<std::mutex> lk(mu);
                copied[(size_t)k] = 1;
            }
            cv.notify_all();
        }
    };
    std::vector<std::thread> pool;
    try {
        for (int w = 0; w < (int)std::min<int64_t>(kWorkers, chunks); w++) pool.emplace_back(work);
    } catch (const std::exception&) {
        // fewer threads than asked for; with none at all this thread copies
    }
    hipError_t e = hipSuccess;
    auto release = [&](int64_t upto) {
        {
            std::lock_guard<std::mutex> lk(mu);
            ready = upto;
        }
        cv.notify_all();
        if (pool.empty())
            for (; next < ready; next++) {
                copy(next);
                copied[(size_t)next] = 1;
            }
    };
    auto wait_copied = [&](int64_t k) {
        std::unique_lock<std::mutex> lk(mu);
        cv.wait(lk, [&] { return copied[(size_t)k] != 0; });
    };
    if (to_device) {
        for (int64_t k = 0; k < chunks && e == hipSuccess; k++) {
            // buffers free for copying: those whose kernel of kBuffers chunks ago is done
            if (k == 0) release(std::min<int64_t>(kBuffers, chunks));
            wait_copied(k);
            e = launch(k);
            if (k + 1 >= kBuffers / 2) {
                const int64_t done = k + 1 - kBuffers / 2;     // its buffer takes chunk done + kBuffers
                if (e == hipSuccess) e = hipEventSynchronize(s->ev[done % kBuffers]);
                if (e == hipSuccess) release(std::min<int64_t>(done + 1 + kBuffers, chunks));
            }
        }
    } else {
        for (int64_t k = 0; k < chunks + kBuffers / 2 && e == hipSuccess; k++) {
            if (k < chunks) {
                if (k >= kBuffers) wait_copied(k - kBuffers);
                e = launch(k);
            }
            const int64_t d = k - kBuffers / 2;
            if (d >= 0 && e == hipSuccess) {
                e = hipEventSynchronize(s->ev[d % kBuffers]);
                if (e == hipSuccess) release(d + 1);
            }
        }
    }
    {
        std::unique_lock<std::mutex> lk(mu);
        // on an error the chunks not yet released are given up
        if (e != hipSuccess) next = chunks;
    }
    cv.notify_all();
    for (auto& t : pool) t.join();
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e == hipSuccess) e = hipGetLastError();
    return e == hipSuccess ? 0 : stage_fail(c, e, "field transfer");
}

}  // namespace mplb
