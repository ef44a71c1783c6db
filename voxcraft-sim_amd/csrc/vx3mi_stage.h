// vx3mi_stage.h -- reading device arrays of four-word records back to the host
// through a pinned buffer.
//
// A kernel on the batch's own stream writes the rows of up to four arrays side by
// side into mapped host memory, a chunk of them at a time while the host unpacks
// the chunk before.  One launch and one wait where a copy of each array into
// pageable memory took a wait for the stream and a staged copy each: the state of
// 64 voxels in FP64 in 12 us instead of 50, a call of ten steps with its state 138 -> 92 us;
// 315,000 voxels in FP32 without four buffers of their own to be paged in first.
// What bounds it: the host's unpacking, and for a few rows the launch and the wait.
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>

#include "vx3mi_batch.h"

namespace vx3mi {

// the stream's device for as long as this lives: what is made on first use belongs to
// it, whichever device the calling thread has at the time
class OnDevice {
    int before = -1;

public:
    explicit OnDevice(hipStream_t stream) {
        int now = -1, its = -1;
        if (hipGetDevice(&now) == hipSuccess && hipStreamGetDevice(stream, &its) == hipSuccess && now != its && hipSetDevice(its) == hipSuccess)
            before = now;
    }
    ~OnDevice() {
        if (before >= 0) (void)hipSetDevice(before);
    }
    OnDevice(const OnDevice &) = delete;
    OnDevice &operator=(const OnDevice &) = delete;
};

template <typename W> struct StageRows {  // arrays of n[k] rows
    const W *src[4];
    int n[4];
};

// rows [i0, i0 + m) of array blockIdx.y to out + m blockIdx.y
template <typename W> __global__ __launch_bounds__(256) void k_stage(StageRows<W> rows, int i0, int m, W *out) {
    const int k = blockIdx.y, i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < m && i0 + i < rows.n[k]) out[(long)k * m + i] = rows.src[k][i0 + i];
}

// One per batch; any thread may read.
template <typename W> class Stage {
    static constexpr int kRows = 16384;  // of all arrays together, per buffer (two of 256 KB or 512 KB)
    std::mutex lock;
    W *host = nullptr;
    int rowsHeld = 0;
    hipEvent_t done[2] = {};

    // room for the rows of a read, one buffer or two, kept for the next (pinning
    // 1 MB takes 0.13 ms: a small batch holds what it needs)
    int ready(hipStream_t stream, int need, bool chunks) {
        if (need <= rowsHeld && !(chunks && !done[1])) return VX3MI_OK;
        OnDevice there(stream);
        for (hipEvent_t &e : done)
            if (chunks && !e) HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        if (need <= rowsHeld) return VX3MI_OK;
        if (host) HIP_TRY(hipHostFree(host));
        host = nullptr;
        rowsHeld = 0;
        HIP_TRY(hipHostMalloc((void **)&host, sizeof(W) * need, hipHostMallocDefault));
        rowsHeld = need;
        return VX3MI_OK;
    }

public:
    Stage() = default;
    Stage(const Stage &) = delete;
    // (reads have ended when they return, so nothing writes the buffer any more)
    ~Stage() {
        if (host) (void)hipHostFree(host);
        for (hipEvent_t e : done)
            if (e) (void)hipEventDestroy(e);
    }

    // The rows of K arrays as they are once the stream's work so far is done:
    // unpack(i0, m, at) for each chunk in order, where row i0 + i (i < m) of array
    // k, if it has one, is at[k * m + i].
    template <typename F> int read(hipStream_t stream, int K, const StageRows<W> &rows, F &&unpack) {
        std::lock_guard<std::mutex> hold(lock);
        int n = 0;
        for (int k = 0; k < K; k++) n = rows.n[k] > n ? rows.n[k] : n;
        if (n == 0) {
            HIP_TRY(hipStreamSynchronize(stream));
            return VX3MI_OK;
        }
        const int chunk = kRows / K;
        const bool chunks = n > chunk;
        int rc = ready(stream, chunks ? 2 * kRows : K * n, chunks);
        if (rc) return rc;
        auto send = [&](int i0, int buf) -> int {
            const int m = n - i0 < chunk ? n - i0 : chunk;
            k_stage<W><<<dim3((m + 255) / 256, K), 256, 0, stream>>>(rows, i0, m, host + buf * kRows);
            HIP_TRY(hipGetLastError());
            if (chunks) HIP_TRY(hipEventRecord(done[buf], stream));
            return VX3MI_OK;
        };
        // (a failure may leave chunks in flight: the stream is waited for)
        auto all = [&]() -> int {
            int rc = send(0, 0);
            for (int i0 = 0, buf = 0; rc == VX3MI_OK && i0 < n; i0 += chunk, buf ^= 1) {
                if (i0 + chunk < n && (rc = send(i0 + chunk, buf ^ 1))) break;
                if (chunks) HIP_TRY(hipEventSynchronize(done[buf]));
                else HIP_TRY(hipStreamSynchronize(stream));
                unpack(i0, n - i0 < chunk ? n - i0 : chunk, (const W *)(host + buf * kRows));
            }
            return rc;
        };
        if ((rc = all())) (void)hipStreamSynchronize(stream);
        return rc;
    }
};

}  // namespace vx3mi
