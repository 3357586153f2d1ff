// transfer.hpp -- cell records between a device array in the device's order and a caller's host array in
// file order, and the few scalars of a step that the host waits for (Board, at the end).
//
// A kernel permutes straight into (or out of) pinned host memory, chunk by chunk, while the host copies the
// chunk before to (or the chunk after from) the caller's pageable array.  What bounds it is the link: about
// 52 GB/s for the kernel's 16-byte stores, and the host's copy, which is as fast, runs beside it.  (A copy
// of the whole array to pageable memory runs at 11-17 GB/s, and a permutation on one host thread at 5.)
// 819,200 2D states (26 MB): 1.1 ms against 14 ms with a staging vector, a pageable copy and a host loop;
// 8,000 states: 17 us against 42.
// Three chunks of TRANSFER_CHUNK doubles per owner, allocated on first use (one, as small as the array, for an
// array that fits), freed with the owner.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>

namespace mstk {

constexpr int64_t TRANSFER_CHUNK = 1 << 18;  // doubles: 2 MiB, 40 us of the link

// dst[i] = element i of the records rec0, rec0 + 1, ... (width doubles each), record r at src + map[r] * width
static __global__ __launch_bounds__(256) void k_records_out(int64_t n, uint32_t width, const int32_t *__restrict__ map,
                                                          const double *__restrict__ src, double *__restrict__ dst) {
    const int64_t i = 2 * ((int64_t)blockIdx.x * 256 + threadIdx.x);
    if (i >= n) return;
    const uint32_t r = (uint32_t)i / width, k = (uint32_t)i % width;  // (a chunk's elements: 32 bits)
    const double a = src[(int64_t)map[r] * width + k];
    if (i + 1 == n) {
        dst[i] = a;
        return;
    }
    const uint32_t r1 = k + 1 == width ? r + 1 : r, k1 = k + 1 == width ? 0 : k + 1;
    *reinterpret_cast<double2 *>(dst + i) = make_double2(a, src[(int64_t)map[r1] * width + k1]);
}

// the inverse: element i of src to record map[i / width] of dst
static __global__ __launch_bounds__(256) void k_records_in(int64_t n, uint32_t width, const int32_t *__restrict__ map,
                                                         const double *__restrict__ src, double *__restrict__ dst) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint32_t r = (uint32_t)i / width, k = (uint32_t)i % width;
    dst[(int64_t)map[r] * width + k] = src[i];
}

struct Transfer {
    static constexpr int SLOTS = 3;
    double *buf[SLOTS] = {};
    hipEvent_t ev[SLOTS] = {};
    int64_t cap = 0;
    int64_t most = 0;  // doubles of the owner's largest usual array

    void release() {
        for (int s = 0; s < SLOTS; s++) {
            if (buf[s]) (void)hipHostFree(buf[s]);
            if (ev[s]) (void)hipEventDestroy(ev[s]);
            buf[s] = nullptr;
            ev[s] = nullptr;
        }
        cap = 0;
    }

    // one slot for an array of at most `total` doubles that fits a chunk, else all of them
    hipError_t ensure(int64_t total) {
        total = std::max(total, most);
        const int64_t want = std::min(total, TRANSFER_CHUNK);
        const int slots = total <= TRANSFER_CHUNK ? 1 : SLOTS;
        if (cap >= want && buf[slots - 1]) return hipSuccess;
        release();
        hipError_t e = hipSuccess;
        for (int s = 0; s < slots && e == hipSuccess; s++) {
            e = hipHostMalloc((void **)&buf[s], sizeof(double) * std::max<int64_t>(want, 2), hipHostMallocDefault);
            if (e == hipSuccess) e = hipEventCreateWithFlags(&ev[s], hipEventDisableTiming);
        }
        if (e != hipSuccess) {
            release();
            return e;
        }
        cap = want;
        return hipSuccess;
    }

    // out[r] = record map[r] of src, r < n (after the stream's earlier work; complete on return)
    hipError_t fetch(hipStream_t st, int64_t n, int width, const int32_t *map, const double *src, double *out) {
        hipError_t e = ensure(n * width);
        if (e != hipSuccess) return e;
        const int64_t per = std::max<int64_t>(1, cap / width), chunks = (n + per - 1) / per;
        auto drain = [&](int64_t c) {
            const hipError_t x = hipEventSynchronize(ev[c % SLOTS]);
            if (x == hipSuccess)
                memcpy(out + c * per * width, buf[c % SLOTS], sizeof(double) * std::min(per, n - c * per) * width);
            return x;
        };
        for (int64_t c = 0; c < chunks; c++) {
            if (c >= SLOTS - 1 && (e = drain(c - (SLOTS - 1))) != hipSuccess) return e;
            const int64_t m = std::min(per, n - c * per) * width;
            hipLaunchKernelGGL(k_records_out, dim3((uint32_t)((m + 511) / 512)), dim3(256), 0, st, m, (uint32_t)width,
                               map + c * per, src, buf[c % SLOTS]);
            if ((e = hipGetLastError()) != hipSuccess) return e;
            if ((e = hipEventRecord(ev[c % SLOTS], st)) != hipSuccess) return e;
        }
        for (int64_t c = std::max<int64_t>(0, chunks - (SLOTS - 1)); c < chunks; c++)
            if ((e = drain(c)) != hipSuccess) return e;
        return hipSuccess;
    }

    // record map[r] of each of the nd arrays dst = in[r], r < n (after the stream's earlier work; complete on return)
    hipError_t put(hipStream_t st, int64_t n, int width, const int32_t *map, const double *in, double *const *dst, int nd) {
        hipError_t e = ensure(n * width);
        if (e != hipSuccess) return e;
        const int64_t per = std::max<int64_t>(1, cap / width), chunks = (n + per - 1) / per;
        for (int64_t c = 0; c < chunks; c++) {
            if (c >= SLOTS && (e = hipEventSynchronize(ev[c % SLOTS])) != hipSuccess) return e;
            const int64_t m = std::min(per, n - c * per) * width;
            memcpy(buf[c % SLOTS], in + c * per * width, sizeof(double) * m);
            for (int d = 0; d < nd; d++) {
                hipLaunchKernelGGL(k_records_in, dim3((uint32_t)((m + 255) / 256)), dim3(256), 0, st, m, (uint32_t)width,
                                   map + c * per, (const double *)buf[c % SLOTS], dst[d]);
                if ((e = hipGetLastError()) != hipSuccess) return e;
            }
            if ((e = hipEventRecord(ev[c % SLOTS], st)) != hipSuccess) return e;
        }
        return hipStreamSynchronize(st);
    }
};

// A context's results of a few words, in pinned host memory: a kernel behind the work stores them and then a sequence
// number, which the host polls.  Waiting so takes 6 us from the launch, a stream synchronisation 11 and a copy into
// pageable memory 11 more.
struct Board {
    double scal[16];
    double mon[8];
    int32_t bad;
    uint32_t seq;
};

// scal and the bad flag to the board; take_bad: the flag is cleared as well
static __global__ __launch_bounds__(64) void k_report(const double *__restrict__ scal, int *__restrict__ bad, int take_bad,
                                                    Board *__restrict__ b, uint32_t seq) {
    const int i = threadIdx.x;
    if (i < 16) b->scal[i] = scal[i];
    if (i == 16) {
        const int v = bad[0];
        b->bad = v;
        if (take_bad && v) bad[0] = 0;
    }
    __threadfence_system();
    __syncthreads();
    if (i == 0) __hip_atomic_store(&b->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

static __global__ void k_store(double *__restrict__ p, double v) { p[0] = v; }

// waits for board sequence number seq, the stream's newest: by polling for about 100 us, then on the stream
inline hipError_t board_wait(const Board *b, uint32_t seq, hipStream_t st) {
    for (int i = 0; i < 2048; i++) {
        if (__atomic_load_n(&b->seq, __ATOMIC_ACQUIRE) == seq) return hipSuccess;
        __builtin_ia32_pause();
    }
    const hipError_t e = hipStreamSynchronize(st);
    if (e != hipSuccess) return e;
    return __atomic_load_n(&b->seq, __ATOMIC_ACQUIRE) == seq ? hipSuccess : hipErrorUnknown;
}

}  // namespace mstk
