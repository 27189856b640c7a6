// mpm_download.hip -- particle rows from the device to a caller's arrays (mpm_download.h).
#include "mpm_download.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>
#include <tuple>
#include <vector>

namespace {

constexpr int FLAG_BYTES = 4096;
static_assert(MPI_NUM_FIELDS % 2 == 0, "int rows are moved two words at a time");

// place in the result -> particle; *bad is set for a place outside it
__global__ void k_places(const int *home, int *inv, long long n, long long homeBase, int *bad) {
    const long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const long long h = home[k] - homeBase;
    if (h < 0 || h >= n) *bad = 1;
    else inv[h] = (int)k;
}

// words w0 .. w0 + cnt of the result (8 bytes: the double rows, then the int rows) into out. Bound by
// the link to the host: consecutive lanes write consecutive words, and the rows are read through inv.
__global__ __launch_bounds__(256) void k_result_words(const double *pos, const double *d, const int *iv, const int *inv,
                                                      long long n, int matShift, long long w0, long long cnt,
                                                      unsigned long long *out) {
    const long long nd = (long long)MPF_NUM_FIELDS * n;
    for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < cnt; k += (long long)gridDim.x * blockDim.x) {
        const long long w = w0 + k;
        unsigned long long v = 0;
        auto particle = [&](long long j) {             // (a hole left by places outside the result is never used)
            const unsigned p = (unsigned)inv[j];
            return p < n ? (long long)p : 0ll;
        };
        if (w < nd) {
            const long long f = w / n, p = particle(w - f * n);
            v = (unsigned long long)__double_as_longlong((f <= MPF_POS_Z ? pos : d)[f * n + p]);
        } else {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const long long e = 2 * (w - nd) + h, q = e / n, p = particle(e - q * n);
                const unsigned x = (unsigned)(iv[q * n + p] - (q == MPI_MAT ? matShift : 0));
                v |= (unsigned long long)x << (32 * h);
            }
        }
        out[k] = v;
    }
}

// a launch's own error, not one that an earlier call left for its caller to read
template <typename... P, typename... A>
hipError_t launch(void (*kernel)(P...), unsigned blocks, hipStream_t s, A... a) {
    std::tuple<P...> values(static_cast<P>(a)...);
    return std::apply([&](auto &...v) {
        void *args[] = {&v...};
        return hipLaunchKernel(reinterpret_cast<const void *>(kernel), dim3(blocks), dim3(256), args, 0, s);
    }, values);
}

// whether the runtime has to copy to p, because the host cannot write there
bool on_device(const void *p) {
    hipPointerAttribute_t a{};
    if (!p) return false;
    const bool clean = hipPeekAtLastError() == hipSuccess;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        if (clean) (void)hipGetLastError();      // memory that the runtime does not know
        return false;
    }
    return a.type == hipMemoryTypeDevice;
}

hipError_t put(void *to, const void *from, size_t bytes, bool device) {
    if (device) return hipMemcpy(to, from, bytes, hipMemcpyHostToDevice);
    std::memcpy(to, from, bytes);
    return hipSuccess;
}

}  // namespace

void RowDownload::free() {
    if (slots) (void)hipHostFree(slots);
    slots = nullptr;
    nslots = 0;
}

hipError_t RowDownload::run(const double *pos, const double *d, const int *iv, const int *home, int *inv, long long n,
                            long long homeBase, int matShift, double *dOut, int32_t *iOut, hipStream_t s) {
    outside = false;
    if (n <= 0) return hipStreamSynchronize(s);
    if (!dOut) return hipErrorInvalidValue;
    const long long nd = (long long)MPF_NUM_FIELDS * n, total = nd + (iOut ? MPI_NUM_FIELDS / 2 * n : 0);
    const long long words = CHUNK / 8, chunks = (total + words - 1) / words;
    const int want = (int)std::min<long long>(THREADS, chunks);
    hipError_t rc = hipSuccess;
    int device = 0;
    if ((rc = hipGetDevice(&device)) != hipSuccess) return rc;
    if (nslots < want) {
        free();
        const bool clean = hipPeekAtLastError() == hipSuccess;
        for (int k = want; !slots && k > 0; k /= 2) {      // as many as the host will pin
            void *p = nullptr;
            if ((rc = hipHostMalloc(&p, FLAG_BYTES + (size_t)k * CHUNK, hipHostMallocCoherent)) != hipSuccess) continue;
            slots = static_cast<char *>(p);
            nslots = k;
        }
        if (clean) (void)hipGetLastError();
        if (!slots) return rc;
    }
    const int threads = std::min(want, nslots);
    volatile int *bad = reinterpret_cast<int *>(slots);
    *bad = 0;
    if ((rc = launch(k_places, (unsigned)((n + 255) / 256), s, home, inv, n, homeBase, reinterpret_cast<int *>(slots))) != hipSuccess)
        return rc;

    const bool dDev = on_device(dOut), iDev = on_device(iOut);
    std::atomic<long long> next{0};
    std::atomic<int> failed{(int)hipSuccess};
    // takes chunks in turn: its launch, the wait for it, the copy; other threads' chunks fill the stream
    auto work = [&](int slot) {
        hipEvent_t done = nullptr;
        hipError_t e = hipSetDevice(device);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&done, hipEventDisableTiming);
        char *at = slots + FLAG_BYTES + (size_t)slot * CHUNK;
        while (e == hipSuccess && failed.load() == (int)hipSuccess) {
            const long long c = next.fetch_add(1);
            if (c >= chunks) break;
            const long long w0 = c * words, cnt = std::min(words, total - w0);
            const unsigned blocks = (unsigned)std::min<long long>((cnt + 255) / 256, 512);
            if ((e = launch(k_result_words, blocks, s, pos, d, iv, inv, n, matShift, w0, cnt,
                            reinterpret_cast<unsigned long long *>(at))) != hipSuccess ||
                (e = hipEventRecord(done, s)) != hipSuccess || (e = hipEventSynchronize(done)) != hipSuccess)
                break;
            if (*bad) { e = hipErrorInvalidValue; break; }
            const long long db = std::max<long long>(0, std::min(cnt, nd - w0));
            if (db) e = put(dOut + w0, at, (size_t)db * 8, dDev);
            if (e == hipSuccess && db < cnt) e = put(iOut + 2 * (w0 + db - nd), at + db * 8, (size_t)(cnt - db) * 8, iDev);
        }
        if (done) (void)hipEventDestroy(done);
        if (e != hipSuccess) failed.store((int)e);
    };
    std::vector<std::thread> team;
    try {
        team.reserve(threads - 1);
        for (int k = 1; k < threads; k++) team.emplace_back(work, k);
    } catch (const std::exception &) {                  // fewer threads than wanted: the others take its chunks
    }
    work(0);
    for (std::thread &t : team) t.join();
    rc = (hipError_t)failed.load();
    const hipError_t end = hipStreamSynchronize(s);     // nothing writes a slot after the return
    outside = *bad != 0;
    return rc != hipSuccess ? rc : end;
}
