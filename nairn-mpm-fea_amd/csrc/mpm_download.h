// mpm_download.h -- particle rows from the device to a caller's arrays, in upload order.
#ifndef MPM_DOWNLOAD_H
#define MPM_DOWNLOAD_H

#include <hip/hip_runtime.h>

#include "mpm_kernels.h"

// Staging of one context's or server's downloads: pinned host slots, one per copying thread. The
// device writes a chunk of the result (gathered into upload order) straight into a slot, and the
// slot's thread copies it on to the caller's pages, so transfers, copies and the first touches of the
// caller's pages overlap. A row at a time through the runtime's pageable copies took 290 ms for 7.08M
// particles (2.2 GB, one thread of copies and page faults); eight threads with 2 MiB chunks take 46
// (48 GB/s, where the link reaches 50; four 59, twelve 46; through a device chunk and a copy engine 63).
// Below one chunk the calling thread does it alone. Pinning the slots costs the first download of an object
// up to 1.3 ms (60k particles: 1.8 ms, then 0.6; the runtime's copies 2.0), and freeing them 0.1 to 0.5 at
// its end. Results collected by several threads at once take turns: 16 of 8k particles 4.5 ms by 16 threads
// and 3.8 one after another (the runtime's copies 4.3 and 8.9), 8 of 64k 7 and 7 (29 and 111). Calls on one object must not overlap.
class RowDownload {
public:
    RowDownload() = default;
    RowDownload(const RowDownload &) = delete;
    RowDownload &operator=(const RowDownload &) = delete;
    ~RowDownload() { free(); }
    void free();
    // The rows of n particles: double rows from d (positions from pos), MPI_* rows from iv, home[] the
    // particles' places in the result (less homeBase), inv n ints of device scratch; matShift is taken
    // off the material numbers. The arrays lie in host memory or, which is slower, in a device's; iOut may
    // be null. Work already on the stream s comes first; returns when the arrays hold the rows. Errors of
    // the runtime come back as they are; hipErrorInvalidValue for a null dOut and if a place lies outside
    // the result, which outside then tells.
    hipError_t run(const double *pos, const double *d, const int *iv, const int *home, int *inv, long long n,
                   long long homeBase, int matShift, double *dOut, int32_t *iOut, hipStream_t s);
    bool outside = false;      // the last run found a place outside its result

private:
    static constexpr int THREADS = 8;
    static constexpr long long CHUNK = 2 << 20;        // bytes
    char *slots = nullptr;                              // pinned; the words before the first slot are a flag
    int nslots = 0;
};

#endif
