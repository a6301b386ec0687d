// Layout kernels and pinned staging of the vectors that cross the C ABI
// (afx_exchange.hpp).
#include "afx_exchange.hpp"

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace afx {

// ----------------------------------------------------------------- kernels --
// A block takes 256 consecutive reference cells: their rows are one contiguous
// stretch, moved with consecutive lanes on consecutive doubles (the host side
// of a PCIe access wants whole 64-byte lines), and the planes are gathered or
// scattered in the device's cell order, where the stretch's cells sit in a few
// tiles.  LDS holds the block's rows in between.  Bound by PCIe for pinned rows
// and by HBM otherwise.  With the host loops and pageable copies that this
// replaces, one residual call of 2M cells (five values per cell up and down,
// 160 MB, of which PCIe needs 2.9 ms) took 33.0 ms, now 5.9; an adjoint and a
// tangent product of 500k cells 20.5 ms, now 5.4; a residual call of 4 096
// cells 108 us, now 77.
namespace {
constexpr int kXBlock = 256;
inline int xblocks(int32_t n) { return (n + kXBlock - 1) / kXBlock; }

template <int NV>
__global__ void __launch_bounds__(kXBlock) k_import_rows(const double* __restrict__ rows,
                                                         const int32_t* __restrict__ old2new, int32_t nT,
                                                         double* __restrict__ planes) {
    __shared__ double sh[NV * kXBlock];
    const int t = threadIdx.x, base = blockIdx.x * kXBlock;
    const int n = min(kXBlock, nT - base);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int e = t + j * kXBlock;
        if (e < NV * n) sh[e] = rows[(size_t)NV * base + e];
    }
    __syncthreads();
    if (t >= n) return;
    const int i = old2new[base + t];
#pragma unroll
    for (int k = 0; k < NV; ++k) planes[(size_t)k * nT + i] = sh[NV * t + k];
}

// value k of device cell i, from planes or from one float4 per cell
__device__ __forceinline__ double cell_value(const double* p, int32_t nT, int i, int k) { return p[(size_t)k * nT + i]; }
__device__ __forceinline__ double cell_value(const float* p, int32_t nT, int i, int k) {
    return (double)p[(size_t)k * nT + i];
}
__device__ __forceinline__ double cell_value(const float4* p, int32_t, int i, int k) {
    return (double)reinterpret_cast<const float*>(p + i)[k];
}

template <typename T, int NV>
__global__ void __launch_bounds__(kXBlock) k_export_rows(const T* __restrict__ cells,
                                                         const int32_t* __restrict__ old2new, int32_t nT,
                                                         double* __restrict__ rows) {
    __shared__ double sh[NV * kXBlock];
    const int t = threadIdx.x, base = blockIdx.x * kXBlock;
    const int n = min(kXBlock, nT - base);
    if (t < n) {
        const int i = old2new[base + t];
#pragma unroll
        for (int k = 0; k < NV; ++k) sh[NV * t + k] = cell_value(cells, nT, i, k);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int e = t + j * kXBlock;
        if (e < NV * n) rows[(size_t)NV * base + e] = sh[e];
    }
}
}  // namespace

hipError_t launch_import_rows(hipStream_t s, const double* rows, const int32_t* old2new, int32_t nT, int nv,
                              double* planes) {
    if (nT <= 0) return hipSuccess;
    if (nv == 4)
        hipLaunchKernelGGL(k_import_rows<4>, dim3(xblocks(nT)), dim3(kXBlock), 0, s, rows, old2new, nT, planes);
    else if (nv == 1)
        hipLaunchKernelGGL(k_import_rows<1>, dim3(xblocks(nT)), dim3(kXBlock), 0, s, rows, old2new, nT, planes);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}
template <typename T>
static hipError_t export_rows(hipStream_t s, const T* planes, const int32_t* old2new, int32_t nT, int nv,
                              double* rows) {
    if (nT <= 0) return hipSuccess;
    if (nv == 4)
        hipLaunchKernelGGL((k_export_rows<T, 4>), dim3(xblocks(nT)), dim3(kXBlock), 0, s, planes, old2new, nT, rows);
    else if (nv == 1)
        hipLaunchKernelGGL((k_export_rows<T, 1>), dim3(xblocks(nT)), dim3(kXBlock), 0, s, planes, old2new, nT, rows);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}
hipError_t launch_export_rows(hipStream_t s, const double* planes, const int32_t* old2new, int32_t nT, int nv,
                              double* rows) {
    return export_rows<double>(s, planes, old2new, nT, nv, rows);
}
hipError_t launch_export_rows(hipStream_t s, const float* planes, const int32_t* old2new, int32_t nT, int nv,
                              double* rows) {
    return export_rows<float>(s, planes, old2new, nT, nv, rows);
}
hipError_t launch_export_rows(hipStream_t s, const float4* cells, const int32_t* old2new, int32_t nT, int nv,
                              double* rows) {
    if (nT <= 0) return hipSuccess;
    if (nv != 4) return hipErrorInvalidValue;
    hipLaunchKernelGGL((k_export_rows<float4, 4>), dim3(xblocks(nT)), dim3(kXBlock), 0, s, cells, old2new, nT, rows);
    return hipGetLastError();
}

// ----------------------------------------------------------------- staging --
struct Staging::Buf {
    int device = -1;
    char* pin = nullptr;
    hipEvent_t ev[kSlots] = {};
    ~Buf() {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
        if (pin) (void)hipHostFree(pin);
    }
};

// Idle buffers, at most kKept of them (8.1 MB each), whatever the number of
// handles and threads; a call that finds none makes its own, and gives it
// back or frees it.
struct StagingPool {
    static constexpr size_t kKept = 4;
    std::mutex mu;
    std::vector<Staging::Buf*> idle;
    long users = 0;

    Staging::Buf* take(int device) {
        std::lock_guard<std::mutex> lock(mu);
        for (size_t k = idle.size(); k-- > 0;)
            if (idle[k]->device == device) {
                Staging::Buf* b = idle[k];
                idle.erase(idle.begin() + (long)k);
                return b;
            }
        return nullptr;
    }
    void give(Staging::Buf* b) {
        {
            std::lock_guard<std::mutex> lock(mu);
            if (users > 0 && idle.size() < kKept) {
                idle.push_back(b);
                return;
            }
        }
        delete b;
    }
    void retain() {
        std::lock_guard<std::mutex> lock(mu);
        if (users++ == 0) idle.reserve(kKept);
    }
    void release() {
        std::vector<Staging::Buf*> go;
        {
            std::lock_guard<std::mutex> lock(mu);
            if (--users == 0) go.swap(idle);
        }
        for (Staging::Buf* b : go) delete b;
    }
};
namespace {
// never destroyed: buffers are freed with the last handle, while the HIP
// runtime is still up
StagingPool& pool() {
    static StagingPool* p = new StagingPool();
    return *p;
}
}  // namespace
thread_local bool t_no_pinned = false;

void staging_retain() { pool().retain(); }
void staging_release() { pool().release(); }

HostMemory::~HostMemory() {
    if (pinned_) (void)hipHostFree(p_);
    else std::free(p_);
}
hipError_t HostMemory::alloc(size_t bytes) {
    if (hipHostMalloc(&p_, t_no_pinned ? size_t(1) << 60 : bytes, hipHostMallocDefault) == hipSuccess) {
        pinned_ = true;
        return hipSuccess;
    }
    (void)hipGetLastError();
    p_ = std::malloc(bytes);
    return p_ ? hipSuccess : hipErrorOutOfMemory;
}

Staging::Staging(hipStream_t s) : s_(s) {
    int dev = 0;
    if ((err_ = hipGetDevice(&dev)) != hipSuccess) return;
    if (!t_no_pinned && (b_ = pool().take(dev))) return;
    b_ = new Buf();
    b_->device = dev;
    const size_t bytes = t_no_pinned ? size_t(1) << 60 : kSlots * kSlotBytes + kScalars * sizeof(double);
    err_ = hipHostMalloc((void**)&b_->pin, bytes, hipHostMallocDefault);
    for (int k = 0; k < kSlots && err_ == hipSuccess; ++k)
        err_ = hipEventCreateWithFlags(&b_->ev[k], hipEventDisableTiming);
    if (err_ != hipSuccess) {
        delete b_;
        b_ = nullptr;
        // the call goes on without: the error must not reach its launches' checks
        (void)hipGetLastError();
    }
}
Staging::~Staging() {
    if (!b_) return;
    if (waited_ || hipStreamSynchronize(s_) == hipSuccess) pool().give(b_);
    else delete b_;
}
hipError_t Staging::wait() {
    const hipError_t e = hipStreamSynchronize(s_);
    waited_ = e == hipSuccess;
    return e;
}
char* Staging::piece(int k) const { return b_->pin + (size_t)k * kSlotBytes; }
double* Staging::scalars() const { return reinterpret_cast<double*>(b_->pin + kSlots * kSlotBytes); }

// Piece c of the vector is worker c % workers's, in one of that worker's own
// slots, so the workers share nothing.  Down: the worker keeps its slots'
// device-to-host copies in flight, waits for each and copies it out.  Up: it
// waits for its slot's previous copy, fills the slot and enqueues.
// Measured at 64 MB on a 16-core share: one host thread moves 14 GB/s into
// freshly allocated memory (page faults) and 28 GB/s into touched memory, the
// PCIe copy of a pinned buffer 56 GB/s; pageable hipMemcpyAsync 4-10 GB/s down
// into fresh memory and 30 GB/s up.
hipError_t Staging::pieces(char* host, char* dev, size_t bytes, bool up) {
    const hipStream_t s = s_;
    const int n = (int)((bytes + kSlotBytes - 1) / kSlotBytes);
    // two slots per worker; one worker up to 4 MB (starting threads costs more)
    const int workers = n <= 4 ? 1 : 4, per = kSlots / workers;
    const int device = b_->device;
    std::atomic<int> failed{(int)hipSuccess};
    auto len = [&](int c) { return std::min(kSlotBytes, bytes - (size_t)c * kSlotBytes); };
    auto work = [&](int w) {
        hipError_t e = hipSetDevice(device);
        auto note = [&](hipError_t r) {
            if (r != hipSuccess && e == hipSuccess) e = r;
        };
        auto slot = [&](int q) { return w + workers * (q % per); };   // of the worker's q-th piece
        const int mine = (n - w + workers - 1) / workers;
        auto copy = [&](int q) {
            const int c = w + workers * q, k = slot(q);
            char* d = dev + (size_t)c * kSlotBytes;
            note(up ? hipMemcpyAsync(d, piece(k), len(c), hipMemcpyHostToDevice, s)
                    : hipMemcpyAsync(piece(k), d, len(c), hipMemcpyDeviceToHost, s));
            note(hipEventRecord(b_->ev[k], s));
        };
        if (!up)
            for (int q = 0; q < std::min(per, mine); ++q) copy(q);
        for (int q = 0; q < mine && e == hipSuccess; ++q) {
            const int c = w + workers * q, k = slot(q);
            char* user = host + (size_t)c * kSlotBytes;
            if (up) {
                if (q >= per) note(hipEventSynchronize(b_->ev[k]));
                std::memcpy(piece(k), user, len(c));
                copy(q);
            } else {
                note(hipEventSynchronize(b_->ev[k]));
                if (e == hipSuccess) std::memcpy(user, piece(k), len(c));
                if (q + per < mine) copy(q + per);
            }
        }
        if (e != hipSuccess) failed.store((int)e);
    };
    std::vector<std::thread> team;
    int started = 1;
    try {
        team.reserve((size_t)workers);
        for (; started < workers; ++started) team.emplace_back(work, started);
    } catch (const std::exception&) {
        // no more threads to be had: this one takes the remaining shares
    }
    work(0);
    for (int w = started; w < workers; ++w) work(w);
    for (std::thread& t : team) t.join();
    // the caller reuses the slots (and its own memory) after this
    const hipError_t last = wait();
    const hipError_t e = (hipError_t)failed.load();
    return e != hipSuccess ? e : last;
}
hipError_t Staging::to_device(const void* host, void* dev, size_t bytes) {
    return pieces(static_cast<char*>(const_cast<void*>(host)), static_cast<char*>(dev), bytes, true);
}
hipError_t Staging::to_host(const void* dev, void* host, size_t bytes) {
    return pieces(static_cast<char*>(host), static_cast<char*>(const_cast<void*>(dev)), bytes, false);
}

}  // namespace afx
