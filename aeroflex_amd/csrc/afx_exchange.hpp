// Vectors crossing the C ABI: the reference's cell order and AoS layout on the
// host side, planes in the device's cell order on the GPU.
//
// The permutation runs on the device.  Between the device and the caller's
// pageable memory the bytes go through pinned staging buffers: vectors of at
// most kDirectBytes in one go, read or written over PCIe by the layout kernel
// itself; larger ones in kSlotBytes pieces copied by a few host threads while
// the next pieces are in flight.
#pragma once
#include <cstddef>
#include <cstdint>
#include <hip/hip_runtime.h>

namespace afx {

constexpr size_t kSlotBytes = size_t(1) << 20;   // one piece of a large transfer
constexpr int kSlots = 8;                         // pieces in flight
constexpr size_t kDirectBytes = 4 * kSlotBytes;   // up to here the kernels access pinned memory themselves
constexpr int kScalars = 64;                      // doubles for norms and flags behind the pieces

// One pinned staging buffer with its events, on the device that was current
// when it was taken.  Taken from a process-wide pool and given back by the
// destructor, which waits for the stream first where the call has queued work
// and not waited for it (an error return); a Staging belongs to one call of one
// thread and one stream.
class Staging {
public:
    explicit Staging(hipStream_t s);
    ~Staging();
    Staging(const Staging&) = delete;
    Staging& operator=(const Staging&) = delete;
    hipError_t status() const { return err_; }
    // waits for the stream; from then on nothing queued reads or writes the buffer
    hipError_t wait();
    // more work on the buffer is about to be queued after a wait
    void queueing() { waited_ = false; }
    char* piece(int k) const;            // host = device address (unified addressing)
    double* scalars() const;
    // caller memory <-> device memory, in pieces; returns once done
    hipError_t to_device(const void* host, void* dev, size_t bytes);
    hipError_t to_host(const void* dev, void* host, size_t bytes);

private:
    hipError_t pieces(char* host, char* dev, size_t bytes, bool up);
    struct Buf;
    friend struct StagingPool;
    Buf* b_ = nullptr;
    hipStream_t s_;
    bool waited_ = false;
    hipError_t err_ = hipSuccess;
};
// A handle's own host memory for asynchronous copies: pinned, or ordinary where no
// pinned memory is to be had (the copies then go through the runtime's staging).
class HostMemory {
public:
    HostMemory() = default;
    ~HostMemory();
    HostMemory(const HostMemory&) = delete;
    HostMemory& operator=(const HostMemory&) = delete;
    hipError_t alloc(size_t bytes);   // once
    void* get() const { return p_; }

private:
    void* p_ = nullptr;
    bool pinned_ = false;
};

// The pool keeps buffers while any solver handle lives: every handle holds one
// reference, and the last one to go frees the idle buffers.
// Test hook, per thread: Staging and HostMemory ask for more pinned memory than there is.
extern thread_local bool t_no_pinned;
void staging_retain();
void staging_release();

// device planes <-> rows of nv values in reference order (nv 4: q(4*i+k); 1: one
// value per cell); old2new: device cell of each reference cell
hipError_t launch_import_rows(hipStream_t s, const double* rows, const int32_t* old2new, int32_t nT, int nv,
                              double* planes);
hipError_t launch_export_rows(hipStream_t s, const double* planes, const int32_t* old2new, int32_t nT, int nv,
                              double* rows);
hipError_t launch_export_rows(hipStream_t s, const float* planes, const int32_t* old2new, int32_t nT, int nv,
                              double* rows);
hipError_t launch_export_rows(hipStream_t s, const float4* cells, const int32_t* old2new, int32_t nT, int nv,
                              double* rows);   // nv 4

}  // namespace afx
