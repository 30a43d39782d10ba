// swg_stage.h -- host arrays to and from the device through a pinned ring.
//
// A pageable hipMemcpy costs about 20 us however small, one after the other,
// and moves 18-38 GB/s; a kernel that reads or writes pinned host memory
// moves about 50 GB/s and takes many arrays in one launch.  A transfer here
// is a list of arrays laid end to end (an "image" of 8-byte words).  It goes
// through the ring chunk by chunk: host memcpy on one side, k_stage (either
// way) on the other, which also turns the callers' (3,n) arrays into the
// device's component arrays and back.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "swg_state.h"

namespace swg {

// One array of a transfer.
struct XferItem {
    void *host;       // caller's array (read by in, written by out)
    int64_t n;        // elements
    int32_t kind;     // 0: n 8-byte words at x; 1: n (3,n) bodies <-> x, y, z; 2: n 4-byte words at x
    void *x, *y, *z;  // device arrays
};

inline XferItem xfer_words(const void *host, const void *dev, int64_t n)
{
    return XferItem{const_cast<void *>(host), n, 0, const_cast<void *>(dev), nullptr, nullptr};
}
inline XferItem xfer_vec3(const double *host, Vec3p v, int64_t n)
{
    return XferItem{const_cast<double *>(host), n, 1, v.x, v.y, v.z};
}
inline XferItem xfer_i32(const int32_t *host, const int32_t *dev, int64_t n)
{
    return XferItem{const_cast<int32_t *>(host), n, 2, const_cast<int32_t *>(dev), nullptr, nullptr};
}

// The ring of one library context: a few chunks of pinned memory, allocated
// at the first transfer and freed with the context.  Used by the thread that
// uses the context, on the context's stream.
class Stage {
  public:
    static constexpr int MAX_ITEMS = 12;  // arrays of one transfer
    static constexpr int SLOTS = 4;
    static constexpr int64_t CHUNK = 1 << 20;  // bytes of a slot
    ~Stage();
    // host -> device on stream st.  The host arrays may be changed as soon as
    // it returns; the device side is stream-ordered.
    hipError_t in(hipStream_t st, const XferItem *items, int n);
    // device -> host, after the work queued on st before; returns when the
    // host arrays hold the data.
    hipError_t out(hipStream_t st, const XferItem *items, int n);

  private:
    hipError_t ready();
    char *pin_ = nullptr;
    hipEvent_t ev_[SLOTS] = {};
    bool busy_[SLOTS] = {};
    int next_ = 0;
};

}  // namespace swg
