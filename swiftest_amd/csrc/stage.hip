// stage.hip -- the pinned transfer ring (swg_stage.h).
#include <algorithm>
#include <cstring>

#include "swg_stage.h"

namespace swg {

namespace {

// the device side of a transfer's arrays: words of the image before item k,
// and where they live
struct Image {
    int n;
    int32_t kind[Stage::MAX_ITEMS];
    int64_t off[Stage::MAX_ITEMS + 1];  // first image word of each item
    int64_t cnt[Stage::MAX_ITEMS];
    void *p[Stage::MAX_ITEMS][3];
};

int64_t words_of(const XferItem &it)
{
    return it.kind == 0 ? it.n : it.kind == 1 ? 3 * it.n : (it.n + 1) / 2;
}
int64_t bytes_of(const XferItem &it) { return it.kind == 0 ? 8 * it.n : it.kind == 1 ? 24 * it.n : 4 * it.n; }

Image image_of(const XferItem *items, int n)
{
    Image im{};
    im.n = n;
    int64_t w = 0;
    for (int k = 0; k < n; k++) {
        im.kind[k] = items[k].kind;
        im.off[k] = w;
        im.cnt[k] = items[k].n;
        im.p[k][0] = items[k].x;
        im.p[k][1] = items[k].y;
        im.p[k][2] = items[k].z;
        w += words_of(items[k]);
    }
    im.off[n] = w;
    return im;
}

// image words [w0, w0 + nw) between the device arrays and `pin`, one word per
// thread: the pinned side is contiguous over the wavefront, the device side
// contiguous (kinds 0 and 2) or three streams a third as dense (kind 1).
// Bound by the host link: 1 MiB in 21 us (50 GB/s) either way.
template <bool IN>
__global__ __launch_bounds__(256) void k_stage(const Image im, int64_t w0, int64_t nw, uint64_t *pin)
{
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= nw) return;
    const int64_t w = w0 + t;
    int k = 0;
    while (k + 1 < im.n && w >= im.off[k + 1]) k++;
    const int64_t q = w - im.off[k];
    if (im.kind[k] == 2) {
        int32_t *a = (int32_t *)im.p[k][0] + 2 * q;
        const bool two = 2 * q + 1 < im.cnt[k];
        if (IN) {
            const uint64_t v = pin[t];
            a[0] = (int32_t)(uint32_t)v;
            if (two) a[1] = (int32_t)(uint32_t)(v >> 32);
        } else {
            pin[t] = (uint64_t)(uint32_t)a[0] | (two ? (uint64_t)(uint32_t)a[1] << 32 : 0);
        }
        return;
    }
    uint64_t *a;
    if (im.kind[k] == 0) {
        a = (uint64_t *)im.p[k][0] + q;
    } else {
        const int64_t body = q / 3;
        a = (uint64_t *)im.p[k][q - 3 * body] + body;
    }
    if (IN) *a = pin[t];
    else pin[t] = *a;
}

// the host side of image words [w0, w0 + nw): between the callers' arrays and
// the slot
void host_copy(const XferItem *items, const Image &im, int64_t w0, int64_t nw, char *pin, bool in)
{
    for (int k = 0; k < im.n; k++) {
        const int64_t a = std::max(w0, im.off[k]), b = std::min(w0 + nw, im.off[k + 1]);
        if (a >= b) continue;
        const int64_t at = 8 * (a - im.off[k]), len = std::min(8 * (b - im.off[k]), bytes_of(items[k])) - at;
        char *h = (char *)items[k].host + at, *p = pin + 8 * (a - w0);
        if (in) std::memcpy(p, h, (size_t)len);
        else std::memcpy(h, p, (size_t)len);
    }
}

}  // namespace

hipError_t Stage::ready()
{
    if (pin_) return hipSuccess;
    hipError_t e = hipSuccess;
    for (int k = 0; k < SLOTS && e == hipSuccess; k++)
        if (!ev_[k]) e = hipEventCreateWithFlags(&ev_[k], hipEventDisableTiming);
    if (e == hipSuccess) e = hipHostMalloc((void **)&pin_, SLOTS * CHUNK);
    return e;
}

Stage::~Stage()
{
    for (int k = 0; k < SLOTS; k++) {
        if (busy_[k]) (void)hipEventSynchronize(ev_[k]);
        if (ev_[k]) (void)hipEventDestroy(ev_[k]);
    }
    if (pin_) (void)hipHostFree(pin_);
}

hipError_t Stage::in(hipStream_t st, const XferItem *items, int n)
{
    const Image im = image_of(items, n);
    if (im.off[n] == 0) return hipSuccess;
    if (hipError_t e = ready()) return e;
    for (int64_t w0 = 0; w0 < im.off[n]; w0 += CHUNK / 8) {
        const int64_t nw = std::min(CHUNK / 8, im.off[n] - w0);
        const int s = next_;
        next_ = (next_ + 1) % SLOTS;
        if (busy_[s]) {
            if (hipError_t e = hipEventSynchronize(ev_[s])) return e;
            busy_[s] = false;
        }
        char *pin = pin_ + s * CHUNK;
        host_copy(items, im, w0, nw, pin, true);
        k_stage<true><<<(int)((nw + 255) / 256), 256, 0, st>>>(im, w0, nw, (uint64_t *)pin);
        if (hipError_t e = hipGetLastError()) return e;
        if (hipError_t e = hipEventRecord(ev_[s], st)) return e;
        busy_[s] = true;
    }
    return hipSuccess;
}

hipError_t Stage::out(hipStream_t st, const XferItem *items, int n)
{
    const Image im = image_of(items, n);
    if (im.off[n] == 0) return hipSuccess;
    if (hipError_t e = ready()) return e;
    const int64_t step = CHUNK / 8, nch = (im.off[n] + step - 1) / step;
    // chunk c goes through slot (first + c) % SLOTS; up to SLOTS chunks are
    // queued ahead of the one the host copies out
    const int first = next_;
    auto queue = [&](int64_t c) -> hipError_t {
        const int s = (int)((first + c) % SLOTS);
        if (busy_[s]) {
            // left by an earlier transfer in: its kernel reads the slot
            if (hipError_t e = hipEventSynchronize(ev_[s])) return e;
        }
        const int64_t w0 = c * step, nw = std::min(step, im.off[n] - w0);
        k_stage<false><<<(int)((nw + 255) / 256), 256, 0, st>>>(im, w0, nw, (uint64_t *)(pin_ + s * CHUNK));
        if (hipError_t e = hipGetLastError()) return e;
        if (hipError_t e = hipEventRecord(ev_[s], st)) return e;
        busy_[s] = true;
        return hipSuccess;
    };
    for (int64_t c = 0; c < std::min<int64_t>(SLOTS, nch); c++)
        if (hipError_t e = queue(c)) return e;
    for (int64_t c = 0; c < nch; c++) {
        const int s = (int)((first + c) % SLOTS);
        if (hipError_t e = hipEventSynchronize(ev_[s])) return e;
        busy_[s] = false;
        const int64_t w0 = c * step, nw = std::min(step, im.off[n] - w0);
        host_copy(items, im, w0, nw, pin_ + s * CHUNK, false);
        if (c + SLOTS < nch)
            if (hipError_t e = queue(c + SLOTS)) return e;
    }
    next_ = (int)((first + nch) % SLOTS);
    return hipSuccess;
}

}  // namespace swg
