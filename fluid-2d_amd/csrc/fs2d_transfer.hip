// fs2d_transfer.hip -- fields in and out of the device: rows between a
// caller's unpadded R x R arrays and the pitched fields.
//
// What bounds it: a transfer from or to pageable host memory, by PCIe and by
// the runtime's own work per call.  A pitched copy of pageable memory
// (hipMemcpy2DAsync) is issued row by row, about 9 us each: 2.4 ms for one
// 256 x 256 field in, 1.7 ms out, whatever its bytes.  So rows are never copied one by
// one here: host arrays move as whole ranges, and a kernel places the rows.
//   * Up to kPinnedStage bytes per call, the arrays are copied into (or out
//     of) a pinned buffer by the host, and one kernel moves all of them
//     between that buffer, read and written over PCIe, and the fields: one
//     launch and one wait per call.  Measured: a 256 x 256 array in, 18 us
//     alone with its launch and wait; 1026 x 1026, 55 us of host copy and 86 us of kernel.
//   * Larger transfers take hipMemcpyAsync on ranges of whole rows (31-35 GB/s in
//     and 18 GB/s out of pageable memory from 1026 x 1026 up: 134 us in) through a
//     device buffer of at most kDeviceStage bytes, which bounds what a handle holds
//     (one array, up to 4 GB, otherwise).  Where no buffer can be had, pitched
//     copies, which need none.  The two ways cost the same at about 4 MB
//     an array; the line lies below that, at 8 MB a call, which also bounds
//     what a handle pins.
// A caller's pointer is dereferenced here, by the host or a kernel, only where that
// is known to be good: pageable memory by the host, and an array that lies whole in
// an allocation of the stream's own device by a kernel.  Any other (pinned or managed
// memory, another device's, a device array given as a host one, one that its allocation
// is too short for) is left to hipMemcpy2DAsync, which orders it on the stream, reaches
// peers, and refuses what it cannot copy.
#include "fs2d_internal.hpp"

#include <algorithm>
#include <cstring>

namespace fs2d {
namespace {

constexpr size_t kPinnedStage = size_t(8) << 20, kDeviceStage = size_t(128) << 20;

// Field blockIdx.z, row blockIdx.y.
__global__ __launch_bounds__(256) void k_copy_rows(RowCopies c, int R, int sp, int dp) {
    const float* __restrict__ s = c.src[blockIdx.z] + (size_t)blockIdx.y * sp;
    float* __restrict__ d = c.dst[blockIdx.z] + (size_t)blockIdx.y * dp;
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j < R) d[j] = s[j];
}

// The stream's device is current while this lives (a handle may be read from a
// thread whose current device is another).
struct OnDeviceOf {
    int saved = -1;
    explicit OnDeviceOf(hipStream_t s) {
        hipDevice_t want = 0;
        int have = 0;
        if (hipStreamGetDevice(s, &want) != hipSuccess || hipGetDevice(&have) != hipSuccess || have == want) return;
        if (hipSetDevice(want) == hipSuccess) saved = have;
    }
    ~OnDeviceOf() {
        if (saved >= 0) (void)hipSetDevice(saved);
    }
};

// Whether the runtime has p: device, pinned or managed memory.
bool registered(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

// Whether [p, p + bytes) lies in one allocation of the stream's device.
bool on_device_of(hipStream_t s, const void* p, size_t bytes) {
    hipPointerAttribute_t a{};
    hipDevice_t dev = 0;
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (hipPointerGetAttributes(&a, p) != hipSuccess || hipStreamGetDevice(s, &dev) != hipSuccess ||
        a.type != hipMemoryTypeDevice || a.device != dev ||
        hipMemGetAddressRange(&base, &size, const_cast<void*>(p)) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    const size_t at = static_cast<const char*>(p) - static_cast<const char*>(base);
    return at <= size && bytes <= size - at;
}

hipError_t pitched_copy(hipStream_t s, const RowCopies& c, int k, int R, int sp, int dp, hipMemcpyKind kind) {
    const size_t f = sizeof(float);
    return hipMemcpy2DAsync(c.dst[k], f * dp, c.src[k], f * sp, f * R, R, kind, s);
}

// `rows` rows of R floats.
hipError_t launch_copy_rows(hipStream_t s, const RowCopies& c, int rows, int R, int sp, int dp) {
    if (c.count <= 0) return hipSuccess;
    const dim3 grid((R + 255) / 256, rows, c.count);
    hipLaunchKernelGGL(k_copy_rows, grid, dim3(256), 0, s, c, R, sp, dp);
    return hipGetLastError();
}

// Arrays of host memory: those that the runtime has are copied by it (at once: a later
// array wins where two overlap, and host arrays follow), the others are left in `rest`.
hipError_t copy_registered(hipStream_t s, const RowCopies& c, int R, int sp, int dp, hipMemcpyKind kind, RowCopies* rest) {
    for (int k = 0; k < c.count; ++k) {
        if (registered(kind == hipMemcpyHostToDevice ? c.src[k] : c.dst[k])) {
            const hipError_t e = pitched_copy(s, c, k, R, sp, dp, kind);
            if (e != hipSuccess) return e;
        } else {
            rest->add(c.src[k], c.dst[k]);
        }
    }
    return hipSuccess;
}

hipError_t grow(float** p, size_t* have, size_t floats, hipStream_t s, bool pinned) {
    if (*have >= floats) return hipSuccess;
    hipError_t e = hipStreamSynchronize(s);  // the old buffer may be in use
    if (e != hipSuccess) return e;
    if (*p) (void)(pinned ? hipHostFree(*p) : hipFree(*p));
    *p = nullptr;
    *have = 0;
    void* q = nullptr;
    e = pinned ? hipHostMalloc(&q, floats * sizeof(float), hipHostMallocDefault) : hipMalloc(&q, floats * sizeof(float));
    if (e != hipSuccess) return e;
    *p = static_cast<float*>(q);
    *have = floats;
    return hipSuccess;
}

// grow, as a question.
bool grown(float** p, size_t* have, size_t floats, hipStream_t s, bool pinned) {
    if (grow(p, have, floats, s, pinned) == hipSuccess) return true;
    (void)hipGetLastError();
    return false;
}

// Rows of R floats that the device buffer takes; 0 where there is none to be had.
int stage_rows(HostStage& h, hipStream_t s, int R) {
    const size_t most = std::max<size_t>(kDeviceStage / sizeof(float) / R, 1);
    const int rows = static_cast<int>(std::min<size_t>(most, R));
    return grown(&h.dev, &h.dev_floats, (size_t)rows * R, s, false) ? rows : 0;
}

}  // namespace

// A later array wins where two destinations overlap, as with copies made one
// after the other: such a set is copied array by array.
hipError_t copy_rows_in_order(hipStream_t s, const RowCopies& c, int R, int P, bool in) {
    const int sp = in ? R : P, dp = in ? P : R;
    const OnDeviceOf device(s);
    const size_t span = (size_t)(R - 1) * dp + R;
    const size_t bytes = sizeof(float) * R * R;  // of a caller's array
    bool apart = true;
    for (int a = 0; a < c.count; ++a)
        for (int b = 0; b < a; ++b) apart = apart && (c.dst[a] + span <= c.dst[b] || c.dst[b] + span <= c.dst[a]);
    RowCopies together;
    hipError_t e;
    for (int a = 0; a < c.count; ++a) {
        RowCopies one;
        one.add(c.src[a], c.dst[a]);
        if (!on_device_of(s, in ? c.src[a] : c.dst[a], bytes)) e = pitched_copy(s, c, a, R, sp, dp, hipMemcpyDeviceToDevice);
        else if (!apart) e = launch_copy_rows(s, one, R, R, sp, dp);
        else {
            together.add(c.src[a], c.dst[a]);
            e = hipSuccess;
        }
        if (e != hipSuccess) return e;
    }
    return launch_copy_rows(s, together, R, R, sp, dp);
}

hipError_t stage_in(HostStage& h, hipStream_t s, const RowCopies& all, int R, int P) {
    const OnDeviceOf device(s);
    const size_t n = (size_t)R * R, bytes = n * sizeof(float);
    RowCopies c;
    hipError_t e = copy_registered(s, all, R, R, P, hipMemcpyHostToDevice, &c);
    if (e != hipSuccess || c.count == 0) return e;
    if (c.count * bytes <= kPinnedStage && grown(&h.pin, &h.pin_floats, c.count * n, s, true)) {
        RowCopies d = c;
        for (int k = 0; k < c.count; ++k) {
            std::memcpy(h.pin + k * n, c.src[k], bytes);
            d.src[k] = h.pin + k * n;
        }
        return launch_copy_rows(s, d, R, R, R, P);
    }
    const int rows = stage_rows(h, s, R);
    for (int k = 0; k < c.count; ++k) {
        if (rows == 0 && (e = pitched_copy(s, c, k, R, R, P, hipMemcpyHostToDevice)) != hipSuccess) return e;
        for (int r = 0; rows && r < R; r += rows) {
            const int m = std::min(rows, R - r);
            RowCopies one;
            one.add(h.dev, c.dst[k] + (size_t)r * P);
            if ((e = hipMemcpyAsync(h.dev, c.src[k] + (size_t)r * R, sizeof(float) * m * R, hipMemcpyHostToDevice, s)) !=
                hipSuccess)
                return e;
            if ((e = launch_copy_rows(s, one, m, R, R, P)) != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

hipError_t stage_out(HostStage& h, hipStream_t s, const RowCopies& all, int R, int P) {
    const OnDeviceOf device(s);
    const size_t n = (size_t)R * R, bytes = n * sizeof(float);
    RowCopies c;
    hipError_t e = copy_registered(s, all, R, P, R, hipMemcpyDeviceToHost, &c);
    if (e != hipSuccess) return e;
    if (c.count == 0) return hipStreamSynchronize(s);
    if (c.count * bytes <= kPinnedStage && grown(&h.pin, &h.pin_floats, c.count * n, s, true)) {
        RowCopies d = c;
        for (int k = 0; k < c.count; ++k) d.dst[k] = h.pin + k * n;
        if ((e = launch_copy_rows(s, d, R, R, P, R)) != hipSuccess) return e;
        if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
        for (int k = 0; k < c.count; ++k) std::memcpy(c.dst[k], h.pin + k * n, bytes);
        return hipSuccess;
    }
    const int rows = stage_rows(h, s, R);
    for (int k = 0; k < c.count; ++k) {
        if (rows == 0 && (e = pitched_copy(s, c, k, R, P, R, hipMemcpyDeviceToHost)) != hipSuccess) return e;
        for (int r = 0; rows && r < R; r += rows) {
            const int m = std::min(rows, R - r);
            RowCopies one;
            one.add(c.src[k] + (size_t)r * P, h.dev);
            if ((e = launch_copy_rows(s, one, m, R, P, R)) != hipSuccess) return e;
            if ((e = hipMemcpyAsync(c.dst[k] + (size_t)r * R, h.dev, sizeof(float) * m * R, hipMemcpyDeviceToHost, s)) !=
                hipSuccess)
                return e;
        }
    }
    return hipStreamSynchronize(s);
}

hipError_t stage_pinned(HostStage& h, hipStream_t s, size_t floats, float** out) {
    *out = nullptr;
    if (floats * sizeof(float) > kPinnedStage) return hipSuccess;
    const OnDeviceOf device(s);
    const hipError_t e = grow(&h.pin, &h.pin_floats, floats, s, true);
    if (e == hipSuccess) *out = h.pin;
    return e;
}

void stage_free(HostStage& h) {
    if (h.pin) (void)hipHostFree(h.pin);
    if (h.dev) (void)hipFree(h.dev);
    h = HostStage{};
}

}  // namespace fs2d
