// readback.hip -- device arrays to caller-owned host memory as doubles.
//
// A read-back is bound by the host: the caller's memory is pageable and
// usually fresh, so the destination's page faults and stores cost more than
// PCIe (67 MB of FP32 field, 134 MB of doubles, at 4096^2).  A kernel
// converts a piece of the array straight into a pinned slot, and several
// host threads, each with a slot of its own, copy the pieces out while the
// others' are on their way; no host pass converts or re-arranges anything, but
// for the small arrays of kCopyMin.
// Measured at 4096^2 against one thread that copied the frame, converted it
// and cut it out: FP32 field 59 -> 3.5 ms, void fraction 74 -> 3.6 ms; 2^22
// radii in the caller's order 16.5 -> 1.2 ms.
#include "brp_internal.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

namespace brp {
namespace {

bool permuted(const PackSrc &s) { return s.kind == PackSrc::kPerm || s.kind == PackSrc::kPermInt; }

// The value at element o of the source.
__host__ __device__ inline double source_value(const PackSrc &s, int64_t o) {
    switch (s.kind) {
        case PackSrc::kFloat: return (double)((const float *)s.src)[o];
        case PackSrc::kPermInt: return (double)((const int *)s.src)[o];
        case PackSrc::kPerm:
        case PackSrc::kDouble: return ((const double *)s.src)[o];
        case PackSrc::kFixed: return (double)((const int64_t *)s.src)[o] * kFgInvScale;
        case PackSrc::kDensity:
            return (1.0 - (double)((const int64_t *)s.src)[o] * kFgInvScale) * s.scale;
        default:  // kSum3
            return ((const double *)s.src)[o] + ((const double *)s.src2)[o] +
                   ((const double *)s.src3)[o];
    }
}

// Element e of the logical array, row-major over nx columns.
__device__ inline double pack_value(const PackSrc &s, int64_t e) {
    if (s.kind == PackSrc::kPerm || s.kind == PackSrc::kPermInt) return source_value(s, s.iperm[e]);
    const int64_t j = e / s.nx, i = e - j * s.nx;
    return source_value(s, frame_off((int)i + s.i0, (int)j + s.j0, s.pitch));
}

__global__ __launch_bounds__(256) void k_pack(PackSrc s, int64_t e0, int n, double *out) {
    for (int k = blockIdx.x * 256 + threadIdx.x; k < n; k += gridDim.x * 256)
        out[k] = pack_value(s, e0 + k);
}

}  // namespace

// A slot of 1 MiB holds a piece for about 20 us of PCIe time, several times a
// launch's latency, and eight of them keep the link busy while most are being
// copied out; the ring is pinned at a handle's first read-back of more than
// `small`, which is pinned with the handle and serves one thread.
constexpr int64_t kSlotDoubles = HostRing::kMaxSmall;
constexpr int kSlots = 8;

// Arrays of more than 16 and up to 64 KiB are copied as they are and converted
// here: the copy engine, which takes copies beyond 16 KiB, is 4 us faster than a
// kernel on an idle stream (into pinned memory 7.8 against 11.9 us at 17 KB, 9.6
// against 12.4 at 64; 2100 radii 13.7 -> 10.5 us, a 30^2 field 13.4 -> 9.7), and
// up to there the conversion takes less.  Behind a kernel it is slower (bubble
// indices, 25 against 18 us).
constexpr size_t kCopyMin = 1 << 14;

void HostRing::release() {
    for (hipEvent_t &e : ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
    if (host) (void)hipHostFree(host);
    host = nullptr;
}

hipError_t HostRing::reserve() {
    if (host) return hipSuccess;
    hipError_t e = hipHostMalloc((void **)&host, sizeof(double) * kSlotDoubles * kSlots,
                                 hipHostMallocDefault);
    if (e != hipSuccess) host = nullptr;
    for (int k = 0; k < kSlots && e == hipSuccess; k++)
        e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
    if (e != hipSuccess) release();
    return e;
}

namespace {
// Elements e0 .. e0 + n of the packed array from a slot to their rows.
void copy_out(const double *buf, int64_t e0, int64_t n, int64_t nx, double *dst, int64_t ld) {
    if (ld == nx) {
        std::memcpy(dst + e0, buf, sizeof(double) * n);
        return;
    }
    for (int64_t k = 0; k < n;) {
        const int64_t j = (e0 + k) / nx, i = (e0 + k) - j * nx;
        const int64_t m = std::min(nx - i, n - k);
        std::memcpy(dst + j * ld + i, buf + k, sizeof(double) * m);
        k += m;
    }
}

hipError_t launch_pack(hipStream_t s, const PackSrc &src, int64_t e0, int n, double *out) {
    hipLaunchKernelGGL(k_pack, dim3(std::min(512, (n + 255) / 256)), dim3(256), 0, s, src, e0, n, out);
    return hipGetLastError();
}

// The bytes from the source's beginning to the end of its last row, or of the
// bubble array; 0 where the kernel has to do it.
size_t source_span(const PackSrc &s, int64_t rows) {
    const size_t elem = s.kind == PackSrc::kFloat || s.kind == PackSrc::kPermInt ? 4 : 8;
    if (permuted(s)) return s.perm ? elem * s.nx : 0;
    return s.kind == PackSrc::kSum3 ? 0 : elem * s.pitch * (rows + s.j0 + 1);
}

// The source's values from a copy of its span.
void convert_out(PackSrc s, const void *copy, int64_t rows, double *dst, int64_t ld) {
    s.src = copy;
    if (permuted(s)) {
        for (int64_t k = 0; k < s.nx; k++) dst[s.perm[k]] = source_value(s, k);
        return;
    }
    for (int64_t j = 0; j < rows; j++) {
        const int64_t o = frame_off(s.i0, (int)j + s.j0, s.pitch);
        for (int64_t i = 0; i < s.nx; i++) dst[j * ld + i] = source_value(s, o + i);
    }
}
}  // namespace

hipError_t read_back(hipStream_t s, int device, HostRing &ring, const PackSrc &src, int64_t rows,
                     double *dst, int64_t ld) {
    const int64_t nx = src.nx, total = nx * rows;
    if (total <= 0) return hipSuccess;
    const std::lock_guard<std::mutex> lock(ring.mu);
    const size_t span = source_span(src, rows);
    if (span > kCopyMin && span <= HostRing::kCopyMax) {
        hipError_t e = hipMemcpyAsync(ring.small, src.src, span, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e == hipSuccess) convert_out(src, ring.small, rows, dst, ld);
        return e;
    }
    if (total <= ring.small_doubles) {
        hipError_t e = launch_pack(s, src, 0, (int)total, ring.small);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e == hipSuccess) copy_out(ring.small, 0, total, nx, dst, ld);
        return e;
    }
    if (hipError_t e = ring.reserve()) return e;
    const int64_t pieces = (total + kSlotDoubles - 1) / kSlotDoubles;
    std::atomic<int64_t> next{0};
    std::atomic<int> failed{(int)hipSuccess};
    auto work = [&](int slot) {
        double *buf = ring.host + slot * kSlotDoubles;
        for (int64_t c; failed == (int)hipSuccess && (c = next++) < pieces;) {
            const int64_t e0 = c * kSlotDoubles;
            const int n = (int)std::min(kSlotDoubles, total - e0);
            hipError_t q = launch_pack(s, src, e0, n, buf);
            if (q == hipSuccess) q = hipEventRecord(ring.ev[slot], s);
            if (q == hipSuccess) q = hipEventSynchronize(ring.ev[slot]);
            if (q != hipSuccess) {
                failed = (int)q;
                return;
            }
            copy_out(buf, e0, n, nx, dst, ld);
        }
    };
    // two pieces or more to a thread; a thread that cannot be had is done without
    const int helpers = (int)std::min<int64_t>(kSlots, pieces / 2) - 1;
    std::vector<std::thread> pool;
    const auto helper = [&](int slot) {
        if (hipError_t d = hipSetDevice(device))  // the current device is per thread
            failed = (int)d;
        else
            work(slot);
    };
    try {
        for (int w = 1; w <= helpers; w++) pool.emplace_back(helper, w);
    } catch (const std::system_error &) {
    } catch (const std::bad_alloc &) {
    }
    work(0);
    for (std::thread &t : pool) t.join();
    return (hipError_t)failed.load();
}

}  // namespace brp
