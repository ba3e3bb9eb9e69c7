// A HIP runtime of two devices in host memory, for tests of the library's host
// code on a machine without a GPU: linked into this program, its functions
// take the place of the runtime's.  Launches compute nothing, but for k_pack
// of FP64 fields.  Streams, events and memory belong to the device that is
// current when they are made; a launch or a record on another device's stream
// is counted, as is memory taken on another device than the test names.
//
//   fake_hip devices   one handle per device, read back, saved and restored
//                      while the other device is current
//   fake_hip threads   two threads read two fields of one handle
//   fake_hip slots     a slot saved again after the window has grown
//   fake_hip rows      a rectangle of more rows than a launch has workgroups in y
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <thread>
#include <vector>

#include "brp_internal.h"
#include "bubbles_rp.h"

namespace {
thread_local int current = 0;
std::atomic<int> foreign{0};    // launches and records on another device's stream
std::atomic<int> expected{-1};  // device on which memory has to be taken, -1: any
std::atomic<int> misplaced{0};
std::atomic<int> taken{0};      // allocations of device memory
std::atomic<int> too_tall{0};   // launches of more than 65535 workgroups in y or z
std::atomic<bool> slow{false};  // waits take a while
struct Handle {
    int device;
};
struct Config {
    dim3 g, b;
    size_t shared;
    hipStream_t s;
};
thread_local Config config;

// kernel names (the library registers its kernels before main's statics are made)
std::map<const void *, std::string> &names() {
    static std::map<const void *, std::string> m;
    return m;
}

int device_of(const void *h) { return h ? ((const Handle *)h)->device : current; }
void pause_a_little() {
    if (slow) std::this_thread::sleep_for(std::chrono::microseconds(200));
}
}  // namespace

extern "C" {
void **__hipRegisterFatBinary(const void *) {
    static void *p;
    return &p;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) {
    names()[host] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shared, hipStream_t s) {
    config = Config{g, b, shared, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shared, hipStream_t *s) {
    *g = config.g;
    *b = config.b;
    *shared = config.shared;
    *s = config.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3, void **args, size_t, hipStream_t s) {
    if (g.y > 65535 || g.z > 65535) too_tall++;
    if (device_of(s) != current) foreign++;
    if (names().at(f).find("k_pack") != std::string::npos) {
        const auto &src = *(const brp::PackSrc *)args[0];
        const int64_t e0 = *(const int64_t *)args[1];
        const int n = *(const int *)args[2];
        double *out = *(double **)args[3];
        if (src.kind == brp::PackSrc::kDouble)
            for (int k = 0; k < n; k++) {
                const int64_t j = (e0 + k) / src.nx, i = (e0 + k) - j * src.nx;
                out[k] = ((const double *)src.src)[brp::frame_off((int)i + src.i0, (int)j + src.j0,
                                                                 src.pitch)];
            }
    }
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
    *d = current;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    if (d < 0 || d > 1) return hipErrorInvalidDevice;
    current = d;
    return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int) {
    *v = a == hipDeviceAttributeMultiprocessorCount ? 256 : 100000;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
    *n = 2;
    return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
    if (expected >= 0 && current != expected) misplaced++;
    taken++;
    *p = std::calloc(n, 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    *p = std::calloc(n, 1);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemset(void *d, int v, size_t n) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static double scratch[1 << 12];
    *p = scratch;
    return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s) {
    *s = (hipStream_t) new Handle{current};
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    delete (Handle *)s;
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
    pause_a_little();
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = (hipEvent_t) new Handle{current};
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete (Handle *)e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (device_of(e) != device_of(s)) foreign++;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) {
    pause_a_little();
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
}  // extern "C"

namespace {
brp_handle *make(int n, bool bubbles) {
    brp_config c;
    brp_config_default(&c);
    c.grid_x = c.grid_y = n;
    c.grid_lx = c.grid_ly = n * 1e-4;
    c.sim_cfl = 0.5;
    c.tr_freq = 1e6;
    c.bub_enable = bubbles;
    c.bub_P0 = 1e5;
    c.bub_T0 = 293.15;
    c.bub_gamma = 1.4;
    c.bub_rho = 1e3;
    c.bub_K0 = 26e-3;
    c.bub_mu = 1e-3;
    brp_handle *h = nullptr;
    if (brp_create(&c, &h) != BRP_OK) {
        std::printf("brp_create: %s\n", brp_last_error(nullptr));
        std::exit(2);
    }
    if (bubbles) {
        const std::vector<double> x(100, 2e-3), R(100, 3e-6);
        if (brp_set_bubbles(h, 100, x.data(), x.data(), R.data(), nullptr, 1e-9) != BRP_OK) {
            std::printf("brp_set_bubbles: %s\n", brp_last_error(h));
            std::exit(2);
        }
    }
    return h;
}

int bad = 0;
void check(const char *what, int n, brp_handle *h, int rc, int device) {
    if (rc != BRP_OK || foreign || misplaced || current != device) {
        std::printf("%s, %d^2: status %d (%s), %d launches or events on a foreign stream, %d "
                    "allocations on another device, current device %d of %d\n",
                    what, n, rc, rc ? brp_last_error(h) : "", foreign.load(), misplaced.load(),
                    current, device);
        bad = 1;
    }
    foreign = misplaced = 0;
    current = device;
}

void devices() {
    for (int n : {48, 400, 700}) {  // the small slot, one thread, several threads
        brp_handle *h[2];
        for (int d = 0; d < 2; d++) {
            current = d;
            h[d] = make(n, true);
            if (brp_prepare(h[d]) != BRP_OK) std::exit(2);
        }
        std::vector<double> out((size_t)(n + 3) * (n + 3));
        for (int cur = 0; cur < 2; cur++)
            for (int d = 0; d < 2; d++) {
                current = cur;
                expected = d;
                check("brp_get_field", n, h[d], brp_get_field(h[d], BRP_FIELD_P0, out.data(), n + 3), cur);
                check("brp_get_bubbles", n, h[d], brp_get_bubbles(h[d], BRP_BUB_R_T, out.data()), cur);
                check("brp_get_bubbles (index)", n, h[d],
                      brp_get_bubbles(h[d], BRP_BUB_IBN_X, out.data()), cur);
                check("brp_save_state", n, h[d], brp_save_state(h[d], cur), cur);
                check("brp_restore_state", n, h[d], brp_restore_state(h[d], cur), cur);
                expected = -1;
            }
        for (brp_handle *q : h) brp_destroy(q);
    }
}

void threads() {
    for (int n : {48, 400, 700}) {
        brp_handle *h = make(n, false);
        const size_t m = (size_t)(n + 3) * (n + 3);
        const int32_t field[2] = {BRP_FIELD_P0, BRP_FIELD_PX};
        std::vector<double> in[2];
        for (int k = 0; k < 2; k++) {
            in[k].resize(m);
            for (size_t q = 0; q < m; q++) in[k][q] = (k ? -1.0 : 1.0) * (double)(q + 1);
            if (brp_set_field(h, field[k], in[k].data(), n + 3) != BRP_OK) std::exit(2);
        }
        slow = true;
        std::atomic<int> wrong{0};
        const auto reader = [&](int k) {
            int nx, ny, i0, j0;
            brp_field_shape(h, field[k], &nx, &ny, &i0, &j0);
            std::vector<double> out(m);
            for (int r = 0; r < 20; r++) {
                if (brp_get_field(h, field[k], out.data(), n + 3) != BRP_OK) wrong++;
                for (int j = 0; j < ny; j++)
                    for (int i = 0; i < nx; i++)
                        if (out[(size_t)j * (n + 3) + i] != in[k][(size_t)j * (n + 3) + i]) {
                            wrong++;
                            j = ny;
                            break;
                        }
            }
        };
        std::thread other(reader, 1);
        reader(0);
        other.join();
        slow = false;
        if (wrong) {
            std::printf("%d^2: %d of 40 reads returned other values\n", n, wrong.load());
            bad = 1;
        }
        brp_destroy(h);
    }
}

void slots() {
    const int n = 200;
    brp_handle *h = make(n, true);
    if (brp_save_state(h, 0) != BRP_OK) std::exit(2);
    std::vector<double> fg((size_t)(n + 2) * (n + 2), 1e-6);
    if (brp_set_field(h, BRP_FIELD_FGN, fg.data(), n + 2) != BRP_OK) std::exit(2);
    taken = 0;
    if (brp_save_state(h, 0) != BRP_OK || taken) {
        std::printf("a slot saved again took memory %d times\n", taken.load());
        bad = 1;
    }
    brp_destroy(h);
}

void rows() {
    // the tallest grid's frame (65 536 cells and its ghosts)
    brp::RectPlan r;
    int64_t a[1], b[1];
    r.add(a, b, sizeof(int64_t));
    brp::launch_copy_rects(nullptr, r, brp::Window{-1, 9, -1, 65537}, 128);
    if (too_tall) {
        std::printf("%d launches of more than 65535 workgroups in y\n", too_tall.load());
        bad = 1;
    }
}
}  // namespace

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "devices")
        devices();
    else if (what == "threads")
        threads();
    else if (what == "slots")
        slots();
    else if (what == "rows")
        rows();
    else
        return 2;
    return bad;
}
