// kernels_copy.hip -- device-to-device copies of many arrays in one launch.
//
// A snapshot is some forty arrays and a recorded step a dozen, most of them
// small: as copy commands each costs its own launch, about 5 us of host and 2.5
// us of device time.  Here one launch copies them all, a workgroup to a tile
// of one array (restore at 64^2 205 -> 14 us, 256^2 197 -> 15, 2048^2 with 2^20 bubbles
// 315 -> 126, which with the void-fraction rows outside the window left out; a 4096^2
// snapshot moves 5.2 TB/s, read and written).
#include "brp_internal.h"

#include <algorithm>

namespace brp {
namespace {

typedef unsigned int u4 __attribute__((ext_vector_type(4)));
constexpr unsigned kTile = 256 * 16 * 8;  // bytes of a workgroup: eight 16-byte pieces a thread

__global__ __launch_bounds__(256) void k_copy_many(CopyPlan c) {
    int lo = 0, hi = c.n - 1;  // the last array whose first tile is not after this one
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (c.tile0[mid] <= blockIdx.x)
            lo = mid;
        else
            hi = mid - 1;
    }
    const size_t at = (size_t)(blockIdx.x - c.tile0[lo]) * kTile;
    const size_t n = min((size_t)kTile, c.bytes[lo] - at);
    const char *src = c.src[lo] ? (const char *)c.src[lo] + at : nullptr;
    char *dst = (char *)c.dst[lo] + at;
    const unsigned pieces = (unsigned)(n / 16);
    u4 v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const unsigned p = threadIdx.x + 256 * k;
        v[k] = src && p < pieces ? ((const u4 *)src)[p] : u4{0, 0, 0, 0};
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const unsigned p = threadIdx.x + 256 * k;
        if (p < pieces) ((u4 *)dst)[p] = v[k];
    }
    const unsigned tail = (unsigned)(n % 16) / 4;  // whole words (the arrays' elements)
    if (threadIdx.x < tail) {
        const size_t o = (size_t)pieces * 16 + 4 * threadIdx.x;
        *(unsigned *)(dst + o) = src ? *(const unsigned *)(src + o) : 0u;
    }
}

// Rows blockIdx.y, blockIdx.y + gridDim.y, ... of rectangle blockIdx.z, from its
// frame to its dense buffer.  (A launch may have 65 536 workgroups in y, the
// tallest frame has 65 539 rows.)
constexpr int kRectRows = 1 << 15;

__global__ __launch_bounds__(256) void k_copy_rects(RectPlan r, Window w, int pitch) {
    const int z = blockIdx.z;
    const int words = (w.i1 - w.i0 + 1) * (r.elem[z] / 4);
    for (int row = blockIdx.y; row <= w.j1 - w.j0; row += gridDim.y) {
        const unsigned *src = (const unsigned *)((const char *)r.src[z] +
                                                 frame_off(w.i0, w.j0 + row, pitch) * r.elem[z]);
        unsigned *dst = (unsigned *)r.dst[z] + (size_t)row * words;
        for (int k = blockIdx.x * 256 + threadIdx.x; k < words; k += gridDim.x * 256) dst[k] = src[k];
    }
}

}  // namespace

void CopyPlan::add(void *d, const void *s, size_t b) {
    if (b == 0) return;
    dst[n] = d;
    src[n] = s;
    bytes[n] = b;
    tile0[n] = tiles;
    tiles += (unsigned)((b + kTile - 1) / kTile);
    n++;
}

void launch_copy_many(hipStream_t s, const CopyPlan &c) {
    if (c.n > 0) hipLaunchKernelGGL(k_copy_many, dim3(c.tiles), dim3(256), 0, s, c);
}

void launch_copy_rects(hipStream_t s, const RectPlan &r, const Window &w, int pitch) {
    if (r.n <= 0 || w.i0 > w.i1 || w.j0 > w.j1) return;
    const int cols = w.i1 - w.i0 + 1;
    const int rows = std::min(kRectRows, w.j1 - w.j0 + 1);
    hipLaunchKernelGGL(k_copy_rects, dim3(std::min(8, (2 * cols + 255) / 256), rows, r.n), dim3(256),
                       0, s, r, w, pitch);
}

}  // namespace brp
