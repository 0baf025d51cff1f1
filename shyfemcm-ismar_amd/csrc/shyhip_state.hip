// shyhip_state.hip -- whole state arrays moved between models and to the host.
//
// launch_copy_arrays: the arrays of a member's state into another model, all
// in one launch (a strided copy each was 3 us of device time and a launch for
// every one of a member's 36 arrays).
// launch_to_host_layout: an array [row][column] of the device into the
// host's layout [column][row] and type, so that a pull is one copy; the host
// used to transpose and convert element by element.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "shyhip_internal.h"

namespace shy {

// ---------------------------------------------------------------- state copies
// Bound by memory: each workgroup copies at most kCopyChunk bytes of one row
// of one array, 16 bytes per work-item and access where both sides are
// aligned to it (a member's rows start anywhere), else 4.
constexpr int kCopyJobs = 48;
constexpr size_t kCopyChunk = 32 * 1024;

struct CopyJob {
    char *d;
    const char *s;
    size_t dp, sp, w;        // row strides and row length in bytes
    unsigned chunks, first;  // workgroups per row, first workgroup
};
struct CopyArgs {
    CopyJob job[kCopyJobs];
    int n;
};

__global__ __launch_bounds__(kThreads) void k_copy_arrays(CopyArgs a) {
    int lo = 0, hi = a.n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) / 2;
        if (a.job[mid].first <= blockIdx.x) lo = mid;
        else hi = mid - 1;
    }
    const CopyJob j = a.job[lo];
    const unsigned idx = blockIdx.x - j.first, row = idx / j.chunks, c = idx % j.chunks;
    const size_t off = (size_t)c * kCopyChunk, len = min(kCopyChunk, j.w - off);
    const char *s = j.s + row * j.sp + off;
    char *d = j.d + row * j.dp + off;
    if (((reinterpret_cast<size_t>(s) | reinterpret_cast<size_t>(d) | len) & 15) == 0) {
        for (size_t i = threadIdx.x; i < len / 16; i += kThreads)
            reinterpret_cast<int4 *>(d)[i] = reinterpret_cast<const int4 *>(s)[i];
    } else {
        for (size_t i = threadIdx.x; i < len / 4; i += kThreads)
            reinterpret_cast<int *>(d)[i] = reinterpret_cast<const int *>(s)[i];
    }
}

int launch_copy_arrays(Model &M, const std::vector<ArrayCopy> &list) {
    CopyArgs a{};
    unsigned blocks = 0;
    auto flush = [&]() -> int {
        if (a.n == 0) return 0;
        hipLaunchKernelGGL(k_copy_arrays, dim3(blocks), dim3(kThreads), 0, M.stream, a);
        HIPCHK(M, hipGetLastError());
        a.n = 0;
        blocks = 0;
        return 0;
    };
    for (const ArrayCopy &x : list) {
        if (x.width == 0 || x.rows == 0) continue;
        CopyJob j{(char *)x.dst, (const char *)x.src, x.dpitch, x.spitch, x.width, 0, blocks};
        size_t rows = x.rows;
        if (x.dpitch == x.width && x.spitch == x.width) {      // one contiguous range
            j.w = x.width * rows;
            rows = 1;
        }
        j.chunks = (unsigned)((j.w + kCopyChunk - 1) / kCopyChunk);
        a.job[a.n++] = j;
        blocks += (unsigned)(j.chunks * rows);
        if (a.n == kCopyJobs && flush()) return 1;
    }
    return flush();
}

// ---------------------------------------------------------------- host layout
// A workgroup takes kHostCols columns: rows read as the device lays them out,
// turned round in LDS, written as one contiguous range.
constexpr int kHostCols = 64;

template <typename S, typename D>
__global__ __launch_bounds__(kThreads) void k_to_host_layout(const S *a, D *out, int rows, int cols, int c0, int nc) {
    extern __shared__ double smem[];
    D *tile = reinterpret_cast<D *>(smem);       // [row][kHostCols + 1]
    const int b0 = blockIdx.x * kHostCols, n = min(kHostCols, nc - b0);
    const int c = threadIdx.x % kHostCols;
    for (int r = threadIdx.x / kHostCols; r < rows; r += kThreads / kHostCols)
        if (c < n) tile[r * (kHostCols + 1) + c] = (D)a[(size_t)r * cols + c0 + b0 + c];
    __syncthreads();
    for (int i = threadIdx.x; i < n * rows; i += kThreads)
        out[(size_t)b0 * rows + i] = tile[(i % rows) * (kHostCols + 1) + i / rows];
}

template <typename S, typename D>
static int to_host_t(Model &M, const void *a, void *out, int rows, int cols, int c0, int nc) {
    hipLaunchKernelGGL((k_to_host_layout<S, D>), dim3((nc + kHostCols - 1) / kHostCols), dim3(kThreads),
                       (size_t)rows * (kHostCols + 1) * sizeof(D), M.stream, (const S *)a, (D *)out, rows, cols, c0, nc);
    HIPCHK(M, hipGetLastError());
    return 0;
}

int launch_to_host_layout(Model &M, const void *a, bool a_double, void *out, bool out_double, int rows, int cols, int c0,
                          int nc) {
    if (a_double)
        return out_double ? to_host_t<double, double>(M, a, out, rows, cols, c0, nc)
                          : to_host_t<double, float>(M, a, out, rows, cols, c0, nc);
    return out_double ? to_host_t<float, double>(M, a, out, rows, cols, c0, nc)
                      : to_host_t<float, float>(M, a, out, rows, cols, c0, nc);
}

}  // namespace shy
