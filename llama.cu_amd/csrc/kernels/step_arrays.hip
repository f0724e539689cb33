// A step's arrays (tokens, positions, block tables, task lists) from host memory, packed into pinned memory, to their places on the device.
//
// What a decode step brings is a few hundred bytes to some tens of kilobytes, spread over arrays of fixed capacity.  One copy of the whole
// capacity is a job of the copy engine with a signal on either side of it, between two steps of the queue: 26 us stood between one captured step and the
// next with it, 10 with this kernel (40 launches replayed; 40,000 entries of capacity, 4,000 in use).  The kernel is bound by one trip over the host's bus, so every
// piece is on its way at once: 16 bytes a thread, the pieces behind one another over the grid.  (5.3 to 7.8 us a launch in steps of 1 to 64 requests.)
#include <string.h>
#include "common.h"

constexpr int ARRAY_PIECES = 24;                 // pieces a launch takes (some 700 bytes of its arguments)
constexpr int ARRAY_BLOCKS = 64;                 // workgroups a launch has at most (each marks that it has read its part; 64 bring 256 KB over in one trip)

// `rows` rows that begin at `at` and then every `stride` entries on the device, at `from` and then every `apart` on the host: the first `cols` of a row's
// `width` entries come over, zeros stand behind them; all in units of 16 bytes
struct ArrayPiece { int at, cols, rows, stride, width, from, apart; };
struct ArrayPieces { ArrayPiece p[ARRAY_PIECES]; };

// Loads that see what the host wrote last, whatever the device's caches hold of the same addresses.
__device__ __forceinline__ uint64_t host_load(const uint64_t *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); }

__global__ void __launch_bounds__(256)
step_arrays_kernel(const uint64_t *__restrict__ host, uint64_t *__restrict__ dev, ArrayPieces pieces, int n_pieces, int total, int *marks, int ticket) {
    for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
        int left = i, k = 0;
        while (k + 1 < n_pieces && left >= pieces.p[k].width * pieces.p[k].rows) { left -= pieces.p[k].width * pieces.p[k].rows; ++k; }
        const ArrayPiece q = pieces.p[k];
        const int col = left % q.width;
        const size_t row = left / q.width, at = 2 * (q.at + row * q.stride + col), from = 2 * (q.from + row * q.apart + col);
        const uint64_t lo = col < q.cols ? host_load(host + from) : 0, hi = col < q.cols ? host_load(host + from + 1) : 0;
        dev[at] = lo;
        dev[at + 1] = hi;
    }
    // The host's memory has been read (what was loaded is behind the barrier, as every wave has it in registers to store it): the host may write there again.  A mark
    // costs the queue nothing, where an event behind every launch took 4 us.
    __syncthreads();
    if (marks && threadIdx.x == 0) __hip_atomic_store(marks + blockIdx.x, ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The address under which the device reads pinned host memory.
LCU_API int lcu_host_on_device(void *host, void **on_device) {
    if (!host || !on_device) return LCU_BAD_ARGUMENT;
    const hipError_t e = hipHostGetDevicePointer(on_device, host, 0);
    if (e != hipSuccess) { (void)hipGetLastError(); return LCU_UNSUPPORTED; }
    return LCU_OK;
}

// dev: an array of `size` 32-bit entries.  pieces: n_pieces times (at, cols, rows, stride, width) in entries, rows as they are and the others multiples of 4,
// cols <= width <= stride (of a single row: any stride): see ArrayPiece.  Where they come from: arrays (null: see below), in ordinary host memory and laid out like dev; what is
// wanted of it is copied to `packed`, one piece behind the other, before anything is launched.  packed: pinned host memory with room for packed_size entries; host: the
// same memory as lcu_host_on_device names it.  Without arrays, host is laid out like dev.  dev, packed, host: 16-byte aligned.
// marks (null: none): ARRAY_BLOCKS ints in pinned host memory, under their address on the device; *n_marks of them, as many as come back, hold `ticket` once all of `host`
// that is wanted has been read.
LCU_API int lcu_step_arrays(const int *arrays, int *packed, long long packed_size, const void *host, void *dev, long long size, const int *pieces, int n_pieces, int *marks,
                            int ticket, int *n_marks, hipStream_t stream) {
    if (n_marks) *n_marks = 0;
    if ((marks && !n_marks) || n_pieces < 0 || size < 0 || (n_pieces && (!host || !dev || !pieces)) || (n_pieces && arrays && !packed) ||
        ((uintptr_t)host | (uintptr_t)dev | (uintptr_t)packed) % 16)
        return LCU_BAD_ARGUMENT;
    int end = 0;                                 // behind the last piece with anything in it: its launch, the last one, leaves the marks
    long long wanted = 0;
    for (int i = 0; i < n_pieces; ++i) {
        const int *p = pieces + 5 * i, at = p[0], cols = p[1], rows = p[2], stride = p[3], width = p[4];
        if (at < 0 || cols < 0 || rows < 0 || stride < 0 || width < cols || (at | cols | stride | width) % 4) return LCU_BAD_ARGUMENT;
        if (width == 0 || rows == 0) continue;
        if ((long long)at + (long long)(rows - 1) * stride + width > size || (rows > 1 && stride < width)) return LCU_BAD_ARGUMENT;
        wanted += (long long)rows * cols;
        end = i + 1;
    }
    if (arrays && wanted > packed_size) return LCU_BAD_ARGUMENT;
    int from = 0;
    for (int done = 0; done < end;) {
        ArrayPieces a{};
        int n = 0;
        long long total = 0;
        for (; n < ARRAY_PIECES && done < end; ++done) {
            const int *p = pieces + 5 * done, at = p[0], cols = p[1], rows = p[2], stride = p[3], width = p[4];
            if (width == 0 || rows == 0) continue;
            a.p[n++] = arrays ? ArrayPiece{at / 4, cols / 4, rows, stride / 4, width / 4, from / 4, cols / 4}
                              : ArrayPiece{at / 4, cols / 4, rows, stride / 4, width / 4, at / 4, stride / 4};
            total += (long long)(width / 4) * rows;
            for (int r = 0; arrays && r < rows; ++r, from += cols) memcpy(packed + from, arrays + at + (size_t)r * stride, (size_t)cols * sizeof(int));
        }
        if (total > 0x7fffffffLL - ARRAY_BLOCKS * 256) return LCU_BAD_ARGUMENT;
        const int blocks = total > ARRAY_BLOCKS * 256 ? ARRAY_BLOCKS : (int)((total + 255) / 256);
        const bool last = done == end;
        step_arrays_kernel<<<blocks, 256, 0, stream>>>((const uint64_t *)host, (uint64_t *)dev, a, n, (int)total, last ? marks : nullptr, ticket);
        LCU_LAUNCH_CHECK();
        if (last && marks) *n_marks = blocks;
    }
    return LCU_OK;
}
