// Stand-ins for the kernel launchers of the built library and for the HIP calls of its host layer (no GPU, nothing is
// computed): they record the memory that a call uses and the allocations that are alive.
#pragma once

#include <cstdint>
#include <cstdlib>
#include <map>
#include <vector>

#include "../../asc-devkit_clone_amd/csrc/launch.h"
#include "ascq.h"

struct Region {
    uintptr_t at;
    size_t bytes;
    const char* what;
};
static std::vector<Region> used;         // by the present call
static std::map<uintptr_t, size_t> heap;  // allocations (addresses only, never dereferenced)
static uintptr_t next_at = 0x100000000ull;
static bool capturing = false;  // the stream of the present call
static int device = 0;
static hipStreamCaptureMode capture_mode = hipStreamCaptureModeGlobal;
static int alloc_not_relaxed = 0;  // hipMalloc / hipFree that would invalidate another stream's capture

static void use(const void* p, size_t bytes, const char* what)
{
    if (bytes) used.push_back({(uintptr_t)p, bytes, what});
}

extern "C" {
hipError_t hipMalloc(void** p, size_t n)
{
    alloc_not_relaxed += capture_mode != hipStreamCaptureModeRelaxed;
    heap[next_at] = n;
    *p = (void*)next_at;
    next_at += (n + 0xFFFFF) / 0x100000 * 0x100000 + 0x100000;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    alloc_not_relaxed += capture_mode != hipStreamCaptureModeRelaxed;
    if (p && !heap.erase((uintptr_t)p)) std::abort();
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDevice(int* d)
{
    *d = device;
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m)
{
    const hipStreamCaptureMode old = capture_mode;
    capture_mode = *m;
    *m = old;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*)
{
    *p = (void*)0x80000000ull;
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s)
{
    *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
}

namespace ascq {
hipError_t launch_pack_rows(const PackRows& a, const PackRows& b, hipStream_t)
{
    if ((uintptr_t)a.dst % 16 != 0 || (uintptr_t)b.dst % 16 != 0) return hipErrorInvalidValue;  // (as the launcher does)
    if (a.dst) use(a.dst, (size_t)a.rows * ((a.cols + 15) / 16 * 16), "packed A");
    if (b.dst) use(b.dst, (size_t)b.rows * ((b.cols + 15) / 16 * 16), "packed B");
    return hipSuccess;
}
hipError_t launch_byte_to_bf16(uint16_t* dst, int64_t ldd, const uint8_t*, int64_t, int64_t rows, int64_t, int, int transpose,
                               hipStream_t)
{
    if ((uintptr_t)dst % 16 != 0) return hipErrorInvalidValue;  // (as the launcher does)
    use(dst, (size_t)(rows * ldd) * 2, transpose ? "packed B (bf16)" : "packed A (bf16)");
    return hipSuccess;
}
hipError_t launch_transpose_i8(uint8_t* dst, const uint8_t*, int64_t rows, int64_t cols, hipStream_t)
{
    use(dst, (size_t)(rows * cols), "transposed A");
    return hipSuccess;
}
hipError_t launch_nz_to_nd(void* dst, const void*, int, int, int64_t rows, int64_t cols, int, hipStream_t)
{
    use(dst, (size_t)(rows * cols), "B from NZ");
    return hipSuccess;
}
template <class G>
static hipError_t gemm(const G& g)
{
    if (g.ws) {
        use(g.ws, decode_split_ws_bytes(g.M, g.N, g.K, g.trans_b), "split partials");
        if (decode_split_ws_bytes(g.M, g.N, g.K, g.trans_b) > g.ws_bytes) use(g.ws, SIZE_MAX / 2, "split partials (room)");
    }
    return hipSuccess;
}
hipError_t launch_gemm_i8(const GemmI8Args& g, hipStream_t) { return gemm(g); }
hipError_t launch_gemm_f8(const GemmF8Args& g, hipStream_t) { return gemm(g); }
}  // namespace ascq

