// common.hpp -- status codes, error reporting and launch helpers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>

#include "../../include/depixel.h"

namespace dpx {

// Records a message as the calling thread's last error and returns `code`.
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// Flags the library knows; the stage and per-frame paths take no indexed frames.
constexpr uint32_t kKnownFlags = DPX_RGB | DPX_TOPDOWN | DPX_ALPHA | DPX_FLIP_OUT | DPX_INDEXED;

// Bytes of a DPX_INDEXED palette: 256 four-byte entries.
constexpr size_t kPaletteBytes = 1024;

// Returns DPX_ENODEV when the process sees no GPU.
int require_device();

// hipMemcpy from the device to host memory that need not be pinned, for
// results of megabytes.
hipError_t download(void* dst, const void* src, size_t n);

// Sizes a context's cell coverage buffer (subdivided items) to at least `bytes`.
int context_reserve_rows(dpx_context* ctx, size_t bytes);

// The samples of a smoothed cell at scale S.  A smoothed vertex is one of the
// cell's hull, a cut point of one of its edges, or the middle between such a
// point and one of the neighbour's hull; over all pairs of hulls that leaves x
// in -48 .. 86 and y in -42 .. 106 (1/64 of a cell; game frames stay within -22
// .. 86, dithers of nearly similar colours do not).  Columns cover_x0(S) .. of
// cover_w(S) <= 32, rows cover_y0(S) .. of cover_h(S); sample k's centre lies at
// (k + 1/2) / S.
constexpr int kReachXLow = -48, kReachXHigh = 86, kReachYLow = -42, kReachYHigh = 106;
constexpr int first_sample(int S, int low)  // the least k with (2 k + 1) 32 >= low S
{
    const int n = low * S - 32;
    return n >= 0 ? (n + 63) / 64 : -(-n / 64);
}
constexpr int last_sample(int S, int high) { return (high * S - 32) / 64; }
constexpr int cover_x0(int S) { return first_sample(S, kReachXLow); }
constexpr int cover_w(int S) { return last_sample(S, kReachXHigh) - cover_x0(S) + 1; }
constexpr int cover_y0(int S) { return first_sample(S, kReachYLow); }
constexpr int cover_h(int S) { return last_sample(S, kReachYHigh) - cover_y0(S) + 1; }

// Coverage words per cell at scale S: nine cell masks of 2 bytes (up to 4x) or
// S bytes (up to 8x), or the sample rows, and a summary.
constexpr size_t cell_row_words(int S)
{
    return S <= 4 ? 5 : S <= 8 ? (9 * (size_t)S + 1 + 3) / 4 : (size_t)cover_h(S) + 1;
}

}  // namespace dpx

#define DPX_HIP(call)                                                                                   \
    do {                                                                                                \
        hipError_t dpx_e_ = (call);                                                                     \
        if (dpx_e_ != hipSuccess)                                                                       \
            return ::dpx::fail(dpx_e_ == hipErrorOutOfMemory ? DPX_ENOMEM : DPX_EHIP, "%s: %s (%s:%d)", \
                               #call, hipGetErrorString(dpx_e_), __FILE__, __LINE__);                   \
    } while (0)

#define DPX_CHECK(cond, ...)                          \
    do {                                              \
        if (!(cond)) return ::dpx::fail(__VA_ARGS__); \
    } while (0)
