// IntLSE fixed-point launchers for gfx950: Q16.16 (fp32 input quantised in the
// kernel, or pre-quantised int32 input) and Q10.6 (int16 input).  The kernels
// and the reduction tree they follow are in lse_int_kernels.hpp.
#include <stdint.h>

#include <type_traits>

#include "../../include/fuselse_amd.h"
#include "fl_status.hpp"
#include "lse_int_kernels.hpp"

namespace fl {

// Calls launch(grid, x, out, acc) for consecutive chunks of rows (one block
// per row), each within one dispatch for blocks of up to 256 threads.
template <typename T, typename LAUNCH>
static void for_row_chunks(const T* x, float* out, int32_t* acc, int64_t B, int64_t N, LAUNCH launch) {
    for_grid_chunks(B, 256, [&](int64_t r0, int64_t rows) {
        launch(dim3((unsigned)rows), x + r0 * N, out + r0, acc ? acc + r0 : nullptr);
    });
}

template <typename T>
static int int_entry_check(const char* name, const T* x, float* out, int64_t B, int64_t N) {
    FL_CHECK(B >= 0 && N >= 0, "%s: negative shape (B=%lld, N=%lld)", name, (long long)B, (long long)N);
    if (B == 0) return ok();
    FL_CHECK(out != nullptr, "%s: out is NULL", name);
    FL_CHECK(x != nullptr || N == 0, "%s: x is NULL", name);
    FL_CHECK((reinterpret_cast<uintptr_t>(x) % sizeof(T)) == 0, "%s: x is not element-aligned", name);
    if (N * (int64_t)sizeof(T) >= ((int64_t)1 << 31))
        return set_error(FL_ERANGE, "%s: rows of %lld elements exceed the 2 GiB buffer range", name, (long long)N);
    return ok();
}

// Whether rows have elements before or after their chunks.
template <int ALIGN, typename T>
static bool edge_rows(const T* x, int64_t N) {
    return N % 4 != 0 || (reinterpret_cast<uintptr_t>(x) & (ALIGN - 1)) != 0;
}

// Whether the short-row kernels take a call: rows of at most 256 chunks, enough
// of them that a wave's longer way through several rows does not show (graph
// replays, Q16.16 fp32 / Q10.6, us, a block per row / short rows: 1024 x 256
// 3.48 / 3.40 -> 3.11 / 2.75, 4096 x 256 6.10 / 4.99 -> 3.25 / 2.86, 65536 x 256
// 62.5 / 41.1 -> 10.2 / 6.7, 65536 x 1024 78.5 / 46.5 -> 40.4 / 19.9; rows with
// edges: 1024 x 255 3.56 / 3.46 -> 5.19 / 3.66, 2048 x 255 4.22 / 4.13 -> 5.22 /
// 3.68, 2048 x 1001 4.66 / 4.17 -> 3.88 / 3.13, 4096 x 255 6.30 / 6.17 -> 5.31 /
// 3.75, 65536 x 255 68.2 / 61.7 -> 14.2 / 8.9).
template <int ALIGN, typename T>
static bool short_rows(const T* x, int64_t B, int64_t N) {
    if (N <= 0 || N / 4 > 256) return false;
    return B >= (!edge_rows<ALIGN>(x, N) ? 1024 : N / 4 > 64 ? 2048 : 4096);
}

// Calls launch(grid, VT, EDGE, first block) for the short-row kernels: VT
// virtual threads a lane hold a row's chunks.
template <int ALIGN, typename T, typename LAUNCH>
static void with_short(const T* x, int64_t B, int64_t N, LAUNCH launch) {
    const bool edge = edge_rows<ALIGN>(x, N);
    const auto go = [&](auto vt) {
        const int64_t per_block = 4 * (8 / vt.value);
        for_grid_chunks((B + per_block - 1) / per_block, 256, [&](int64_t b0, int64_t nb) {
            if (edge)
                launch(dim3((unsigned)nb), vt, std::true_type{}, b0);
            else
                launch(dim3((unsigned)nb), vt, std::false_type{}, b0);
        });
    };
    if (N / 4 <= 64)
        go(std::integral_constant<int, 1>{});
    else if (N / 4 <= 128)
        go(std::integral_constant<int, 2>{});
    else
        go(std::integral_constant<int, 4>{});
}

template <typename SRC>
static void launch_q16_short(const typename SRC::T* x, float* out, int32_t* acc_out, int64_t B, int64_t N, int use_lut,
                             hipStream_t st) {
    with_short<16>(x, B, N, [&](dim3 g, auto vt, auto edge, int64_t b0) {
        if (use_lut)
            intlse_q16_short_rows<SRC, true, vt.value, edge.value><<<g, dim3(256), 0, st>>>(x, out, acc_out, B, N, b0);
        else
            intlse_q16_short_rows<SRC, false, vt.value, edge.value><<<g, dim3(256), 0, st>>>(x, out, acc_out, B, N, b0);
    });
}

}  // namespace fl

using namespace fl;

extern "C" int fl_intlse_q16_f32(const float* x, float* out, int32_t* acc_out, int64_t B, int64_t N, int use_lut,
                                 void* stream) {
    const char* name = "fl_intlse_q16_f32";
    if (int rc = int_entry_check(name, x, out, B, N)) return rc;
    if (B == 0) return ok();
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (short_rows<16>(x, B, N)) {
        launch_q16_short<SrcF32>(x, out, acc_out, B, N, use_lut, st);
        return launch_status(name);
    }
    for_row_chunks(x, out, acc_out, B, N, [&](dim3 g, const float* xc, float* oc, int32_t* ac) {
        with_prefetch(g.x, 16, [&](auto d) {
            if (use_lut)
                intlse_q16_rows<SrcF32, true, d.value><<<g, dim3(256), 0, st>>>(xc, oc, ac, N);
            else
                intlse_q16_rows<SrcF32, false, d.value><<<g, dim3(256), 0, st>>>(xc, oc, ac, N);
        });
    });
    return launch_status(name);
}

extern "C" int fl_intlse_q16_i32(const int32_t* q, float* out, int32_t* acc_out, int64_t B, int64_t N, int use_lut,
                                 void* stream) {
    const char* name = "fl_intlse_q16_i32";
    if (int rc = int_entry_check(name, q, out, B, N)) return rc;
    if (B == 0) return ok();
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (short_rows<16>(q, B, N)) {
        launch_q16_short<SrcI32>(q, out, acc_out, B, N, use_lut, st);
        return launch_status(name);
    }
    for_row_chunks(q, out, acc_out, B, N, [&](dim3 g, const int32_t* qc, float* oc, int32_t* ac) {
        with_prefetch(g.x, 16, [&](auto d) {
            if (use_lut)
                intlse_q16_rows<SrcI32, true, d.value><<<g, dim3(256), 0, st>>>(qc, oc, ac, N);
            else
                intlse_q16_rows<SrcI32, false, d.value><<<g, dim3(256), 0, st>>>(qc, oc, ac, N);
        });
    });
    return launch_status(name);
}

extern "C" int fl_intlse_q10_6(const int16_t* q, float* out, int32_t* acc_out, int64_t B, int64_t N, void* stream) {
    const char* name = "fl_intlse_q10_6";
    if (int rc = int_entry_check(name, q, out, B, N)) return rc;
    if (B == 0) return ok();
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (short_rows<8>(q, B, N)) {
        with_short<8>(q, B, N, [&](dim3 g, auto vt, auto edge, int64_t b0) {
            intlse_q10_6_short_rows<vt.value, edge.value><<<g, dim3(256), 0, st>>>(q, out, acc_out, B, N, b0);
        });
        return launch_status(name);
    }
    const bool paired = (reinterpret_cast<uintptr_t>(q) & 15u) == 0 && N % 8 == 0 && N > 0 && N <= 32768 && B >= 2048;
    for_row_chunks(q, out, acc_out, B, N, [&](dim3 g, const int16_t* qc, float* oc, int32_t* ac) {
        if (paired)
            intlse_q10_6_rows_paired<kQ10PairedAhead><<<g, dim3(128), 0, st>>>(qc, oc, ac, N);
        else
            with_prefetch(g.x, 8, [&](auto d) { intlse_q10_6_rows<d.value><<<g, dim3(256), 0, st>>>(qc, oc, ac, N); });
    });
    return launch_status(name);
}
