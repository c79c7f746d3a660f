// Device execution of an application's stencil functor table.
//
// The reference compiles each application's functor header (heat_3D/stencil.h,
// kmeans/stencil.h) with GPU_KERNEL defined and calls the functors through a
// __constant__ function-pointer table, one call per cell
// (kmeans/lib/compute_cuda.cu:30-100).  Here the application compiles the same
// header into a HIP translation unit and names its table:
//
//     #define GPU_KERNEL
//     #include "stencil.h"
//     #include "gpu/stencil_table.hpp"
//     static const int kUnit[] = {4};                  // element bytes per entry
//     static const int kSameAs[] = {PAT_STENCIL_HEAT}; // or -1
//     PAT_STENCIL_TABLE(FGPU::stencil_function_table, kUnit, kSameAs)
//
// With CONSTANT = __device__ constexpr (pattern_api.h) the table is a
// compile-time array, so each index becomes its own kernel with the functor
// called directly and inlined.  A workgroup takes 256 consecutive cells of the
// interior's rows and 1 to 4 planes.  The library's stencil handle calls the table's
// sweep() once per step on its two halo-inclusive grids (pat_stencil_set_table).
#ifndef PAT_GPU_STENCIL_TABLE_HPP_
#define PAT_GPU_STENCIL_TABLE_HPP_

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>
#include <utility>

#include "gpu/stencil_planes.hpp"
#include "pattern.h"

namespace pat_gpu {

struct StencilGrid {
    int size[3];       // halo-inclusive extents, dimension 0 fastest
    int lo[3], hi[3];  // interior cells [lo, hi) per dimension
};

// The reference has a 5-argument functor (with parameter,
// heat_3D/stencil.h:32) and a 4-argument one (kmeans/stencil.h:32).
template <typename F>
__device__ __forceinline__ void call_stencil(F f, void *in, void *out, int *offset, int *size, void *param)
{
    if constexpr (std::is_invocable_v<F, void *, void *, int *, int *, void *>)
        f(in, out, offset, size, param);
    else
        f(in, out, offset, size);
}

// t / d for 0 <= t < 2^31: the product with the reciprocal, rounded down, is
// short by one at most.  (The compiler's division of two numbers known only at
// run time took half of a sweep.)
struct Divisor {
    int d;
    unsigned m;
};
inline Divisor divisor(int d) { return {d, 0xffffffffu / (unsigned)d}; }
__device__ __forceinline__ int divide(int t, Divisor v)
{
    const int q = (int)__umulhi((unsigned)t, v.m);
    return t - q * v.d >= v.d ? q + 1 : q;
}

// A thread takes P planes of one column: the functor inlined P times, with the
// grids known not to overlap, lets the compiler load a neighbour once for all
// of them.  Bound by loads and their misses in L2: 200 x 186 x 210, W = 3 star,
// 17.0 us a sweep against 26.5 with one cell a thread in 64 x 4 blocks dealt to
// the XCDs in turn (every XCD then fetches every plane); 300^3 FP32 heat 37.0
// against 87.8, 300 x 280 x 290 FP64 heat 112 against 138 (3.5 TB/s).  Without
// the XCDs' chunks: 23.8, 65.4 and 111; in 64 x 4 blocks, whose last column of
// blocks is nearly empty at 200 and 300: 19.5, 35.8 and 119.
template <class Tab, int I, int P>
__global__ __launch_bounds__(kStencilCells) void stencil_sweep(const void *__restrict__ in, void *__restrict__ out,
                                                     StencilGrid g, const void *param, Divisor blocks, Divisor nx,
                                                     int plane)
{
    // workgroups are dealt to the 8 XCDs in turn: each takes a run of planes
    const int per = (int)gridDim.x / 8, bid = (int)blockIdx.x;
    const int t = bid < per * 8 ? bid % 8 * per + bid / 8 : bid;
    const int tz = divide(t, blocks), i = (t - tz * blocks.d) * kStencilCells + (int)threadIdx.x;
    const int z = g.lo[2] + tz * P;
    if (i >= plane) return;
    const int row = divide(i, nx);
    const int x = g.lo[0] + i - row * nx.d, y = g.lo[1] + row;
    auto cell = [&](int zz) {
        int offset[3] = {x, y, zz};
        int size[3] = {g.size[0], g.size[1], g.size[2]};
        Tab::template call<I>(const_cast<void *>(in), out, offset, size, const_cast<void *>(param));
    };
    if (z + P <= g.hi[2]) {
#pragma unroll
        for (int p = 0; p < P; p++) cell(z + p);
    } else {
        for (int zz = z; zz < g.hi[2]; zz++) cell(zz);
    }
}

template <class Tab, int I>
int stencil_launch(const void *in, void *out, const StencilGrid &grid, const void *param, hipStream_t st)
{
    if constexpr (!Tab::template valid<I>()) {
        return PAT_ERR_UNSUPPORTED;
    } else {
        const int nx = grid.hi[0] - grid.lo[0], ny = grid.hi[1] - grid.lo[1], nz = grid.hi[2] - grid.lo[2];
        const int P = stencil_planes(nx, ny, nz);
        const int chunks = (nz + P - 1) / P;
        // rows per launch: indexes within a plane and workgroups below 2^31
        const int rows = (int)std::max<int64_t>(1, std::min<int64_t>(ny, (1LL << 30) / ((int64_t)nx * chunks)));
        for (int y0 = 0; y0 < ny; y0 += rows) {
            StencilGrid g = grid;
            g.lo[1] = grid.lo[1] + y0;
            g.hi[1] = std::min(grid.hi[1], g.lo[1] + rows);
            const int plane = nx * (g.hi[1] - g.lo[1]), blocks = (plane + kStencilCells - 1) / kStencilCells;
            auto launch = [&](auto planes) {
                hipLaunchKernelGGL((stencil_sweep<Tab, I, decltype(planes)::value>), dim3((unsigned)(blocks * chunks)),
                                   dim3(kStencilCells), 0, st, in, out, g, param, divisor(blocks), divisor(nx), plane);
            };
            if (P == 4) launch(std::integral_constant<int, 4>{});
            else if (P == 2) launch(std::integral_constant<int, 2>{});
            else launch(std::integral_constant<int, 1>{});
            if (hipGetLastError() != hipSuccess) return PAT_ERR_HIP;
        }
        return PAT_OK;
    }
}

template <class Tab, std::size_t... I>
int stencil_dispatch(int idx, const void *in, void *out, const StencilGrid &g, const void *param, hipStream_t st,
                     std::index_sequence<I...>)
{
    int rc = PAT_ERR_UNSUPPORTED;
    ((idx == (int)I ? (void)(rc = stencil_launch<Tab, (int)I>(in, out, g, param, st)) : (void)0), ...);
    return rc;
}

// pat_stencil_table::sweep for table Tab: one sweep of functor idx over the
// interior of a grid of extents size[0..ndims-1] with halo width 'width'.
template <class Tab>
int stencil_sweep_entry(int idx, const void *in, void *out, const int32_t *size, int ndims, int width,
                        const void *param, void *stream)
{
    if (!in || !out || !size || ndims < 1 || ndims > 3 || width < 0) return PAT_ERR_INVALID;
    StencilGrid g;
    for (int d = 0; d < 3; d++) {
        const bool used = d < ndims;
        g.size[d] = used ? size[d] : 1;
        g.lo[d] = used ? width : 0;
        g.hi[d] = used ? size[d] - width : 1;
        if (g.hi[d] <= g.lo[d]) return PAT_ERR_INVALID;
    }
    if (g.hi[2] - g.lo[2] > 65535) return PAT_ERR_UNSUPPORTED;  // as pat_stencil_create
    return stencil_dispatch<Tab>(idx, in, out, g, param, (hipStream_t)stream,
                                 std::make_index_sequence<(std::size_t)Tab::count>{});
}

}  // namespace pat_gpu

// Defines pat_app_stencil_table() for the application's table TABLE (a
// __device__ constexpr array of stencil functors), with UNIT[i] the element
// bytes functor i reads and writes and SAME_AS[i] the library's tuned functor
// that computes the same bits (PAT_STENCIL_HEAT) or -1.
#define PAT_STENCIL_TABLE(TABLE, UNIT, SAME_AS)                                                                  \
    namespace {                                                                                                  \
    struct PatStencilTab {                                                                                       \
        static constexpr int count = (int)(sizeof(TABLE) / sizeof(TABLE[0]));                                    \
        template <int I>                                                                                         \
        static constexpr bool valid()                                                                            \
        {                                                                                                        \
            return TABLE[I] != nullptr;                                                                          \
        }                                                                                                        \
        template <int I>                                                                                         \
        __device__ static void call(void *in, void *out, int *offset, int *size, void *param)                    \
        {                                                                                                        \
            pat_gpu::call_stencil(TABLE[I], in, out, offset, size, param);                                       \
        }                                                                                                        \
    };                                                                                                           \
    static_assert(sizeof(UNIT) / sizeof(UNIT[0]) == PatStencilTab::count, "one element size per table entry");  \
    static_assert(sizeof(SAME_AS) / sizeof(SAME_AS[0]) == PatStencilTab::count, "one same-as entry per functor"); \
    }                                                                                                            \
    extern "C" const pat_stencil_table *pat_app_stencil_table(void)                                              \
    {                                                                                                            \
        static const pat_stencil_table t = {PatStencilTab::count, UNIT, SAME_AS,                                 \
                                            &pat_gpu::stencil_sweep_entry<PatStencilTab>};                       \
        return &t;                                                                                               \
    }

#endif
