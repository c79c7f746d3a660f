// The planes that a thread of a functor table's sweep takes
// (api/gpu/stencil_table.hpp); the library reports them as the tile's depth
// (pat_stencil_tile).
#ifndef PAT_GPU_STENCIL_PLANES_HPP_
#define PAT_GPU_STENCIL_PLANES_HPP_

#include <cstdint>

namespace pat_gpu {

constexpr int kStencilCells = 256;  // cells of the interior's rows, one after another, per workgroup

// More planes a thread save loads, fewer leave more wavefronts: 4 planes from 8
// workgroups per CU (128^3 FP32 heat 5.8 us a sweep, 6.2 with 2; 64^3 star 3.4
// and 3.4), 2 from 1 per CU (100^3 star 4.9, 5.6 with 1; at 32^3 star 3.1, 3.0
// with 1).  nx, ny, nz: the interior.
inline int stencil_planes(int64_t nx, int64_t ny, int64_t nz)
{
    const int64_t blocks = (nx * ny + kStencilCells - 1) / kStencilCells;
    if (blocks * ((nz + 3) / 4) >= 2048) return nz >= 4 ? 4 : 1;
    return blocks * ((nz + 1) / 2) >= 256 && nz >= 2 ? 2 : 1;
}

}  // namespace pat_gpu

#endif
