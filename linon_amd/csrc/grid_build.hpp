// Device build of the uniform grid (grid_build.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "device/grid_sat.hpp"

namespace linon {

// Device arrays of a built grid (owned by the caller once returned).
struct DeviceGrid {
    unsigned* cell_start = nullptr;  // ncells + 1
    unsigned* cell_faces = nullptr;  // refs, ascending face ids per cell
    unsigned char* dist = nullptr;   // ncells, Chebyshev cell distance to occupancy, capped at 255
    float* tris = nullptr;           // 12 floats per face: v0, v1 - v0, v2 - v0 (float4 each)
    size_t refs = 0;
    void release();
};

// The x pass of the distance field: 64-cell masks of a row of nx cells, and their LDS bytes for
// a block's four rows.
__host__ __device__ constexpr int dist_x_chunks(int nx) { return (nx + 63) / 64; }
__host__ __device__ constexpr unsigned dist_x_lds(int nx) { return 4u * (unsigned)dist_x_chunks(nx) * 8u; }

// Blocks of 256 lanes for the kernels with 16 lanes a face or a lane a reference, which stride over
// what is left: a launch holds fewer than 2^32 lanes, 2^28 faces' worth, and 16,384 blocks are
// eight times what the device runs at once.
constexpr unsigned stride_blocks(size_t lanes) {
    return (unsigned)(lanes < (size_t{1} << 22) ? (lanes + 255) / 256 : size_t{1} << 14);
}

// Builds the grid of geometry `g` (from grid_geometry, which also validated the mesh) on the
// device: uploads the mesh, counts, scans, fills, sorts and computes the distance field on
// stream s, synchronising twice.  On failure `err` is set and nothing is allocated.
// `refuse_alloc` > 0: the build's allocation of that number asks for a petabyte (tests of full
// memory); a build makes GRID_BUILD_ALLOCS of them.
constexpr int GRID_BUILD_ALLOCS = 6;
enum class GridResult {
    BUILT,
    NO_ROOM,    // the device has no memory for the grid or the build's scratch
    TOO_LARGE,  // more references than a grid holds
    FAILED      // any other error of HIP's
};
GridResult build_grid_device(const GridGeom& g, const float* h_xyz, uint32_t nv, const uint32_t* h_faces, uint32_t nf,
                             hipStream_t s, int refuse_alloc, DeviceGrid& out, std::string& err);

}  // namespace linon
