// C entry points of the host code the grid builds share, for tests/test_grid_rules.py (g++, no GPU).
#include <string>

#include "grid.hpp"
#include "grid_build.hpp"

extern "C" {

int grid_dims(const float* xyz, uint32_t nv, const uint32_t* faces, uint32_t nf, int resolution, int* dims) {
    linon::GridGeom g;
    std::string err;
    if (!linon::grid_geometry(xyz, nv, faces, nf, resolution, g, err)) return 0;
    for (int k = 0; k < 3; ++k) dims[k] = g.dim[k];
    return 1;
}

int row_mask_chunks(int nx) { return linon::dist_x_chunks(nx); }
unsigned row_mask_bytes(int nx) { return linon::dist_x_lds(nx); }
unsigned stride_blocks(size_t lanes) { return linon::stride_blocks(lanes); }

int grid_is_tiny(const float* xyz, uint32_t nv, const uint32_t* faces, uint32_t nf, int resolution) {
    linon::GridGeom g;
    std::string err;
    if (!linon::grid_geometry(xyz, nv, faces, nf, resolution, g, err)) return -1;
    return linon::grid_is_tiny(g, xyz, faces, nf);
}
}
