// Device build of the uniform grid (the host build in grid.cpp computes the same arrays):
//   1. overlap: 16 lanes per face test its cells; which of them it overlaps is kept as a bit mask,
//      how many as the face's count.  A face with more than 256 cells in range gets a wave, one
//      with more than 8192 (a wall) is spread over the blocks;
//   2. exclusive scan of the face counts -> where each face's references stand, and their total;
//   3. place: every reference takes its slot in its cell (an atomic counter per cell) and is
//      recorded as (cell, slot, face);
//   4. exclusive scan of the cell counts -> cell_start;
//   5. each reference goes to its cell's list, then to its rank there (how many of the list's
//      faces have a smaller id; long lists are sorted): the host build's ascending order;
//   6. Chebyshev distance field: the distance along x from each row's occupancy bits, then min-max
//      passes along y and z.
// The overlap decisions are those of the shared double-precision separating-axis test with
// contraction off (FaceTest below settles nearly all of them with a fraction of its arithmetic),
// so every array equals the host build's.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <vector>

#include "device/grid_sat.hpp"
#include "grid_build.hpp"

namespace linon {

namespace {

constexpr int kScanBlock = 1024;  // elements per block of the local scan (256 lanes x 4)

__device__ __forceinline__ void load_face(const float* xyz, const uint32_t* faces, uint32_t f, double v[3][3]) {
    for (int j = 0; j < 3; ++j) {
        const float* p = xyz + 3 * (size_t)faces[3 * (size_t)f + j];
        for (int k = 0; k < 3; ++k) v[j][k] = (double)p[k];
    }
}

// Faces whose cell range holds more than kMidFaceCells cells are tested by a wave each, those with
// more than kHugeFaceCells by many blocks: a wall of the Cornell box spans 3 x 256^2 cells of the
// 256^3 grid, a face of a displaced icosphere a handful to a few hundred.  Above 8192 cells a lone
// wave becomes the launch's tail (the Cornell box's inner faces in 128^3 cells: 97 us with the line
// at 16384, 16 us with it at 2048), while faces spread over blocks cost each block the face's set-up
// (1.3 M faces, many of 2048 to 8192 cells in 256^3: 3.2 ms with the line at 2048).
constexpr size_t kMidFaceCells = 256, kHugeFaceCells = 8192;

constexpr int kFaceLanes = 16;  // lanes per face in the overlap test: 16 cells a lane at most
static_assert(kMidFaceCells == (size_t)kFaceLanes * 16, "a lane's cells fill a 16-bit mask");

__device__ __forceinline__ size_t range_cells(const int c0[3], const int c1[3]) {
    return (size_t)(c1[0] - c0[0] + 1) * (size_t)(c1[1] - c0[1] + 1) * (size_t)(c1[2] - c0[2] + 1);
}

// Cell k of a face's range, x fastest.  At most 1024^3 cells, or a little more where a dimension's
// count rounds up past the resolution: 32 bits hold every index.
struct FaceCells {
    int x0, y0, z0;
    unsigned sx, sxy;
    __device__ __forceinline__ FaceCells(const int c0[3], const int c1[3])
        : x0(c0[0]), y0(c0[1]), z0(c0[2]), sx((unsigned)(c1[0] - c0[0] + 1)),
          sxy(sx * (unsigned)(c1[1] - c0[1] + 1)) {}
    __device__ __forceinline__ void at(unsigned k, int& x, int& y, int& z) const {
        const unsigned kz = k / sxy, r = k - kz * sxy, ky = r / sx;
        x = x0 + (int)(r - ky * sx);
        y = y0 + (int)ky;
        z = z0 + (int)kz;
    }
};

__device__ __forceinline__ unsigned cell_index(const GridGeom& g, int x, int y, int z) {
    return ((unsigned)z * (unsigned)g.dim[1] + (unsigned)y) * (unsigned)g.dim[0] + (unsigned)x;
}

struct Reference {
    unsigned cell, slot, face;
};

// The separating-axis test of one face with what depends on the face alone computed once: the
// projections of the three vertices on each of the 13 axes, widened by the box's half extent.  A
// cell is then settled by the projection of its centre, about 70 double-precision operations
// where face_in_cell takes 350, unless some axis comes within a slack of its threshold, which
// covers the rounding of both computations; those cells take face_in_cell itself.  With |vertices|,
// |centres| <= S both projections onto an edge axis are off by less than 2^-46 S^2, onto the normal
// by less than 2^-42 S^3, and onto a box axis by 2^-50 S; the slacks are 8 times that and more.  For
// a mesh about the origin about one cell in 10^11 comes so close.  They grow with the distance from
// the origin, not the mesh's size, and a face without area has a normal of zero, which always does:
// 327,716 faces in 256^3 cells take 6.4 ms about the origin, 9.6 at 100 units from it and 9.7 at
// 1000, 7.1 without area (by face_in_cell alone, one lane a face, 14.7, 20.5, 14.7 and 13.8).  An
// axis that is exactly zero (an edge along it: the difference of equal coordinates is zero in both
// computations) separates nothing and has infinite thresholds.
struct FaceTest {
    double e[3][3];            // edges
    double lo[9], hi[9];       // thresholds of the edge axes (3 j + i: edge j x unit vector i)
    double blo[3], bhi[3];     // of the box axes
    double n[3], nlo, nhi;     // the normal and its thresholds
    double slack_e, slack_b, slack_n;

    __device__ __forceinline__ FaceTest(const GridGeom& g, const double v[3][3]) {
        const double h = 0.5 * g.cs + g.margin;
        double S = 0.0;
        for (int k = 0; k < 3; ++k)
            S = gs_max(S, gs_max(gs_abs((double)g.lo[k]), gs_abs((double)g.hi[k])));
        S += g.cs + g.margin;  // the grid's box, which holds every vertex, and a cell more
        slack_e = S * S * 0x1p-43;
        slack_b = S * 0x1p-46;
        slack_n = S * S * S * 0x1p-38;
        for (int k = 0; k < 3; ++k) {
            e[0][k] = v[1][k] - v[0][k];
            e[1][k] = v[2][k] - v[1][k];
            e[2][k] = v[0][k] - v[2][k];
            blo[k] = gs_min(v[0][k], gs_min(v[1][k], v[2][k])) - h;
            bhi[k] = gs_max(v[0][k], gs_max(v[1][k], v[2][k])) + h;
        }
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double q0 = along(j, i, v[0]), q1 = along(j, i, v[1]), q2 = along(j, i, v[2]);
                const double p = e[j][(i + 1) % 3], q = e[j][(i + 2) % 3];
                const double r = h * (gs_abs(p) + gs_abs(q));
                const bool none = p == 0.0 && q == 0.0;
                lo[3 * j + i] = none ? -__builtin_inf() : gs_min(q0, gs_min(q1, q2)) - r;
                hi[3 * j + i] = none ? __builtin_inf() : gs_max(q0, gs_max(q1, q2)) + r;
            }
        n[0] = e[0][1] * e[1][2] - e[0][2] * e[1][1];
        n[1] = e[0][2] * e[1][0] - e[0][0] * e[1][2];
        n[2] = e[0][0] * e[1][1] - e[0][1] * e[1][0];
        const double d = n[0] * v[0][0] + n[1] * v[0][1] + n[2] * v[0][2];
        const double r = h * (gs_abs(n[0]) + gs_abs(n[1]) + gs_abs(n[2]));
        nlo = d - r;
        nhi = d + r;
    }
    // projection on edge j x unit vector i, up to sign: e_(i+1) x_(i+2) - e_(i+2) x_(i+1)
    __device__ __forceinline__ double along(int j, int i, const double x[3]) const {
        const int a = (i + 1) % 3, b = (i + 2) % 3;
        return e[j][a] * x[b] - e[j][b] * x[a];
    }
    __device__ __forceinline__ bool in_cell(const GridGeom& g, const double v[3][3], int x, int y, int z) const {
        const double c[3] = {(double)g.lo[0] + (x + 0.5) * g.cs, (double)g.lo[1] + (y + 0.5) * g.cs,
                             (double)g.lo[2] + (z + 0.5) * g.cs};
        double ge = -__builtin_inf(), gb = -__builtin_inf();  // widest gaps
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double s = along(j, i, c);
                ge = __builtin_fmax(ge, __builtin_fmax(lo[3 * j + i] - s, s - hi[3 * j + i]));
            }
#pragma unroll
        for (int k = 0; k < 3; ++k) gb = __builtin_fmax(gb, __builtin_fmax(blo[k] - c[k], c[k] - bhi[k]));
        const double s = n[0] * c[0] + n[1] * c[1] + n[2] * c[2];
        const double gn = __builtin_fmax(nlo - s, s - nhi);
        if (ge > slack_e || gb > slack_b || gn > slack_n) return false;
        if (ge < -slack_e && gb < -slack_b && gn < -slack_n) return true;
        return face_in_cell(g, v, x, y, z);
    }
};

// Lists the faces that face_overlap_kernel leaves alone: mid ones from the front of big[nf], huge
// ones from its back; nbig[0] and nbig[1] count them.  One atomic per class and block of 1024 faces: they all
// go to two addresses, about 9 ns each.
__global__ void __launch_bounds__(1024) classify_kernel(GridGeom g, const float* xyz, const uint32_t* faces,
                                                        uint32_t nf, unsigned* big, unsigned* nbig) {
    __shared__ unsigned base[2][16];
    const size_t f = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const unsigned wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    size_t cells = 0;
    if (f < nf) {
        double v[3][3];
        load_face(xyz, faces, (uint32_t)f, v);
        int c0[3], c1[3];
        face_cell_range(g, v, c0, c1);
        if (c1[0] >= c0[0] && c1[1] >= c0[1] && c1[2] >= c0[2]) cells = range_cells(c0, c1);
    }
    const bool huge = cells > kHugeFaceCells, mid = cells > kMidFaceCells && !huge;
    const unsigned long long m = __ballot(mid), h = __ballot(huge);
    if (lane == 0) {
        base[0][wave] = (unsigned)__popcll(m);
        base[1][wave] = (unsigned)__popcll(h);
    }
    __syncthreads();
    if (threadIdx.x < 2) {
        unsigned* c = base[threadIdx.x];
        unsigned n = 0;
        for (int w = 0; w < 16; ++w) n += c[w];
        unsigned at = n ? atomicAdd(nbig + threadIdx.x, n) : 0u;
        for (int w = 0; w < 16; ++w) {
            const unsigned k = c[w];
            c[w] = at;
            at += k;
        }
    }
    __syncthreads();
    const unsigned long long below = (1ull << lane) - 1ull;
    if (mid) big[base[0][wave] + (unsigned)__popcll(m & below)] = (unsigned)f;
    if (huge) big[nf - 1u - (base[1][wave] + (unsigned)__popcll(h & below))] = (unsigned)f;
}

// Overlap test, 16 lanes per face: lane s tests cells s, s + 16, ... of the face's range and keeps
// bit i for cell s + 16 i.  One lane per face left a 20,516-face mesh 80 blocks, each lane testing
// up to 256 cells one after another (0.5 ms, twice: the second time to place them).
__global__ void __launch_bounds__(256) face_overlap_kernel(GridGeom g, const float* xyz, const uint32_t* faces,
                                                           uint32_t nf, unsigned short* masks, unsigned* count) {
    const unsigned sub = threadIdx.x % kFaceLanes;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < (size_t)nf * kFaceLanes; t += stride) {
        const size_t f = t / kFaceLanes;
        double v[3][3];
        load_face(xyz, faces, (uint32_t)f, v);
        int c0[3], c1[3];
        face_cell_range(g, v, c0, c1);
        unsigned mask = 0;
        // (an empty range, outside the grid, cannot happen: the grid encloses every face)
        if (c1[0] >= c0[0] && c1[1] >= c0[1] && c1[2] >= c0[2]) {
            const size_t cells = range_cells(c0, c1);
            if (cells <= kMidFaceCells) {
                const FaceCells C(c0, c1);
                const FaceTest T(g, v);
                int x, y, z;
                for (unsigned k = sub, i = 0; k < (unsigned)cells; k += kFaceLanes, ++i) {
                    C.at(k, x, y, z);
                    if (T.in_cell(g, v, x, y, z)) mask |= 1u << i;
                }
            }
        }
        masks[t] = (unsigned short)mask;
        unsigned n = (unsigned)__popc(mask);
        for (int off = kFaceLanes / 2; off > 0; off >>= 1) n += __shfl_xor(n, off, kFaceLanes);
        if (sub == 0) count[f] = n;  // 0 for a listed face: its own kernel adds its references
    }
}

// A reference's slot in its cell.
__device__ __forceinline__ Reference take_slot(unsigned cell, unsigned face, unsigned* cell_count) {
    return Reference{cell, atomicAdd(cell_count + cell, 1u), face};
}

// The references the overlap test found, from the masks (16 lanes per face as there).
__global__ void __launch_bounds__(256) face_place_kernel(GridGeom g, const float* xyz, const uint32_t* faces,
                                                         uint32_t nf, const unsigned short* masks,
                                                         const unsigned* first, unsigned* cell_count, Reference* refs) {
    const unsigned sub = threadIdx.x % kFaceLanes;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < (size_t)nf * kFaceLanes; t += stride) {
        const size_t f = t / kFaceLanes;
        unsigned mask = masks[t];
        const unsigned n = (unsigned)__popc(mask);
        unsigned upto = n;  // inclusive prefix over the face's lanes
        for (unsigned off = 1; off < (unsigned)kFaceLanes; off <<= 1) {
            const unsigned x = __shfl_up(upto, off, kFaceLanes);
            if (sub >= off) upto += x;
        }
        if (!mask) continue;
        double v[3][3];
        load_face(xyz, faces, (uint32_t)f, v);
        int c0[3], c1[3];
        face_cell_range(g, v, c0, c1);
        const FaceCells C(c0, c1);
        Reference* out = refs + first[f] + (upto - n);
        int x, y, z;
        for (; mask; mask &= mask - 1) {
            C.at(sub + kFaceLanes * (unsigned)(__ffs((int)mask) - 1), x, y, z);
            *out++ = take_slot(cell_index(g, x, y, z), (unsigned)f, cell_count);
        }
    }
}

// The mid faces, a wave each (grid-stride over the list), or, with Huge, the huge ones:
// blockIdx.x strides over the faces, the lanes of all blockIdx.y over a face's cell range.  Count
// (PLACE = false), or place the references of a face from first[face] on: a wave that has its face
// to itself counts along, the blocks of a huge one share a cursor.  (One block per face took 6.3 ms
// for 1.3 M displaced-icosphere faces and the Cornell box in 256^3 cells, most of it in the 12
// walls.)
template <bool Huge, bool PLACE>
__global__ void __launch_bounds__(256) big_overlap_kernel(GridGeom g, const float* xyz, const uint32_t* faces,
                                                          uint32_t nf, const unsigned* big, const unsigned* nbig,
                                                          unsigned* count, const unsigned* first, unsigned* cursor,
                                                          unsigned* cell_count, Reference* refs) {
    const unsigned n = nbig[Huge ? 1 : 0];
    const unsigned lane = threadIdx.x & 63;
    const unsigned wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned begin = Huge ? blockIdx.x : blockIdx.x * 4 + wave;
    const unsigned stride = Huge ? gridDim.x : gridDim.x * 4;
    for (unsigned i = begin; i < n; i += stride) {
        const unsigned f = big[Huge ? nf - 1u - i : i];
        double v[3][3];
        load_face(xyz, faces, f, v);
        int c0[3], c1[3];
        face_cell_range(g, v, c0, c1);
        const FaceCells C(c0, c1);
        const FaceTest T(g, v);
        const unsigned cells = (unsigned)range_cells(c0, c1);
        unsigned found = 0;
        // 64 neighbouring cells at a time, so that a wave's lanes stay together for the ballot
        const unsigned k_begin = Huge ? (blockIdx.y * 4 + wave) * 64 : 0, k_stride = Huge ? gridDim.y * 256 : 64;
        for (unsigned k0 = k_begin; k0 < cells; k0 += k_stride) {
            const unsigned k = k0 + lane;
            int x = 0, y = 0, z = 0;
            bool in = k < cells;
            if (in) {
                C.at(k, x, y, z);
                in = T.in_cell(g, v, x, y, z);
            }
            const unsigned long long lanes = __ballot(in);
            if (!lanes) continue;
            if (PLACE) {
                unsigned base = found;
                if (Huge) {
                    if (lane == 0) base = atomicAdd(cursor + i, (unsigned)__popcll(lanes));
                    base = __shfl(base, 0, 64);
                }
                if (in)
                    refs[(size_t)first[f] + base + (unsigned)__popcll(lanes & ((1ull << lane) - 1ull))] =
                        take_slot(cell_index(g, x, y, z), f, cell_count);
            }
            found += (unsigned)__popcll(lanes);
        }
        if (!PLACE && lane == 0) {
            if (!Huge)
                count[f] = found;
            else if (found)
                atomicAdd(count + f, found);
        }
    }
}

// Each reference to its slot of its cell's list.
__global__ void __launch_bounds__(256) list_kernel(const Reference* refs, size_t n, const unsigned* cell_start,
                                                   unsigned* list) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const Reference r = refs[i];
        list[(size_t)cell_start[r.cell] + r.slot] = r.face;
    }
}

// Each reference to its rank in its cell: the ascending order of the face ids (distinct in a
// cell).  A lane compares against its cell's whole list, so a list of L faces takes L^2
// comparisons side by side, where an insertion sort by one lane takes as many in a chain (0.9 ms
// for 1.3 M faces in 256^3 cells).  Lists beyond kLongList are left to long_list_kernel; their
// cells go to long_cells.
constexpr unsigned kLongList = 256;
__global__ void __launch_bounds__(256) rank_kernel(const Reference* refs, size_t n, const unsigned* cell_start,
                                                   const unsigned* list, unsigned* cell_faces, unsigned* long_cells,
                                                   unsigned* nlong) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const Reference r = refs[i];
        const unsigned b = cell_start[r.cell], e = cell_start[r.cell + 1];
        if (e - b > kLongList) {
            if (r.slot == 0) long_cells[atomicAdd(nlong, 1u)] = r.cell;
            continue;
        }
        unsigned rank = 0;
        for (unsigned j = b; j < e; ++j) rank += list[j] < r.face ? 1u : 0u;
        cell_faces[(size_t)b + rank] = r.face;
    }
}

// Sorts each long list, a block of 1024 a list: radix passes of 8 bits, lowest first, between `list`
// and `cell_faces`, an odd number of them so that the last ends in cell_faces.  Ranked like the short
// ones, L faces in the same C cells take C L^2 comparisons: 4,000 triangles across the grid, all in
// the same 16,766 of 128^3 cells, 4.0 s for the whole build; so 8 ms, and 10,000 of them 20 ms (the
// host build 2.5 s).
__global__ void __launch_bounds__(1024) long_list_kernel(const unsigned* cell_start, unsigned* list,
                                                         unsigned* cell_faces, const unsigned* long_cells,
                                                         const unsigned* nlong, int passes) {
    __shared__ unsigned at[256], wave_at[16][256];
    const unsigned t = threadIdx.x, wave = t >> 6, lane = t & 63;
    for (unsigned i = blockIdx.x; i < *nlong; i += gridDim.x) {
        const unsigned b = cell_start[long_cells[i]], n = cell_start[long_cells[i] + 1] - b;
        for (int p = 0; p < passes; ++p) {
            const unsigned* in = (p & 1 ? cell_faces : list) + b;
            unsigned* out = (p & 1 ? list : cell_faces) + b;
            const int shift = 8 * p;
            auto digit = [&](unsigned x) { return shift < 32 ? (x >> shift) & 255u : 0u; };
            if (t < 256) at[t] = 0;
            __syncthreads();
            for (unsigned j = t; j < n; j += 1024) atomicAdd(&at[digit(in[j])], 1u);
            __syncthreads();
            // where each digit's faces begin: one wave, four digits a lane
            if (t < 64) {
                unsigned c[4], sum = 0;
                for (int k = 0; k < 4; ++k) {
                    c[k] = at[4 * t + k];
                    sum += c[k];
                }
                unsigned upto = sum;
                for (unsigned off = 1; off < 64; off <<= 1) {
                    const unsigned x = __shfl_up(upto, off, 64);
                    if (lane >= off) upto += x;
                }
                unsigned begin = upto - sum;
                for (int k = 0; k < 4; ++k) {
                    at[4 * t + k] = begin;
                    begin += c[k];
                }
            }
            for (unsigned j0 = 0; j0 < n; j0 += 1024) {
                for (unsigned k = t; k < 16 * 256; k += 1024) wave_at[k >> 8][k & 255] = 0;
                __syncthreads();
                const bool have = j0 + t < n;
                const unsigned x = have ? in[j0 + t] : 0u, d = digit(x);
                unsigned long long same = __ballot(have);  // the wave's lanes of this digit
                for (int bit = 0; bit < 8; ++bit) {
                    const unsigned long long set = __ballot(d >> bit & 1u);
                    same &= d >> bit & 1u ? set : ~set;
                }
                const unsigned before = (unsigned)__popcll(same & ((1ull << lane) - 1ull));
                if (have && before == 0) wave_at[wave][d] = (unsigned)__popcll(same);
                __syncthreads();
                if (t < 256) {
                    unsigned o = at[t];
                    for (int w = 0; w < 16; ++w) {
                        const unsigned k = wave_at[w][t];
                        wave_at[w][t] = o;
                        o += k;
                    }
                    at[t] = o;
                }
                __syncthreads();
                if (have) out[wave_at[wave][d] + before] = x;
                __syncthreads();  // before the counts are cleared, and before the next pass reads `out`
            }
        }
    }
}

__device__ __forceinline__ unsigned long long block_inclusive_scan(unsigned long long v, unsigned long long* s) {
    const int t = threadIdx.x;
    s[t] = v;
    __syncthreads();
    for (int off = 1; off < (int)blockDim.x; off <<= 1) {
        const unsigned long long x = t >= off ? s[t - off] : 0ull;
        __syncthreads();
        s[t] += x;
        __syncthreads();
    }
    return s[t];
}

// Exclusive scan inside each block of kScanBlock counts; block totals to bsum.
__global__ void __launch_bounds__(256) scan_local_kernel(const unsigned* in, size_t n, unsigned long long* out,
                                                         unsigned long long* bsum) {
    __shared__ unsigned long long s[256];
    const size_t base = (size_t)blockIdx.x * kScanBlock + (size_t)threadIdx.x * 4;
    unsigned long long v[4], t = 0;
    for (int k = 0; k < 4; ++k) {
        v[k] = base + k < n ? in[base + k] : 0u;
        t += v[k];
    }
    const unsigned long long incl = block_inclusive_scan(t, s);
    unsigned long long run = incl - t;
    for (int k = 0; k < 4; ++k) {
        if (base + k < n) out[base + k] = run;
        run += v[k];
    }
    if (threadIdx.x == blockDim.x - 1) bsum[blockIdx.x] = incl;
}

// Exclusive scan of the nb block totals in place (one block, each lane a contiguous chunk);
// the grand total to *total.
__global__ void __launch_bounds__(1024) scan_sums_kernel(unsigned long long* bsum, size_t nb,
                                                         unsigned long long* total) {
    __shared__ unsigned long long s[1024];
    const size_t chunk = (nb + blockDim.x - 1) / blockDim.x;
    const size_t b0 = (size_t)threadIdx.x * chunk, b1 = b0 + chunk < nb ? b0 + chunk : nb;
    unsigned long long t = 0;
    for (size_t i = b0; i < b1; ++i) t += bsum[i];
    const unsigned long long incl = block_inclusive_scan(t, s);
    unsigned long long run = incl - t;
    for (size_t i = b0; i < b1; ++i) {
        const unsigned long long x = bsum[i];
        bsum[i] = run;
        run += x;
    }
    if (threadIdx.x == blockDim.x - 1) *total = incl;
}

__global__ void __launch_bounds__(256) scan_finish_kernel(const unsigned long long* local,
                                                          const unsigned long long* bsum, size_t n, unsigned* out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = (unsigned)(local[i] + bsum[i / kScanBlock]);
}

__global__ void __launch_bounds__(256) fill_u32_kernel(unsigned* p, size_t n, unsigned value) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

// Distance along x to the nearest occupied cell of the row (capped at 255), one wave per row: the
// row's occupancy as 64-bit masks, in which every lane finds the nearest set bit on either side.
// (A sweep of each row by one lane took 76 us for 128^3 cells, 374 us for 256^3.)  The masks are
// sized by the launch, dist_x_lds(nx) bytes: a row can be longer than the resolution, whose cells
// are counted up from rounded bounds (1025 for 1024 over x in [0, 0.02f]).
__global__ void __launch_bounds__(256) dist_x_kernel(const unsigned* cell_start, int nx, size_t rows,
                                                     unsigned char* a) {
    extern __shared__ unsigned long long row_masks[];
    const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    const size_t row = (size_t)blockIdx.x * 4 + wave;
    const bool in = row < rows;
    const size_t base = row * (size_t)nx;
    const int chunks = dist_x_chunks(nx);
    unsigned long long* bits = row_masks + wave * chunks;
    for (int c = 0; c < chunks; ++c) {
        const int x = 64 * c + lane;
        const bool occ = in && x < nx && cell_start[base + x + 1] > cell_start[base + x];
        const unsigned long long m = __ballot(occ);
        if (lane == 0) bits[c] = m;
    }
    __syncthreads();
    if (!in) return;
    for (int c = 0; c < chunks; ++c) {
        const int x = 64 * c + lane;
        if (x >= nx) break;
        int d = 255;
        // left, the cell itself included: the highest set bit at or below it
        unsigned long long m = bits[c] & (~0ull >> (63 - lane));
        for (int k = c;;) {
            if (m) {
                d = min(d, x - (64 * k + 63 - __clzll((long long)m)));
                break;
            }
            if (--k < 0 || x - (64 * k + 63) >= 255) break;
            m = bits[k];
        }
        // right: the lowest set bit at or above it
        m = bits[c] & (~0ull << lane);
        for (int k = c;;) {
            if (m) {
                d = min(d, 64 * k + __ffsll((long long)m) - 1 - x);
                break;
            }
            if (++k >= chunks || 64 * k - x >= 255) break;
            m = bits[k];
        }
        a[base + x] = (unsigned char)d;
    }
}

// out[i] = min over j of max(|i - j|, in[j]) along y (axis 1) or z (axis 2), one lane per cell,
// searched outwards from i until the offset alone reaches the best value.  Neighbouring lanes are
// neighbours in x, so every load of the search is coalesced.  (One lane per line, 16,384 of them
// for 128^3 cells, took 418 us a pass, 1.7 ms for 256^3.)
__global__ void __launch_bounds__(256) dist_minmax_kernel(const unsigned char* in, unsigned char* out, int nx,
                                                          int ny, int nz, int axis) {
    const size_t cell = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (cell >= (size_t)nx * ny * nz) return;
    const unsigned row = (unsigned)cell / (unsigned)nx;  // fewer than 2^32 cells
    const int i = (int)(axis == 1 ? row % (unsigned)ny : row / (unsigned)ny);
    const int n = axis == 1 ? ny : nz;
    const size_t s = axis == 1 ? (size_t)nx : (size_t)nx * ny;
    const unsigned char* p = in + cell;
    int best = *p;
    // (past both ends of the line nothing is left that could be smaller)
    for (int dlt = 1; dlt < best && (i - dlt >= 0 || i + dlt < n); ++dlt) {
        int g = 255;
        if (i - dlt >= 0) g = min(g, (int)p[-(ptrdiff_t)((size_t)dlt * s)]);
        if (i + dlt < n) g = min(g, (int)p[(size_t)dlt * s]);
        best = min(best, max(dlt, g));
    }
    out[cell] = (unsigned char)best;
}

// Per-face (v0, v1 - v0, v2 - v0) as three float4 (f32 subtraction, as the shader's edges).
__global__ void __launch_bounds__(256) pack_faces_kernel(const float* xyz, const uint32_t* faces, uint32_t nf,
                                                         float4* tris) {
    const size_t f = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= nf) return;
    const float* a = xyz + 3 * (size_t)faces[3 * f];
    const float* b = xyz + 3 * (size_t)faces[3 * f + 1];
    const float* c = xyz + 3 * (size_t)faces[3 * f + 2];
    tris[3 * f] = make_float4(a[0], a[1], a[2], 0.0f);
    tris[3 * f + 1] = make_float4(b[0] - a[0], b[1] - a[1], b[2] - a[2], 0.0f);
    tris[3 * f + 2] = make_float4(c[0] - a[0], c[1] - a[1], c[2] - a[2], 0.0f);
}

unsigned blocks_for(size_t n, unsigned per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

void DeviceGrid::release() {
    for (void** p : {(void**)&cell_start, (void**)&cell_faces, (void**)&dist, (void**)&tris}) {
        if (*p) (void)hipFree(*p);
        *p = nullptr;
    }
    refs = 0;
}

namespace {

// A sequence of arrays in one allocation, each 256-byte aligned: declare them, allocate, then ask
// for the pointers in the same order.
struct Arena {
    std::vector<size_t> at;
    size_t bytes = 0;
    char* base = nullptr;
    template <class T>
    int add(size_t n) {
        at.push_back(bytes);
        bytes += (std::max<size_t>(n, 1) * sizeof(T) + 255) / 256 * 256;
        return (int)at.size() - 1;
    }
    template <class Alloc>
    hipError_t allocate(Alloc& alloc) {
        return alloc(&base, bytes);
    }
    template <class T>
    T* get(int i) const {
        return reinterpret_cast<T*>(base + at[(size_t)i]);
    }
    ~Arena() {
        if (base) (void)hipFree(base);
    }
};

}  // namespace

GridResult build_grid_device(const GridGeom& g, const float* h_xyz, uint32_t nv, const uint32_t* h_faces, uint32_t nf,
                             hipStream_t s, int refuse_alloc, DeviceGrid& out, std::string& err) {
    out.release();
    (void)hipGetLastError();  // an earlier call's error is not this build's: its launches are checked below
    const size_t nx = (size_t)g.dim[0], ny = (size_t)g.dim[1], nz = (size_t)g.dim[2];
    const size_t nc = nx * ny * nz;
    const size_t longest = std::max<size_t>(nc, nf);
    const size_t max_blocks = (longest + kScanBlock - 1) / kScanBlock;
    Arena A, R;
    const int i_xyz = A.add<float>(3 * (size_t)nv), i_faces = A.add<uint32_t>(3 * (size_t)nf);
    const int i_masks = A.add<unsigned short>((size_t)nf * kFaceLanes);
    const int i_count = A.add<unsigned>(nf), i_first = A.add<unsigned>(nf), i_big = A.add<unsigned>(nf);
    const int i_cursor = A.add<unsigned>(nf), i_cells = A.add<unsigned>(nc);
    const int i_local = A.add<unsigned long long>(longest), i_bsum = A.add<unsigned long long>(max_blocks);
    const int i_total = A.add<unsigned long long>(1), i_nbig = A.add<unsigned>(3), i_tmp = A.add<unsigned char>(nc);
    GridResult result = GridResult::BUILT;
    auto check = [&](hipError_t e, const char* what) {
        if (e == hipSuccess) return true;
        err = std::string("device grid build: ") + what + ": " + hipGetErrorString(e);
        result = e == hipErrorOutOfMemory ? GridResult::NO_ROOM : GridResult::FAILED;
        return false;
    };
    int allocs = 0;
    auto alloc = [&](auto** p, size_t bytes) {
        return hipMalloc(p, ++allocs == refuse_alloc ? size_t{1} << 50 : bytes);
    };
    auto build = [&]() {
        if (!check(A.allocate(alloc), "alloc") || !check(alloc(&out.cell_start, (nc + 1) * 4), "alloc") ||
            !check(alloc(&out.dist, nc), "alloc") ||
            !check(alloc(&out.tris, std::max<size_t>(1, (size_t)nf) * 48), "alloc"))
            return false;
        float* d_xyz = A.get<float>(i_xyz);
        uint32_t* d_faces = A.get<uint32_t>(i_faces);
        unsigned short* d_masks = A.get<unsigned short>(i_masks);
        unsigned *d_count = A.get<unsigned>(i_count), *d_first = A.get<unsigned>(i_first);
        unsigned *d_big = A.get<unsigned>(i_big), *d_nbig = A.get<unsigned>(i_nbig);
        unsigned *d_cursor = A.get<unsigned>(i_cursor), *d_cells = A.get<unsigned>(i_cells);
        unsigned long long *d_local = A.get<unsigned long long>(i_local), *d_bsum = A.get<unsigned long long>(i_bsum);
        unsigned long long* d_total = A.get<unsigned long long>(i_total);
        unsigned char* d_tmp = A.get<unsigned char>(i_tmp);
        // exclusive scan of n counts into `to`, their total into d_total
        auto scan = [&](const unsigned* counts, size_t n, unsigned* to) {
            const size_t nb = (n + kScanBlock - 1) / kScanBlock;
            hipLaunchKernelGGL(scan_local_kernel, dim3((unsigned)nb), dim3(256), 0, s, counts, n, d_local, d_bsum);
            hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(1024), 0, s, d_bsum, nb, d_total);
            hipLaunchKernelGGL(scan_finish_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, s, d_local, d_bsum, n, to);
        };
        hipLaunchKernelGGL(fill_u32_kernel, dim3(blocks_for(nc, 256)), dim3(256), 0, s, d_cells, nc, 0u);
        unsigned long long total = 0;
        const dim3 mid_grid((unsigned)std::max<size_t>(1, std::min<size_t>(((size_t)nf + 3) / 4, 4096)));
        const dim3 huge_grid((unsigned)std::max<size_t>(1, std::min<size_t>(nf, 64)), 64);
        const unsigned face_blocks = stride_blocks((size_t)nf * kFaceLanes);
        if (nf) {
            if (nv && !check(hipMemcpyAsync(d_xyz, h_xyz, 3 * (size_t)nv * 4, hipMemcpyHostToDevice, s), "upload"))
                return false;
            if (!check(hipMemcpyAsync(d_faces, h_faces, 3 * (size_t)nf * 4, hipMemcpyHostToDevice, s), "upload"))
                return false;
            hipLaunchKernelGGL(fill_u32_kernel, dim3(1), dim3(256), 0, s, d_nbig, (size_t)3, 0u);
            hipLaunchKernelGGL(fill_u32_kernel, dim3(blocks_for(nf, 256)), dim3(256), 0, s, d_cursor, (size_t)nf, 0u);
            hipLaunchKernelGGL(classify_kernel, dim3(blocks_for(nf, 1024)), dim3(1024), 0, s, g, d_xyz, d_faces, nf,
                               d_big, d_nbig);
            hipLaunchKernelGGL(face_overlap_kernel, dim3(face_blocks), dim3(256), 0, s, g, d_xyz, d_faces, nf, d_masks,
                               d_count);
            big_overlap_kernel<false, false><<<mid_grid, 256, 0, s>>>(g, d_xyz, d_faces, nf, d_big, d_nbig, d_count,
                                                                      nullptr, nullptr, nullptr, nullptr);
            big_overlap_kernel<true, false><<<huge_grid, 256, 0, s>>>(g, d_xyz, d_faces, nf, d_big, d_nbig, d_count,
                                                                      nullptr, nullptr, nullptr, nullptr);
            scan(d_count, nf, d_first);
            hipLaunchKernelGGL(pack_faces_kernel, dim3(blocks_for(nf, 256)), dim3(256), 0, s, d_xyz, d_faces, nf,
                               reinterpret_cast<float4*>(out.tris));
            if (!check(hipGetLastError(), "overlap launch") ||
                !check(hipMemcpyAsync(&total, d_total, 8, hipMemcpyDeviceToHost, s), "total") ||
                !check(hipStreamSynchronize(s), "overlap"))
                return false;
            if (total > 0xFFFFFFFFull) {
                err = "grid has more than 2^32 face references; lower the resolution";
                result = GridResult::TOO_LARGE;
                return false;
            }
        }
        const int i_refs = R.add<Reference>((size_t)total), i_list = R.add<unsigned>((size_t)total);
        const int i_long = R.add<unsigned>((size_t)total / kLongList);
        if (!check(alloc(&out.cell_faces, std::max<size_t>(1, (size_t)total) * 4), "alloc")) return false;
        out.refs = (size_t)total;
        if (total) {
            if (!check(R.allocate(alloc), "alloc")) return false;
            Reference* d_refs = R.get<Reference>(i_refs);
            unsigned *d_list = R.get<unsigned>(i_list), *d_long = R.get<unsigned>(i_long);
            hipLaunchKernelGGL(face_place_kernel, dim3(face_blocks), dim3(256), 0, s, g, d_xyz, d_faces, nf,
                               (const unsigned short*)d_masks, (const unsigned*)d_first, d_cells, d_refs);
            big_overlap_kernel<false, true><<<mid_grid, 256, 0, s>>>(g, d_xyz, d_faces, nf, d_big, d_nbig, nullptr,
                                                                     d_first, nullptr, d_cells, d_refs);
            big_overlap_kernel<true, true><<<huge_grid, 256, 0, s>>>(g, d_xyz, d_faces, nf, d_big, d_nbig, nullptr,
                                                                     d_first, d_cursor, d_cells, d_refs);
            scan(d_cells, nc, out.cell_start);
            hipLaunchKernelGGL(list_kernel, dim3(stride_blocks((size_t)total)), dim3(256), 0, s,
                               (const Reference*)d_refs, (size_t)total, (const unsigned*)out.cell_start, d_list);
            hipLaunchKernelGGL(fill_u32_kernel, dim3(1), dim3(256), 0, s, out.cell_start + nc, (size_t)1,
                               (unsigned)total);
            hipLaunchKernelGGL(rank_kernel, dim3(stride_blocks((size_t)total)), dim3(256), 0, s,
                               (const Reference*)d_refs, (size_t)total, (const unsigned*)out.cell_start,
                               (const unsigned*)d_list, out.cell_faces, d_long, d_nbig + 2);
            if (nf > kLongList) {  // (a shorter mesh has no such list)
                int passes = 1;
                while (passes < 4 && (nf - 1) >> (8 * passes)) ++passes;
                hipLaunchKernelGGL(long_list_kernel, dim3(512), dim3(1024), 0, s, (const unsigned*)out.cell_start,
                                   d_list, out.cell_faces, (const unsigned*)d_long, (const unsigned*)(d_nbig + 2),
                                   passes | 1);
            }
        } else {
            hipLaunchKernelGGL(fill_u32_kernel, dim3(blocks_for(nc + 1, 256)), dim3(256), 0, s, out.cell_start, nc + 1,
                               0u);
        }
        hipLaunchKernelGGL(dist_x_kernel, dim3(blocks_for(ny * nz, 4)), dim3(256), dist_x_lds((int)nx), s,
                           (const unsigned*)out.cell_start, (int)nx, ny * nz, out.dist);
        hipLaunchKernelGGL(dist_minmax_kernel, dim3(blocks_for(nc, 256)), dim3(256), 0, s,
                           (const unsigned char*)out.dist, d_tmp, (int)nx, (int)ny, (int)nz, 1);
        hipLaunchKernelGGL(dist_minmax_kernel, dim3(blocks_for(nc, 256)), dim3(256), 0, s,
                           (const unsigned char*)d_tmp, out.dist, (int)nx, (int)ny, (int)nz, 2);
        return check(hipGetLastError(), "place/distance launch") &&
               check(hipStreamSynchronize(s), "place/distance");
    };
    if (!build()) {
        (void)hipStreamSynchronize(s);  // nothing may still run on what is freed
        out.release();
        (void)hipGetLastError();  // it has been reported: the next launch's check must not find it
    }
    return result;
}

}  // namespace linon
