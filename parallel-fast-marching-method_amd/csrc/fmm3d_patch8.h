// fmm3d_patch8.h -- the LDS cells of a layer of an 8 x 8 patch, one node per
// lane of a wavefront, two halo nodes deep on four sides (no corners: the
// stencil is a cross).  Plain integer functions, for the kernels and for a CPU
// program that goes through them.
#pragma once

#ifndef FMM3D_HD
#define FMM3D_HD __host__ __device__ __forceinline__
#endif

namespace fmm3d {

struct Patch8 {
    static constexpr int P = 8;
    static constexpr int LZ = P + 5;                // odd row stride: phi neighbours spread over banks
    static constexpr int CELLS = (P + 4) * LZ;
    // lanes without a node read a stencil like the others, but of spare cells
    // behind the patch; lanes without a halo node write one of those
    static constexpr int OUT = CELLS + LZ;
    static constexpr int HALO_OUT = CELLS + 2 * LZ;
    static constexpr int SIZE = OUT + 2 * LZ + 1;
    static_assert(OUT - 2 * LZ >= 0 && OUT + 2 * LZ < SIZE && HALO_OUT < SIZE, "a spare lane's stencil stays in the array");

    // cell of patch row hx, column hz, both counted from the halo's first
    static FMM3D_HD int cell(int hx, int hz) { return hx * LZ + hz; }
    // the cell of lane (lx, lz); in: it has a node
    static FMM3D_HD int own(int lx, int lz, bool in) { return in ? cell(lx + 2, lz + 2) : OUT; }
    // the halo node of lane t: its row and column from the halo's first
    static FMM3D_HD void halo(int t, int* hx, int* hz)
    {
        const int side = t >> 4, d = (t >> 3) & 1, e = t & 7;
        *hx = side == 0 ? 1 - d : side == 1 ? P + 2 + d : 2 + e;
        *hz = side == 2 ? 1 - d : side == 3 ? P + 2 + d : 2 + e;
    }
};

}  // namespace fmm3d
