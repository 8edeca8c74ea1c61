// fmm3d_look.h -- which columns a wavefront of the fixed-point check reads.
//
// The check gives each slot whole blocks of 256 columns, a wavefront 64 of
// them from f0 on, a lane one.  A slot has NL = nnx * nnz columns, rarely a
// multiple of 256, so a slot's last block can have wavefronts without a
// column (f0 >= NL) and one with fewer than 64.  Plain integer functions: the
// kernel forms its addresses with them, and a CPU program can go through all
// of a grid's.
#pragma once
#include <stddef.h>

#ifndef FMM3D_HD
#define FMM3D_HD __host__ __device__ __forceinline__
#endif

namespace fmm3d {

// Whether the wavefront whose first column is f0 has any: one without leaves
// before its first load.
FMM3D_HD bool look_has_columns(size_t f0, size_t NL) { return f0 < NL; }

// The late inputs of a column (ix, iz): per axis the step to its first and
// second neighbour outside its patch, unless that one lies in the patch it
// waits for (at patch index - f along the axis; f 0: none) or outside the
// slot's grid; 0 where the input is not late.  A patch has eight rows at
// least, so late inputs lie on one side of the node only.
struct LookLate {
    int dx[2], dz[2];
};
FMM3D_HD LookLate look_late(int ix, int iz, int snx, int snz, int px, int pz, int fx, int fz)
{
    LookLate r = { { 0, 0 }, { 0, 0 } };
    const int pxo = ix / px, pzo = iz / pz;
    for (int k = 0; k < 2; ++k)
        for (int s = 1; s >= -1; s -= 2) {   // the lower side last: it is the one taken
            const int jx = ix + s * (k + 1), jz = iz + s * (k + 1);
            if (jx >= 0 && jx < snx && jx / px != pxo && !(fx != 0 && jx / px == pxo - fx)) r.dx[k] = s * (k + 1);
            if (jz >= 0 && jz < snz && jz / pz != pzo && !(fz != 0 && jz / pz == pzo - fz)) r.dz[k] = s * (k + 1);
        }
    return r;
}

// Columns are counted from this many rows before the wavefront's first one: 2,
// so that those of late inputs are not negative.  0 where a row is so long
// that two of them on either side pass 32 bits of bytes: the check then reads
// no late inputs and evaluates every node.
FMM3D_HD int look_rows(int nnz, size_t bytes) { return ((size_t)4 * nnz + 64) * bytes <= 0xffffffffu ? 2 : 0; }

// The column a lane reads for itself (dx = dz = 0) or as a late input (rows 2).
// A lane without a column of its own reads the wavefront's first.
FMM3D_HD unsigned look_node(int rows, int nnz, int lane, bool on, int dx, int dz)
{
    return on ? (unsigned)((rows + dx) * nnz + lane + dz) : (unsigned)(rows * nnz);
}

}  // namespace fmm3d
