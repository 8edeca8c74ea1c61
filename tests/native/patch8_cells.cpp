// The LDS cells the one-node-per-lane walks read and write, from the functions
// the kernels form them with.
#define FMM3D_HD inline
#include "../../parallel-fast-marching-method_amd/csrc/fmm3d_patch8.h"

using namespace fmm3d;

// A patch with nx x nz nodes (1..8 each) whose halo reaches rows r0..r1 and
// columns c0..c1 of the grid around it.  out: the lowest and highest cell any
// lane touches, the array's size, and the faults found: two lanes that write
// one cell of the patch or its halo, a stencil cell of a lane with a node that
// is neither a node, a halo node, nor left at its start value.
extern "C" void patch8_cells(int nx, int nz, int r0, int r1, int c0, int c1, int* out)
{
    int lo = 0, hi = 0, faults = 0;
    static int writes[1024];
    for (int& w : writes) w = 0;
    auto touch = [&](int c) { lo = c < lo ? c : lo; hi = c > hi ? c : hi; return c; };
    for (int t = 0; t < 64; ++t) {
        const int lx = t / Patch8::P, lz = t % Patch8::P;
        const bool in = lx < nx && lz < nz;
        const int own = touch(Patch8::own(lx, lz, in));
        if (in) ++writes[own];
        int hx, hz;
        Patch8::halo(t, &hx, &hz);
        const bool ok = hx - 2 >= r0 && hx - 2 <= r1 && hz - 2 >= c0 && hz - 2 <= c1;
        // a halo cell that is one of the patch's own nodes would be written twice
        const int ridx = touch(ok ? Patch8::cell(hx, hz) : Patch8::HALO_OUT);
        if (ok) ++writes[ridx];
        // the stencil, of lanes without a node too
        const int step[8] = { -Patch8::LZ, -2 * Patch8::LZ, Patch8::LZ, 2 * Patch8::LZ, -1, -2, 1, 2 };
        for (int s : step) touch(own + s);
        for (int k = 0; k < 8 && in; ++k) {
            const int d = k & 1 ? 2 : 1, up = k & 2 ? d : -d;
            const int ex = k < 4 ? lx + 2 + up : lx + 2, ez = k < 4 ? lz + 2 : lz + 2 + up;
            if (own + step[k] != Patch8::cell(ex, ez) || ex < 0 || ex >= Patch8::P + 4 || ez < 0 || ez >= Patch8::P + 4) ++faults;
        }
    }
    for (int c = 0; c < Patch8::CELLS; ++c) faults += writes[c] > 1;
    out[0] = lo;
    out[1] = hi;
    out[2] = Patch8::SIZE;
    out[3] = faults;
}
