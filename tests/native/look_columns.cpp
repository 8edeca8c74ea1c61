// The columns the fixed-point check's look reads, from the functions its
// kernel forms them with: every wavefront of a slot, every lane, in the
// kernel's order.
#define FMM3D_HD inline
#include "../../parallel-fast-marching-method_amd/csrc/fmm3d_look.h"

using namespace fmm3d;

// The lowest and the highest column of the slot any lane reads (out[0],
// out[1]), the columns that are some lane's own (out[2]) and, of their late
// inputs, those that are not the neighbour itself (out[3]).
extern "C" void look_extent(int nnx, int nnz, int snx, int snz, int px, int pz, int fx, int fz, long long* out)
{
    const size_t NL = (size_t)nnx * nnz, nb = (NL + 255) / 256;
    long long lo = (long long)NL, hi = -1, own = 0, wrong = 0;
    for (size_t block = 0; block < nb; ++block)
        for (int wave = 0; wave < 4; ++wave) {
            const size_t f0 = block * 256 + 64 * wave;
            if (!look_has_columns(f0, NL)) continue;
            for (int lane = 0; lane < 64; ++lane) {
                const size_t f = f0 + lane;
                const int ix = (int)(f / nnz), iz = (int)(f - (size_t)ix * nnz);
                const bool on = f < NL && ix < snx && iz < snz;
                LookLate late = { { 0, 0 }, { 0, 0 } };
                if (on) late = look_late(ix, iz, snx, snz, px, pz, fx, fz);
                const long long base = (long long)f0 - 2 * (long long)nnz;
                auto read = [&](int dx, int dz) {
                    const long long c = base + look_node(2, nnz, lane, on, dx, dz);
                    lo = c < lo ? c : lo;
                    hi = c > hi ? c : hi;
                    return c;
                };
                const long long c = read(0, 0);
                own += on && c == (long long)f;
                for (int k = 0; k < 2; ++k) {
                    const long long x = read(late.dx[k], 0), z = read(0, late.dz[k]);
                    wrong += on && (x != (long long)(ix + late.dx[k]) * nnz + iz || z != (long long)ix * nnz + iz + late.dz[k]);
                }
            }
        }
    out[0] = lo;
    out[1] = hi;
    out[2] = own;
    out[3] = wrong;
}

// Whether every offset a lane of a wavefront forms for rows nnz long, times the
// size of a value, is the exact one in 32 bits.
extern "C" int look_fits(int nnz, int bytes)
{
    const int rows = look_rows(nnz, (size_t)bytes);
    for (int lane = 0; lane < 64; ++lane)
        for (int dx = -rows; dx <= rows; ++dx)
            for (int dz = rows ? -2 : 0; dz <= (rows ? 2 : 0); ++dz) {
                const unsigned o = look_node(rows, nnz, lane, true, dx, dz);
                const long long exact = (long long)(rows + dx) * nnz + lane + dz;
                if (exact >= 0 && (unsigned long long)(o * (unsigned)bytes) != (unsigned long long)exact * (unsigned)bytes) return 0;
            }
    return 1;
}
