// fmm3d_update.h -- one node update of the column walks: the minimum over the
// octants of a node's stencil, from one of them where that one is certain.
#pragma once
#include <limits>
#include <type_traits>

#include "fmm3d_device.h"

namespace fmm3d {

// The two sides of one axis of a node's stencil: the first and second
// neighbours' values towards the lower index (l1, l2) and the higher one
// (h1, h2), inf outside the grid, and whether the first ones exist.
template <typename R> struct AxisSides {
    R l1, l2, h1, h2;
    bool lin, hin;
};

// float32 helpers for the axis-sum octant form: fused multiply-subtract,
// hardware square root and reciprocal (about 1 ulp each).
template <typename R> __device__ __forceinline__ R fused_mul_sub(R a, R b, R c) { return fma(a, b, -c); }
template <typename R> __device__ __forceinline__ R fast_sqrt(R x) { return sqrt(x); }
template <> __device__ __forceinline__ float fast_sqrt<float>(float x) { return __builtin_amdgcn_sqrtf(x); }
template <typename R> __device__ __forceinline__ R fast_rcp(R x) { return R(1) / x; }
template <> __device__ __forceinline__ float fast_rcp<float>(float x) { return __builtin_amdgcn_rcpf(x); }

// Octant minimum in the axis-sum form (FAST): for the counted sides of an
// octant sum (c*T - D)^2 / H^2 = s^2 with c, D, H = (1, t1, h) first order
// and (3, 4 t1 - t2, 2 h) second order, i.e. A T^2 - 2 B T + C = 0 with
// A = sum (c/H)^2, B = sum (c/H)(D/H), C = sum (D/H)^2 - s^2; the larger
// root with the discriminant clamped at zero.  This is the reference's
// octant quadratic after the substitution T = (X + D_L)/c_L on its leading
// axis (fm3dt_parallel.f90:535-1004), so the two agree up to rounding.
// Octants through a missing side are skipped, octants with no counted side
// give nothing, as in the reference: the first carry A = NaN, the second
// A = B = 0 and so T = 0 * inf = NaN, and the running minimum is fmin,
// which passes over a NaN.  Values arrive shifted by the smallest counted
// neighbour.
//
// One octant usually decides.  With at most one side counted per axis, the
// octant of the counted sides has the least solution, since the others leave
// out some of its squared terms and so reach s^2 later.  In the computed
// values that is certain where each counted term alpha T - beta is positive
// (so T is a root and not where the discriminant was clamped) and its square
// exceeds the rounding of the whole sum, a few units in the last place of
// M = A T^2 + sum beta^2 + s^2 <= 3 (sum beta^2 + s^2); the margin asked for
// is 2^8 of them.  Where an axis' term is not certain, the octant without it
// is evaluated too, and where both sides of an axis count, the octants of
// either (float32: all eight in either case), so that every value is the
// minimum over all eight octants to the last bit.  Measured against eight
// octants each time: 6 % of the wavefronts' passes need more than one in the
// first sweep of 50 float32 plane waves at 201^3, which went from 5.55 to 3.33
// G VALU instructions; in k_column, eight float64 sources at 31x110x140 went
// from 9.0 to 5.4 ms and a local source at 61^3 from 53 to 30 ms.

// The octant of one side per axis (ord 0: none; t1, t2 relative to a common
// time), its solution and the axes whose term is not certain (bits).
// h2: squared spacings; kt: as octant_one's (float64).
template <typename R, bool FAST>
__device__ __forceinline__ R octant_eval(const Side<R> p[3], const R h2[3], const R ih[3], R s2, R kt, unsigned* weak)
{
    if constexpr (FAST) {
        R pa[3], pb[3], paa[3], pbb[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const bool cnt = p[a].ord != 0, sec = p[a].ord == 2;
            const R num = sec ? fma(R(-0.5), p[a].t2, p[a].t1 + p[a].t1) : p[a].t1;
            pa[a] = ih[a] * (cnt ? (sec ? R(1.5) : R(1)) : R(0));
            pb[a] = cnt ? num * ih[a] : R(0);
            paa[a] = pa[a] * pa[a];
            pbb[a] = pb[a] * pb[a];
        }
        const R A = paa[0] + (paa[1] + paa[2]), B = pa[0] * pb[0] + (pa[1] * pb[1] + pa[2] * pb[2]);
        const R bb = pbb[1] + pbb[2], C = (pbb[0] - s2) + bb;
        R disc = fused_mul_sub(B, B, A * C);
        const bool clamped = !(disc > R(0));   // T is no root then, and no term certain
        disc = clamped ? R(0) : disc;
        const R T = (B + fast_sqrt(disc)) * fast_rcp(A);
        const R thr = R(0x1.8p-15) * (pbb[0] + bb + s2);
        unsigned w = clamped ? 7u : 0u;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const R g = fma(pa[a], T, -pb[a]);
            w |= (p[a].ord != 0 && !(g * fabs(g) > thr)) ? 1u << a : 0u;
        }
        *weak = w;
        return T;
    } else {
        return octant_one(p, h2, s2, kt, R(0x1p-40) * s2, weak);
    }
}

// All eight octants in the axis-sum form, side by side: cheap in float32 (a
// hardware square root and reciprocal each), where a node's own, one after the
// other, gained nothing (201^3, 50 plane waves, a solve: 13.4 ms with those
// where one axis is in doubt, 13.2 so).  Per side (a, b, c) = (alpha^2,
// alpha*beta, beta^2); a missing side carries a = NaN, and fmin passes over the
// octants through it.
template <typename R, bool SHIFT, typename G>
__device__ __forceinline__ R octants_eight(int fom, R top, R sh, G gather, const R ih[3], R s2)
{
    struct Coef { R a, b, c; };
    auto coef = [&](R w1, R w2, bool in, R ihx) {
        // selects on plain values keep this branch-free
        const bool cnt = SHIFT ? w1 <= top : w1 < top, sec = fom && w1 > w2;
        const R u1 = w1 - sh, u2 = w2 - sh;
        const R num = sec ? fma(R(-0.5), u2, u1 + u1) : u1;
        const R al = ihx * (cnt ? (sec ? R(1.5) : R(1)) : R(0));
        const R be = cnt ? num * ihx : R(0);
        return Coef{ in ? al * al : R(__builtin_nan("")), al * be, be * be };
    };
    R best = Lim<R>::inf();
    const AxisSides<R> r = gather(0), x = gather(1), z = gather(2);
    Coef cr[2] = { coef(r.l1, r.l2, r.lin, ih[0]), coef(r.h1, r.h2, r.hin, ih[0]) };
    const Coef cx[2] = { coef(x.l1, x.l2, x.lin, ih[1]), coef(x.h1, x.h2, x.hin, ih[1]) };
    const Coef cz[2] = { coef(z.l1, z.l2, z.lin, ih[2]), coef(z.h1, z.h2, z.hin, ih[2]) };
    cr[0].c -= s2;
    cr[1].c -= s2;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const R Axz = cx[j].a + cz[k].a, Bxz = cx[j].b + cz[k].b, Cxz = cx[j].c + cz[k].c;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const R A = cr[i].a + Axz, B = cr[i].b + Bxz, C = cr[i].c + Cxz;
                R disc = fused_mul_sub(B, B, A * C);
                disc = disc > R(0) ? disc : R(0);
                best = fmin(best, (B + fast_sqrt(disc)) * fast_rcp(A));
            }
        }
    return best;
}

// The minimum over the octants of a node whose one octant, of solution best,
// was not certain on the axes weak, or has both sides of an axis counted
// (sides counted below top, times relative to sh), where an octant is dear
// (float64).  Per axis, role 0 is the lower side and role 1 the other: its
// octants differ where both sides count (both), and where role 1 leaves the
// axis out while role 0 counts (drop).  The other octants of the counted sides
// come first, then those without one or more of the axes some of them left
// uncertain; each lane goes through its own (their sets differ from node to
// node), so the wavefront takes the most that one node needs (eight plane waves
// at 31x110x140, a call: 8.1 ms with the set its nodes need together, 4.5 so;
// the first sweep took 5.2 ms with all eight octants and 3.3 with that set).
// The stencil is gathered again for each, so that this path holds few
// registers.
template <typename R, bool SHIFT, typename G>
__device__ __forceinline__ R octants_more(int fom, R top, R sh, G gather, const R h2[3], const R ih[3], R s2, R kt,
                                          R best, unsigned weak)
{
    auto counts = [&](R v) { return SHIFT ? v <= top : v < top; };
    unsigned both = 0, drop = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const AxisSides<R> g = gather(a);
        const bool lo = g.l1 <= g.h1, ob = counts(lo ? g.h1 : g.l1);
        both |= ob ? 1u << a : 0u;
        drop |= !ob && counts(lo ? g.l1 : g.h1) && (lo ? g.hin : g.lin) ? 1u << a : 0u;
    }
    unsigned unsure = weak & drop;
    // todo: the octants left, a bit for each set of axes in role 1
    unsigned todo = subsets(both) & ~1u;
    for (bool first = true;;) {
        if (!todo && first) { first = false; todo = subsets(both | unsure) & ~subsets(both); }
        if (!todo) break;
        const unsigned m = __ffs(todo) - 1;
        todo &= todo - 1;
        asm volatile("" ::: "memory");
        Side<R> p[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const AxisSides<R> g = gather(a);
            const bool lo = g.l1 <= g.h1, other = (m >> a) & 1;
            const R o1 = lo ? g.h1 : g.l1, o2 = lo ? g.h2 : g.l2, q1 = lo ? g.l1 : g.h1, q2 = lo ? g.l2 : g.h2;
            const R t1 = other ? o1 : q1, t2 = other ? o2 : q2;   // a dropped axis' other side does not count
            p[a].ord = counts(t1) ? (fom && t1 > t2 ? 2 : 1) : 0;
            p[a].t1 = p[a].ord ? t1 - sh : R(0);
            p[a].t2 = p[a].ord == 2 ? t2 - sh : R(0);
        }
        if (!(p[0].ord | p[1].ord | p[2].ord)) continue;
        unsigned w;
        const R T = octant_eval<R, false>(p, h2, ih, s2, kt, &w);
        if (T < best) best = T;
        if (first) unsure |= w & drop;
    }
    return best;
}

// One node update.  gather(a) gives axis a's sides of the stencil (every axis
// has at least two nodes).  FAST selects the axis-sum octant form; otherwise
// the reference's leading-axis form in the CPU oracle's operation order.
// h, ih: spacings and their reciprocals along r, x, z.  free: whether the node
// is one to update (the value returned for another one is not to be used).
// EIGHT (float32): all eight octants at once.  *more, if asked for: whether one
// octant left some node of the wavefront in doubt.
// The walks whose lanes hold more than one node, and the hyperplane walk, take
// eight in float32: their many nodes a wavefront leave few passes where one
// decides (201^3, 20 sources, 16 x 16 patches / 8 x 16 / hyperplane, a call:
// 19.0 / 13.4 / 122 ms with one octant first, 15.8 / 12.1 / 90.6 so).
template <typename R, bool FAST, bool SHIFT, bool EIGHT = false, typename G>
__device__ __forceinline__ R col_update(int fom, R tc, G gather, const R h[3], const R ih[3], R slown, bool free = true,
                                        bool* more = nullptr)
{
    const R inf = Lim<R>::inf();
    // per axis the lower side (t1, t2) -- the counted one, where one counts --
    // and the least of the other sides: at or below the node, two count
    R t1[3], t2[3], other = inf;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const AxisSides<R> g = gather(a);
        const bool lo = g.l1 <= g.h1;
        t1[a] = lo ? g.l1 : g.h1;
        t2[a] = lo ? g.l2 : g.h2;
        const R o = lo ? g.h1 : g.l1;
        other = o < other ? o : other;
    }
    // an unknown node counts every known neighbour: its value compares as the
    // largest finite one where equal values count, as inf where they do not
    const R top = SHIFT ? (tc < inf ? tc : std::numeric_limits<R>::max()) : tc;
    auto counts = [&](R v) { return SHIFT ? v <= top : v < top; };
    const R low = t1[0] < t1[1] ? (t1[0] < t1[2] ? t1[0] : t1[2]) : (t1[1] < t1[2] ? t1[1] : t1[2]);
    const bool known = counts(low);   // some neighbour counts
    const R sh = SHIFT ? low : R(0);
    const R s2 = slown * slown;
    const R h2[3] = { h[0] * h[0], h[1] * h[1], h[2] * h[2] };
    R kt = R(0);
    Side<R> p[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        p[a].ord = counts(t1[a]) ? (fom && t1[a] > t2[a] ? 2 : 1) : 0;
        p[a].t1 = FAST || p[a].ord ? t1[a] - sh : R(0);
        p[a].t2 = FAST || p[a].ord == 2 ? t2[a] - sh : R(0);
        kt += R(0x1.2p-38) * ih[a] * ih[a];   // the largest (c / H)^2: 9/4
    }
    R best;
    if constexpr (EIGHT) {
        best = octants_eight<R, SHIFT>(fom, top, sh, gather, ih, s2);
    } else {
        unsigned weak;
        best = octant_eval<R, FAST>(p, h2, ih, s2, kt, &weak);
        const bool doubt = (weak || counts(other)) && known && free;
        if (more) *more = __any(doubt);
        if (doubt) {
            if constexpr (FAST) best = octants_eight<R, SHIFT>(fom, top, sh, gather, ih, s2);
            else best = octants_more<R, SHIFT>(fom, top, sh, gather, h2, ih, s2, kt, best, weak);
        }
    }
    if (SHIFT && best < inf) best = sh + best;
    return known ? best : inf;
}

}  // namespace fmm3d
