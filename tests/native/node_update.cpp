// The walks' node update against a plain enumeration of the eight octants in
// the same arithmetic, on random stencils.
#include <hip/hip_runtime.h>

#include <random>

#include "../../parallel-fast-marching-method_amd/csrc/fmm3d_update.h"

using namespace fmm3d;

int lane_ulp = 0;

namespace {

template <typename R> struct Node {
    R tc, v1[3][2], v2[3][2];   // the node; per axis and side the first and second neighbour
    bool in[3][2];
    R h[3], slown;
};

// One octant, sides s[a] of the axes; in float32 the sums' order of the
// axis-sum form, in float64 octant_solve.  NaN where it gives nothing.
template <typename R, bool FAST>
R octant(const Side<R> p[3], const Node<R>& n, bool* clamped)
{
    const R nan = (R)NAN;
    if (p[0].ord < 0 || p[1].ord < 0 || p[2].ord < 0 || !(p[0].ord | p[1].ord | p[2].ord)) return nan;
    if constexpr (FAST) {
        R al[3], be[3], bb[3];
        for (int a = 0; a < 3; ++a) {
            const R ih = R(1) / n.h[a];
            const R num = p[a].ord == 2 ? fma(R(-0.5), p[a].t2, p[a].t1 + p[a].t1) : p[a].t1;
            al[a] = ih * (p[a].ord == 2 ? R(1.5) : p[a].ord == 1 ? R(1) : R(0));
            be[a] = p[a].ord ? num * ih : R(0);
            bb[a] = be[a] * be[a];
        }
        const R A = al[0] * al[0] + (al[1] * al[1] + al[2] * al[2]);
        const R B = al[0] * be[0] + (al[1] * be[1] + al[2] * be[2]);
        const R C = (bb[0] - n.slown * n.slown) + (bb[1] + bb[2]);
        R disc = fma(B, B, -(A * C));
        *clamped |= !(disc > R(0));
        disc = disc > R(0) ? disc : R(0);
        return (B + lane_sqrt(disc)) * lane_rcp(A);
    } else {
        return octant_solve<R>(p[0], p[1], p[2], n.h[0], n.h[1], n.h[2], n.slown);
    }
}

template <typename R, bool FAST, bool SHIFT>
R eight(int fom, const Node<R>& n, int* nlow, bool* clamped)
{
    const R inf = Lim<R>::inf();
    bool cnt[3][2];
    R sh = inf;
    for (int a = 0; a < 3; ++a)
        for (int s = 0; s < 2; ++s) {
            const R v = n.v1[a][s];
            cnt[a][s] = n.in[a][s] && (SHIFT ? v <= n.tc && v < inf : v < n.tc);
            if (cnt[a][s] && v < sh) sh = v;
        }
    if (!(sh < inf)) return inf;
    if (!SHIFT) sh = R(0);
    R best = inf;
    *nlow = 0;
    for (int o = 0; o < 8; ++o) {
        Side<R> p[3];
        for (int a = 0; a < 3; ++a) {
            const int s = (o >> a) & 1;
            const bool sec = cnt[a][s] && fom && n.v2[a][s] < inf && n.v1[a][s] > n.v2[a][s];
            p[a].ord = !n.in[a][s] ? -1 : sec ? 2 : cnt[a][s] ? 1 : 0;
            p[a].t1 = cnt[a][s] ? n.v1[a][s] - sh : R(0);
            p[a].t2 = sec ? n.v2[a][s] - sh : R(0);
        }
        const R T = octant<R, FAST>(p, n, clamped);
        if (T == best) ++*nlow;
        if (T < best) { best = T; *nlow = 1; }
    }
    return SHIFT && best < inf ? sh + best : best;
}

template <typename R> bool same(R a, R b) { return memcmp(&a, &b, sizeof a) == 0; }

// out: updates that differ, nodes with both sides of an axis counted, with a
// clamped octant, with several least octants, unknown, with a side outside
template <typename R, bool FAST, bool SHIFT>
void run(long n, unsigned seed, int fom, long long* out)
{
    std::mt19937_64 rng(seed);
    auto uni = [&](double lo, double hi) { return lo + (hi - lo) * (double)(rng() >> 11) * 0x1p-53; };
    auto pick = [&](int k) { return (int)(rng() % (unsigned)k); };
    const R inf = Lim<R>::inf();
    for (long i = 0; i < n; ++i) {
        Node<R> d;
        d.slown = (R)uni(0.08, 0.4);
        for (R& h : d.h) h = (R)uni(0.5, 12.0);
        // a wave of unit slowness vector g about time t0, kinks and noise on it
        double g[3], gg = 0.0;
        for (double& x : g) { x = pick(4) ? uni(-1.0, 1.0) : 0.0; gg += x * x; }
        for (double& x : g) x *= gg > 0.0 ? (double)d.slown / std::sqrt(gg) : 0.0;
        const double t0 = pick(3) ? uni(-3.0, 3.0) : uni(0.0, 600.0);
        const int kind = pick(8);
        const double noise = kind < 2 ? 0.0 : kind < 5 ? 1e-6 : kind < 7 ? 0.3 : 30.0;
        const double grain = kind == 4 || kind == 5 ? 0x1p-22 : kind == 6 ? 0.25 : 0.0;   // ties
        auto val = [&](double x) {
            x += noise * uni(-1.0, 1.0);
            if (grain > 0.0) x = std::nearbyint(x / grain) * grain;
            return (R)x;
        };
        const int kink = pick(6);   // an axis on which both sides run ahead, or behind
        for (int a = 0; a < 3; ++a)
            for (int s = 0; s < 2; ++s) {
                const double dir = kink == a ? -std::fabs(g[a]) : kink == a + 3 ? std::fabs(g[a]) : (s ? g[a] : -g[a]);
                d.in[a][s] = pick(12) != 0;
                if (s == 1 && !d.in[a][0]) d.in[a][1] = true;   // an axis has two nodes at least
                d.v1[a][s] = d.in[a][s] && pick(10) ? val(t0 + dir * d.h[a]) : inf;
                d.v2[a][s] = d.in[a][s] && pick(10) ? val(t0 + 2.0 * dir * d.h[a]) : inf;
                if (pick(20) == 0) d.v2[a][s] = d.v1[a][s];
            }
        d.tc = val(t0);
        switch (pick(6)) {
        case 0: d.tc = inf; break;                                     // not reached yet
        case 1: d.tc = d.v1[pick(3)][pick(2)]; break;                  // on a neighbour
        case 2: d.tc = (R)(t0 + 40.0); break;                          // late: everything counts
        case 3: d.tc = (R)(t0 - uni(0.0, 3.0)); break;                 // early: little does
        }
        const R ih[3] = { R(1) / d.h[0], R(1) / d.h[1], R(1) / d.h[2] };
        auto gather = [&](int a) { return AxisSides<R>{ d.v1[a][0], d.v2[a][0], d.v1[a][1], d.v2[a][1], d.in[a][0], d.in[a][1] }; };
        int nlow = 0, two = 0, outside = 0;
        bool clamped = false;
        const R want = eight<R, FAST, SHIFT>(fom, d, &nlow, &clamped);
        const R got = col_update<R, FAST, SHIFT>(fom, d.tc, gather, d.h, ih, d.slown);
        const R all = col_update<R, FAST, SHIFT, FAST>(fom, d.tc, gather, d.h, ih, d.slown);
        out[0] += !same(want, got) || !same(want, all);
        for (int a = 0; a < 3; ++a) {
            two |= d.v1[a][0] < d.tc && d.v1[a][1] < d.tc;
            outside |= !d.in[a][0] || !d.in[a][1];
        }
        out[1] += two;
        out[2] += clamped;
        out[3] += nlow > 1;
        out[4] += !(d.tc < inf);
        out[5] += outside;
    }
}

}  // namespace

extern "C" void node_update(int f32, int order, long n, unsigned seed, int ulp, long long* out)
{
    lane_ulp = ulp;
    for (int k = 0; k < 6; ++k) out[k] = 0;
    if (f32) run<float, true, true>(n, seed, order, out);
    else run<double, false, false>(n, seed, order, out);
}
