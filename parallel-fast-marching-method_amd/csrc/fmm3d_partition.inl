// fmm3d_partition.inl -- the reference's 2x2x2 partitioned teleseismic solve
// on the device (FMM3D_REFERENCE_PARTITION).  Included by fmm3d_solver.hip.
//
// fm3dt_parallel splits the grid over a 2x2x2 layout of ranks (F:6127-6171)
// and, per source, repeats passes (F:6397-6435) until the largest change of
// a pass is at most the float32 literal 1e-5 (F:6403):
//   1. every rank that marched in the previous pass sends its two planes next
//      to each face; a receiving rank relaxes its face nodes from them, one
//      face after the other, each face node once, in the order of a heap
//      keyed by the near ghost value (order_overlap + fouds2_<face>,
//      F:157-386, 1100-2825);
//   2. if any face node was accepted, the rank reclassifies its nodes
//      against the smallest and largest accepted value (F:387-415) and
//      marches its heap to empty (local_fmm, F:78-155), with stencils that
//      end at the rank's own faces (F:708-710).
// Pass 0 is start_fmm: the bottom face is injected and the bottom rank(s)
// with the smallest face minimum march from it (F:6894-6961).
//
// Here all eight blocks of every source live in one field per source, and
// the two sequential parts run in parallel forms that give the same values:
//   - face relaxation (k_pt_face): in heap order a face node reads the new
//     value of each in-plane neighbour (first or second) with a smaller key
//     that is in the heap, the old value of every other; so it can be
//     computed once those neighbours are done.  One workgroup per
//     (source, block) runs rounds over the nodes the round before made
//     ready.  Key ties go by face index.
//   - the march (k_pt_walk): the pop-order update.  The march freezes the
//     nodes alive at its start and gives every other node the minimum of its
//     starting value and the octant candidates computed each time a
//     neighbour pops, from the neighbours alive then.  A neighbour pops
//     before the node iff its value is below the node's value so far: the
//     update walks the known neighbours in increasing value, one joins while
//     it is below the running minimum, and after each join the octants
//     through it give a candidate.  The result depends on the neighbours
//     only, so Jacobi passes cannot cycle, and they settle where the march
//     does.  One wavefront per 8 x 8 patch column of a block walks the
//     block's layers, alternating direction per sweep, and sweeps repeat
//     until one changes nothing.
// The CPU oracle restates both forms (or_relax_tele_part) and checks them
// against the heap forms (or_fmm_tele_part, which reproduces the reference's
// rtravel.out bit for bit).
//
// Node velocities and metric terms use each block's own offset arithmetic,
// as the ranks compute them (F:540-543, 6989-7038), so the float64 values
// are the reference's.  Unknown times are +inf (the reference's 0); an
// unknown ghost enters a face update as 0, as in the reference.

namespace {

constexpr int PT_FACE_AXIS[6] = { 1, 1, 2, 2, 0, 0 };   // faces: left, right, in, out, up, down
constexpr int PT_FACE_SIDE[6] = { -1, 1, -1, 1, -1, 1 };
constexpr int PT_P = 8;                                 // patch edge of the block walk
constexpr int PT_FACE_THREADS = 1024;

// Block layout: per axis the first index of the second block.  The first
// block takes the extra node of an odd count (the reference's rank sizes).
struct PartGeo {
    int n[3];
    int cut[3];
    __host__ __device__ int lo(int a, int b) const { return b ? cut[a] : 0; }
    __host__ __device__ int len(int a, int b) const { return b ? n[a] - cut[a] : cut[a]; }
};

__host__ __device__ inline void pt_coord(int blk, int c[3]) { c[0] = blk >> 2; c[1] = (blk >> 1) & 1; c[2] = blk & 1; }

// the in-plane axes of face k, (outer, inner) in the reference's loop order
__host__ __device__ inline void pt_face_axes(int k, int& outer, int& inner)
{
    const int a = PT_FACE_AXIS[k];
    if (a == 1) { outer = 0; inner = 2; }
    else if (a == 2) { outer = 0; inner = 1; }
    else { outer = 1; inner = 2; }
}

static PartGeo part_geo(const Grid& g)
{
    PartGeo p;
    p.n[0] = g.nnr; p.n[1] = g.nnx; p.n[2] = g.nnz;
    for (int a = 0; a < 3; ++a) p.cut[a] = (p.n[a] + 1) / 2;
    return p;
}

}  // namespace

// Device state of the partitioned mode, owned by the context.
struct PartState {
    int cap = 0;                    // slots the arrays hold
    size_t nfmax = 0;               // largest face of a block (nodes)
    double* Tprev = nullptr;        // field at the start of the pass (ghosts, change)
    double* T0 = nullptr;           // march start: -value for heap nodes, value otherwise
    uint32_t* hbits = nullptr;      // nodes accepted by this pass's face relaxation (the heap)
    int* on = nullptr;              // per slot: passes continue
    int* dsend = nullptr;           // per slot x block: marched in the previous pass
    int* march = nullptr;           // per slot x block: marches in this pass
    double* mini = nullptr;         // per slot x block: smallest heap value
    int* stamp = nullptr;           // per slot x block x patch: last sweep that changed a value
    int* prog = nullptr;            // per slot x block x patch: sweep * (nnr + 1) + layers finished
    int* flow = nullptr;            // per slot: signs of the lateral flow (theta, phi)
    int* chg = nullptr;             // per slot: the sweep changed a value
    int* pstart = nullptr;          // per slot: first sweep of its current pass
    unsigned long long* err = nullptr;   // per slot: largest change of the pass (bits of a double)
    int* seed = nullptr;            // pass 0: (slot, node) pairs of the heap seeds
    int nseed_cap = 0;
    double* slo = nullptr;          // slowness, block arithmetic
    double* hx = nullptr;           // nnr
    double* hz = nullptr;           // nnr x nnx
    bool model = false;             // slo / hx / hz are those of the resident model
    int* h_chg = nullptr;           // pinned host copies
    unsigned long long* h_err = nullptr;
    std::vector<int> passes;        // per slot: passes of the last solve
};

namespace {

// Node velocity with a block's offset arithmetic (F:6989-7038 on a rank's
// local indices); slowness in solver layout.
__global__ void k_pt_gridder(Grid g, PartGeo p, const double* __restrict__ velv, double* __restrict__ slo)
{
    const long total = (long)g.nnr * g.nnx * g.nnz;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
        const int kz = (int)(i % g.nnz), kx = (int)((i / g.nnz) % g.nnx), kr = (int)(i / ((long)g.nnz * g.nnx));
        const int k3[3] = { kr, kx, kz };
        int off[3], l[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            off[a] = k3[a] >= p.cut[a] ? p.cut[a] + 1 : 1;    // 1-based global index of local index 1
            l[a] = k3[a] - off[a] + 2;                         // 1-based local index
        }
        const double h = g.rgor - (off[0] - 1) * g.dnr - (l[0] - 1) * g.dnr;
        const double hr = g.gor - g.rgor + (off[0] - 1) * g.dnr + (l[0] - 1) * g.dnr;
        const double th = g.rgox + (off[1] - 1) * g.dnx + (l[1] - 1) * g.dnx;
        const double ph = g.rgoz + (off[2] - 1) * g.dnz + (l[2] - 1) * g.dnz;
        const int NR = g.nvr + 2, NX = g.nvx + 2, NZ = g.nvz + 2;
        const int ri = (int)floor(hr / g.dvr) + 1;
        double wr[4], wx[4], wz[4];
        bspline4(((g.gor - (ri - 1) * g.dvr) - h) / g.dvr, wr);
        const int xi = (int)floor((th - g.gox) / g.dvx) + 1;
        bspline4((th - g.gox - (xi - 1) * g.dvx) / g.dvx, wx);
        const int zi = (int)floor((ph - g.goz) / g.dvz) + 1;
        bspline4((ph - g.goz - (zi - 1) * g.dvz) / g.dvz, wz);
        double acc_z = 0.0;
        for (int a = 0; a < 4; ++a) {
            const int iz = min(max(zi - 1 + a, 0), NZ - 1);
            double acc_x = 0.0;
            for (int b = 0; b < 4; ++b) {
                const int ix = min(max(xi - 1 + b, 0), NX - 1);
                const double* col = velv + ((size_t)iz * NX + ix) * NR;
                double acc_r = 0.0;
                for (int c = 0; c < 4; ++c) acc_r += wr[c] * col[min(max(ri - 1 + c, 0), NR - 1)];
                acc_x += wx[b] * acc_r;
            }
            acc_z += wz[a] * acc_x;
        }
        slo[i] = 1.0 / acc_z;
    }
}

// Bottom-face injection (start_fmm, F:6914-6939): values > 0 known, the
// rest unknown; every other node unknown.
__global__ void k_pt_inject(int nnr, int nnx, int nnz, int nslots, const double* __restrict__ faces, double* __restrict__ T)
{
    const size_t NL = (size_t)nnx * nnz, N = NL * nnr;
    const size_t total = (size_t)nslots * N;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const size_t s = i / N, q = i - s * N;
        double v = __builtin_huge_val();
        if (q >= (size_t)(nnr - 1) * NL) {
            const double f = faces[s * NL + (q - (size_t)(nnr - 1) * NL)];
            if (f > 0.0) v = f;
        }
        T[i] = v;
    }
}

// heap membership of the pass-0 seeds: (slot, node) pairs
__global__ void k_pt_setbits(int n, const int* __restrict__ sn, size_t words, uint32_t* __restrict__ bits)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t node = (size_t)sn[2 * i + 1];
    atomicOr(bits + (size_t)sn[2 * i] * words + (node >> 5), 1u << (node & 31));
}

struct PartArgs {
    double* T;
    double* Tprev;
    double* T0;
    uint32_t* hbits;
    const double* slo;
    const double* hx;
    const double* hz;
    double hr;             // radial spacing
    PartGeo p;
    int nslots;
    int fom;
    size_t N, words;
    const int* on;
    int* dsend;
    int* march;
    double* mini;
    int* stamp;
    int* prog;
    const int* flow;
    int spin_limit;        // polls before a wait on a neighbour is given up
    int* chg;
    int* pstart;
    unsigned long long* err;
    size_t nfmax;
    int npx, npz;          // patches per block per axis (the larger block's)
    int iter;              // sweep number
    int maxpass;           // Jacobi passes per layer at most
    unsigned long long* updates;
};

__device__ __forceinline__ bool pt_hbit(const uint32_t* hb, size_t q) { return (hb[q >> 5] >> (q & 31)) & 1u; }

__device__ __forceinline__ size_t pt_idx(const PartGeo& p, int r, int x, int z)
{
    return ((size_t)r * p.n[1] + x) * p.n[2] + z;
}

// ---------------------------------------------------------------- face relaxation

// One octant of a face node's value from ghost face k (F:1100-1400): the ghost
// side of the face axis A always counts (second order iff near ghost > far
// ghost), the other side of that axis is not used; an in-plane neighbour
// counts iff known and below the node (or the node unknown), second order iff
// its second neighbour is known and below it; face updates are mixed order
// whatever the .in file says (F:197-383).  Neighbours beyond the block are out
// of bounds: inf, as no octant.  so, si: the octant's sides (-1, 1) of the
// in-plane axes.
__device__ __forceinline__ double pt_face_octant(const PartArgs& a, const double* __restrict__ P, const double* T, int A,
                                                 int outer, int inner, int side, int so, int si, const int c[3],
                                                 const int lo[3], const int len[3])
{
    const double inf = __builtin_huge_val();
    const ptrdiff_t NL = (ptrdiff_t)a.p.n[1] * a.p.n[2];
    const size_t me = pt_idx(a.p, c[0], c[1], c[2]);
    const double tc = T[me];
    bool ok = true;
    Side<double> sd[3];
    // the values before any is used: their loads are in flight together
    double v1[3], v2[3];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        const ptrdiff_t st = ax == 0 ? NL : ax == 1 ? (ptrdiff_t)a.p.n[2] : 1;
        const int d = ax == A ? side : ax == outer ? so : si;
        const int q1 = c[ax] + d - lo[ax], q2 = c[ax] + 2 * d - lo[ax];
        const bool in1 = ax == A || (q1 >= 0 && q1 < len[ax]), in2 = ax == A || (q2 >= 0 && q2 < len[ax]);
        const double* F = ax == A ? P : T;
        const size_t m1 = in1 ? me + d * st : me, m2 = in2 ? me + 2 * d * st : me;
        v1[ax] = F[m1];
        v2[ax] = F[m2];
        ok = ok && in1;
        v2[ax] = in2 ? v2[ax] : inf;
    }
    const double hx = a.hx[c[0]], hz = a.hz[(size_t)c[0] * a.p.n[1] + c[1]], slown = a.slo[me];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        Side<double>& S = sd[ax];
        if (ax == A) {   // an unknown ghost enters as 0
            S.t1 = v1[ax] < inf ? v1[ax] : 0.0;
            const double gf = v2[ax] < inf ? v2[ax] : 0.0;
            S.ord = S.t1 > gf ? 2 : 1;
            S.t2 = S.ord == 2 ? gf : 0.0;
        } else {
            const bool cnt = v1[ax] < inf && v1[ax] < tc;
            S.ord = cnt ? (v1[ax] > v2[ax] ? 2 : 1) : 0;
            S.t1 = cnt ? v1[ax] : 0.0;
            S.t2 = S.ord == 2 ? v2[ax] : 0.0;
        }
    }
    return ok ? octant_solve<double>(sd[0], sd[1], sd[2], a.hr, hx, hz, slown) : inf;
}

// The faces of every block whose neighbour across them marched in the previous
// pass, one after the other: one workgroup per (slot, block).  In heap order a
// node reads the new value of its in-plane heap neighbours of smaller key, so
// it is ready once they are done.  Dynamic LDS: per node the neighbours (bits)
// it still waits for, the queue of ready nodes in the order they became so,
// and a bit for the nodes in the heap.  A round takes what the round before
// made ready, four lanes a node, each one of its octants; of two neighbours
// one waits for the other, so no round reads a value it writes.  A round of
// some 25 ready nodes is latency: with every thread looking through its own
// nodes for ready ones, each wavefront ran the whole update for one or two
// lanes, and a pass over the eight sources at 31x110x140 took 4840 us in six
// launches, one a face; 493 this way (a face of 3850 nodes: 160).
__global__ void __launch_bounds__(PT_FACE_THREADS) k_pt_face(PartArgs a)
{
    extern __shared__ unsigned pt_lds[];
    __shared__ int cnt[3];   // nodes made ready by the round before, this round, cleared for the next
    const int slot = blockIdx.x >> 3, blk = blockIdx.x & 7;
    if (slot >= a.nslots || !a.on[slot]) return;
    int bc[3];
    pt_coord(blk, bc);
    int lo[3], len[3];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) { lo[ax] = a.p.lo(ax, bc[ax]); len[ax] = a.p.len(ax, bc[ax]); }
    double* T = a.T + (size_t)slot * a.N;
    const double* P = a.Tprev + (size_t)slot * a.N;
    uint32_t* hb = a.hbits + (size_t)slot * a.words;
    const double inf = __builtin_huge_val();
    const int t = threadIdx.x;
    unsigned* dep = pt_lds;                                            // a byte per node
    unsigned* heap = dep + (a.nfmax + 3) / 4;                          // a bit per node
    unsigned short* queue = (unsigned short*)(heap + (a.nfmax + 31) / 32);
    const int NBo[8] = { -1, 1, -2, 2, 0, 0, 0, 0 }, NBi[8] = { 0, 0, 0, 0, -1, 1, -2, 2 };   // q ^ 1: the opposite one
#pragma unroll 1
    for (int k = 0; k < 6; ++k) {
        const int A = PT_FACE_AXIS[k], side = PT_FACE_SIDE[k];
        const int across = (A == 0 ? bc[0] : A == 1 ? bc[1] : bc[2]) + side;
        if (across < 0 || across > 1) continue;
        if (!a.dsend[slot * 8 + (blk ^ (4 >> A))]) continue;
        int outer, inner;
        pt_face_axes(k, outer, inner);
        const int no = outer == 0 ? len[0] : len[1], ni = inner == 1 ? len[1] : len[2], nf = no * ni;
        const int lA = A == 0 ? lo[0] : A == 1 ? lo[1] : lo[2], nA = A == 0 ? len[0] : A == 1 ? len[1] : len[2];
        const int fa = side < 0 ? lA : lA + nA - 1;     // the face plane
        auto node_of = [&](int io, int ii, int plane, int c[3]) {
            c[0] = A == 0 ? plane : lo[0] + io;                                   // the outer axis, unless the face's
            c[1] = A == 1 ? plane : lo[1] + (A == 0 ? io : ii);
            c[2] = A == 2 ? plane : lo[2] + ii;
        };
        auto key_of = [&](int io, int ii) {
            int c[3];
            node_of(io, ii, fa + side, c);
            const double v = P[pt_idx(a.p, c[0], c[1], c[2])];
            return v < inf ? v : 0.0;
        };
        // the heap of this face: nodes whose near ghost is below them (or unknown nodes)
        __syncthreads();
        for (int w = t; w < (nf + 31) / 32; w += PT_FACE_THREADS) heap[w] = 0u;
        for (int w = t; w < (nf + 3) / 4; w += PT_FACE_THREADS) dep[w] = 0u;
        if (t < 3) cnt[t] = 0;
        __syncthreads();
        for (int fi = t; fi < nf; fi += PT_FACE_THREADS) {
            const int io = fi / ni, ii = fi - io * ni;
            int c[3];
            node_of(io, ii, fa, c);
            if (key_of(io, ii) < T[pt_idx(a.p, c[0], c[1], c[2])]) atomicOr(heap + (fi >> 5), 1u << (fi & 31));
        }
        __syncthreads();
        // what each waits for: in-plane heap neighbours (first and second) of smaller (key, index)
        for (int fi = t; fi < nf; fi += PT_FACE_THREADS) {
            if (!((heap[fi >> 5] >> (fi & 31)) & 1u)) continue;
            const int io = fi / ni, ii = fi - io * ni;
            const double ki = key_of(io, ii);
            unsigned m = 0;
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int jo = io + NBo[q], ji = ii + NBi[q];
                if (jo < 0 || jo >= no || ji < 0 || ji >= ni) continue;
                const int fj = jo * ni + ji;
                if (!((heap[fj >> 5] >> (fj & 31)) & 1u)) continue;
                const double kj = key_of(jo, ji);
                if (kj < ki || (kj == ki && fj < fi)) m |= 1u << q;
            }
            if (m) atomicOr(dep + (fi >> 2), m << (8 * (fi & 3)));
            else queue[atomicAdd(cnt, 1)] = (unsigned short)fi;
        }
        // every round but the last takes at least one node
        int head = 0;
#pragma unroll 1
        for (int round = 0, at = 0; round <= nf; ++round) {
            __syncthreads();
            const int tail = head + cnt[at], nx = at == 2 ? 0 : at + 1;
            if (head == tail) break;
            if (t == 0) cnt[nx == 2 ? 0 : nx + 1] = 0;
            for (int e = head + (t >> 2); e < tail; e += PT_FACE_THREADS / 4) {
                const int fi = queue[e], io = fi / ni, ii = fi - io * ni;
                int c[3];
                node_of(io, ii, fa, c);
                const size_t me = pt_idx(a.p, c[0], c[1], c[2]);
                double best = pt_face_octant(a, P, T, A, outer, inner, side, t & 1 ? 1 : -1, t & 2 ? 1 : -1, c, lo, len);
                const double old = T[me];
                best = fmin(best, __shfl_xor(best, 1));
                best = fmin(best, __shfl_xor(best, 2));
                // acceptance as F:1378, strict on the down face (F:2817); unknown old accepts
                const bool acc = (k == 5) ? (old > best || !(old < inf)) : (old >= best || !(old < inf));
                if ((t & 3) == 0 && acc) {
                    T[me] = best;
                    atomicOr(hb + (me >> 5), 1u << (me & 31));
                }
                // two of the neighbours each: those that wait for this node alone are ready
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int q = (t & 3) + 4 * h;
                    const int step = (t & 1 ? 1 : -1) * (t & 2 ? 2 : 1);
                    const int jo = io + (h ? 0 : step), ji = ii + (h ? step : 0);
                    if (jo < 0 || jo >= no || ji < 0 || ji >= ni) continue;
                    const int fj = jo * ni + ji, sh = 8 * (fj & 3);
                    const unsigned bit = 1u << (q ^ 1);
                    const unsigned was = (atomicAnd(dep + (fj >> 2), ~(bit << sh)) >> sh) & 255u;
                    if (was == bit) queue[tail + atomicAdd(cnt + nx, 1)] = (unsigned short)fj;
                }
            }
            head = tail;
            at = nx;
        }
        __threadfence_block();
    }
}

// Per (slot, block): whether any node is in the heap (the block marches this
// pass) and the smallest heap value (F:387-389).  Heap nodes lie on the
// block's faces.
__global__ void __launch_bounds__(256) k_pt_mark(PartArgs a)
{
    __shared__ double s_min[256];
    __shared__ int s_any[256];
    const int slot = blockIdx.x >> 3, blk = blockIdx.x & 7;
    if (slot >= a.nslots || !a.on[slot]) return;
    int bc[3], lo[3], len[3];
    pt_coord(blk, bc);
    for (int ax = 0; ax < 3; ++ax) { lo[ax] = a.p.lo(ax, bc[ax]); len[ax] = a.p.len(ax, bc[ax]); }
    const double* T = a.T + (size_t)slot * a.N;
    const uint32_t* hb = a.hbits + (size_t)slot * a.words;
    double mn = __builtin_huge_val();
    int any = 0;
    for (int f = 0; f < 6; ++f) {
        const int A = PT_FACE_AXIS[f];
        int outer, inner;
        pt_face_axes(f, outer, inner);
        const int plane = PT_FACE_SIDE[f] < 0 ? lo[A] : lo[A] + len[A] - 1;
        const int nf = len[outer] * len[inner];
        for (int fi = threadIdx.x; fi < nf; fi += 256) {
            int c[3];
            c[A] = plane; c[outer] = lo[outer] + fi / len[inner]; c[inner] = lo[inner] + fi % len[inner];
            const size_t q = pt_idx(a.p, c[0], c[1], c[2]);
            if (pt_hbit(hb, q)) { any = 1; mn = fmin(mn, T[q]); }
        }
    }
    s_min[threadIdx.x] = mn;
    s_any[threadIdx.x] = any;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            s_min[threadIdx.x] = fmin(s_min[threadIdx.x], s_min[threadIdx.x + w]);
            s_any[threadIdx.x] |= s_any[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        a.march[slot * 8 + blk] = s_any[0];
        a.mini[slot * 8 + blk] = s_min[0];
    }
}

// The march's starting state for the marching blocks: T0 = -value for heap
// nodes (they pop), +value otherwise (+inf unknown).
__global__ void k_pt_start(PartArgs a)
{
    const size_t total = (size_t)a.nslots * a.N;
    const size_t NL = (size_t)a.p.n[1] * a.p.n[2];
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const size_t s = i / a.N, q = i - s * a.N;
        if (!a.on[s]) continue;
        const int r = (int)(q / NL), x = (int)((q / a.p.n[2]) % a.p.n[1]), z = (int)(q % a.p.n[2]);
        const int blk = ((r >= a.p.cut[0]) << 2) | ((x >= a.p.cut[1]) << 1) | (z >= a.p.cut[2]);
        if (!a.march[s * 8 + blk]) continue;
        const double v = a.T[i];
        a.T0[i] = pt_hbit(a.hbits + s * a.words, q) ? -v : v;
    }
}

// ---------------------------------------------------------------- the march as a relaxation

// Pop-order update (see the file comment).  gather(a) gives axis a's sides
// (inf unknown or outside the block, and whether the first neighbours are
// inside it); t0 the starting value (inf unknown).  Second order on a side iff
// its second neighbour is known and below the first (F:645-707).  tc, the
// value so far, only says which sides to expect: the result depends on the
// neighbours alone.
//
// The joins meet every octant of joined sides when the last of its sides
// joins; an axis is left out of it if one of the axis' sides inside the block
// has not joined by then.  So take the sides below a guess of the result, and
// fin, the least of t0 and the solutions of their octants: if all of them are
// below fin, every one joins, and if every other side is at or above it, none
// follows, and fin is the result to the last bit.  With one side per axis
// taken and every term certain (octant_one), no octant of fewer sides is below
// the octant of all of them: one octant decides.  Otherwise the octants of
// either side of an axis, and those without an axis whose term is not certain,
// are evaluated too.  The guesses are the value so far, then the last fin; a
// node none settles takes the joins one by one.  (Eight sources at 31x110x140,
// two models: 261 and 181 ms with all octants of every join at every node, 124
// and 73 ms with these; with the patches in flow order, 48 and 21 ms where the
// lanes take the octants that any of them needs, 38 and 16 ms each its own.)
template <typename G>
__device__ __forceinline__ double pt_pop_update(int fom, double t0, double tc, G gather, double hr, double hx,
                                                double hz, const double ih[3], double slown)
{
    const double inf = __builtin_huge_val();
    const double h2[3] = { hr * hr, hx * hx, hz * hz }, s2 = slown * slown;
    // the largest (c / H)^2: 9/4
    const double kt = 0x1.2p-38 * (ih[0] * ih[0] + ih[1] * ih[1] + ih[2] * ih[2]), ks = 0x1p-40 * s2;
    double guess = tc < t0 ? tc : t0;
    bool ok = false;
#pragma unroll 1
    for (int attempt = 0; attempt < 4 && !ok; ++attempt) {
        Side<double> p[3];
        double last = -inf, next = inf;   // the latest side taken, the earliest left
        unsigned taken = 0, both = 0;     // axes with a side taken, with two
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const AxisSides<double> g = gather(a);
            const bool lo = g.l1 <= g.h1;
            const double t1 = lo ? g.l1 : g.h1, t2 = lo ? g.l2 : g.h2, o = lo ? g.h1 : g.l1;
            const bool take = t1 < guess, two = o < guess;
            p[a].ord = take ? (fom && t1 > t2 ? 2 : 1) : 0;
            p[a].t1 = take ? t1 : 0.0;
            p[a].t2 = p[a].ord == 2 ? t2 : 0.0;
            const double left = two ? inf : take ? o : t1, got = two ? o : t1;
            next = left < next ? left : next;
            last = take && got > last ? got : last;
            taken |= take ? 1u << a : 0u;
            both |= two ? 1u << a : 0u;
        }
        unsigned weak;
        double T = octant_one(p, h2, s2, kt, ks, &weak);
        double fin = taken && T < t0 ? T : t0;
        weak &= taken;
        if (weak | both) {
            // todo: the octants left, bit (c, d): c the axes whose other side is
            // taken instead, d the axes left out; each lane takes its own.  First
            // those of all taken axes, then the others their weak axes ask for
            unsigned open = weak;
            unsigned long long todo = 0;
#pragma unroll
            for (int c = 1; c < 8; ++c) todo |= (c & ~both) ? 0ull : 1ull << (8 * c);
#pragma unroll 1
            for (bool first = true;;) {
                if (!todo && first) {
                    first = false;
#pragma unroll
                    for (unsigned c = 0; c < 8; ++c)
                        todo |= (c & ~both) ? 0ull
                                            : (unsigned long long)(subsets(open & ~c) & ~(1u | 1u << taken)) << (8 * c);
                }
                if (!todo) break;
                const unsigned m = __ffsll(todo) - 1, c = m >> 3, d = m & 7;
                todo &= todo - 1;
                Side<double> r[3];
                double top = -inf;        // the last of this octant's sides to join, and its place
                int at = -1;
                bool reached = true;
                double before[3];         // per axis left out: when its last side inside the block joins
                asm volatile("" ::: "memory");   // the stencil is read again, not kept
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    const AxisSides<double> g = gather(a);
                    const bool lo = g.l1 <= g.h1, other = (c >> a) & 1, out = (d >> a) & 1;
                    const double o1 = lo ? g.h1 : g.l1, o2 = lo ? g.h2 : g.l2, q1 = lo ? g.l1 : g.h1, q2 = lo ? g.l2 : g.h2;
                    const double t1 = other ? o1 : q1, t2 = other ? o2 : q2;
                    const bool use = ((taken >> a) & 1) && !out;
                    r[a].ord = use ? (fom && t1 > t2 ? 2 : 1) : 0;
                    r[a].t1 = use ? t1 : 0.0;
                    r[a].t2 = r[a].ord == 2 ? t2 : 0.0;
                    if (use && t1 >= top) { top = t1; at = a; }
                    before[a] = !out ? inf : (lo ? g.hin : g.lin) ? ((both >> a) & 1 ? o1 : inf) : q1;
                }
#pragma unroll
                for (int a = 0; a < 3; ++a)
                    if (before[a] < top || (before[a] == top && a < at)) reached = false;
                if (!reached) continue;
                unsigned w;
                T = octant_one(r, h2, s2, kt, ks, &w);
                if (T < fin) fin = T;
                if (first) open |= w & taken;
            }
        }
        ok = last < fin && next >= fin;
        guess = fin;
    }
    if (ok) return guess;
    // the joins, in (value, side) order
    double cur = t0;
    unsigned joined = 0;
#pragma unroll 1
    for (int i = 0; i < 6; ++i) {
        int j = -1;
        double vj = inf;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const AxisSides<double> g = gather(a);
            if (g.l1 < vj && !((joined >> (2 * a)) & 1)) { vj = g.l1; j = 2 * a; }
            if (g.h1 < vj && !((joined >> (2 * a + 1)) & 1)) { vj = g.h1; j = 2 * a + 1; }
        }
        if (j < 0 || !(vj < cur)) break;
        joined |= 1u << j;
        // the octants through side j
#pragma unroll 1
        for (int o = 0; o < 8; ++o) {
            if (((o >> (j >> 1)) & 1) != (j & 1)) continue;
            asm volatile("" ::: "memory");   // the stencil is read again, not kept
            Side<double> p[3];
            bool in = true;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const AxisSides<double> g = gather(a);
                const bool hi = (o >> a) & 1;
                const double t1 = hi ? g.h1 : g.l1, t2 = hi ? g.h2 : g.l2;
                const bool on = (joined >> (2 * a + (hi ? 1 : 0))) & 1;
                in = in && (hi ? g.hin : g.lin);
                p[a].ord = on ? (fom && t1 > t2 ? 2 : 1) : 0;
                p[a].t1 = on ? t1 : 0.0;
                p[a].t2 = p[a].ord == 2 ? t2 : 0.0;
            }
            if (!in) continue;
            unsigned weak;
            const double T = octant_one(p, h2, s2, kt, ks, &weak);
            if (T < cur) cur = T;
        }
    }
    return cur;
}

// One sweep of the march relaxation over the marching blocks: a wavefront
// per (slot, block, 8 x 8 patch column).  Per layer it stages the patch with
// a two-node ring (inside the block; one halo value per lane, no corners) and
// relaxes it with Jacobi passes until a pass changes nothing; a lane keeps the
// two layers its column walked just before and the two ahead in registers.  A
// patch column runs in the first sweep of a pass, or when it or a lateral
// neighbour changed a value in the sweep before.  It waits, layer by layer,
// for its upstream neighbours along the source's lateral flow, so that one
// sweep carries a value through the whole block; the sweeps' order does not
// change where they settle (eight sources at 31x110x140, two models: 140 and
// 101 sweeps, 84 and 56 ms without the waits; 55 and 28 sweeps, 48 and 21 ms
// with them, before each lane took its own octants).
__global__ void __launch_bounds__(64, 4) k_pt_walk(PartArgs a)
{
    constexpr int LZ = Patch8::LZ;
    static_assert(PT_P == Patch8::P, "one node per lane");
    __shared__ double cur[Patch8::SIZE];
    const int ppb = a.npx * a.npz;
    // patch by patch in flow order, over all slots and blocks: the neighbours
    // a patch waits for start before it
    const int sb = blockIdx.x % (8 * a.nslots), slot = sb >> 3, blk = sb & 7, rank = blockIdx.x / (8 * a.nslots);
    if (!a.on[slot] || !a.march[slot * 8 + blk]) return;
    int bc[3], lo[3], len[3];
    pt_coord(blk, bc);
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) { lo[ax] = a.p.lo(ax, bc[ax]); len[ax] = a.p.len(ax, bc[ax]); }
    const int npxb = (len[1] + PT_P - 1) / PT_P, npzb = (len[2] + PT_P - 1) / PT_P;
    const int ri = rank / a.npz, rj = rank % a.npz;
    if (ri >= npxb || rj >= npzb) return;
    const int fx = a.flow[2 * slot] < 0 ? -1 : 1, fz = a.flow[2 * slot + 1] < 0 ? -1 : 1;
    const int pxi = fx > 0 ? ri : npxb - 1 - ri, pzi = fz > 0 ? rj : npzb - 1 - rj, pi = pxi * a.npz + pzi;
    int* pg = a.prog + ((size_t)slot * 8 + blk) * ppb;
    const int iter = a.iter;
    const bool first = iter == a.pstart[slot];
    const int pbase = iter * (a.p.n[0] + 1);
    int* st = a.stamp + ((size_t)slot * 8 + blk) * ppb;
    const int t = threadIdx.x;
    {
        int m = st[pi];
        if (pxi > 0) m = max(m, st[pi - a.npz]);
        if (pxi < npxb - 1) m = max(m, st[pi + a.npz]);
        if (pzi > 0) m = max(m, st[pi - 1]);
        if (pzi < npzb - 1) m = max(m, st[pi + 1]);
        if (!first && __builtin_amdgcn_readfirstlane(m) < iter - 1) {
            // an idle patch is finished with every layer of this sweep
            if (t == 0) __hip_atomic_store(pg + pi, pbase + len[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
    }
    // the upstream neighbours: lanes 0..31 read the theta one's counter, the
    // others the phi one's (done: none there, or no longer waited for)
    constexpr int done = 0x7fffffff;
    int seen_x = ri > 0 ? 0 : done, seen_z = rj > 0 ? 0 : done;
    const int pgo = t < 32 ? (ri > 0 ? pi - fx * a.npz : pi) : rj > 0 ? pi - fz : pi;
    const double inf = __builtin_huge_val();
    const size_t NL = (size_t)a.p.n[1] * a.p.n[2];
    double* T = a.T + (size_t)slot * a.N;
    const double* T0 = a.T0 + (size_t)slot * a.N;
    const double mini = a.mini[slot * 8 + blk];
    const bool down = ((iter - a.pstart[slot]) & 1) != 0;   // the first sweep of a pass walks upward
    const int dn = down ? 1 : -1;
    const int x0 = lo[1] + pxi * PT_P, z0 = lo[2] + pzi * PT_P;
    const int xe = lo[1] + len[1], ze = lo[2] + len[2];        // block ends (exclusive)
    const int lx = t / PT_P, lz = t % PT_P;
    const int gx = x0 + lx, gz = z0 + lz;
    const bool in = gx < xe && gz < ze;
    const size_t coff = in ? (size_t)gx * a.p.n[2] + gz : (size_t)x0 * a.p.n[2] + z0;
    const int own = Patch8::own(lx, lz, in);
    const int hrow = min(gx, xe - 1);
    int ridx;
    size_t roff;
    {
        int hx_, hz_;
        Patch8::halo(t, &hx_, &hz_);
        const int rx = x0 + hx_ - 2, rz = z0 + hz_ - 2;
        const bool ok = rx >= lo[1] && rx < xe && rz >= lo[2] && rz < ze;
        ridx = ok ? Patch8::cell(hx_, hz_) : Patch8::HALO_OUT;
        roff = ok ? (size_t)rx * a.p.n[2] + rz : coff;
    }
    for (int e = t; e < Patch8::SIZE; e += 64) cur[e] = inf;
    const bool inx0 = gx - 1 >= lo[1], inx1 = gx + 1 < xe, inz0 = gz - 1 >= lo[2], inz1 = gz + 1 < ze;
    bool anyv = false;
    unsigned long long nupd = 0;
    const ptrdiff_t step = (ptrdiff_t)dn * (ptrdiff_t)NL;
    int ir = down ? lo[0] : lo[0] + len[0] - 1;
    size_t lay = (size_t)ir * NL;
    double b1 = inf, b2 = inf;   // the walk starts at a block face: nothing before it
    double cv = T[lay + coff], n1 = len[0] > 1 ? T[lay + step + coff] : inf;
    for (int q = 0; q < len[0]; ++q, ir += dn, lay += step) {
        // wait (bounded) until the upstream patches have finished this layer
        const int need = pbase + q + 1;
        for (int spins = 0; min(seen_x, seen_z) < need;) {
            const int v = __hip_atomic_load(pg + pgo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (seen_x != done) seen_x = __builtin_amdgcn_readlane(v, 0);
            if (seen_z != done) seen_z = __builtin_amdgcn_readlane(v, 32);
            if (min(seen_x, seen_z) >= need) break;
            if (++spins > a.spin_limit) {
                if (seen_x < need) seen_x = done;
                if (seen_z < need) seen_z = done;
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        asm volatile("" ::: "memory");   // what follows is read after the wait
        // lateral ring: neighbouring patches of the same block may be writing it
        const double hv = __hip_atomic_load(T + lay + roff, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const double n2 = q + 2 < len[0] ? T[lay + 2 * step + coff] : inf;
        const double s0 = T0[lay + coff];
        const double slown = a.slo[lay + coff];
        const double hzl = a.hz[(size_t)ir * a.p.n[1] + hrow];
        const double hxl = a.hx[ir];
        // fixed: alive at the march's start (a known non-heap node at or below the heap minimum)
        const bool free = in && !(s0 > 0.0 && s0 < inf && s0 <= mini);
        const double t0 = s0 < 0.0 ? -s0 : s0;
        const double ih[3] = { 1.0 / a.hr, 1.0 / hxl, 1.0 / hzl };
        const double orig = cv;
        double tc = cv;
        cur[own] = tc;
        cur[ridx] = hv;
        __builtin_amdgcn_wave_barrier();
        int npass = 0;
#pragma unroll 1
        for (int pass = 0; pass < a.maxpass; ++pass) {
            auto gather = [&](int ax) {
                AxisSides<double> g;
                if (ax == 0) {   // the layers above (ir-1) and below (ir+1)
                    const bool ahead = q + 1 < len[0];
                    g = { down ? b1 : n1, down ? b2 : n2, down ? n1 : b1, down ? n2 : b2, down ? q > 0 : ahead, down ? ahead : q > 0 };
                } else if (ax == 1) {
                    g = { cur[own - LZ], cur[own - 2 * LZ], cur[own + LZ], cur[own + 2 * LZ], inx0, inx1 };
                } else {
                    g = { cur[own - 1], cur[own - 2], cur[own + 1], cur[own + 2], inz0, inz1 };
                }
                return g;
            };
            double nv = tc;
            if (free) nv = pt_pop_update(a.fom, t0, tc, gather, a.hr, hxl, hzl, ih, slown);
            // every lane has read its stencil before any lane writes (one wavefront)
            __builtin_amdgcn_wave_barrier();
            const bool moved = nv != tc;
            cur[own] = nv;
            tc = nv;
            __builtin_amdgcn_wave_barrier();
            ++npass;
            if (!__ballot(moved)) break;
        }
        nupd += (unsigned long long)npass;
        if (tc != orig) __hip_atomic_store(T + lay + coff, tc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__ballot(tc != orig)) anyv = true;
        b2 = b1; b1 = tc;
        cv = n1; n1 = n2;
        // publish the layer once its stores have completed
        __builtin_amdgcn_s_waitcnt(0);
        if (t == 0) __hip_atomic_store(pg + pi, need, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (t != 0) return;
    if (nupd) atomicAdd(a.updates, nupd * (unsigned long long)(min(PT_P, xe - x0) * min(PT_P, ze - z0)));
    if (anyv) {
        st[pi] = iter;
        atomicOr(a.chg + slot, 1);
    }
}

// Largest change of the pass per slot: max |T - Tprev| over the grid with
// unknown values taken as 0, the reference's error_calculate (F:6963-6987).
__global__ void __launch_bounds__(256) k_pt_err(PartArgs a)
{
    __shared__ double s_m[256];
    const int slot = blockIdx.y;
    double m = 0.0;
    if (a.on[slot]) {
        const double* T = a.T + (size_t)slot * a.N;
        const double* P = a.Tprev + (size_t)slot * a.N;
        for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < a.N; i += (size_t)gridDim.x * blockDim.x) {
            const double x = T[i] < __builtin_huge_val() ? T[i] : 0.0;
            const double y = P[i] < __builtin_huge_val() ? P[i] : 0.0;
            m = fmax(m, fabs(x - y));
        }
    }
    s_m[threadIdx.x] = m;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s_m[threadIdx.x] = fmax(s_m[threadIdx.x], s_m[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0 && s_m[0] > 0.0)
        atomicMax(a.err + slot, (unsigned long long)__double_as_longlong(s_m[0]));
}

// per slot: copy the field to Tprev and clear the heap bits (passes continuing)
__global__ void k_pt_pass_begin(PartArgs a)
{
    const size_t total = (size_t)a.nslots * a.N;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const size_t s = i / a.N;
        if (!a.on[s]) continue;
        a.Tprev[i] = a.T[i];
        const size_t q = i - s * a.N;
        if (q < a.words) a.hbits[s * a.words + q] = 0u;
    }
}

// per slot: the blocks that marched this pass send next pass; the pass's
// first sweep number; the change flags cleared
__global__ void k_pt_pass_end(PartArgs a, int next_iter)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.nslots * 8) return;
    const int s = i >> 3;
    if (!a.on[s]) return;
    a.dsend[i] = a.march[i];
    if ((i & 7) == 0) {
        a.pstart[s] = next_iter;
        a.err[s] = 0ull;
    }
}

__global__ void k_pt_fill_int(int* p, size_t n, int v)
{
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_pt_fill_u32(uint32_t* p, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = 0u;
}

}  // namespace

// ---------------------------------------------------------------- host driver

// the block-arithmetic slowness is recomputed before the next partitioned solve
static void part_model_changed(PartState* ps)
{
    if (ps) ps->model = false;
}

static void part_free(PartState* ps)
{
    if (!ps) return;
    (void)hipFree(ps->Tprev); (void)hipFree(ps->T0); (void)hipFree(ps->hbits);
    (void)hipFree(ps->on); (void)hipFree(ps->dsend); (void)hipFree(ps->march); (void)hipFree(ps->mini);
    (void)hipFree(ps->stamp); (void)hipFree(ps->prog); (void)hipFree(ps->flow);
    (void)hipFree(ps->chg); (void)hipFree(ps->pstart); (void)hipFree(ps->err);
    (void)hipFree(ps->seed); (void)hipFree(ps->slo); (void)hipFree(ps->hx); (void)hipFree(ps->hz);
    (void)hipHostFree(ps->h_chg); (void)hipHostFree(ps->h_err);
    delete ps;
}

// Metric tables with each block's offset arithmetic (F:540-543): a node at
// global index k of block b (local index l = k - off + 2, off its first
// global index) has ri = rgor - (off-1) dnr - (l-1) dnr + earth.
static void part_metrics(const Grid& g, const PartGeo& p, std::vector<double>& hx, std::vector<double>& hz)
{
    hx.assign(g.nnr, 0.0);
    hz.assign((size_t)g.nnr * g.nnx, 0.0);
    for (int kr = 0; kr < g.nnr; ++kr) {
        const int off0 = kr >= p.cut[0] ? p.cut[0] + 1 : 1, l0 = kr - off0 + 2;
        const double ri = g.rgor - (off0 - 1) * g.dnr - (l0 - 1) * g.dnr + g.earth;
        hx[kr] = ri * g.dnx;
        for (int kx = 0; kx < g.nnx; ++kx) {
            const int off1 = kx >= p.cut[1] ? p.cut[1] + 1 : 1, l1 = kx - off1 + 2;
            const double sth = sin(g.rgox + (off1 - 1) * g.dnx + (l1 - 1) * g.dnx);
            hz[(size_t)kr * g.nnx + kx] = ri * sth * g.dnz;
        }
    }
}

static int part_prepare(fmm3d_ctx* c, int nsrc)
{
    const Grid& g = c->g;
    const PartGeo p = part_geo(g);
    if (!c->part) c->part = new PartState();
    PartState& ps = *c->part;
    const size_t N = c->N, words = (N + 31) / 32;
    if (!ps.model) {
        if (!ps.slo) {
            HIPCHK(c, dalloc(&ps.slo, N * sizeof(double)));
            HIPCHK(c, dalloc(&ps.hx, (size_t)g.nnr * sizeof(double)));
            HIPCHK(c, dalloc(&ps.hz, (size_t)g.nnr * g.nnx * sizeof(double)));
            HIPCHK(c, hipHostMalloc((void**)&ps.h_chg, 4096 * sizeof(int), hipHostMallocDefault));
            HIPCHK(c, hipHostMalloc((void**)&ps.h_err, 4096 * sizeof(unsigned long long), hipHostMallocDefault));
        }
        std::vector<double> hx, hz;
        part_metrics(g, p, hx, hz);
        HIPCHK(c, hipMemcpy(ps.hx, hx.data(), hx.size() * sizeof(double), hipMemcpyHostToDevice));
        HIPCHK(c, hipMemcpy(ps.hz, hz.data(), hz.size() * sizeof(double), hipMemcpyHostToDevice));
        const long total = (long)N;
        k_pt_gridder<<<(int)std::min<long>((total + 255) / 256, 65536), 256, 0, c->stream>>>(g, p, c->d_velv, ps.slo);
        HIPCHK(c, hipGetLastError());
        HIPCHK(c, hipStreamSynchronize(c->stream));
        ps.model = true;
    }
    if (ps.cap < nsrc) {
        (void)hipFree(ps.Tprev); (void)hipFree(ps.T0); (void)hipFree(ps.hbits);
        (void)hipFree(ps.on); (void)hipFree(ps.dsend); (void)hipFree(ps.march); (void)hipFree(ps.mini);
        (void)hipFree(ps.stamp); (void)hipFree(ps.prog); (void)hipFree(ps.flow);
        (void)hipFree(ps.chg); (void)hipFree(ps.pstart); (void)hipFree(ps.err);
        ps.Tprev = ps.T0 = nullptr; ps.hbits = nullptr; ps.on = ps.dsend = ps.march = nullptr;
        ps.mini = nullptr; ps.stamp = ps.prog = ps.flow = ps.chg = ps.pstart = nullptr; ps.err = nullptr;
        ps.cap = 0;
        size_t nf = 0;
        for (int k = 0; k < 6; ++k) {
            int outer, inner;
            pt_face_axes(k, outer, inner);
            nf = std::max(nf, (size_t)p.len(outer, 0) * p.len(inner, 0));
        }
        ps.nfmax = nf;
        if (nf > 32768) return fail(c, FMM3D_E_ARG, "partitioned solve: block faces of %zu nodes exceed 32768", nf);
        const int npx = (p.len(1, 0) + PT_P - 1) / PT_P, npz = (p.len(2, 0) + PT_P - 1) / PT_P;
        HIPCHK(c, dalloc(&ps.Tprev, (size_t)nsrc * N * sizeof(double)));
        HIPCHK(c, dalloc(&ps.T0, (size_t)nsrc * N * sizeof(double)));
        HIPCHK(c, dalloc(&ps.hbits, (size_t)nsrc * words * sizeof(uint32_t)));
        HIPCHK(c, dalloc(&ps.on, (size_t)nsrc * sizeof(int)));
        HIPCHK(c, dalloc(&ps.dsend, (size_t)nsrc * 8 * sizeof(int)));
        HIPCHK(c, dalloc(&ps.march, (size_t)nsrc * 8 * sizeof(int)));
        HIPCHK(c, dalloc(&ps.mini, (size_t)nsrc * 8 * sizeof(double)));
        HIPCHK(c, dalloc(&ps.stamp, (size_t)nsrc * 8 * npx * npz * sizeof(int)));
        HIPCHK(c, dalloc(&ps.prog, (size_t)nsrc * 8 * npx * npz * sizeof(int)));
        HIPCHK(c, dalloc(&ps.flow, (size_t)nsrc * 2 * sizeof(int)));
        HIPCHK(c, dalloc(&ps.chg, (size_t)nsrc * sizeof(int)));
        HIPCHK(c, dalloc(&ps.pstart, (size_t)nsrc * sizeof(int)));
        HIPCHK(c, dalloc(&ps.err, (size_t)nsrc * sizeof(unsigned long long)));
        ps.cap = nsrc;
    }
    return FMM3D_OK;
}

// The partitioned solve of nsrc bottom faces (host copies in `faces`, device
// copies in c->d_faces) into slots 0 .. nsrc-1 (float64 fields).
static int part_run(fmm3d_ctx* c, int nsrc, const double* faces, int order)
{
    const Grid& g = c->g;
    const PartGeo p = part_geo(g);
    if (nsrc > 4096) return fail(c, FMM3D_E_ARG, "partitioned solve: at most 4096 sources per call");
    for (int a_ = 0; a_ < 3; ++a_)
        if (p.len(a_, 1) < 3)
            return fail(c, FMM3D_E_ARG, "partitioned solve: each of the 2x2x2 blocks needs >= 3 nodes per axis");
    int rc = part_prepare(c, nsrc);
    if (rc) return rc;
    PartState& ps = *c->part;
    const size_t N = c->N, words = (N + 31) / 32, NL = (size_t)g.nnx * g.nnz;
    const int npx = (p.len(1, 0) + PT_P - 1) / PT_P, npz = (p.len(2, 0) + PT_P - 1) / PT_P;
    double* T = (double*)c->sl.T;
    PartArgs a{};
    a.T = T; a.Tprev = ps.Tprev; a.T0 = ps.T0; a.hbits = ps.hbits; a.slo = ps.slo; a.hx = ps.hx; a.hz = ps.hz;
    a.hr = g.dnr; a.p = p; a.nslots = nsrc; a.fom = order == FMM3D_ORDER_MIXED ? 1 : 0; a.N = N; a.words = words;
    a.on = ps.on; a.dsend = ps.dsend; a.march = ps.march; a.mini = ps.mini; a.stamp = ps.stamp;
    a.prog = ps.prog; a.flow = ps.flow; a.spin_limit = c->spin_limit; a.chg = ps.chg;
    a.pstart = ps.pstart; a.err = ps.err; a.nfmax = ps.nfmax; a.npx = npx; a.npz = npz;
    a.maxpass = 16; a.updates = c->d_visits + 1;
    hipStream_t st = c->stream;
    const int gsz = (int)std::min<size_t>(((size_t)nsrc * N + 255) / 256, 65536);
    // pass 0: injection; the bottom block(s) holding the smallest face minimum march from it
    k_pt_inject<<<gsz, 256, 0, st>>>(g.nnr, g.nnx, g.nnz, nsrc, c->d_faces, T);
    k_fill_real<double><<<gsz, 256, 0, st>>>(ps.Tprev, (size_t)nsrc * N, __builtin_huge_val());
    k_pt_fill_u32<<<gsz, 256, 0, st>>>(ps.hbits, (size_t)nsrc * words);
    k_pt_fill_int<<<(nsrc * 8 * npx * npz + 255) / 256, 256, 0, st>>>(ps.stamp, (size_t)nsrc * 8 * npx * npz, -1000);
    k_pt_fill_int<<<(nsrc * 8 * npx * npz + 255) / 256, 256, 0, st>>>(ps.prog, (size_t)nsrc * 8 * npx * npz, 0);
    std::vector<int> flow((size_t)nsrc * 2), march((size_t)nsrc * 8, 0), seeds, on(nsrc, 1), zeros((size_t)nsrc * 8, 0);
    std::vector<double> mini((size_t)nsrc * 8, __builtin_huge_val());
    for (int s = 0; s < nsrc; ++s) {
        const double* f = faces + (size_t)s * NL;
        lateral_flow(g, f, &flow[2 * (size_t)s]);
        int have[4] = { 0, 0, 0, 0 }, seed[4] = { -1, -1, -1, -1 };
        double tmin[4] = { 0, 0, 0, 0 };
        for (int q = 0; q < 4; ++q) {
            const int bx = q >> 1, bz = q & 1;
            for (int ix = p.lo(1, bx); ix < p.lo(1, bx) + p.len(1, bx); ++ix)
                for (int iz = p.lo(2, bz); iz < p.lo(2, bz) + p.len(2, bz); ++iz) {
                    const double v = f[(size_t)ix * g.nnz + iz];
                    if (v > 0.0 && (!have[q] || v < tmin[q])) {
                        tmin[q] = v;
                        have[q] = 1;
                        seed[q] = (int)((size_t)(g.nnr - 1) * NL + (size_t)ix * g.nnz + iz);
                    }
                }
        }
        for (int q = 0; q < 4; ++q) {
            if (!have[q]) continue;
            bool smaller = false;
            for (int o = 0; o < 4; ++o)
                if (have[o] && tmin[q] > tmin[o]) smaller = true;
            if (smaller) continue;
            march[(size_t)s * 8 + 4 + q] = 1;
            seeds.push_back(s);
            seeds.push_back(seed[q]);
        }
    }
    if ((int)seeds.size() / 2 > ps.nseed_cap) {
        (void)hipFree(ps.seed);
        ps.seed = nullptr;
        ps.nseed_cap = 0;
        HIPCHK(c, dalloc(&ps.seed, seeds.size() * sizeof(int)));
        ps.nseed_cap = (int)seeds.size() / 2;
    }
    const int nseed = (int)seeds.size() / 2;
    if (nseed) HIPCHK(c, hipMemcpyAsync(ps.seed, seeds.data(), seeds.size() * sizeof(int), hipMemcpyHostToDevice, st));
    HIPCHK(c, hipMemcpyAsync(ps.flow, flow.data(), flow.size() * sizeof(int), hipMemcpyHostToDevice, st));
    HIPCHK(c, hipMemcpyAsync(ps.march, march.data(), march.size() * sizeof(int), hipMemcpyHostToDevice, st));
    HIPCHK(c, hipMemcpyAsync(ps.mini, mini.data(), mini.size() * sizeof(double), hipMemcpyHostToDevice, st));
    HIPCHK(c, hipMemcpyAsync(ps.on, on.data(), on.size() * sizeof(int), hipMemcpyHostToDevice, st));
    HIPCHK(c, hipMemcpyAsync(ps.dsend, zeros.data(), zeros.size() * sizeof(int), hipMemcpyHostToDevice, st));
    k_pt_fill_int<<<(nsrc + 255) / 256, 256, 0, st>>>(ps.pstart, (size_t)nsrc, 1);
    HIPCHK(c, hipMemsetAsync(ps.err, 0, (size_t)nsrc * sizeof(unsigned long long), st));
    if (nseed) k_pt_setbits<<<(nseed + 255) / 256, 256, 0, st>>>(nseed, ps.seed, words, ps.hbits);
    HIPCHK(c, hipGetLastError());
    // the host vectors above are pageable: the copies must land before they go
    HIPCHK(c, hipStreamSynchronize(st));

    const double tol = (double)1.0e-5f;   // F:6403, a default-real literal
    const int walk_blocks = nsrc * 8 * npx * npz;
    const size_t face_lds = (ps.nfmax + 3) / 4 * 4 + (ps.nfmax + 31) / 32 * 4 + 2 * ps.nfmax;
    int iter = 1;
    long total_sweeps = 0;
    ps.passes.assign(nsrc, 0);
    const int max_pass = 1000;
    for (int pass = 0; pass <= max_pass; ++pass) {
        if (pass > 0) {
            k_pt_pass_begin<<<gsz, 256, 0, st>>>(a);
            k_pt_face<<<nsrc * 8, PT_FACE_THREADS, face_lds, st>>>(a);
            k_pt_mark<<<nsrc * 8, 256, 0, st>>>(a);
        }
        k_pt_start<<<gsz, 256, 0, st>>>(a);
        HIPCHK(c, hipGetLastError());
        // the march: sweeps until one changes nothing in every slot
        for (int sw = 0;; ++sw) {
            if (sw >= 100000) return fail(c, FMM3D_E_NOCONV, "partitioned solve: pass %d did not settle", pass);
            k_pt_fill_int<<<(nsrc + 255) / 256, 256, 0, st>>>(ps.chg, (size_t)nsrc, 0);
            a.iter = iter;
            k_pt_walk<<<walk_blocks, 64, 0, st>>>(a);
            HIPCHK(c, hipGetLastError());
            HIPCHK(c, hipMemcpyAsync(ps.h_chg, ps.chg, nsrc * sizeof(int), hipMemcpyDeviceToHost, st));
            HIPCHK(c, hipStreamSynchronize(st));
            ++iter;
            ++total_sweeps;
            bool any = false;
            for (int s = 0; s < nsrc; ++s) any |= ps.h_chg[s] != 0;
            if (!any) break;
        }
        k_pt_err<<<dim3(64, nsrc), 256, 0, st>>>(a);
        HIPCHK(c, hipMemcpyAsync(ps.h_err, ps.err, nsrc * sizeof(unsigned long long), hipMemcpyDeviceToHost, st));
        HIPCHK(c, hipStreamSynchronize(st));
        int live = 0;
        for (int s = 0; s < nsrc; ++s) {
            if (!on[s]) continue;
            ps.passes[s] = pass;
            double e;
            memcpy(&e, &ps.h_err[s], sizeof e);
            if (!(e > tol)) on[s] = 0;
            live += on[s];
        }
        // blocks that marched send next pass; slots whose change is within the tolerance stop
        k_pt_pass_end<<<(nsrc * 8 + 255) / 256, 256, 0, st>>>(a, iter);
        HIPCHK(c, hipMemcpyAsync(ps.on, on.data(), on.size() * sizeof(int), hipMemcpyHostToDevice, st));
        HIPCHK(c, hipStreamSynchronize(st));
        if (!live) break;
        if (pass == max_pass) return fail(c, FMM3D_E_NOCONV, "partitioned solve: %d passes without settling", max_pass);
    }
    c->stats.sweeps = (int32_t)total_sweeps;
    int mp = 0;
    for (int s = 0; s < nsrc; ++s) mp = std::max(mp, ps.passes[s]);
    c->stats.phase_sweeps[0] = mp;
    return FMM3D_OK;
}
