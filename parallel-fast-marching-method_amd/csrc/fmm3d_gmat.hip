// fmm3d_gmat.hip -- the Frechet matrix G resident on the device and the
// sparse products subinv's subspace step takes with it (subinv.f90:
// 612-620 G^T d, 759-790 G a / Cd then G^T, 829-850 the same for the
// projected matrix).
//
// subinv reads frechet.out into CSR (rows = traveltimes, 1-based columns =
// vertices, subinv.f90:346-399), builds the transpose column by column with
// the rows of a column in ascending order (subinv.f90:457-475), and sums in
// single precision, entry by entry in that order.  Here the CSR is uploaded
// once; the transpose comes from a stable radix sort of the entries by
// column (for rows with ascending columns, the order subinv builds); the
// products run 16 lanes per column (G^T x) or per row (G x / cd), each a
// sequential float32 sum in subinv's order without contraction, so they
// are subinv's numbers.
#include <hip/hip_runtime.h>

#include <stdint.h>
#include <string.h>

#include <cstring>
#include <rocprim/device/device_radix_sort.hpp>

#include <string>
#include <vector>

#include "../../include/fmm3d.h"

struct fmm3d_gmat {
    int device = 0;
    hipStream_t stream = nullptr;
    int64_t nrows = 0, ncols = 0, nnz = 0;
    int64_t* rp = nullptr;      // CSR
    int32_t* col = nullptr;     // 0-based columns
    float* val = nullptr;
    int64_t* cp = nullptr;      // CSC: ncols+1 offsets
    int32_t* row = nullptr;     // rows ascending within a column
    float* tval = nullptr;
    float* x = nullptr;         // staging of one product's input and output
    float* y = nullptr;
    float* cd = nullptr;
    std::string err;
};

namespace {

thread_local std::string g_gmat_err;

int gfail(fmm3d_gmat* m, int code, const std::string& msg)
{
    if (m) m->err = msg;
    else g_gmat_err = msg;
    return code;
}

// the row of every CSR entry
__global__ void k_entry_rows(int64_t nrows, const int64_t* __restrict__ rp, int32_t* __restrict__ erow)
{
    for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < nrows; r += (int64_t)gridDim.x * blockDim.x)
        for (int64_t k = rp[r]; k < rp[r + 1]; ++k) erow[k] = (int32_t)r;
}

// column offsets of the column-sorted entries: cp[c] = first entry of column c
__global__ void k_col_offsets(int64_t nnz, int64_t ncols, const int32_t* __restrict__ scol, int64_t* __restrict__ cp)
{
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k <= nnz; k += (int64_t)gridDim.x * blockDim.x) {
        const int64_t c0 = k == 0 ? -1 : scol[k - 1];
        const int64_t c1 = k == nnz ? ncols : scol[k];
        for (int64_t c = c0 + 1; c <= c1; ++c) cp[c] = k;
    }
}

__global__ void k_gather_t(int64_t nnz, const int32_t* __restrict__ perm, const int32_t* __restrict__ erow,
                           const float* __restrict__ val, int32_t* __restrict__ row, float* __restrict__ tval)
{
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < nnz; k += (int64_t)gridDim.x * blockDim.x) {
        const int32_t e = perm[k];
        row[k] = erow[e];
        tval[k] = val[e];
    }
}

// s + p(lane J of the own 16 lanes), for J = 0 .. 15 in order
template <int J> __device__ __forceinline__ float add16(float s, float p)
{
    if constexpr (J > 0) s = add16<J - 1>(s, p);
    return s + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(p), 0x150 + J, 0xf, 0xf, false));   // row_newbcast:J
}

// The sum of one list's products, its entries k .. k1 - 1 in order: every lane
// of the 16 that share the list gets it (l: the lane's place in them).  They
// load and multiply 64 entries side by side, and each then adds the 64 products
// in order, so only the additions are serial, one instruction for an entry of
// each of the wavefront's four lists.  (An entry past the end adds +0, which
// changes no sum: one that starts from +0 is never -0.)
__device__ __forceinline__ float list_sum16(int64_t k, int64_t k1, int l, const int32_t* __restrict__ idx,
                                            const float* __restrict__ val, const float* __restrict__ x)
{
    float s = 0.0f;
    int32_t c[4];
    float v[4];
    auto fetch = [&](int64_t at) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int64_t e = at + 16 * j + l;
            const bool in = e < k1;
            c[j] = in ? idx[e] : -1;
            v[j] = in ? val[e] : 0.0f;
        }
    };
    fetch(k);
    while (__ballot(k < k1)) {
        float p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) p[j] = c[j] >= 0 ? v[j] * x[c[j]] : 0.0f;
        k += 64;
        fetch(k);   // the next entries are on their way during the sum
#pragma unroll
        for (int j = 0; j < 4; ++j) s = add16<15>(s, p[j]);
    }
    return s;
}

// y(i) = (sum over list i of val(k) x(idx(k)), in list order) / cd(i): G^T x over
// the columns, rows ascending (subinv.f90:612-616), G x / cd over the rows, in
// file order (subinv.f90:759-767).  Sixteen lanes per list.  Bound by latency:
// a list of 250 entries is four rounds of two dependent loads.  15000 x 19683,
// 3.75M entries, G^T x and G x: one thread per list, its loads a list apart,
// 594 and 151 us; one wavefront per list, two instructions an entry, 45 each;
// 23 so.
__global__ void __launch_bounds__(256) k_ordered_sums(int64_t n, const int64_t* __restrict__ ptr, const int32_t* __restrict__ idx,
                                                      const float* __restrict__ val, const float* __restrict__ x,
                                                      const float* __restrict__ cd, float* __restrict__ y)
{
    const int l = threadIdx.x & 15;
    const int64_t step = (int64_t)gridDim.x * 16;
    // the four lists of a wavefront stay together (i0: its first), so that the broadcasts run with all lanes
    for (int64_t i0 = blockIdx.x * (int64_t)16 + (threadIdx.x >> 6) * 4; i0 < n; i0 += step) {
        const int64_t i = i0 + ((threadIdx.x >> 4) & 3);
        int64_t k = 0, k1 = 0;
        if (i < n) { k = ptr[i]; k1 = ptr[i + 1]; }
        const float s = list_sum16(k, k1, l, idx, val, x);
        if (l == 0 && i < n) y[i] = cd ? s / cd[i] : s;
    }
}

// The same where lists are short on average: a lane per list of at most
// SHORT_LIST entries, then the wavefront's longer ones, four at a time.
constexpr int SHORT_LIST = 32;
__global__ void __launch_bounds__(256) k_ordered_sums_short(int64_t n, const int64_t* __restrict__ ptr, const int32_t* __restrict__ idx,
                                                            const float* __restrict__ val, const float* __restrict__ x,
                                                            const float* __restrict__ cd, float* __restrict__ y)
{
    const int lane = threadIdx.x & 63;
    const int64_t step = (int64_t)gridDim.x * 256;
    for (int64_t i0 = blockIdx.x * (int64_t)256 + (threadIdx.x & ~63); i0 < n; i0 += step) {
        const int64_t i = i0 + lane;
        int64_t k = 0, k1 = 0;
        if (i < n) { k = ptr[i]; k1 = ptr[i + 1]; }
        const bool small = k1 - k <= SHORT_LIST;
        if (i < n && small) {
            float s = 0.0f;
            for (int64_t e = k; e < k1; ++e) s = s + val[e] * x[idx[e]];
            y[i] = cd ? s / cd[i] : s;
        }
        for (unsigned long long left = __ballot(!small); left;) {
            // the 16 lanes' list: of those left, as many taken before as lower sixteens
            unsigned long long own = left;
            for (int g = 0; g < 4; ++g) {
                if (g < lane >> 4) own &= own - 1;
                left &= left - 1;
            }
            const int from = own ? __ffsll(own) - 1 : 0;
            const int64_t a = __shfl(k, from), b = __shfl(k1, from);
            const float s = list_sum16(a, own ? b : a, lane & 15, idx, val, x);
            if (own && (lane & 15) == 0) y[i0 + from] = cd ? s / cd[i0 + from] : s;
        }
    }
}

int grid_of(int64_t n) { return (int)std::min<int64_t>((n + 255) / 256, 65536); }

// Lists of fewer than this many entries on average take a lane each.  A call
// with sixteen lanes a list / a lane a list, us: 1,000,000 rows of 2 entries
// 479 / 406, of 4 471 / 437, of 8 479 / 451, 500,000 of 16 254 / 315; the
// columns of 1,000,000, mean 0.1 (few rows of a large model) 322 / 289, 2
// 352 / 311, 8 348 / 346, 16 385 / 517.
constexpr int SHORT_MEAN = 8;

void ordered_sums(hipStream_t st, int64_t n, int64_t nnz, const int64_t* ptr, const int32_t* idx, const float* val,
                  const float* x, const float* cd, float* y)
{
    if (nnz < SHORT_MEAN * n) k_ordered_sums_short<<<grid_of(n), 256, 0, st>>>(n, ptr, idx, val, x, cd, y);
    else k_ordered_sums<<<(int)std::min<int64_t>((n + 15) / 16, 65536), 256, 0, st>>>(n, ptr, idx, val, x, cd, y);
}

}  // namespace

extern "C" const char* fmm3d_gmat_last_error(const fmm3d_gmat* m) { return m ? m->err.c_str() : g_gmat_err.c_str(); }

extern "C" int fmm3d_gmat_create(int device, int64_t nrows, int64_t ncols, const int64_t* row_ptr, const int32_t* cols,
                                 const float* vals, fmm3d_gmat** out)
{
    if (!out || nrows < 0 || ncols <= 0 || !row_ptr) return gfail(nullptr, FMM3D_E_ARG, "fmm3d_gmat_create: bad arguments");
    *out = nullptr;
    const int64_t nnz = row_ptr[nrows];
    if (row_ptr[0] != 0 || nnz < 0 || nnz > INT32_MAX || ncols > INT32_MAX || nrows > INT32_MAX)
        return gfail(nullptr, FMM3D_E_ARG, "fmm3d_gmat_create: row_ptr must start at 0 and hold < 2^31 entries");
    if (nnz > 0 && (!cols || !vals)) return gfail(nullptr, FMM3D_E_ARG, "fmm3d_gmat_create: null entries");
    std::vector<int32_t> c0((size_t)nnz);
    for (int64_t r = 0; r < nrows; ++r) {
        if (row_ptr[r + 1] < row_ptr[r]) return gfail(nullptr, FMM3D_E_ARG, "fmm3d_gmat_create: row_ptr decreases");
        for (int64_t k = row_ptr[r]; k < row_ptr[r + 1]; ++k) {
            if (cols[k] < 1 || cols[k] > ncols)
                return gfail(nullptr, FMM3D_E_ARG, "fmm3d_gmat_create: column " + std::to_string(cols[k]) + " out of 1.." +
                                                       std::to_string(ncols));
            if (k > row_ptr[r] && cols[k] <= cols[k - 1])
                return gfail(nullptr, FMM3D_E_ARG, "fmm3d_gmat_create: columns must ascend within a row");
            c0[k] = cols[k] - 1;
        }
    }
    if (hipSetDevice(device) != hipSuccess) return gfail(nullptr, FMM3D_E_DEVICE, "fmm3d_gmat_create: hipSetDevice failed");
    fmm3d_gmat* m = new fmm3d_gmat();
    m->device = device;
    m->nrows = nrows; m->ncols = ncols; m->nnz = nnz;
    int32_t *erow = nullptr, *iota = nullptr, *perm = nullptr, *scol = nullptr;
    void* tmp = nullptr;
    size_t tmp_bytes = 0;
    const size_t nz = (size_t)std::max<int64_t>(nnz, 1);
    hipError_t e = hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipMalloc(&m->rp, (nrows + 1) * sizeof(int64_t));
    if (e == hipSuccess) e = hipMalloc(&m->col, nz * sizeof(int32_t));
    if (e == hipSuccess) e = hipMalloc(&m->val, nz * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&m->cp, (ncols + 1) * sizeof(int64_t));
    if (e == hipSuccess) e = hipMalloc(&m->row, nz * sizeof(int32_t));
    if (e == hipSuccess) e = hipMalloc(&m->tval, nz * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&m->x, std::max<int64_t>(nrows, ncols) * sizeof(float) + 256);
    if (e == hipSuccess) e = hipMalloc(&m->y, std::max<int64_t>(nrows, ncols) * sizeof(float) + 256);
    if (e == hipSuccess) e = hipMalloc(&m->cd, std::max<int64_t>(nrows, 1) * sizeof(float));
    if (e == hipSuccess) e = hipMalloc(&erow, nz * sizeof(int32_t));
    if (e == hipSuccess) e = hipMalloc(&iota, nz * sizeof(int32_t));
    if (e == hipSuccess) e = hipMalloc(&perm, nz * sizeof(int32_t));
    if (e == hipSuccess) e = hipMalloc(&scol, nz * sizeof(int32_t));
    if (e == hipSuccess) e = hipMemcpyAsync(m->rp, row_ptr, (nrows + 1) * sizeof(int64_t), hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess && nnz) e = hipMemcpyAsync(m->col, c0.data(), nnz * sizeof(int32_t), hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess && nnz) e = hipMemcpyAsync(m->val, vals, nnz * sizeof(float), hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess && nnz) {
        std::vector<int32_t> h((size_t)nnz);
        for (int64_t k = 0; k < nnz; ++k) h[k] = (int32_t)k;
        e = hipMemcpyAsync(iota, h.data(), nnz * sizeof(int32_t), hipMemcpyHostToDevice, m->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(m->stream);   // h is pageable and goes out of scope
    }
    if (e == hipSuccess && nnz) {
        k_entry_rows<<<grid_of(nrows), 256, 0, m->stream>>>(nrows, m->rp, erow);
        e = hipGetLastError();
    }
    // stable sort by column: within a column the entries keep their CSR (row) order
    int bits = 1;
    while (bits < 32 && (int64_t(1) << bits) < ncols) ++bits;
    if (e == hipSuccess && nnz)
        e = rocprim::radix_sort_pairs(nullptr, tmp_bytes, m->col, scol, iota, perm, (size_t)nnz, 0, bits, m->stream);
    if (e == hipSuccess && nnz) e = hipMalloc(&tmp, std::max<size_t>(tmp_bytes, 1));
    if (e == hipSuccess && nnz)
        e = rocprim::radix_sort_pairs(tmp, tmp_bytes, m->col, scol, iota, perm, (size_t)nnz, 0, bits, m->stream);
    if (e == hipSuccess) {
        k_col_offsets<<<grid_of(nnz + 1), 256, 0, m->stream>>>(nnz, ncols, scol, m->cp);
        e = hipGetLastError();
    }
    if (e == hipSuccess && nnz) {
        k_gather_t<<<grid_of(nnz), 256, 0, m->stream>>>(nnz, perm, erow, m->val, m->row, m->tval);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    (void)hipFree(erow); (void)hipFree(iota); (void)hipFree(perm); (void)hipFree(scol); (void)hipFree(tmp);
    if (e != hipSuccess) {
        std::string msg = std::string("fmm3d_gmat_create: ") + hipGetErrorString(e);
        fmm3d_gmat_destroy(m);
        return gfail(nullptr, e == hipErrorOutOfMemory ? FMM3D_E_NOMEM : FMM3D_E_DEVICE, msg);
    }
    *out = m;
    return FMM3D_OK;
}

extern "C" int fmm3d_gmat_destroy(fmm3d_gmat* m)
{
    if (!m) return FMM3D_OK;
    (void)hipSetDevice(m->device);
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    (void)hipFree(m->rp); (void)hipFree(m->col); (void)hipFree(m->val); (void)hipFree(m->cp); (void)hipFree(m->row);
    (void)hipFree(m->tval); (void)hipFree(m->x); (void)hipFree(m->y); (void)hipFree(m->cd);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
    return FMM3D_OK;
}

extern "C" int fmm3d_gmat_gtx(fmm3d_gmat* m, const float* x, float* y)
{
    if (!m || !x || !y) return gfail(m, FMM3D_E_ARG, "fmm3d_gmat_gtx: null argument");
    hipError_t e = hipSetDevice(m->device);
    if (e == hipSuccess && m->nrows) e = hipMemcpyAsync(m->x, x, m->nrows * sizeof(float), hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess) {
        ordered_sums(m->stream, m->ncols, m->nnz, m->cp, m->row, m->tval, m->x, nullptr, m->y);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(y, m->y, m->ncols * sizeof(float), hipMemcpyDeviceToHost, m->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    if (e != hipSuccess) return gfail(m, FMM3D_E_DEVICE, std::string("fmm3d_gmat_gtx: ") + hipGetErrorString(e));
    return FMM3D_OK;
}

extern "C" int fmm3d_gmat_gx(fmm3d_gmat* m, const float* x, const float* cd, float* y)
{
    if (!m || !x || !y) return gfail(m, FMM3D_E_ARG, "fmm3d_gmat_gx: null argument");
    hipError_t e = hipSetDevice(m->device);
    if (e == hipSuccess) e = hipMemcpyAsync(m->x, x, m->ncols * sizeof(float), hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess && cd && m->nrows) e = hipMemcpyAsync(m->cd, cd, m->nrows * sizeof(float), hipMemcpyHostToDevice, m->stream);
    if (e == hipSuccess && m->nrows) {
        ordered_sums(m->stream, m->nrows, m->nnz, m->rp, m->col, m->val, m->x, cd ? m->cd : nullptr, m->y);
        e = hipGetLastError();
    }
    if (e == hipSuccess && m->nrows) e = hipMemcpyAsync(y, m->y, m->nrows * sizeof(float), hipMemcpyDeviceToHost, m->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    if (e != hipSuccess) return gfail(m, FMM3D_E_DEVICE, std::string("fmm3d_gmat_gx: ") + hipGetErrorString(e));
    return FMM3D_OK;
}
