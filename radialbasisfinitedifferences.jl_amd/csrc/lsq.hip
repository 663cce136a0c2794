// lsq.hip -- device kernels of the sparse solve D x = b behind `D \ f` in the
// reference's PDE harness (test/poisson_test.jl:75-121,
// test/mesh_import_test.jl:150): a least-squares solve when D has more rows
// than columns (oversampled collocation, Y != X), a plain solve when square.
//
// The solver is CGLS (conjugate gradients on the normal equations,
// Hestenes-Stiefel form) on the column-equilibrated matrix D~ = D C,
// C = diag(1 / ||D e_j||), with x = x0 + C z.  One iteration is two kernels:
//   1. p = s + (gamma / gamma_old) p,  q = D~ p,              |q|^2
//   2. a = gamma / |q|^2,  z += a p,  r -= a q,  s = D~^T r,  gamma' = |s|^2
// Each product forms the vector it gathers from (p, r) entry by entry as it
// reads it, with the rounding of the stored copy that the kernel also writes.
// D~^T is stored as a CSR of its own, so both products are row gathers with
// no atomics.  The systems are small (3.8 MB of D at 10,201 x 2,601): an
// iteration is bound by its dependent launches, not by bytes.  A kernel leaves
// its block sums of a squared norm in a list that every block of the next one
// adds up in the same order (at most 1,024 values: two loads a thread), so there
// is no fence, counter or last block, the scalars never leave the device and a
// solve is bitwise reproducible.  Four kernels an iteration with a last-block
// sum in the two products took 12 + 5 + 12 + 5 us, 31 us an iteration; the two
// take 4.4 + 4.8 us, 10.3 us an iteration (10,201 x 2,601, 204,020 entries).
//
// For systems whose dense copy fits the device, the direct method writes D
// into a column-major dense array and calls rocSOLVER's QR least-squares
// routine (gels), which gives `\`'s answer to rounding for both shapes.
// rocSOLVER is opened at run time, so the library keeps linking only the HIP
// runtime; without it the direct method reports that it is unsupported.
#include <dlfcn.h>

#include <mutex>

#include <rocblas/rocblas.h>      // types and prototypes only
#include <rocsolver/rocsolver.h>  // (the symbols come from dlsym)

#include "device_common.hpp"
#include "internal.hpp"

namespace rbffd {

__device__ __forceinline__ double wave_sum_f64(double v)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

constexpr int kLsqThreads = 512;

// Sum of v over the block, in every thread (fixed order)
__device__ __forceinline__ double block_sum(double v)
{
    __shared__ double wsum[kLsqThreads / 64];
    v = wave_sum_f64(v);
    __syncthreads();  // wsum may still be read from an earlier sum
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < kLsqThreads / 64; ++w) s += wsum[w];
    return s;
}

__device__ __forceinline__ double list_sum(const double *partial, int n)
{
    double v = 0.0;
    for (int i = threadIdx.x; i < n; i += kLsqThreads) v += partial[i];
    return block_sum(v);
}

// One product of an iteration over CSR rows, G lanes a row: with
// v = x + c y of the pairs uw formed where they are read (one 16-byte load an
// entry: two loads took 203 against 196 us an iteration at 640,000 x 160,000),
// A v and the block sums of its squares to sum_out; v itself is stored too.
//   FIRST: pairs (s, p), v the new p, A v = q, c = gamma / gamma_old (gamma: the
//     sum of sum_in, also kept in *gam; *gam_old is 0 for the first step);
//   else:  pairs (r, q), v the new r, A v = s, c = -gamma / |q|^2 (|q|^2: the sum
//     of sum_in), and z -= c p.
// The outputs are halves of pairs as well: stride 2.
// A wave walks its rows in passes of 64 / G (a wave-uniform loop, so the
// lane-group sums always run with the whole wave).
template <int G, bool FIRST>
__global__ __launch_bounds__(kLsqThreads) void lsq_product_kernel(LsqProduct a)
{
    constexpr int RPW = 64 / G, PRE = 2;
    const long tid = blockIdx.x * (long)kLsqThreads + threadIdx.x, nthreads = (long)gridDim.x * kLsqThreads;
    const int lane = threadIdx.x & 63, sub = lane % G;
    const long base0 = (tid >> 6) * RPW, stride = (nthreads >> 6) * RPW;
    // the first row's first entries do not need c: their chain of loads
    // (row pointer, column, vector) runs beside the sum's (0.5 us of 5.4)
    long p0 = 0, p1 = 0;
    double fv[PRE];
    double2 fx[PRE];
    if (base0 + lane / G < a.rows) { p0 = a.rowptr[base0 + lane / G]; p1 = a.rowptr[base0 + lane / G + 1]; }
#pragma unroll
    for (int e = 0; e < PRE; ++e) {
        const long p = p0 + sub + G * e;
        fv[e] = 0.0;
        fx[e] = double2{0.0, 0.0};
        if (p < p1) {
            fv[e] = a.val[p];
            fx[e] = a.uw[a.col[p]];
        }
    }
    const double total = list_sum(a.sum_in, a.nsum_in);
    double c;
    if constexpr (FIRST) {
        const double old = *a.gam_old;
        c = old > 0.0 ? total / old : 0.0;
        if (blockIdx.x == 0 && threadIdx.x == 0) *a.gam = total;
    } else {
        c = total > 0.0 ? -(*a.gam / total) : 0.0;
    }
    for (long i = tid; i < a.nv; i += nthreads) {
        const double2 x = a.uw[i];
        a.vnew[2 * i] = __builtin_fma(c, x.y, x.x);
    }
    if constexpr (!FIRST)
        for (long i = tid; i < a.nz; i += nthreads) a.z[i] = __builtin_fma(-c, a.p[2 * i], a.z[i]);
    double sq = 0.0;
    for (long base = base0; base < a.rows; base += stride) {
        const long row = base + lane / G;
        const bool live = row < a.rows;
        double acc = 0.0;
        long p = 0, end = 0;
        if (base == base0) {
#pragma unroll
            for (int e = 0; e < PRE; ++e)
                if (p0 + sub + G * e < p1) acc = __builtin_fma(fv[e], __builtin_fma(c, fx[e].y, fx[e].x), acc);
            p = p0 + sub + G * PRE;
            end = p1;
        } else if (live) {
            p = a.rowptr[row] + sub;
            end = a.rowptr[row + 1];
        }
        for (; p < end; p += G) {
            const double2 x = a.uw[a.col[p]];
            acc = __builtin_fma(a.val[p], __builtin_fma(c, x.y, x.x), acc);
        }
        acc = G == 64 ? wave_sum_f64(acc) : group_sum_f64<G == 64 ? 32 : G>(acc);
        if (live && sub == 0) {
            a.y[2 * row] = acc;
            sq = __builtin_fma(acc, acc, sq);
        }
    }
    sq = block_sum(sq);
    if (threadIdx.x == 0) a.sum_out[blockIdx.x] = sq;
}

// *out = the sum of a list of block sums
__global__ __launch_bounds__(kLsqThreads) void lsq_sum_kernel(const double *partial, int n, double *out)
{
    const double s = list_sum(partial, n);
    if (threadIdx.x == 0) *out = s;
}

void launch_lsq_sum(const double *partial, int n, double *out, hipStream_t s)
{
    lsq_sum_kernel<<<1, kLsqThreads, 0, s>>>(partial, n, out);
}

// Lanes per row: two passes or so over an average row.
static int lsq_lanes(long rows, long nnz)
{
    const long avg = rows > 0 ? nnz / rows : 0;
    return avg < 12 ? 8 : (avg < 64 ? 16 : 64);
}

int lsq_blocks(long rows, long nnz)
{
    const long b = (rows * lsq_lanes(rows, nnz) + kLsqThreads - 1) / kLsqThreads;
    return (int)std::max<long>(1, std::min<long>(kLsqBlocks, b));
}

void launch_lsq_product(const LsqProduct &a, long nnz, bool first, hipStream_t s)
{
    const unsigned nb = (unsigned)lsq_blocks(a.rows, nnz);
    const int g = lsq_lanes(a.rows, nnz);
    if (first) {
        if (g == 8) lsq_product_kernel<8, true><<<nb, kLsqThreads, 0, s>>>(a);
        else if (g == 16) lsq_product_kernel<16, true><<<nb, kLsqThreads, 0, s>>>(a);
        else lsq_product_kernel<64, true><<<nb, kLsqThreads, 0, s>>>(a);
    } else {
        if (g == 8) lsq_product_kernel<8, false><<<nb, kLsqThreads, 0, s>>>(a);
        else if (g == 16) lsq_product_kernel<16, false><<<nb, kLsqThreads, 0, s>>>(a);
        else lsq_product_kernel<64, false><<<nb, kLsqThreads, 0, s>>>(a);
    }
}

// ---- set-up and finish
// row_of[p] = row of CSR entry p
__global__ void row_of_kernel(const int64_t *rowptr, long M, int *row_of)
{
    const long r = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (r >= M) return;
    for (long p = rowptr[r]; p < rowptr[r + 1]; ++p) row_of[p] = (int)r;
}

void launch_row_of(const int64_t *rowptr, long M, int *row_of, hipStream_t s)
{
    if (M > 0) row_of_kernel<<<(unsigned)((M + 255) / 256), 256, 0, s>>>(rowptr, M, row_of);
}

// dst[i] = src[idx[i]]
__global__ void gather_i32_kernel(const int *src, const int *idx, long n, int *dst)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[idx[i]];
}

void launch_gather_i32(const int *src, const int *idx, long n, int *dst, hipStream_t s)
{
    if (n > 0) gather_i32_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(src, idx, n, dst);
}

// scale[j] = 1 / ||row j of the transpose|| (0 for an empty or all-zero column)
__global__ void col_scale_kernel(const int64_t *tptr, long N, const double *tval, double *scale)
{
    const long j = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (j >= N) return;
    double s = 0.0;
    for (long p = tptr[j]; p < tptr[j + 1]; ++p) s = __builtin_fma(tval[p], tval[p], s);
    scale[j] = s > 0.0 ? 1.0 / __builtin_sqrt(s) : 0.0;
}

void launch_col_scale(const int64_t *tptr, long N, const double *tval, double *scale, hipStream_t s)
{
    if (N > 0) col_scale_kernel<<<(unsigned)((N + 255) / 256), 256, 0, s>>>(tptr, N, tval, scale);
}

// out[p] = v[p] * scale[col[p]]
__global__ void scale_cols_kernel(const int *col, long nnz, const double *scale, const double *v, double *out)
{
    const long p = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (p < nnz) out[p] = v[p] * scale[col[p]];
}

void launch_scale_cols(const int *col, long nnz, const double *scale, const double *v, double *out, hipStream_t s)
{
    if (nnz > 0) scale_cols_kernel<<<(unsigned)((nnz + 255) / 256), 256, 0, s>>>(col, nnz, scale, v, out);
}

// out = (x, 0) pairs
__global__ void lsq_pair_kernel(const double *x, long n, double2 *out)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) out[i] = double2{x[i], 0.0};
}

void launch_lsq_pair(const double *x, long n, double2 *out, hipStream_t s)
{
    if (n > 0) lsq_pair_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(x, n, out);
}

// y = x (n entries)
__global__ void copy_f64_kernel(const double *x, long n, double *y)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) y[i] = x[i];
}

void launch_copy_f64(const double *x, long n, double *y, hipStream_t s)
{
    if (n > 0) copy_f64_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(x, n, y);
}

// x[j] += scale[j] * z[j]
__global__ void lsq_finish_kernel(long N, const double *scale, const double *z, double *x)
{
    const long j = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (j < N) x[j] = __builtin_fma(scale[j], z[j], x[j]);
}

void launch_lsq_finish(long N, const double *scale, const double *z, double *x, hipStream_t s)
{
    if (N > 0) lsq_finish_kernel<<<(unsigned)((N + 255) / 256), 256, 0, s>>>(N, scale, z, x);
}

__global__ void fill_f64_kernel(double *p, long n, double v)
{
    const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

void launch_fill_f64(double *p, long n, double v, hipStream_t s)
{
    if (n > 0) fill_f64_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(p, n, v);
}

// ---- direct method
// A (column-major, leading dimension M) += the entries of CSR row r
__global__ void densify_kernel(long M, const int64_t *rowptr, const int *col, const double *val, double *A)
{
    const long r = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (r >= M) return;
    for (long p = rowptr[r]; p < rowptr[r + 1]; ++p) A[(long)col[p] * M + r] += val[p];
}

namespace {

struct SolverLib {
    decltype(&rocblas_create_handle) create = nullptr;
    decltype(&rocblas_destroy_handle) destroy = nullptr;
    decltype(&rocblas_set_stream) set_stream = nullptr;
    decltype(&rocsolver_dgels) dgels = nullptr;
};

const SolverLib *solver_lib()
{
    static std::once_flag once;
    static SolverLib lib;
    std::call_once(once, [] {
        void *hb = dlopen("librocblas.so.5", RTLD_NOW | RTLD_LOCAL);
        if (!hb) hb = dlopen("/opt/rocm/lib/librocblas.so.5", RTLD_NOW | RTLD_LOCAL);
        void *hs = dlopen("librocsolver.so.0", RTLD_NOW | RTLD_LOCAL);
        if (!hs) hs = dlopen("/opt/rocm/lib/librocsolver.so.0", RTLD_NOW | RTLD_LOCAL);
        if (!hb || !hs) return;
        SolverLib l;
        l.create = (decltype(l.create))dlsym(hb, "rocblas_create_handle");
        l.destroy = (decltype(l.destroy))dlsym(hb, "rocblas_destroy_handle");
        l.set_stream = (decltype(l.set_stream))dlsym(hb, "rocblas_set_stream");
        l.dgels = (decltype(l.dgels))dlsym(hs, "rocsolver_dgels");
        if (l.create && l.destroy && l.set_stream && l.dgels) lib = l;
    });
    return lib.dgels ? &lib : nullptr;
}

}  // namespace

bool dense_solver_available() { return solver_lib() != nullptr; }

void dense_solver_destroy(void *handle)
{
    const SolverLib *L = solver_lib();
    if (L && handle) (void)L->destroy((rocblas_handle)handle);
}

int dense_lsq(void **handle, long M, long N, const int64_t *rowptr, const int *col, const double *vals,
              const double *b, double *x, double *A, double *B, int *info, hipStream_t s)
{
    const SolverLib *L = solver_lib();
    if (!L) throw Error{2, "solve: the direct method needs rocSOLVER (librocsolver.so.0), which did not load"};
    if (!*handle) {
        rocblas_handle h = nullptr;
        if (L->create(&h) != rocblas_status_success) throw Error{3, "solve: rocblas_create_handle failed"};
        *handle = h;
    }
    rocblas_handle h = (rocblas_handle)*handle;
    if (L->set_stream(h, s) != rocblas_status_success) throw Error{3, "solve: rocblas_set_stream failed"};
    launch_fill_f64(A, M * N, 0.0, s);
    densify_kernel<<<(unsigned)((M + 255) / 256), 256, 0, s>>>(M, rowptr, col, vals, A);
    launch_copy_f64(b, M, B, s);
    RBFFD_HIP(hipGetLastError());
    const rocblas_status st = L->dgels(h, rocblas_operation_none, (rocblas_int)M, (rocblas_int)N, 1, A,
                                       (rocblas_int)M, B, (rocblas_int)M, info);
    if (st != rocblas_status_success) throw Error{3, "solve: rocsolver_dgels failed (status " + std::to_string((int)st) + ")"};
    launch_copy_f64(B, N, x, s);
    int hinfo = 0;
    RBFFD_HIP(hipMemcpyAsync(&hinfo, info, sizeof(int), hipMemcpyDeviceToHost, s));
    RBFFD_HIP(hipStreamSynchronize(s));
    return hinfo;
}

// A X = I by QR: X = inv(A)
__global__ void identity_kernel(long n, double *X)
{
    const long e = blockIdx.x * (long)blockDim.x + threadIdx.x;
    if (e < n * n) X[e] = (e % (n + 1) == 0) ? 1.0 : 0.0;
}

int dense_inverse(void **handle, long n, double *Aw, double *Ainv, int *info, hipStream_t s)
{
    const SolverLib *L = solver_lib();
    if (!L) throw Error{2, "inverse: needs rocSOLVER (librocsolver.so.0), which did not load"};
    if (!*handle) {
        rocblas_handle h = nullptr;
        if (L->create(&h) != rocblas_status_success) throw Error{3, "inverse: rocblas_create_handle failed"};
        *handle = h;
    }
    rocblas_handle h = (rocblas_handle)*handle;
    if (L->set_stream(h, s) != rocblas_status_success) throw Error{3, "inverse: rocblas_set_stream failed"};
    identity_kernel<<<(unsigned)((n * n + 255) / 256), 256, 0, s>>>(n, Ainv);
    RBFFD_HIP(hipGetLastError());
    const rocblas_status st = L->dgels(h, rocblas_operation_none, (rocblas_int)n, (rocblas_int)n, (rocblas_int)n, Aw,
                                       (rocblas_int)n, Ainv, (rocblas_int)n, info);
    if (st != rocblas_status_success) throw Error{3, "inverse: rocsolver_dgels failed (status " + std::to_string((int)st) + ")"};
    int hinfo = 0;
    RBFFD_HIP(hipMemcpyAsync(&hinfo, info, sizeof(int), hipMemcpyDeviceToHost, s));
    RBFFD_HIP(hipStreamSynchronize(s));
    return hinfo;
}

}  // namespace rbffd
