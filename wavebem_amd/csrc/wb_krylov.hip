// wb_krylov.hip -- Arnoldi building blocks for one or several GMRES instances.
//
// Vectors are split into chunks of KCHUNK entries, one workgroup per chunk; reductions
// produce one partial per chunk and are finished, in chunk order, by the consumer, so every
// result is deterministic.  blockIdx.y selects the instance (right-hand side) of a batch;
// each instance has its own Krylov basis, work vector and partials at the given strides, and
// an optional activity flag lets converged instances sit out.
//
// Orthogonalization is classical Gram-Schmidt with one re-orthogonalization pass (CGS2):
//   h1 = V^T z, z -= V h1, h2 = V^T z, z -= V h2, h = h1 + h2, s = |z|, v_new = z / s
// (dot_partials, then update_dot twice, then finalize); it spans the same Krylov space as
// the modified Gram-Schmidt of deal.II's SolverGMRES with two global reductions per step.
// The chunk partials of a pass are summed by every workgroup of the next kernel, in one
// fixed order (reduce_partials), which saves a launch per reduction (8 instances at 61k
// and about 8 basis vectors: 11.7 us for the pass, against 7.4 + 10.7 us with the sums in a
// kernel of their own).
#include "wb_internal.h"

namespace wb {

namespace {

constexpr int KTHREADS = 256;
constexpr int KPER = 1;  // 256-entry chunks: about n/256 workgroups per reduction
constexpr int KCHUNK = KTHREADS * KPER;

__device__ __forceinline__ double ksum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

template <typename T>
__device__ void chunk_dots(const T *__restrict__ V, size_t ldv, int kcount,
                           const T *__restrict__ zs /*LDS chunk*/, int base, int m,
                           double *__restrict__ P, int part)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int k = wave; k < kcount; k += KTHREADS / 64) {
        const T *vk = V + (size_t)k * ldv + base;
        double s = 0.0;
        for (int e = lane; e < m; e += 64) s += (double)vk[e] * (double)zs[e];
        s = ksum(s);
        if (lane == 0) P[(size_t)part * KMAX + k] = s;
    }
}

template <typename T>
__global__ __launch_bounds__(KTHREADS) void k_dot_partials(const T *__restrict__ V, size_t ldv,
                                                           size_t sV, int kcount,
                                                           const T *__restrict__ z, size_t sZ,
                                                           int n, double *__restrict__ P,
                                                           const int *__restrict__ active)
{
    __shared__ T zs[KCHUNK];
    const int b = blockIdx.y;
    if (active && !active[b]) return;
    V += b * sV;
    z += b * sZ;
    P += (size_t)b * gridDim.x * KMAX;
    const int base = blockIdx.x * KCHUNK;
    const int m = min(KCHUNK, n - base);
    for (int e = threadIdx.x; e < KCHUNK; e += KTHREADS) zs[e] = e < m ? z[base + e] : (T)0;
    __syncthreads();
    chunk_dots(V, ldv, kcount, zs, base, m, P, blockIdx.x);
}

// h[k] = sum over the nparts chunk partials P[p][k] (k < kcount), by one workgroup:
// with kw = kcount rounded up to a power of two, thread (k, q) = (t % kw, t / kw) sums
// every (KTHREADS / kw)-th partial from q on, and the KTHREADS / kw sums of each k are then
// added in q order.  The order depends only on kcount and nparts, so every workgroup that
// runs it gets the same bits.
__device__ __forceinline__ void reduce_partials(int kcount, const double *__restrict__ P,
                                                int nparts, double *red /*LDS, KTHREADS*/,
                                                double *h /*LDS, KMAX*/)
{
    int kw = 1;
    while (kw < kcount) kw <<= 1;
    const int nq = KTHREADS / kw;
    const int k = threadIdx.x % kw, q = threadIdx.x / kw;
    double s0 = 0.0, s1 = 0.0;
    if (k < kcount) {
        int p = q;
        for (; p + nq < nparts; p += 2 * nq) {
            s0 += P[(size_t)p * KMAX + k];
            s1 += P[(size_t)(p + nq) * KMAX + k];
        }
        if (p < nparts) s0 += P[(size_t)p * KMAX + k];
    }
    red[threadIdx.x] = s0 + s1;
    __syncthreads();
    if ((int)threadIdx.x < kcount) {
        double t = red[threadIdx.x];
        for (int j = 1; j < nq; ++j) t += red[j * kw + threadIdx.x];
        h[threadIdx.x] = t;
    }
}

// z -= V h;  then optional partial dots (Pout) and partial |z|^2 (normp).  h is formed here
// from the nparts chunk partials Pin of the previous pass by every workgroup
// (reduce_partials), workgroup 0 also storing it to hsave.
template <typename T>
__global__ __launch_bounds__(KTHREADS) void k_update_dot(const T *__restrict__ V, size_t ldv,
                                                         size_t sV, int kcount,
                                                         size_t sH, T *__restrict__ z,
                                                         size_t sZ, int n,
                                                         double *__restrict__ Pout,
                                                         double *__restrict__ normp,
                                                         const int *__restrict__ active,
                                                         const double *__restrict__ Pin,
                                                         double *__restrict__ hsave)
{
    __shared__ double h[KMAX];
    __shared__ T zs[KCHUNK];
    __shared__ double red[KTHREADS / 64];
    __shared__ double rpart[KTHREADS];
    const int b = blockIdx.y;
    if (active && !active[b]) return;
    const int nparts = gridDim.x;
    V += b * sV;
    z += b * sZ;
    if (Pout) Pout += (size_t)b * nparts * KMAX;
    if (normp) normp += (size_t)b * nparts;
    const int base = blockIdx.x * KCHUNK;
    const int m = min(KCHUNK, n - base);
    reduce_partials(kcount, Pin + (size_t)b * nparts * KMAX, nparts, rpart, h);
    __syncthreads();
    if (blockIdx.x == 0)
        for (int k = threadIdx.x; k < kcount; k += KTHREADS) hsave[b * sH + k] = h[k];
    double nrm = 0.0;
    for (int e = threadIdx.x; e < KCHUNK; e += KTHREADS) {
        T v = (T)0;
        if (e < m) {
            double a = (double)z[base + e];
            for (int k = 0; k < kcount; ++k) a -= h[k] * (double)V[(size_t)k * ldv + base + e];
            v = (T)a;
            z[base + e] = v;
            nrm += (double)v * (double)v;
        }
        zs[e] = v;
    }
    __syncthreads();
    if (Pout) chunk_dots(V, ldv, kcount, zs, base, m, Pout, blockIdx.x);
    if (normp) {
        nrm = ksum(nrm);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = nrm;
        __syncthreads();
        if (threadIdx.x == 0) {
            double s = 0.0;
            for (int w = 0; w < KTHREADS / 64; ++w) s += red[w];
            normp[blockIdx.x] = s;
        }
    }
}

// hmap[k] = h1[k] + h2[k] (k < kcount), hmap[kcount] = sqrt(sum Pn); vout = z / hmap[kcount].
// Every workgroup forms the norm itself, wavefront-parallel and in the same order.
// hmap is coherent pinned host memory (instance b at sHmap entries): every thread of
// workgroup 0 writes its entries and fences at system scope, then thread 0 publishes seq
// after them, so a host that reads seq (acquire) sees the column.
// With xcl (single instance), vout is also written to xcl[pos[i]] (FP32).
template <typename T>
__global__ __launch_bounds__(KTHREADS) void k_finalize(int kcount, const double *__restrict__ h1,
                                                       const double *__restrict__ h2,
                                                       size_t sHin,
                                                       const double *__restrict__ Pn, int nparts,
                                                       const T *__restrict__ z, size_t sZ,
                                                       int n, T *__restrict__ vout, size_t sV,
                                                       const int *__restrict__ active,
                                                       double *__restrict__ hmap,
                                                       unsigned long long *__restrict__ hseq,
                                                       unsigned long long seq,
                                                       float *__restrict__ xcl,
                                                       const int *__restrict__ pos,
                                                       size_t sHmap)
{
    __shared__ double snorm;
    const int b = blockIdx.y;
    if (active && !active[b]) return;
    if (h1) h1 += b * sHin;
    if (h2) h2 += b * sHin;
    Pn += (size_t)b * nparts;
    z += b * sZ;
    if (vout) vout += b * sV;
    hmap += b * sHmap;
    hseq += b * sHmap;
    if (threadIdx.x < 64) {
        double s = 0.0;
        for (int p = threadIdx.x; p < nparts; p += 64) s += Pn[p];
        s = ksum(s);
        if (threadIdx.x == 0) snorm = sqrt(s);
    }
    __syncthreads();
    const double nv = snorm;
    if (blockIdx.x == 0) {
        for (int k = threadIdx.x; k < kcount; k += KTHREADS)
            hmap[k] = (h1 ? h1[k] : 0.0) + (h2 ? h2[k] : 0.0);
        if (threadIdx.x == 0) hmap[kcount] = nv;
        __threadfence_system();
        __syncthreads();
        if (threadIdx.x == 0)
            __hip_atomic_store(hseq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (vout) {
        const double inv = nv > 0 ? 1.0 / nv : 0.0;
        const int base = blockIdx.x * KCHUNK;
        const int m = min(KCHUNK, n - base);
        for (int e = threadIdx.x; e < m; e += KTHREADS) {
            const T v = (T)((double)z[base + e] * inv);
            vout[base + e] = v;
            if (xcl) {
                const int ps = pos[base + e];
                if (ps >= 0) xcl[ps] = (float)v;
            }
        }
    }
}

// One Arnoldi step of a small problem in one workgroup: both passes, the norm, the new
// basis vector and the publication (as k_dot_partials, k_update_dot twice and k_finalize, with
// the same roundings of z; the sums of a dot are formed by one wavefront in a fixed order).
// One launch in place of four, which cost about 5 us each whatever the size; the basis is
// read four times through one CU, so only up to ARNOLDI1_BYTES of it (launch_arnoldi1).
constexpr int A1_THREADS = 1024;

template <typename T>
__global__ __launch_bounds__(A1_THREADS) void k_arnoldi1(
    const T *__restrict__ V, size_t ldv, int kcount, const T *__restrict__ z, int n,
    T *__restrict__ vout, double *__restrict__ hmap,
    unsigned long long *__restrict__ hseq, unsigned long long seq, float *__restrict__ xcl,
    const int *__restrict__ pos)
{
    __shared__ T zs[ARNOLDI1_MAX_N];
    __shared__ double h[2][KMAX];
    __shared__ double red[A1_THREADS / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int e = tid; e < n; e += A1_THREADS) zs[e] = z[e];
    double nrm = 0.0;
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
        __syncthreads();
        for (int k = wave; k < kcount; k += A1_THREADS / 64) {
            const T *vk = V + (size_t)k * ldv;
            double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
            int e = lane;
            for (; e + 192 < n; e += 256) {
                s0 += (double)vk[e] * (double)zs[e];
                s1 += (double)vk[e + 64] * (double)zs[e + 64];
                s2 += (double)vk[e + 128] * (double)zs[e + 128];
                s3 += (double)vk[e + 192] * (double)zs[e + 192];
            }
            for (; e < n; e += 64) s0 += (double)vk[e] * (double)zs[e];
            const double s = ksum((s0 + s1) + (s2 + s3));
            if (lane == 0) h[pass][k] = s;
        }
        __syncthreads();
        for (int e = tid; e < n; e += A1_THREADS) {
            double a = (double)zs[e];
            for (int k = 0; k < kcount; ++k) a -= h[pass][k] * (double)V[(size_t)k * ldv + e];
            const T v = (T)a;
            zs[e] = v;
            if (pass == 1) nrm += (double)v * (double)v;
        }
    }
    nrm = ksum(nrm);
    if (lane == 0) red[wave] = nrm;
    __syncthreads();
    double t = 0.0;
    for (int w = 0; w < A1_THREADS / 64; ++w) t += red[w];
    const double nv = sqrt(t);
    for (int k = tid; k <= kcount; k += A1_THREADS)
        hmap[k] = k < kcount ? h[0][k] + h[1][k] : nv;
    __threadfence_system();
    __syncthreads();
    if (tid == 0) __hip_atomic_store(hseq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    const double inv = nv > 0 ? 1.0 / nv : 0.0;
    for (int e = tid; e < n; e += A1_THREADS) {
        const T v = (T)((double)zs[e] * inv);
        vout[e] = v;
        if (xcl) {
            const int ps = pos[e];
            if (ps >= 0) xcl[ps] = (float)v;
        }
    }
}

// x += sum_i y_i v_i   (x may be double while V is float)
struct Coefficients {
    double v[KMAX];
};

template <typename T, typename TX>
__global__ void k_axpy_basis(const T *__restrict__ V, size_t ldv, int kcount, Coefficients y,
                             TX *__restrict__ x, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double a = (double)x[i];
    for (int k = 0; k < kcount; ++k) a += y.v[k] * (double)V[(size_t)k * ldv + i];
    x[i] = (TX)a;
}

template <typename T>
__global__ __launch_bounds__(KTHREADS) void k_norm2_partials(const T *__restrict__ x, size_t sX,
                                                             int n, double *__restrict__ P,
                                                             const int *__restrict__ active)
{
    __shared__ double red[KTHREADS / 64];
    const int b = blockIdx.y;
    if (active && !active[b]) return;
    x += b * sX;
    P += (size_t)b * gridDim.x;
    const int base = blockIdx.x * KCHUNK;
    const int m = min(KCHUNK, n - base);
    double s = 0.0;
    for (int e = threadIdx.x; e < m; e += KTHREADS) {
        const double v = (double)x[base + e];
        s += v * v;
    }
    s = ksum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < KTHREADS / 64; ++w) t += red[w];
        P[blockIdx.x] = t;
    }
}

}  // namespace

int krylov_partials_blocks(int n) { return (n + KCHUNK - 1) / KCHUNK; }

void launch_dot_partials(int is_float, const void *V, size_t ldv, int kcount, const void *z,
                         int n, double *P, hipStream_t s, int batch, size_t sV, size_t sZ,
                         const int *active)
{
    dim3 grid(krylov_partials_blocks(n), batch);
    if (is_float)
        hipLaunchKernelGGL(k_dot_partials<float>, grid, dim3(KTHREADS), 0, s, (const float *)V,
                           ldv, sV, kcount, (const float *)z, sZ, n, P, active);
    else
        hipLaunchKernelGGL(k_dot_partials<double>, grid, dim3(KTHREADS), 0, s, (const double *)V,
                           ldv, sV, kcount, (const double *)z, sZ, n, P, active);
}

void launch_update_dot(int is_float, const void *V, size_t ldv, int kcount, void *z, int n,
                       const double *Pin, double *hsave, double *Pout, double *normp,
                       hipStream_t s, int batch, size_t sV, size_t sZ, size_t sH,
                       const int *active)
{
    dim3 grid(krylov_partials_blocks(n), batch);
    if (is_float)
        hipLaunchKernelGGL(k_update_dot<float>, grid, dim3(KTHREADS), 0, s, (const float *)V,
                           ldv, sV, kcount, sH, (float *)z, sZ, n, Pout, normp, active, Pin,
                           hsave);
    else
        hipLaunchKernelGGL(k_update_dot<double>, grid, dim3(KTHREADS), 0, s, (const double *)V,
                           ldv, sV, kcount, sH, (double *)z, sZ, n, Pout, normp, active, Pin,
                           hsave);
}

void launch_finalize(int is_float, int kcount, const double *h1, const double *h2,
                     const double *Pn, void *z, int n, void *vout, double *hmap,
                     unsigned long long *hseq, unsigned long long seq, hipStream_t s, int batch,
                     size_t sZ, size_t sV, size_t sHin, size_t sHmap, const int *active,
                     float *xcl, const int *pos)
{
    // without a new vector one workgroup per instance has all there is to do
    const int parts = krylov_partials_blocks(n);
    dim3 grid(vout ? parts : 1, batch);
    if (is_float)
        hipLaunchKernelGGL(k_finalize<float>, grid, dim3(KTHREADS), 0, s, kcount, h1, h2, sHin,
                           Pn, parts, (const float *)z, sZ, n, (float *)vout, sV, active, hmap,
                           hseq, seq, xcl, pos, sHmap);
    else
        hipLaunchKernelGGL(k_finalize<double>, grid, dim3(KTHREADS), 0, s, kcount, h1, h2, sHin,
                           Pn, parts, (const double *)z, sZ, n, (double *)vout, sV, active,
                           hmap, hseq, seq, (float *)nullptr, pos, sHmap);
}

// Whether an Arnoldi step with kcount basis vectors goes to k_arnoldi1: the basis it reads
// four times through one CU stays within ARNOLDI1_BYTES.  Steps of the FP32-IR solve, limits
// of 40, 160 and 400 KB: 2.10, 2.08, 2.11 ms at 1,083 dofs (2.41 with four launches always),
// 2.63, 2.58, 2.60 at 2,915 (2.81); FP64 at 2,915 2.15, 2.14, 2.21 (2.19).
bool arnoldi1_fits(int is_float, int kcount, int n)
{
    return n <= ARNOLDI1_MAX_N && (size_t)kcount * n * (is_float ? 4 : 8) <= ARNOLDI1_BYTES;
}

void launch_arnoldi1(int is_float, const void *V, size_t ldv, int kcount, const void *z, int n,
                     void *vout, double *hmap, unsigned long long *hseq,
                     unsigned long long seq, hipStream_t s, float *xcl, const int *pos)
{
    if (is_float)
        hipLaunchKernelGGL(k_arnoldi1<float>, dim3(1), dim3(A1_THREADS), 0, s, (const float *)V,
                           ldv, kcount, (const float *)z, n, (float *)vout, hmap, hseq, seq,
                           xcl, pos);
    else
        hipLaunchKernelGGL(k_arnoldi1<double>, dim3(1), dim3(A1_THREADS), 0, s,
                           (const double *)V, ldv, kcount, (const double *)z, n, (double *)vout,
                           hmap, hseq, seq, (float *)nullptr, pos);
}

void launch_axpy_basis(int is_float, const void *V, size_t ldv, int kcount, const double *y,
                       void *x, int x_is_float, int n, hipStream_t s)
{
    Coefficients yv;
    for (int k = 0; k < kcount; ++k) yv.v[k] = y[k];
    const dim3 grid((n + 255) / 256);
    if (is_float && x_is_float)
        hipLaunchKernelGGL((k_axpy_basis<float, float>), grid, dim3(256), 0, s, (const float *)V,
                           ldv, kcount, yv, (float *)x, n);
    else if (is_float)
        hipLaunchKernelGGL((k_axpy_basis<float, double>), grid, dim3(256), 0, s,
                           (const float *)V, ldv, kcount, yv, (double *)x, n);
    else
        hipLaunchKernelGGL((k_axpy_basis<double, double>), grid, dim3(256), 0, s,
                           (const double *)V, ldv, kcount, yv, (double *)x, n);
}

void launch_norm2_partials(int is_float, const void *x, int n, double *P, hipStream_t s,
                           int batch, size_t sX, const int *active)
{
    dim3 grid(krylov_partials_blocks(n), batch);
    if (is_float)
        hipLaunchKernelGGL(k_norm2_partials<float>, grid, dim3(KTHREADS), 0, s, (const float *)x,
                           sX, n, P, active);
    else
        hipLaunchKernelGGL(k_norm2_partials<double>, grid, dim3(KTHREADS), 0, s,
                           (const double *)x, sX, n, P, active);
}

}  // namespace wb
