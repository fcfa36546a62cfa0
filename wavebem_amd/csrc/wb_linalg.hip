// wb_linalg.hip -- bandwidth-bound kernels of the GMRES path on gfx950.
//
// Column-selected GEMV: BEMProblem::vmult (source/bem_problem.cc:621-670) computes
//   dst = -G (surface .* src) + H (other .* src) + alpha .* other .* src
// and compute_rhs (:673-717) the complementary selection.  Every column j needs either
// G(:,j) or H(:,j), never both, so one kernel reads exactly n entries per row: for each
// group of 4 columns a 4-bit mask says which matrix each column comes from; groups that
// agree (all but the few at a Dirichlet/Neumann boundary in the device ordering) issue
// one vector load from the selected matrix.  Rows run one per (wave, row slot) with
// wavefront shuffle reductions; constrained rows (ConstrainedOperator,
// include/constrained_matrix.h:73-86) are skipped; blocks of the same launch write their lines.
#include "wb_internal.h"
#include "wb_device.h"

namespace wb {

__device__ __forceinline__ double wave_sum(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

__device__ __forceinline__ float wave_sumf(float v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

__device__ __forceinline__ double bf16_to_double(uint16_t b)
{
    return (double)__uint_as_float((uint32_t)b << 16);
}

// native clang vector types (usable with the nontemporal load builtins)
typedef double dvec4 __attribute__((ext_vector_type(4)));
typedef float fvec4 __attribute__((ext_vector_type(4)));
typedef unsigned short uvec4 __attribute__((ext_vector_type(4)));

// ------------------------------------------------------------------ constraint rows
template <typename T>
__global__ void k_constraint_rows(int n_lines, const int *__restrict__ rows,
                                  const int *__restrict__ ptr, const int *__restrict__ cols,
                                  const double *__restrict__ w, const double *__restrict__ inhom,
                                  int mode_inhom, const T *__restrict__ x, T *__restrict__ y)
{
    const int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l >= n_lines) return;
    const int r = rows[l];
    if (mode_inhom) {
        y[r] = (T)inhom[l];
        return;
    }
    y[r] = (T)line_value({n_lines, rows, ptr, cols, w}, l, x);
}

// op[i] = alpha[i] (1 - s[i]), rhs[i] = -alpha[i] s[i] for a 0/1 mask s
__global__ void k_diag_from_mask(int n, const double *__restrict__ alpha,
                                 const double *__restrict__ s, double *__restrict__ op,
                                 double *__restrict__ rhs)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    op[i] = alpha[i] * (1.0 - s[i]);
    rhs[i] = alpha[i] * -s[i];
}

void launch_diag_from_mask(int n, const double *alpha, const double *s, double *op, double *rhs,
                           hipStream_t st)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_diag_from_mask, dim3((n + 255) / 256), dim3(256), 0, st, n, alpha, s, op,
                       rhs);
}

// a[i] = v[i] where mask[i] == 0, b[i] = v[i] where mask[i] != 0
__global__ void k_scatter_mask(int n, const uint8_t *__restrict__ mask,
                               const double *__restrict__ v, double *__restrict__ a,
                               double *__restrict__ b)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (mask[i]) b[i] = v[i];
    else a[i] = v[i];
}

void launch_scatter_mask(int n, const uint8_t *mask, const double *v, double *a, double *b,
                         hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_scatter_mask, dim3((n + 255) / 256), dim3(256), 0, s, n, mask, v, a, b);
}

void launch_constraint_rows(int is_float, int n_lines, const int *rows, const int *ptr,
                            const int *cols, const double *w, const double *inhom, int mode_inhom,
                            const void *x, void *y, hipStream_t s)
{
    if (n_lines <= 0) return;
    dim3 grid((n_lines + 255) / 256);
    if (is_float)
        hipLaunchKernelGGL(k_constraint_rows<float>, grid, dim3(256), 0, s, n_lines, rows, ptr,
                           cols, w, inhom, mode_inhom, (const float *)x, (float *)y);
    else
        hipLaunchKernelGGL(k_constraint_rows<double>, grid, dim3(256), 0, s, n_lines, rows, ptr,
                           cols, w, inhom, mode_inhom, (const double *)x, (double *)y);
}

// ------------------------------------------------------------------ block Jacobi
// Diagonal blocks of the preconditioner matrix of BEMProblem::assemble_preconditioner
// (source/bem_problem.cc:1107-1149): column i holds H(j,i) (+alpha_i on the diagonal)
// for a Neumann column, -G(j,i) for a Dirichlet column; constrained rows are identity
// rows.  Inverted by Gauss-Jordan elimination with partial pivoting, blocks of 64 in one
// wavefront's registers, others in LDS; stored column-major (binv[c*bs + r]) so the apply
// kernel reads it coalesced.
constexpr int BJ_THREADS = 256;

// entry (j, i) of the preconditioner matrix, device indices
__device__ __forceinline__ double bj_entry(int j, int i, const void *__restrict__ Gv,
                                           const void *__restrict__ Hv,
                                           const uint16_t *__restrict__ Glo,
                                           const uint16_t *__restrict__ Hlo, int precision,
                                           size_t ld, const double *__restrict__ alpha,
                                           const double *__restrict__ surface,
                                           const uint8_t *__restrict__ constrained)
{
    if (constrained[j]) return i == j ? 1.0 : 0.0;
    const size_t off = (size_t)j * ld + i;
    const bool neu = surface[i] == 0.0;
    double v;
    if (precision == WB_PREC_FP64)
        v = ((const double *)(neu ? Hv : Gv))[off];
    else
        v = (double)((const float *)(neu ? Hv : Gv))[off] +
            (double)__uint_as_float((uint32_t)(neu ? Hlo : Glo)[off] << 16);
    return neu ? v + (i == j ? alpha[i] : 0.0) : -v;
}

// Blocks of 64 unknowns, one wavefront each, lane = row, the row in registers.  In-place
// Gauss-Jordan with the columns rotated by one at every step, so that the pivot column is
// always register 0 and the loop body serves all steps; rows stay where they are (step k's
// pivot row is the unused row with the largest entry, as partial pivoting's), and the write-out puts row
// and column k of the result at (k, pivot row of step k).  Serial chain: 64 steps of a
// wavefront maximum and 63 register updates; the LDS form takes nine barriers per step,
// 0.23 ms for any number of blocks up to the CUs'; this one 0.12.
__global__ __launch_bounds__(64) void k_block_jacobi_build64(
    int n, const void *__restrict__ Gv, const void *__restrict__ Hv,
    const uint16_t *__restrict__ Glo, const uint16_t *__restrict__ Hlo, int precision, size_t ld,
    const double *__restrict__ alpha, const double *__restrict__ surface,
    const uint8_t *__restrict__ constrained, double *__restrict__ binv, float *__restrict__ binv32)
{
    __shared__ double t[64 * 65];
    __shared__ int piv[64];
    const int lane = threadIdx.x, base = blockIdx.x * 64, m = min(64, n - base);
    for (int r = 0; r < 64; ++r)
        t[r * 65 + lane] = r < m && lane < m
                               ? bj_entry(base + r, base + lane, Gv, Hv, Glo, Hlo, precision, ld,
                                          alpha, surface, constrained)
                               : (r == lane ? 1.0 : 0.0);
    __syncthreads();
    double a[64];
#pragma unroll
    for (int j = 0; j < 64; ++j) a[j] = t[lane * 65 + j];
    int step = -1;  // the step this row was the pivot of
    for (int k = 0; k < 64; ++k) {
        // unused rows before used ones, then the larger entry, then the smaller row
        double best = step >= 0 ? -2.0 : fabs(a[0]);
        if (!(best >= 0.0) && step < 0) best = -1.0;  // NaN
        int p = lane;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const double ob = __shfl_xor(best, o, 64);
            const int op = __shfl_xor(p, o, 64);
            if (ob > best || (ob == best && op < p)) {
                best = ob;
                p = op;
            }
        }
        p = __builtin_amdgcn_readfirstlane(p);
        const bool mine = lane == p;
        if (mine) step = k;
        if (lane == 0) piv[k] = p;
        auto bcast = [&](double v) {
            const unsigned long long u = __double_as_longlong(v);
            const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)u, p);
            const unsigned hi = __builtin_amdgcn_readlane((int)(unsigned)(u >> 32), p);
            return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
        };
        const double d = bcast(a[0]);
        const double inv = d != 0.0 ? 1.0 / d : 0.0;
        // other rows: a_j - f inv a_pj, pivot column -f inv; the pivot row: a_j inv, inv
        const double c = mine ? -inv : a[0] * inv, keep = mine ? 0.0 : 1.0;
#pragma unroll
        for (int j = 1; j < 64; ++j) a[j - 1] = __builtin_fma(-c, bcast(a[j]), a[j] * keep);
        a[63] = -c;
    }
    __syncthreads();
    double *out = binv + (size_t)blockIdx.x * 64 * 64;
    float *out32 = binv32 + (size_t)blockIdx.x * 64 * 64;
#pragma unroll
    for (int j = 0; j < 64; ++j) {
        const int e = piv[j] * 64 + step;
        out[e] = a[j];
        out32[e] = (float)a[j];
    }
}

__global__ __launch_bounds__(BJ_THREADS) void k_block_jacobi_build(
    int n, int bs, const void *__restrict__ Gv, const void *__restrict__ Hv,
    const uint16_t *__restrict__ Glo, const uint16_t *__restrict__ Hlo, int precision, size_t ld,
    const double *__restrict__ alpha, const double *__restrict__ surface,
    const uint8_t *__restrict__ constrained, double *__restrict__ binv, float *__restrict__ binv32)
{
    extern __shared__ double sm[];
    double *A = sm;                                // bs x bs, row-major
    double *colk = sm + (size_t)bs * bs;           // bs: column k before elimination
    int *piv = (int *)(sm + (size_t)bs * bs + bs);  // bs
    __shared__ int red_i[1];
    const int b = blockIdx.x;
    const int base = b * bs;
    const int m = min(bs, n - base);
    const int tid = threadIdx.x;
    for (int e = tid; e < bs * bs; e += BJ_THREADS) {
        const int rl = e / bs, cl = e % bs;
        double v = (rl == cl) ? 1.0 : 0.0;
        if (rl < m && cl < m)
            v = bj_entry(base + rl, base + cl, Gv, Hv, Glo, Hlo, precision, ld, alpha, surface,
                         constrained);
        A[e] = v;
    }
    __syncthreads();
    (void)gj_invert_lds<BJ_THREADS>(A, colk, piv, red_i, bs);
    double *out = binv + (size_t)b * bs * bs;
    float *out32 = binv32 + (size_t)b * bs * bs;
    for (int e = tid; e < bs * bs; e += BJ_THREADS) {
        const int rl = e / bs, cl = e % bs;
        out[cl * bs + rl] = A[e];
        out32[cl * bs + rl] = (float)A[e];
    }
}

void launch_block_jacobi_build(int n, int bs, const void *G, const void *H, const void *Glo,
                               const void *Hlo, int precision, size_t ld, const double *alpha,
                               const double *surface, const uint8_t *constrained, double *binv,
                               float *binv32, hipStream_t s)
{
    const int nb = (n + bs - 1) / bs;
    if (bs == 64) {
        hipLaunchKernelGGL(k_block_jacobi_build64, dim3(nb), dim3(64), 0, s, n, G, H,
                           (const uint16_t *)Glo, (const uint16_t *)Hlo, precision, ld, alpha,
                           surface, constrained, binv, binv32);
        return;
    }
    const size_t smem = sizeof(double) * (bs * bs + bs) + sizeof(int) * bs;
    hipLaunchKernelGGL(k_block_jacobi_build, dim3(nb), dim3(BJ_THREADS), smem, s, n, bs, G, H,
                       (const uint16_t *)Glo, (const uint16_t *)Hlo, precision, ld, alpha,
                       surface, constrained, binv, binv32);
}

// y_blk = Binv_blk x_blk for k vectors (column stride ldx); one thread per block row.
// With C (the coarse-space part of the two-level preconditioner, CS_MAX entries per
// vector): y_i += z_a for the aggregate a = i / agg of row i, z_a = sum_b Aci[a][b] C[v][b]
// (Aci row-major nc x nc; with trans, Aci^T for the transposed system), formed by the
// block for the at most three aggregates its rows touch (bs <= 128, agg >= 64), the
// partial products reduced in a fixed order.
template <typename T>
__global__ void k_block_jacobi_apply(int n, int bs, const T *__restrict__ binv,
                                     const T *__restrict__ x, T *__restrict__ y, int k, size_t ldx,
                                     int trans, const double *__restrict__ C,
                                     const T *__restrict__ Aci, int nc, int agg)
{
    extern __shared__ char smraw[];
    T *xs = (T *)smraw;
    __shared__ double zred[2][3];
    __shared__ double zs[3];
    const int b = blockIdx.x, r = threadIdx.x, base = b * bs;
    const int m = min(bs, n - base);
    const T *B = binv + (size_t)b * bs * bs;
    const int a0 = C ? base / agg : 0, na = C ? (base + m - 1) / agg - a0 + 1 : 0;
    for (int v = 0; v < k; ++v) {
        if (r < bs) xs[r] = (r < m) ? x[(size_t)v * ldx + base + r] : (T)0;
        for (int q = 0; q < na; ++q) {
            const int a = a0 + q;
            const double *c = C + (size_t)v * CS_MAX;
            double p = 0.0;
            // row a of Ac^-1, or with trans (the adjoint) column a, i.e. row a of Ac^-T
            for (int bb = r; bb < nc; bb += blockDim.x)
                p += (double)(trans ? Aci[(size_t)bb * nc + a] : Aci[(size_t)a * nc + bb]) * c[bb];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) p += __shfl_xor(p, off, 64);
            if ((r & 63) == 0) zred[r >> 6][q] = p;
        }
        __syncthreads();
        if (r < na) zs[r] = blockDim.x > 64 ? zred[0][r] + zred[1][r] : zred[0][r];
        __syncthreads();
        if (r < m) {
            T acc = 0;
            if (trans)  // the transposed block inverse, for the adjoint system
                for (int c = 0; c < m; ++c) acc += B[r * bs + c] * xs[c];
            else
                for (int c = 0; c < m; ++c) acc += B[c * bs + r] * xs[c];
            if (C) acc = (T)((double)acc + zs[(base + r) / agg - a0]);
            y[(size_t)v * ldx + base + r] = acc;
        }
        __syncthreads();
    }
}

void launch_block_jacobi_apply(int is_float, int n, int bs, const void *binv, const void *x,
                               void *y, int k, size_t ldx, hipStream_t s, int trans,
                               const double *C, const void *Aci, int nc, int agg)
{
    const int nb = (n + bs - 1) / bs;
    const int threads = bs <= 64 ? 64 : 128;
    if (is_float)
        hipLaunchKernelGGL(k_block_jacobi_apply<float>, dim3(nb), dim3(threads),
                           sizeof(float) * bs, s, n, bs, (const float *)binv, (const float *)x,
                           (float *)y, k, ldx, trans, C, (const float *)Aci, nc, agg);
    else
        hipLaunchKernelGGL(k_block_jacobi_apply<double>, dim3(nb), dim3(threads),
                           sizeof(double) * bs, s, n, bs, (const double *)binv,
                           (const double *)x, (double *)y, k, ldx, trans, C,
                           (const double *)Aci, nc, agg);
}

// elementwise ops on n entries:
//  0: c(d) = a(d) - b(d)          1: c(f) = (float) a(d)          2: c(d) += a(f)
//  3: c(d) = a(d) * alpha         4: c(d) = a(d) * b(d)            5: c(f) = a(f) * alpha
//  6: c(d) = 0                    7: c(f) = 0                      8: c(d) = b(d) - a(d)
//  9: c(f) = b(f) - a(f)
__global__ void k_vec_ops(int op, int n, const void *__restrict__ a, const void *__restrict__ b,
                          void *__restrict__ c, double alpha)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double *ad = (const double *)a, *bd = (const double *)b;
    const float *af = (const float *)a;
    double *cd = (double *)c;
    float *cf = (float *)c;
    switch (op) {
    case 0: cd[i] = ad[i] - bd[i]; break;
    case 1: cf[i] = (float)ad[i]; break;
    case 2: cd[i] += (double)af[i]; break;
    case 3: cd[i] = ad[i] * alpha; break;
    case 4: cd[i] = ad[i] * bd[i]; break;
    case 5: cf[i] = (float)((double)af[i] * alpha); break;
    case 6: cd[i] = 0.0; break;
    case 7: cf[i] = 0.0f; break;
    case 8: cd[i] = bd[i] - ad[i]; break;
    case 9: cf[i] = ((const float *)b)[i] - af[i]; break;
    default: break;
    }
}

void launch_vec_ops(int op, int n, const void *a, const void *b, void *c, double alpha,
                    hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_vec_ops, dim3((n + 255) / 256), dim3(256), 0, s, op, n, a, b, c, alpha);
}

// gather: dst[i] = src[idx[i]];  scatter: dst[idx[i]] = src[i]
__global__ void k_permute(int n, const int *__restrict__ idx, const double *__restrict__ src,
                          double *__restrict__ dst, int gather)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (gather)
        dst[i] = src[idx[i]];
    else
        dst[idx[i]] = src[i];
}

void launch_permute(int n, const int *idx, const double *src, double *dst, int gather,
                    hipStream_t s)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_permute, dim3((n + 255) / 256), dim3(256), 0, s, n, idx, src, dst, gather);
}

}  // namespace wb
