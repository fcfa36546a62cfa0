// wb_project.hip -- L2 projections onto the continuous Q1 space of the dofs, on the device.
//
// Replaces the UMFPACK mass-matrix solves of
//   ComputationalDomain::compute_normals        (source/computational_domain.cc:1525-1620),
//   NumericalTowingTank::compute_normals_at_nodes (source/numerical_towing_tank.cc:3358-3433),
//   BEMProblem::compute_surface_gradients       (source/bem_problem.cc:1154-1290),
//   FreeSurface::compute_potential_gradients    (source/free_surface.cc:9271-9400):
//   sum_j M_ij x_j = sum_c sum_q phi_i(q) f(q) JxW(q),  M_ij = sum_c sum_q phi_i phi_j JxW,
// with f = the cell normal (normals) or the surface gradient of the Q1 interpolant of u
// (gradients; plus n psi for the complete potential gradient), one scalar mass matrix for the three components (the reference's vector
// mass matrix couples only equal components).
//
// The mass matrix stays in element form: ten values per cell (the symmetric 4x4 block),
// applied row by row through the node -> cell incidence in a fixed order, so the product
// needs no atomics and is bit-reproducible.  The six right-hand sides (normal x,y,z and
// gradient x,y,z) are solved together by Jacobi-preconditioned CG; vectors are [n][6].
// Every kernel is HBM/latency-bound and tiny next to the assembly (n * 6 doubles per
// vector); the point is to keep the geometry on the device and the host out of the loop.
#include "wb_internal.h"
#include "wb_device.h"

namespace wb {

namespace {

constexpr int NCOL = 6;
constexpr int PB = 256;  // threads per block of the row kernels

// packed index of the symmetric 4x4 element block, a <= b
__host__ __device__ constexpr int msym(int a, int b)
{
    return a <= b ? a * 4 - a * (a - 1) / 2 + (b - a) : b * 4 - b * (b - 1) / 2 + (a - b);
}

// one thread per cell: element mass block (10) and element right-hand sides (4 x 6)
// With psi (dphi/dn at the dofs), the gradient columns take the complete potential
// gradient n psi + surface gradient of u (FreeSurface::compute_potential_gradients,
// source/free_surface.cc:9325-9344).
__global__ void k_proj_cells(const double *__restrict__ X, const int *__restrict__ cell_int,
                             const int8_t *__restrict__ orient, const double *__restrict__ u,
                             const double *__restrict__ psi, int nc, int nq,
                             const double *__restrict__ qpts, const double *__restrict__ qw,
                             double *__restrict__ emass, double *__restrict__ erhs)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nc) return;
    double v[4][3], uc[4] = {0, 0, 0, 0}, pc[4] = {0, 0, 0, 0};
    for (int k = 0; k < 4; ++k) {
        const int d = cell_int[4 * c + k];
        for (int e = 0; e < 3; ++e) v[k][e] = X[3 * d + e];
        if (u) uc[k] = u[d];
        if (psi) pc[k] = psi[d];
    }
    const double so = orient[c] < 0 ? -1.0 : 1.0;
    double m[10], r[4][NCOL];
    for (int k = 0; k < 10; ++k) m[k] = 0.0;
    for (int k = 0; k < 4; ++k)
        for (int e = 0; e < NCOL; ++e) r[k][e] = 0.0;
    for (int q = 0; q < nq; ++q) {
        double sh[4], dx[4], de[4];
        q1_shape(qpts[2 * q], qpts[2 * q + 1], sh, dx, de);
        double a[3] = {0, 0, 0}, b[3] = {0, 0, 0};
        double ux = 0.0, ue = 0.0, pq = 0.0;
        for (int k = 0; k < 4; ++k) {
            for (int e = 0; e < 3; ++e) {
                a[e] += dx[k] * v[k][e];
                b[e] += de[k] * v[k][e];
            }
            ux += dx[k] * uc[k];
            ue += de[k] * uc[k];
            pq += sh[k] * pc[k];
        }
        const double g00 = a[0] * a[0] + a[1] * a[1] + a[2] * a[2];
        const double g01 = a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
        const double g11 = b[0] * b[0] + b[1] * b[1] + b[2] * b[2];
        const double det = g00 * g11 - g01 * g01;
        const double jxw = sqrt(det) * qw[q];
        const double nn[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2],
                              a[0] * b[1] - a[1] * b[0]};
        const double ns = so / sqrt(nn[0] * nn[0] + nn[1] * nn[1] + nn[2] * nn[2]);
        // surface gradient of the interpolant: J (J^T J)^-1 (du/dxi, du/deta)
        const double ca = (g11 * ux - g01 * ue) / det, cb = (g00 * ue - g01 * ux) / det;
        double f[NCOL];
        for (int e = 0; e < 3; ++e) {
            f[e] = nn[e] * ns * jxw;
            f[3 + e] = (ca * a[e] + cb * b[e] + nn[e] * ns * pq) * jxw;
        }
        for (int i = 0; i < 4; ++i) {
            for (int j = i; j < 4; ++j) m[msym(i, j)] += sh[i] * sh[j] * jxw;
            for (int e = 0; e < NCOL; ++e) r[i][e] += sh[i] * f[e];
        }
    }
    for (int k = 0; k < 10; ++k) emass[10 * (size_t)c + k] = m[k];
    for (int i = 0; i < 4; ++i)
        for (int e = 0; e < NCOL; ++e) erhs[(size_t)(4 * c + i) * NCOL + e] = r[i][e];
}

// right-hand side and inverse diagonal per row, gathered over the incident cells
__global__ void k_proj_rows(const int *__restrict__ inc_ptr, const int *__restrict__ inc_item,
                            const double *__restrict__ emass, const double *__restrict__ erhs,
                            int n, double *__restrict__ B, double *__restrict__ dinv)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double b[NCOL] = {0, 0, 0, 0, 0, 0}, d = 0.0;
    for (int p = inc_ptr[i]; p < inc_ptr[i + 1]; ++p) {
        const int it = inc_item[p], c = it >> 2, a = it & 3;
        d += emass[10 * (size_t)c + msym(a, a)];
        for (int e = 0; e < NCOL; ++e) b[e] += erhs[(size_t)it * NCOL + e];
    }
    for (int e = 0; e < NCOL; ++e) B[(size_t)i * NCOL + e] = b[e];
    dinv[i] = d > 0.0 ? 1.0 / d : 0.0;
}

// The CG kernels work on PR rows per block, eight lanes per row, lane e < 6 for column e: a
// thread per row walked six columns of sixteen neighbours in 43 blocks at 11k dofs.
constexpr int PR = PB / 8;

// sums over the block's rows of K values per thread, for every column: out[k * NCOL + e]
template <int K>
__device__ __forceinline__ void block_sum(double (&v)[K], double (*lds)[K][8],
                                          double *__restrict__ out)
{
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
        for (int o = 8; o < 64; o <<= 1) v[k] += __shfl_xor(v[k], o, 64);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane < 8)
#pragma unroll
        for (int k = 0; k < K; ++k) lds[wv][k][lane] = v[k];
    __syncthreads();
    if (threadIdx.x < K * NCOL) {
        const int k = threadIdx.x / NCOL, e = threadIdx.x % NCOL;
        out[threadIdx.x] = ((lds[0][k][e] + lds[1][k][e]) + lds[2][k][e]) + lds[3][k][e];
    }
}

// totals of the block partials part[nb][K], broadcast through LDS (out, K values): the PB / K
// threads of each k add every (PB / K)-th partial, and their sums are added in thread order
// (the same bits in every block).  A serial sum by K threads took 10 us for 43 partials.
// Every block reads all n / PR partials, so a launch reads n^2: small beside the rows' own
// latency up to the sizes that a context can hold.  One compute_potential_gradients, against
// a thread per row and 256 rows per block: 2.15 -> 1.22 ms at 11k dofs, 4.3 -> 2.4 at 40k,
// 5.8 -> 3.9 at 59k, 9.1 -> 7.0 at 95k, 11.6 -> 9.4 at 121k (the FP32-IR matrices of 155k
// fill the card).
template <int K>
__device__ __forceinline__ void sum_parts(const double *__restrict__ part, int nb, double *out)
{
    constexpr int T = PB / K;  // threads per k
    __shared__ double sh[K * T];
    const int k = threadIdx.x % K, t = threadIdx.x / K;
    if (t < T) {
        double s = 0.0;
#pragma unroll 4
        for (int b = t; b < nb; b += T) s += part[(size_t)b * K + k];
        sh[t * K + k] = s;
    }
    __syncthreads();
    if (t == 0) {
        double s = sh[k];
#pragma unroll
        for (int j = 1; j < T; ++j) s += sh[j * K + k];
        out[k] = s;
    }
    __syncthreads();
}

// state: rho[2][6] (by iteration parity), bb[6], rr[6]; part2 = partials r.z, r.r of the
// last update.  Records rho and r.r of iteration iter (and b.b at iteration 0).
__device__ __forceinline__ void proj_record(const double *tot, int iter, double *state)
{
    if (threadIdx.x < NCOL) {
        const int e = threadIdx.x;
        state[(iter & 1) * NCOL + e] = tot[e];
        if (iter == 0) state[2 * NCOL + e] = tot[NCOL + e];
        state[3 * NCOL + e] = tot[NCOL + e];
    }
}

// the record alone, for the host's convergence check between iterations
__global__ void __launch_bounds__(PB) k_proj_record(const double *__restrict__ part2, int nb,
                                                    int iter, double *__restrict__ state)
{
    __shared__ double tot[2 * NCOL];
    sum_parts<2 * NCOL>(part2, nb, tot);
    proj_record(tot, iter, state);
}

// The direction and its product in one pass: beta = rho / rho_old, P = Z + beta Pold (P = Z
// at iteration 0), formed for every neighbour of the row as it is read, Q = M P, partial P.Q.
__global__ void __launch_bounds__(PB) k_proj_apply(
    const int *__restrict__ inc_ptr, const int *__restrict__ inc_item,
    const int *__restrict__ cell_int, const double *__restrict__ emass,
    const double *__restrict__ part2, int nb, double *__restrict__ state, int iter,
    const double *__restrict__ Z, const double *__restrict__ Pold, int n,
    double *__restrict__ P, double *__restrict__ Q, double *__restrict__ part)
{
    __shared__ double tot[2 * NCOL];
    __shared__ double lds[PB / 64][1][8];
    sum_parts<2 * NCOL>(part2, nb, tot);
    const int i = blockIdx.x * PR + threadIdx.x / 8, e = threadIdx.x & 7;
    const bool live = i < n && e < NCOL;
    double beta = 0.0;
    if (e < NCOL && iter > 0) {
        const double rho = state[((iter - 1) & 1) * NCOL + e];
        beta = rho > 0.0 ? tot[e] / rho : 0.0;
    }
    if (blockIdx.x == 0) proj_record(tot, iter, state);  // the other parity than read above
    double acc[1] = {0.0};
    if (live) {
        auto dir = [&](size_t o) { return iter > 0 ? Z[o] + beta * Pold[o] : Z[o]; };
        double q = 0.0;
        for (int p = inc_ptr[i]; p < inc_ptr[i + 1]; ++p) {
            const int it = inc_item[p], c = it >> 2, a = it & 3;
            const double *m = emass + 10 * (size_t)c;
#pragma unroll
            for (int b = 0; b < 4; ++b)
                q += m[msym(a, b)] * dir((size_t)cell_int[4 * c + b] * NCOL + e);
        }
        const size_t o = (size_t)i * NCOL + e;
        const double pv = dir(o);
        P[o] = pv;
        Q[o] = q;
        acc[0] = pv * q;
    }
    block_sum<1>(acc, lds, part + (size_t)blockIdx.x * NCOL);
}

// alpha = rho / (p.q); x += alpha p; r -= alpha q; z = D^-1 r; partials r.z, r.r
__global__ void __launch_bounds__(PB) k_proj_update(
    const double *__restrict__ part, int nb, const double *__restrict__ state, int iter,
    const double *__restrict__ P, const double *__restrict__ Q, const double *__restrict__ dinv,
    int n, double *__restrict__ Xs, double *__restrict__ R, double *__restrict__ Z,
    double *__restrict__ part2)
{
    __shared__ double tot[NCOL];
    __shared__ double lds[PB / 64][2][8];
    sum_parts<NCOL>(part, nb, tot);
    const int i = blockIdx.x * PR + threadIdx.x / 8, e = threadIdx.x & 7;
    double acc[2] = {0.0, 0.0};
    if (i < n && e < NCOL) {
        const double rho = state[(iter & 1) * NCOL + e], pq = tot[e];
        const double alpha = pq > 0.0 ? rho / pq : 0.0;
        const size_t o = (size_t)i * NCOL + e;
        Xs[o] += alpha * P[o];
        const double r = R[o] - alpha * Q[o];
        R[o] = r;
        const double z = dinv[i] * r;
        Z[o] = z;
        acc[0] = r * z;
        acc[1] = r * r;
    }
    block_sum<2>(acc, lds, part2 + (size_t)blockIdx.x * 2 * NCOL);
}

// x = 0, r = b, z = D^-1 b, partials r.z, r.r
__global__ void __launch_bounds__(PB) k_proj_init(const double *__restrict__ B,
                                                  const double *__restrict__ dinv, int n,
                                                  double *__restrict__ Xs, double *__restrict__ R,
                                                  double *__restrict__ Z,
                                                  double *__restrict__ part2)
{
    __shared__ double lds[PB / 64][2][8];
    const int i = blockIdx.x * PR + threadIdx.x / 8, e = threadIdx.x & 7;
    double acc[2] = {0.0, 0.0};
    if (i < n && e < NCOL) {
        const double di = dinv[i];
        const size_t o = (size_t)i * NCOL + e;
        const double r = B[o];
        Xs[o] = 0.0;
        R[o] = r;
        Z[o] = di * r;
        acc[0] = r * di * r;
        acc[1] = r * r;
    }
    block_sum<2>(acc, lds, part2 + (size_t)blockIdx.x * 2 * NCOL);
}

}  // namespace

int proj_blocks(int n) { return (n + PR - 1) / PR; }

void launch_proj_setup(const double *X, const int *cell_int, const int8_t *orient,
                       const double *u, const double *psi, int nc, int nq, const double *qpts,
                       const double *qw, const int *inc_ptr, const int *inc_item, int n,
                       double *emass, double *erhs, double *B, double *dinv, hipStream_t s)
{
    hipLaunchKernelGGL(k_proj_cells, dim3((nc + 127) / 128), dim3(128), 0, s, X, cell_int,
                       orient, u, psi, nc, nq, qpts, qw, emass, erhs);
    hipLaunchKernelGGL(k_proj_rows, dim3((n + PB - 1) / PB), dim3(PB), 0, s, inc_ptr, inc_item,
                       emass, erhs, n, B, dinv);
}

void launch_proj_cg_start(const double *B, const double *dinv, int n, double *Xs, double *R,
                          double *Z, double *part2, double *state, hipStream_t s)
{
    const int nb = proj_blocks(n);
    hipLaunchKernelGGL(k_proj_init, dim3(nb), dim3(PB), 0, s, B, dinv, n, Xs, R, Z, part2);
    hipLaunchKernelGGL(k_proj_record, dim3(1), dim3(PB), 0, s, part2, nb, 0, state);
}

// One iteration in two launches, the directions in P[iter & 1] (P[1 - iter & 1] the last
// ones): at 11k dofs 36 -> 16 us per iteration.
void launch_proj_cg_iter(const int *inc_ptr, const int *inc_item, const int *cell_int,
                         const double *emass, const double *dinv, int n, int iter, double *Xs,
                         double *R, double *Z, double *const P[2], double *Q, double *part,
                         double *part2, double *state, hipStream_t s)
{
    const int nb = proj_blocks(n);
    double *Pn = P[iter & 1];
    hipLaunchKernelGGL(k_proj_apply, dim3(nb), dim3(PB), 0, s, inc_ptr, inc_item, cell_int,
                       emass, part2, nb, state, iter, Z, P[1 - (iter & 1)], n, Pn, Q, part);
    hipLaunchKernelGGL(k_proj_update, dim3(nb), dim3(PB), 0, s, part, nb, state, iter, Pn, Q,
                       dinv, n, Xs, R, Z, part2);
}

// state as of the start of iteration iter, for the host's convergence check
void launch_proj_cg_state(const double *part2, int n, int iter, double *state, hipStream_t s)
{
    hipLaunchKernelGGL(k_proj_record, dim3(1), dim3(PB), 0, s, part2, proj_blocks(n), iter,
                       state);
}

}  // namespace wb
