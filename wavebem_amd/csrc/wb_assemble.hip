// wb_assemble.hip -- dense single-layer G and double-layer H assembly on gfx950.
//
// Replaces the loops of BEMProblem::assemble_system (source/bem_problem.cc:106-590):
//   G_ij = sum_{c ni j} sum_q  phi_{j,c}(q) JxW_cq / (4 pi |y_cq - x_i|)
//   H_ij = sum_{c ni j} sum_q  phi_{j,c}(q) (x_i - y_cq).n_cq JxW_cq / (4 pi |y_cq - x_i|^3)
// (LaplaceKernel::kernels, include/laplace_kernel.h:45-64), with the regular QGauss
// rule on cells that do not touch x_i and QGaussOneOverR on the cells that do
// (double-node membership test, source/bem_problem.cc:214-230).
//
// Regular cells: one wavefront owns 64 collocation rows (lane = row).  Cell quadrature
// data is wave-uniform and arrives through scalar loads; each lane forms the 4+4 local G/H
// values of the current cell for its row and adds them to register (G) and lane-private
// LDS (H) accumulators, which leave through LDS as whole row segments, written once.
//  * Strips (k_assemble_strips): on logically structured patches a workgroup sweeps a run
//    of grid lines of at most 8 dofs, four gaps between lines at a time; every cell is
//    evaluated once per strip task it touches (about 1.1 times at 40k dofs) and its updates
//    go to fixed slots.
//  * Tiles (k_assemble_tiles): elsewhere, column tiles of up to TILE_COLS dofs and every
//    cell touching the tile, with wave-uniform slot indices.
// Both evaluate every cell with the regular rule; the singular kernel replaces the
// regular part of each singular (row, cell) pair by its QGaussOneOverR integral.
#include "wb_internal.h"
#include "wb_device.h"

#include <type_traits>

namespace wb {

__device__ __forceinline__ void split_hilo(double v, float &hi, uint16_t &lo)
{
    hi = (float)v;
    float r = (float)(v - (double)hi);
    // r is rounded to FP32 first, then to bf16 (nearest even, v_cvt_pk_bf16_f32 on
    // gfx950); the empty asm keeps the compiler from merging the two roundings into one
    // emulated FP64 -> bf16 rounding, which costs eight more instructions
    asm volatile("" : "+v"(r));
    lo = __builtin_bit_cast(uint16_t, (__bf16)r);
}

__device__ __forceinline__ double join_hilo(float hi, uint16_t lo)
{
    return (double)hi + (double)__uint_as_float((uint32_t)lo << 16);
}

// Factors from the sums of cell_local_values to the entries of G and H: 1/(4 pi), the sign
// of H, and the powers of two of FAST's 2/r.
template <bool FAST> struct RuleScale {
    static constexpr double g = FAST ? 0.5 * INV4PI : INV4PI;
    static constexpr double h = FAST ? -0.125 * INV4PI : -INV4PI;
};

// pointers to global memory that stay so through an opaque asm (a generic one would be stored
// to with flat instructions)
template <typename T> using glob = __attribute__((address_space(1))) T *;
typedef glob<char> glob_bytes;

// ------------------------------------------------------------------ cell geometry
// deal.II FEValues<2,3> with a Q1 mapping: x = sum phi_k v_k, a = dx/dxi, b = dx/deta,
// JxW = sqrt(det(J^T J)) w, n = orient (a x b)/|a x b|.
// Record: y(3), sn n*JxW(3), sj JxW, sj xi*JxW (xi = first reference coordinate of the
// point).  sn = sj = 1, or the factors that make the strip kernel's sums the entries
// themselves (RuleScale).
__global__ void k_cell_geometry(const double *__restrict__ X, const int *__restrict__ cell_int,
                                const int8_t *__restrict__ orient, int n_slots, int nq,
                                const double *__restrict__ qpts, const double *__restrict__ qw,
                                double *__restrict__ cellq, const int *__restrict__ slot_cell,
                                double sn, double sj)
{
    const int gid = blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= n_slots * nq) return;
    const int slot = gid / nq, q = gid % nq;
    const int c = slot_cell ? slot_cell[slot] : slot;
    if (c < 0) return;
    const double xi = qpts[2 * q], eta = qpts[2 * q + 1];
    const double phi[4] = {(1 - xi) * (1 - eta), xi * (1 - eta), (1 - xi) * eta, xi * eta};
    const double dxi[4] = {-(1 - eta), (1 - eta), -eta, eta};
    const double deta[4] = {-(1 - xi), -xi, (1 - xi), xi};
    double x[3] = {0, 0, 0}, a[3] = {0, 0, 0}, b[3] = {0, 0, 0};
    for (int k = 0; k < 4; ++k) {
        const int v = cell_int[4 * c + k];
        for (int d = 0; d < 3; ++d) {
            const double p = X[3 * v + d];
            x[d] += phi[k] * p;
            a[d] += dxi[k] * p;
            b[d] += deta[k] * p;
        }
    }
    const double g00 = a[0] * a[0] + a[1] * a[1] + a[2] * a[2];
    const double g01 = a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
    const double g11 = b[0] * b[0] + b[1] * b[1] + b[2] * b[2];
    const double jxw = sqrt(g00 * g11 - g01 * g01) * qw[q];
    double nn[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]};
    const double nl = sqrt(nn[0] * nn[0] + nn[1] * nn[1] + nn[2] * nn[2]);
    const double s = (orient[c] < 0 ? -1.0 : 1.0) / nl;
    double *r = cellq + (size_t)gid * 8;
    r[0] = x[0];
    r[1] = x[1];
    r[2] = x[2];
    r[3] = nn[0] * s * jxw * sn;
    r[4] = nn[1] * s * jxw * sn;
    r[5] = nn[2] * s * jxw * sn;
    r[6] = jxw * sj;
    r[7] = xi * jxw * sj;
}

void launch_cell_geometry(const double *X, const int *cell_int, const int8_t *orient,
                          int n_slots, int nq, const double *qpts, const double *qw,
                          double *cellq, hipStream_t s, const int *slot_cell, int strip_precision)
{
    const bool fast = strip_precision == WB_PREC_FP32_IR;
    const double sn = strip_precision < 0 ? 1.0 : fast ? RuleScale<true>::h : RuleScale<false>::h;
    const double sj = strip_precision < 0 ? 1.0 : fast ? RuleScale<true>::g : RuleScale<false>::g;
    const long total = (long)n_slots * nq;
    if (total <= 0) return;
    hipLaunchKernelGGL(k_cell_geometry, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, X,
                       cell_int, orient, n_slots, nq, qpts, qw, cellq, slot_cell, sn, sj);
}

// ------------------------------------------------------------------ regular cells
// Q = points per direction of the tensor rule (NQ = Q*Q, point q = i + Q*j, i fastest).
// The Q1 shape values factor as phi_k(q) = a_k(xi_i) b_k(eta_j), so the four local sums
// are formed per rule row j from S0 = sum_i (1-xi_i) t_ij and S1 = sum_i xi_i t_ij:
// only the Q Gauss nodes are needed (kept in SGPRs).
//
// The TC tile columns of each lane's row: G in a TC-wide register vector, H in LDS.  A
// cell's four tile-local columns are wave-uniform, so G is updated with s_set_gpr_idx
// register moves and H with one no-return LDS add per column; both are lane-private, so
// there is no contention and the summation order is fixed.  Keeping H out of the registers
// is what lets four waves share a SIMD.
// Measured at 41k dofs (FP64 assembly): 3 waves per SIMD with both accumulator tiles in
// registers 67 ms; 4 waves with the H tile in LDS 51 ms (the few spilled registers of the
// 4-wave budget cost less than the lost occupancy).
#ifndef WB_ASM_WAVES
#define WB_ASM_WAVES 4  // requested waves per SIMD for the column-tile kernel
#endif
// The four local G and H values of one cell for the lane's collocation point x:
// g_k = sum_q phi_k(q) JxW_q / |y_q - x|, h_k = sum_q phi_k(q) (y_q - x).N_q / |y_q - x|^3
// (N = n JxW; the 1/(4 pi) factors and the sign of H are RuleScale's, applied at the tile
// kernel's write-out and in the strip kernel's records).
// rec: the cell's NQ records (wave-uniform, read by scalar loads).
// FAST: the values are stored as FP32 hi + bf16 lo, and 1/r takes one Newton step
// (rsqrt2_f64_newton1) instead of the third-order one; g then comes out times 2 and h
// times 8 (RuleScale puts the powers of two back).
// TOUCH: once a batch has arrived, one word of each 64-byte line of the next batch is touched (the
// next cell's first records after the last batch; the arrays have REC_PAD records more),
// so that the next batch finds its lines in the scalar cache: 27.5 -> 26.5 ms for the
// FP32-IR assembly at 41k dofs.  A whole second batch does not fit the scalar registers.
template <int Q, bool FAST, bool TOUCH>
__device__ __forceinline__ void cell_local_values(const double *rec, double x0, double x1,
                                                  double x2, const PhiTable &nodes,
                                                  double (&g)[4], double (&h)[4])
{
    constexpr int B = Q <= 4 ? 4 : (Q + 1) / 2;  // points per batch of scalar loads
    // larger rules keep their row loop: unrolled, they spill hundreds of registers
    constexpr int JU = Q <= 4 ? Q : 1;
    double g0 = 0, g1 = 0, g2 = 0, g3 = 0, h0 = 0, h1 = 0, h2 = 0, h3 = 0;
#pragma unroll JU
    for (int j = 0; j < Q; ++j) {
        double sg = 0, sg1 = 0, sh = 0, sh1 = 0;
        // The records of B points arrive in one batch of scalar loads:
        // scalar loads return out of order, so every use of one waits for all
        // outstanding ones (lgkmcnt(0)), and batching divides those waits.
#pragma unroll
        for (int i = 0; i < Q; i += B) {
            double rr[8 * B];
#pragma unroll
            for (int k = 0; k < 8 * B; ++k)
                rr[k] = (i + k / 8 < Q) ? rec[(i + Q * j) * 8 + k] : 0.0;
            int touch[B];
            if constexpr (TOUCH) {
                asm volatile("" ::"s"(rr[0]));  // the batch has arrived
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < B; ++k)
                    touch[k] = *(const int *)(rec + 8 * ((i + B < Q ? i + B : Q) + Q * j + k));
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int u = 0; u < B; ++u) {
                if (i + u >= Q) break;
                const double *r = rr + 8 * u;
                const double R0 = r[0] - x0, R1 = r[1] - x1, R2 = r[2] - x2;
                const double r2 = __builtin_fma(R0, R0, __builtin_fma(R1, R1, R2 * R2));
                const double ri = FAST ? rsqrt2_f64_newton1(r2) : rsqrt_f64(r2);
                sg = __builtin_fma(ri, r[6], sg);   // sum JxW / r
                sg1 = __builtin_fma(ri, r[7], sg1); // sum xi JxW / r
                const double dn = __builtin_fma(R0, r[3], __builtin_fma(R1, r[4], R2 * r[5]));
                const double thv = (dn * ri) * (ri * ri);
                sh += thv;
                sh1 = __builtin_fma(nodes.phi[i + u], thv, sh1);
            }
            if constexpr (TOUCH) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < B; ++k) asm volatile("" ::"s"(touch[k]));
            }
        }
        const double sg0 = sg - sg1, sh0 = sh - sh1;  // sum (1 - xi_i) t
        const double eta = nodes.phi[j], ome = 1.0 - eta;
        g0 = __builtin_fma(ome, sg0, g0);
        g1 = __builtin_fma(ome, sg1, g1);
        g2 = __builtin_fma(eta, sg0, g2);
        g3 = __builtin_fma(eta, sg1, g3);
        h0 = __builtin_fma(ome, sh0, h0);
        h1 = __builtin_fma(ome, sh1, h1);
        h2 = __builtin_fma(eta, sh0, h2);
        h3 = __builtin_fma(eta, sh1, h3);
    }
    g[0] = g0;
    g[1] = g1;
    g[2] = g2;
    g[3] = g3;
    h[0] = h0;
    h[1] = h1;
    h[2] = h2;
    h[3] = h3;
}

template <int Q, int TC, int OUT>
__global__ __launch_bounds__(TILE_ROWS) __attribute__((amdgpu_waves_per_eu(WB_ASM_WAVES)))
void k_assemble_tiles(
    const double *__restrict__ xrow, const double *__restrict__ cellq,
    const int *__restrict__ tile_ptr, const int *__restrict__ tile_cell,
    const int *__restrict__ tile_cols, const int *__restrict__ tile_start, int n, int n_tiles,
    size_t ld, PhiTable nodes,
    void *__restrict__ Gv, void *__restrict__ Hv, uint16_t *__restrict__ Glo,
    uint16_t *__restrict__ Hlo, double *__restrict__ hsum_part)
{
    constexpr int NQ = Q * Q;
    static_assert(TC == 16, "tile width");
    typedef double accv __attribute__((ext_vector_type(16)));
    // [column][row] tile in LDS, row stride ACC_LD (68: the remapped row-segment reads of
    // the write-out hit distinct banks); holds the H accumulators, then stages G
    constexpr int ACC_LD = TILE_ROWS + 4;
    __shared__ double lacc[TC * ACC_LD];
    const int lane = threadIdx.x;
    const int rb = blockIdx.x;
    const int tg = blockIdx.y;
    const int row = rb * TILE_ROWS + lane;
    const int rr = row < n ? row : n - 1;
    const double x0 = xrow[3 * rr], x1 = xrow[3 * rr + 1], x2 = xrow[3 * rr + 2];
    double hs_total = 0.0;
    const int t_begin = tg * TILES_PER_WG;
    const int t_end = min(n_tiles, t_begin + TILES_PER_WG);
    for (int tile = t_begin; tile < t_end; ++tile) {
        accv aG = 0.0;
#pragma unroll
        for (int c = 0; c < TC; ++c) lacc[c * ACC_LD + lane] = 0.0;
        // c is wave-uniform: the G vector index becomes an s_set_gpr_idx register move; the
        // H entry is a lane-private LDS word, updated by a no-return LDS add (ds_add_f64)
        auto upd = [&](int c, double g, double h) {
            aG[c & 15] += g;
            __hip_atomic_fetch_add(&lacc[(c & 15) * ACC_LD + lane], h, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WAVEFRONT);
        };
        double hs = 0.0;
        const int p0 = tile_ptr[tile], p1 = tile_ptr[tile + 1];
        for (int p = p0; p < p1; ++p) {
            const int cell = __builtin_amdgcn_readfirstlane(tile_cell[p]);
            const int cols = __builtin_amdgcn_readfirstlane(tile_cols[p]);
            const double *rec = cellq + (size_t)cell * (NQ * 8);
            double gl[4], hl[4];
            cell_local_values<Q, OUT == 1, false>(rec, x0, x1, x2, nodes, gl, hl);
            const double g0 = gl[0], g1 = gl[1], g2 = gl[2], g3 = gl[3];
            const double h0 = hl[0], h1 = hl[1], h2 = hl[2], h3 = hl[3];
            const int c0 = (int)(int8_t)(cols & 0xff);
            const int c1 = (int)(int8_t)((cols >> 8) & 0xff);
            const int c2 = (int)(int8_t)((cols >> 16) & 0xff);
            const int c3 = (int)(int8_t)((cols >> 24) & 0xff);
            if (c0 >= 0) {
                upd(c0, g0, h0);
                hs += h0;
            }
            if (c1 >= 0) {
                upd(c1, g1, h1);
                hs += h1;
            }
            if (c2 >= 0) {
                upd(c2, g2, h2);
                hs += h2;
            }
            if (c3 >= 0) {
                upd(c3, g3, h3);
                hs += h3;
            }
        }
        // Write-out through LDS: H (already there), then G parked by each lane; lanes are
        // remapped to (row, column) so every store instruction writes whole row segments.
        const int c_begin = tile_start[tile];
        const int ncols = min(TC, tile_start[tile + 1] - c_begin);
#pragma unroll
        for (int m = 1; m >= 0; --m) {
            const double scale = m == 0 ? RuleScale<OUT == 1>::g : RuleScale<OUT == 1>::h;
            __syncthreads();
            if (m == 0) {
#pragma unroll
                for (int c = 0; c < TC; ++c) lacc[c * ACC_LD + lane] = aG[c];
            }
            __syncthreads();
            constexpr int RPI = TILE_ROWS / TC;  // rows per store instruction
            const int cl = lane % TC, rsub = lane / TC;
#pragma unroll
            for (int r0 = 0; r0 < TILE_ROWS; r0 += RPI) {
                const int rl = r0 + rsub;
                const int grow = rb * TILE_ROWS + rl;
                if (grow < n && cl < ncols) {
                    const double v = lacc[cl * ACC_LD + rl] * scale;
                    const size_t off = (size_t)grow * ld + c_begin + cl;
                    if (OUT == 0) {
                        ((double *)(m == 0 ? Gv : Hv))[off] = v;
                    } else {
                        float hi;
                        uint16_t lo;
                        split_hilo(v, hi, lo);
                        ((float *)(m == 0 ? Gv : Hv))[off] = hi;
                        (m == 0 ? Glo : Hlo)[off] = lo;
                    }
                }
            }
        }
        hs_total += hs;
    }
    if (row < n) hsum_part[(size_t)tg * n + row] = hs_total * RuleScale<OUT == 1>::h;
}

template <int Q>
static void launch_tiles_q(int precision, const double *xrow, const double *cellq,
                           const int *tile_ptr, const int *tile_cell, const int *tile_cols,
                           const int *tile_start, int n, int n_tiles, size_t ld,
                           const PhiTable &nodes, void *G, void *H, void *Glo, void *Hlo,
                           double *hsum_part, hipStream_t s)
{
    dim3 grid((n + TILE_ROWS - 1) / TILE_ROWS, (n_tiles + TILES_PER_WG - 1) / TILES_PER_WG);
    if (precision == WB_PREC_FP64)
        hipLaunchKernelGGL((k_assemble_tiles<Q, TILE_COLS, 0>), grid, dim3(TILE_ROWS), 0, s, xrow,
                           cellq, tile_ptr, tile_cell, tile_cols, tile_start, n, n_tiles, ld,
                           nodes, G, H, (uint16_t *)Glo, (uint16_t *)Hlo, hsum_part);
    else
        hipLaunchKernelGGL((k_assemble_tiles<Q, TILE_COLS, 1>), grid, dim3(TILE_ROWS), 0, s, xrow,
                           cellq, tile_ptr, tile_cell, tile_cols, tile_start, n, n_tiles, ld,
                           nodes, G, H, (uint16_t *)Glo, (uint16_t *)Hlo, hsum_part);
}

// nodes.phi[0..q_order-1] = 1-D Gauss nodes on [0,1] of the regular rule.  Tiles of up to
// 16 columns share the 16-wide register tile (tc only shapes the tiles on the host).
void launch_assemble_tiles(int precision, int q_order, int tc, const double *xrow,
                           const double *cellq, const int *tile_ptr, const int *tile_cell,
                           const int *tile_cols, const int *tile_start, int n, int n_tiles,
                           size_t ld, const PhiTable &nodes, void *G, void *H, void *Glo,
                           void *Hlo, double *hsum_part, hipStream_t s)
{
    (void)tc;
#define WB_TILES(QV)                                                                           \
    case QV:                                                                                   \
        launch_tiles_q<QV>(precision, xrow, cellq, tile_ptr, tile_cell, tile_cols, tile_start, \
                           n, n_tiles, ld, nodes, G, H, Glo, Hlo, hsum_part, s);               \
        break;
    switch (q_order) {
        WB_TILES(1)
        WB_TILES(2)
        WB_TILES(3)
        WB_TILES(4)
        WB_TILES(5)
        WB_TILES(6)
    default: break;
    }
#undef WB_TILES
}

// ------------------------------------------------------------------ regular cells, strips
// A workgroup owns 64 collocation rows (lane = row) and one strip task: the lines 0 ..
// L - 1 (grid rows of at most STRIP_W consecutive dofs) of a run of levels of a structured
// patch.  Gap t holds the cells between lines t and t + 1, t = -1 .. L - 1 (line -1 and line
// L belong to the neighbouring tasks).  The records are built from cell_int_s, whose vertex
// order puts the position direction first, so the cell at position k of gap t adds its local
// values 0, 1 to positions k - 1, k of line t ("lo") and 2, 3 to positions k - 1, k of line
// t + 1 ("up").
//
// The four wavefronts take four consecutive gaps at a time.  A wavefront walks its nine cell
// positions (unrolled): G values add up in registers at fixed slots; an H value is complete
// once the next position is done and goes straight to LDS.  Line t is then lo of gap t plus
// up of gap t - 1 (the neighbouring wavefront's, or kept from the last round), and the four
// lines leave together: 32 consecutive columns per row, so a store instruction fills whole
// 128-byte lines (FP32: 2 rows x 32 columns).
//
// Bound: FP64 issue at the clock the power limit leaves (20.6 FP64 operations and one
// v_rsq_f64 per point and row; at 41k dofs 93% of the issue slots at 2.08 GHz, where the one
// wavefront per task form below had 76% at 2.06).  Measured at 41k dofs, FP32-IR / FP64:
//   32.4 / 31.0 ms  one wavefront per task and 64 rows, one line (8 columns) stored at a time;
//   28.8 / 28.4     with the next gap's records touched a gap ahead: the wavefronts of an XCD
//                   walk a task side by side, and every new line made all of them wait for
//                   one L2 miss;
//   26.9 / 27.7     this form.  Without its stores it takes 22 ms: the 8-column segments left
//                   the L2 2.3 times over (47.7 GB for 20.4 GB of entries; 31.4 GB now).
// A small mesh gets four times as many wavefronts, each a quarter as long: 0.75 -> 0.19 ms
// at 2,915 dofs, 0.27 -> 0.08 ms at 1,083.
// Three wavefronts per SIMD hold everything in registers; at four, a spilled register reloaded
// between the stores waits for all of them (loads and stores share one in-order counter).
//
// LDS, in regions of STRIP_W x 64 doubles: LO[4] by wavefront, UP[5] by gap modulo 5 (the
// fifth is the last round's), and the G part's own kept UP: 10 x 4 KB.  A CU holds three
// workgroups, by their registers (the LDS would take four).  Slot p of a region holds row r
// at (r ^ 2 p ^ 16 parity): the write-out reads 16 columns (two lines of different parity)
// x 2 rows per half wavefront from distinct banks.
// Every cell is evaluated once per task it touches: once inside a strip, twice on the
// boundary between two strips or two tasks of one strip.
constexpr int STRIP_REGION = STRIP_W * TILE_ROWS;  // doubles

// The LDS word of position p for a row word of position 0 (byte offsets): slot p holds row
// r at r ^ 2 p.  Opaque, so that the sixteen offsets of a gap are formed when needed and not
// held in registers.
__device__ __forceinline__ double *strip_word(double *lds, int word0, int p)
{
    asm volatile("" : "+v"(word0));
    return (double *)((char *)lds + ((word0 ^ (16 * p)) + 512 * p));
}

// Positions K .. STRIP_W of one gap.  lo, up: G sums by position; wlo, wup: this lane's
// words of position 0 of the H regions; cl, cu: H values of the previous cell still waiting
// for this one; hs: the row sum of H over the positions of lines t (lm_lo) and t + 1 (lm_up)
// that belong to the task.
template <int Q, int K, bool FAST>
__device__ __forceinline__ void strip_gap_cells(int cmask, int lm_lo, int lm_up,
                                                const double *grec, double x0, double x1,
                                                double x2, const PhiTable &nodes,
                                                double (&lo)[STRIP_W], double (&up)[STRIP_W],
                                                double *lds, int wlo, int wup,
                                                double cl, double cu, double &hs)
{
    if constexpr (K <= STRIP_W) {
        double nl = 0.0, nu = 0.0;
        if constexpr (K < STRIP_W) lo[K] = up[K] = 0.0;
        if (cmask & (1 << K)) {
            double g[4], h[4];
            cell_local_values<Q, FAST, true>(grec + K * (Q * Q * 8), x0, x1, x2, nodes, g, h);
            if constexpr (K >= 1) {
                lo[K - 1] += g[0];
                up[K - 1] += g[2];
                cl += h[0];
                cu += h[2];
            }
            if constexpr (K < STRIP_W) {
                lo[K] = g[1];
                up[K] = g[3];
            }
            nl = h[1];
            nu = h[3];
        }
        if constexpr (K >= 1) {
            constexpr int P = K - 1;
            *strip_word(lds, wlo, P) = cl;
            *strip_word(lds, wup, P) = cu;
            if (lm_lo & (1 << P)) hs += cl;
            if (lm_up & (1 << P)) hs += cu;
        }
        strip_gap_cells<Q, K + 1, FAST>(cmask, lm_lo, lm_up, grec, x0, x1, x2, nodes, lo, up, lds,
                                        wlo, wup, nl, nu, hs);
    }
}

template <int Q, int OUT>
__global__ __launch_bounds__(TILE_ROWS * STRIP_WAVES)
__attribute__((amdgpu_waves_per_eu(3)))
void k_assemble_strips(const double *__restrict__ xrow, const double *__restrict__ recs,
                       const int2 *__restrict__ tasks, const int4 *__restrict__ gaps, int n,
                       size_t ld, PhiTable nodes, void *__restrict__ Gv, void *__restrict__ Hv,
                       uint16_t *__restrict__ Glo, uint16_t *__restrict__ Hlo,
                       double *__restrict__ hsum_part)
{
    constexpr int NQ = Q * Q;
    constexpr int KS = STRIP_W + 1;  // cell positions per gap
    constexpr int NW = STRIP_WAVES, NU = NW + 1;
    static_assert(NW == 4 && STRIP_W == 8 && TILE_ROWS == 64, "the write-out's lane map");
    __shared__ double lds[(NW + NU + 1) * STRIP_REGION];
    // LO[wv], UP[gap % 5], UPG: G's UP of the last round's last gap
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row0 = blockIdx.x * TILE_ROWS;
    const int task = blockIdx.y;
    const int row = row0 + lane;
    const int rr = row < n ? row : n - 1;
    const double x0 = xrow[3 * rr], x1 = xrow[3 * rr + 1], x2 = xrow[3 * rr + 2];
    const int2 T = tasks[task];
    const int g0 = __builtin_amdgcn_readfirstlane(T.x);
    const int ng = __builtin_amdgcn_readfirstlane(T.y);
    // wait for the row's coordinates here: loads and stores share one in-order counter, so a
    // wait for them inside the loop would wait for the last round's stores as well
    asm volatile("" ::"v"(x0), "v"(x1), "v"(x2));
    double hs = 0.0;
    auto line_mask = [&](int t) {  // positions of line t (the gap's index in the task)
        return t < ng ? __builtin_amdgcn_readfirstlane(gaps[g0 + t].z) : 0;
    };
    int u5 = 0;  // (round's first gap) modulo 5
    for (int j0 = 0; j0 < ng; j0 += NW) {
        const int j = j0 + wv;  // this wavefront's gap
        const int uw = (u5 + wv) % NU;
        // this lane's words of position 0 in LO[wv] and UP[uw] (bytes)
        const int wlo = 8 * (wv * STRIP_REGION + (lane ^ (16 * (wv & 1))));
        const int wup = 8 * ((NW + uw) * STRIP_REGION + (lane ^ (16 * (uw & 1))));
        double lo[STRIP_W], up[STRIP_W];
        {
            // touch the records of the wavefront's next gap (one word per 64-byte line): the
            // wavefronts of an XCD walk the same task side by side, and without this each new
            // line makes all of them wait for one L2 miss
            constexpr int LINES = KS * NQ, PF = (LINES + 63) / 64;
            float pf[PF];
            const double *nrec = recs + (size_t)(g0 + min(j + NW, ng - 1)) * KS * (NQ * 8);
#pragma unroll
            for (int k = 0; k < PF; ++k)
                pf[k] = *(const float *)(nrec + 8 * min(lane + 64 * k, LINES - 1));
            int cmask = 0;
            const double *grec = recs;
            if (j < ng) {
                cmask = __builtin_amdgcn_readfirstlane(gaps[g0 + j].x);
                grec = recs + (size_t)(g0 + j) * KS * (NQ * 8);
            }
            strip_gap_cells<Q, 0, OUT == 1>(
                cmask, line_mask(j), line_mask(j + 1), grec, x0, x1, x2, nodes, lo, up, lds, wlo,
                wup, 0.0, 0.0, hs);
#pragma unroll
            for (int k = 0; k < PF; ++k) asm volatile("" ::"v"(pf[k]));
        }
        // Write-out: this lane's column c of the round's lines (line l, position pos) and
        // row offset rsub; rows 16 wv .. 16 wv + 15, two per step.  The lane number is made
        // opaque here so that none of this is held in registers across the cells: a register
        // spilled there is reloaded between the stores, and each reload waits for them.
        int ln = threadIdx.x & 63;
        asm volatile("" : "+v"(ln));
        const int c = (ln & 15) + 16 * (ln >> 5), rsub = (ln >> 4) & 1;
        const int m0 = line_mask(j0), m1 = line_mask(j0 + 1), m2 = line_mask(j0 + 2),
                  m3 = line_mask(j0 + 3);
        int l = c >> 3, pos = c & 7, cols = 32;
        if ((m0 & m1 & m2 & m3) != 255) {
            const int e0 = __builtin_popcount(m0), e1 = e0 + __builtin_popcount(m1),
                      e2 = e1 + __builtin_popcount(m2);
            cols = e2 + __builtin_popcount(m3);
            l = (c >= e0) + (c >= e1) + (c >= e2);
            const int lm = l == 0 ? m0 : l == 1 ? m1 : l == 2 ? m2 : m3;
            int rank = c - (l == 0 ? 0 : l == 1 ? e0 : l == 2 ? e1 : e2);
            pos = 0;
#pragma unroll
            for (int p = 0; p < STRIP_W; ++p) {  // the position of the rank-th present dof
                const int bit = (lm >> p) & 1;
                if (bit && rank == 0) pos = p;
                rank -= bit;
            }
        }
        const int first = m0 ? 0 : m1 ? 1 : m2 ? 2 : 3;
        const int col0 = j0 + first < ng ? __builtin_amdgcn_readfirstlane(gaps[g0 + j0 + first].y)
                                         : 0;
        int ul = u5 + l + NU - 1;  // UP region of gap j0 + l - 1
        ul -= ul >= 2 * NU ? 2 * NU : ul >= NU ? NU : 0;
        const int r0 = 16 * wv + rsub;  // this lane's first row in the block
        // LDS bytes of (pos, r0); step it flips the row bits 2 it, which r0 leaves clear
        const int plo = 8 * (l * STRIP_REGION + pos * TILE_ROWS + (r0 ^ (2 * pos) ^ (16 * (l & 1))));
        const int pup = 8 * ((NW + ul) * STRIP_REGION + pos * TILE_ROWS +
                             (r0 ^ (2 * pos) ^ (16 * (ul & 1))));
        // line 0 finds G's up part of the last round in UPG
        const int pug = l == 0 ? pup + 8 * (NU - ul) * STRIP_REGION : pup;
        // the first gap of a task (line -1) has no line, so l = 0 of round 0 is never read
        const int steps = c >= cols ? 0 : min(TILE_ROWS / (2 * NW), (n - row0 - r0 + 1) / 2);
        // bytes of the lane's entry from the first row of the block (64 rows fit 32 bits) and
        // wave-uniform row steps; the running row pointers are opaque, or their multiples
        // of 2 ld would be kept (and spilled) over the cells
        typedef typename std::conditional<OUT == 0, double, float>::type MT;
        const unsigned vb = ((unsigned)r0 * (unsigned)ld + (unsigned)(col0 + c)) * sizeof(MT);
        auto write_out = [&](int pu, void *Mb, uint16_t *Mlob) {
            glob_bytes M = (glob_bytes)Mb + (size_t)row0 * ld * sizeof(MT);
            glob_bytes Mlo = (glob_bytes)Mlob + (size_t)row0 * ld * 2;
            // four steps' LDS reads in flight together
            constexpr int NS = TILE_ROWS / (2 * NW), NB = 4;
#pragma unroll
            for (int ib = 0; ib < NS; ib += NB) {
                double a[NB], b[NB];
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    a[k] = *(const double *)((const char *)lds + (plo ^ (16 * (ib + k))));
                    b[k] = *(const double *)((const char *)lds + (pu ^ (16 * (ib + k))));
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < NB; ++k) {
                    asm volatile("" : "+s"(M));
                    if (OUT == 1) asm volatile("" : "+s"(Mlo));
                    const double v = a[k] + b[k];
                    if (ib + k < steps) {
                        if (OUT == 0) {
                            *(glob<MT>)(M + vb) = v;
                        } else {
                            float hi;
                            uint16_t lo16;
                            split_hilo(v, hi, lo16);
                            *(glob<MT>)(M + vb) = hi;
                            *(glob<uint16_t>)(Mlo + vb / 2) = lo16;
                        }
                    }
                    M += 2 * ld * sizeof(MT);
                    Mlo += 4 * ld;
                }
            }
        };
        __syncthreads();
        write_out(pup, Hv, Hlo);
        __syncthreads();
        // G takes H's place; H's UP of the round's last gap stays for the next round, so G's
        // goes to UPG once the last round's has been read
#pragma unroll
        for (int p = 0; p < STRIP_W; ++p) {
            *strip_word(lds, wlo, p) = lo[p];
            if (wv != NW - 1) *strip_word(lds, wup, p) = up[p];
        }
        __syncthreads();
        write_out(pug, Gv, Glo);
        __syncthreads();
        if (wv == NW - 1) {
            // with the parity of UP[uw], as line 0 of the next round reads it
#pragma unroll
            for (int p = 0; p < STRIP_W; ++p)
                *strip_word(lds + (NU - uw) * STRIP_REGION, wup, p) = up[p];
        }
        u5 = (u5 + NW) % NU;
    }
    // row sums of H, wavefront by wavefront
    __syncthreads();
    lds[threadIdx.x] = hs;
    __syncthreads();
    if (wv == 0 && row < n) {
        double s = hs;
#pragma unroll
        for (int w = 1; w < NW; ++w) s += lds[w * 64 + lane];
        hsum_part[(size_t)task * n + row] = s;
    }
}

void launch_assemble_strips(int precision, int q_order, const double *xrow, const double *recs,
                            const int *tasks, const int *gaps, int n, int n_tasks, size_t ld,
                            const PhiTable &nodes, void *G, void *H, void *Glo, void *Hlo,
                            double *hsum_part, hipStream_t s)
{
    if (n_tasks <= 0) return;
    dim3 grid((n + TILE_ROWS - 1) / TILE_ROWS, n_tasks);  // row blocks of a task side by side
#define WB_STRIPS(QV)                                                                          \
    case QV:                                                                                   \
        if (precision == WB_PREC_FP64)                                                         \
            hipLaunchKernelGGL((k_assemble_strips<QV, 0>), grid, dim3(TILE_ROWS * STRIP_WAVES), 0, s, xrow,  \
                               recs, (const int2 *)tasks, (const int4 *)gaps, n, ld, nodes, G, \
                               H, (uint16_t *)Glo, (uint16_t *)Hlo, hsum_part);                \
        else                                                                                   \
            hipLaunchKernelGGL((k_assemble_strips<QV, 1>), grid, dim3(TILE_ROWS * STRIP_WAVES), 0, s, xrow,  \
                               recs, (const int2 *)tasks, (const int4 *)gaps, n, ld, nodes, G, \
                               H, (uint16_t *)Glo, (uint16_t *)Hlo, hsum_part);                \
        break;
    switch (q_order) {
        WB_STRIPS(1)
        WB_STRIPS(2)
        WB_STRIPS(3)
        WB_STRIPS(4)
        WB_STRIPS(5)
        WB_STRIPS(6)
    default: break;
    }
#undef WB_STRIPS
}

// ------------------------------------------------------------------ singular cells
// Sixteen lanes per row: for each cell touching x_i (first coincident vertex j*), they share
// the points of the QGaussOneOverR rule of vertex j*, with full FEValues geometry at every
// point (source/bem_problem.cc:475-525), and those of the regular rule, whose values are
// taken off (the regular kernels evaluate every cell with QGauss, which keeps the singular
// test out of their inner loop); the sums are added over the lanes in a fixed order and go
// into row i.  One thread per row walked 66 points per pair in a chain: 0.10 ms at 1,083
// dofs and 0.22 ms at 41k; now 0.02 at 1,083.
constexpr int SING_LANES = 16;

template <int OUT>
__global__ __launch_bounds__(256) void k_assemble_singular(
    const double *__restrict__ X, const int *__restrict__ cell_int,
    const int8_t *__restrict__ orient, const int *__restrict__ sing_ptr,
    const int *__restrict__ sing_cell, const int *__restrict__ sing_vtx, int n, int ns,
    const double *__restrict__ rule, const double *__restrict__ cellq, int nq,
    const double *__restrict__ qpts, size_t ld, void *__restrict__ Gv, void *__restrict__ Hv,
    uint16_t *__restrict__ Glo, uint16_t *__restrict__ Hlo, double *__restrict__ hsum_sing)
{
    const int i = (blockIdx.x * blockDim.x + threadIdx.x) / SING_LANES;
    const int sl = threadIdx.x % SING_LANES;
    if (i >= n) return;  // whole groups of lanes
    const double x0 = X[3 * i], x1 = X[3 * i + 1], x2 = X[3 * i + 2];
    double hs = 0.0;
    for (int p = sing_ptr[i]; p < sing_ptr[i + 1]; ++p) {
        const int c = sing_cell[p], vtx = sing_vtx[p];
        int vid[4];
        double v[4][3];
        for (int k = 0; k < 4; ++k) {
            vid[k] = cell_int[4 * c + k];
            for (int d = 0; d < 3; ++d) v[k][d] = X[3 * vid[k] + d];
        }
        const double sgn = orient[c] < 0 ? -1.0 : 1.0;
        const double *ru = rule + (size_t)vtx * ns * 3;
        double lv[8] = {0, 0, 0, 0, 0, 0, 0, 0};  // G, then H
        for (int q = sl; q < ns; q += SING_LANES) {
            const double xi = ru[3 * q], eta = ru[3 * q + 1], w = ru[3 * q + 2];
            const double phi[4] = {(1 - xi) * (1 - eta), xi * (1 - eta), (1 - xi) * eta, xi * eta};
            const double dxi[4] = {-(1 - eta), (1 - eta), -eta, eta};
            const double deta[4] = {-(1 - xi), -xi, (1 - xi), xi};
            double y[3] = {0, 0, 0}, a[3] = {0, 0, 0}, b[3] = {0, 0, 0};
            for (int k = 0; k < 4; ++k)
                for (int d = 0; d < 3; ++d) {
                    y[d] += phi[k] * v[k][d];
                    a[d] += dxi[k] * v[k][d];
                    b[d] += deta[k] * v[k][d];
                }
            const double g00 = a[0] * a[0] + a[1] * a[1] + a[2] * a[2];
            const double g01 = a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
            const double g11 = b[0] * b[0] + b[1] * b[1] + b[2] * b[2];
            const double jxw = sqrt(g00 * g11 - g01 * g01) * w;
            double nn[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2],
                            a[0] * b[1] - a[1] * b[0]};
            const double nl = sqrt(nn[0] * nn[0] + nn[1] * nn[1] + nn[2] * nn[2]);
            const double R0 = y[0] - x0, R1 = y[1] - x1, R2 = y[2] - x2;
            const double r2 = R0 * R0 + R1 * R1 + R2 * R2;
            const double ri = rsqrt_f64(r2);
            const double dn = (R0 * nn[0] + R1 * nn[1] + R2 * nn[2]) * (sgn / nl);
            const double tg = ri * jxw;
            const double th = dn * ri * ri * ri * jxw;
            for (int k = 0; k < 4; ++k) {
                lv[k] = __builtin_fma(tg, phi[k], lv[k]);
                lv[4 + k] = __builtin_fma(th, phi[k], lv[4 + k]);
            }
        }
        // the regular-rule part the regular kernels added for this pair (same kernel; it
        // cancels up to rounding)
        const double *rec = cellq + (size_t)c * nq * 8;
        for (int q = sl; q < nq; q += SING_LANES) {
            const double *r = rec + 8 * q;
            const double xi = qpts[2 * q], eta = qpts[2 * q + 1];
            const double phi[4] = {(1 - xi) * (1 - eta), xi * (1 - eta), (1 - xi) * eta, xi * eta};
            const double R0 = r[0] - x0, R1 = r[1] - x1, R2 = r[2] - x2;
            const double ri = rsqrt_f64(__builtin_fma(R0, R0, __builtin_fma(R1, R1, R2 * R2)));
            const double dn = __builtin_fma(R0, r[3], __builtin_fma(R1, r[4], R2 * r[5]));
            const double tg = ri * r[6], th = (dn * ri) * (ri * ri);
            for (int k = 0; k < 4; ++k) {
                lv[k] = __builtin_fma(-tg, phi[k], lv[k]);
                lv[4 + k] = __builtin_fma(-th, phi[k], lv[4 + k]);
            }
        }
#pragma unroll
        for (int o = SING_LANES / 2; o > 0; o >>= 1)
#pragma unroll
            for (int k = 0; k < 8; ++k) lv[k] += __shfl_xor(lv[k], o, 64);
        // every lane holds the sums: lane k < 4 adds entry vid[k] of G, lane 4 + k of H; of
        // lanes with the same entry (a cell that names a dof twice) the first adds their sum
        const int vk = sl & 2 ? (sl & 1 ? vid[3] : vid[2]) : (sl & 1 ? vid[1] : vid[0]);
        double add = 0.0;
        bool first = sl < 8;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool same = vid[j] == vk;
            add += same ? (sl < 4 ? lv[j] : lv[4 + j]) : 0.0;
            first = first && !(same && j < (sl & 3));
        }
        if (first) {
            const size_t off = (size_t)i * ld + vk;
            void *M = sl < 4 ? Gv : Hv;
            add *= sl < 4 ? INV4PI : -INV4PI;
            if (OUT == 0) {
                ((double *)M)[off] += add;
            } else {
                uint16_t *L = sl < 4 ? Glo : Hlo;
                float hi;
                uint16_t lo;
                split_hilo(join_hilo(((float *)M)[off], L[off]) + add, hi, lo);
                ((float *)M)[off] = hi;
                L[off] = lo;
            }
        }
        for (int k = 0; k < 4; ++k) hs += lv[4 + k] * (-INV4PI);
        // the next cell shares vertices with this one under other k: what a lane has stored is
        // another lane's load there (one wavefront: program order of its memory operations)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    if (sl == 0) hsum_sing[i] = hs;
}

void launch_assemble_singular(int precision, const double *X, const int *cell_int,
                              const int8_t *orient, const int *sing_ptr, const int *sing_cell,
                              const int *sing_vtx, int n, int ns, const double *rule,
                              const double *cellq, int nq, const double *qpts, size_t ld,
                              void *G, void *H, void *Glo, void *Hlo, double *hsum_sing,
                              hipStream_t s)
{
    dim3 grid((int)(((long)n * SING_LANES + 255) / 256));
    if (precision == WB_PREC_FP64)
        hipLaunchKernelGGL(k_assemble_singular<0>, grid, dim3(256), 0, s, X, cell_int, orient,
                           sing_ptr, sing_cell, sing_vtx, n, ns, rule, cellq, nq, qpts, ld, G, H,
                           (uint16_t *)Glo, (uint16_t *)Hlo, hsum_sing);
    else
        hipLaunchKernelGGL(k_assemble_singular<1>, grid, dim3(256), 0, s, X, cell_int, orient,
                           sing_ptr, sing_cell, sing_vtx, n, ns, rule, cellq, nq, qpts, ld, G, H,
                           (uint16_t *)Glo, (uint16_t *)Hlo, hsum_sing);
}

// alpha_i = -(sum over tile groups of the regular H row sums + singular H row sum)
// alpha_i = -(sum over tile groups of the partial row sums + singular part).  A block
// owns 64 rows; its 4 wavefronts sum interleaved quarters of the partials and the quarters
// are added in a fixed order, so the result does not depend on scheduling.
__global__ __launch_bounds__(256) void k_alpha_reduce(const double *__restrict__ part,
                                                      int n_parts,
                                                      const double *__restrict__ sing, int n,
                                                      double *__restrict__ alpha)
{
    __shared__ double q[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + lane;
    double s = 0.0;
    if (i < n)
        for (int p = wave; p < n_parts; p += 4) s += part[(size_t)p * n + i];
    q[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && i < n) alpha[i] = -(((q[0][lane] + q[1][lane]) + (q[2][lane] + q[3][lane])) + sing[i]);
}

void launch_alpha_reduce(const double *hsum_part, int n_parts, const double *hsum_sing, int n,
                         double *alpha, hipStream_t s)
{
    hipLaunchKernelGGL(k_alpha_reduce, dim3((n + 63) / 64), dim3(256), 0, s, hsum_part, n_parts,
                       hsum_sing, n, alpha);
}

}  // namespace wb
