// Solution evaluation at barycentric points common to all cells (fem3DapplyL,
// eval.inl:84-100, core.inl:370-405).
//
// One lane per cell: its geometry and DOF values are read once for all points
// (one lane per (cell, point) read them q times, from q addresses per cell),
// the basis at the points is evaluated by the workgroup into LDS from the
// points in the kernel's arguments (no table in device memory to allocate,
// copy and wait for), and the values go through LDS so that the workgroup
// stores whole ranges.  What bounds it then is the values written and the
// gathers of nodes and DOFs.  P2 gradients at 4 points of 663,552 cells: call
// 157 us -> 33 us (3.4 TB/s).
#pragma once

#include "element_kernels.h"

namespace anifem {

constexpr int kMaxApplyPoints = 96;

// The points of one call, by value: 3 KB of kernel arguments.
struct ApplyPoints {
    double xyl[4 * kMaxApplyPoints];
};

__host__ __device__ constexpr int apply_nf0(int fem) {
    return fem == ANIFEM_FEM_P0 || fem == ANIFEM_FEM_B4 ? 1
           : fem == ANIFEM_FEM_P2                       ? 10
           : fem == ANIFEM_FEM_P3                       ? 20
           : fem == ANIFEM_FEM_B2 || fem == ANIFEM_FEM_ND0 ? 6
                                                        : 4;
}

// Row of the stage per cell: an odd number of values, so that the lanes of a
// wave write different banks.
__host__ __device__ inline int apply_stage_row(int pc, int dim) { return (pc * dim) | 1; }

// Workgroups that a launch has room for (four per CU).
constexpr int64_t kApplyGroups = 1024;

// Points per pass, by the stage's share of the LDS.  32 KB keeps five workgroups
// on a CU; 60 KB where even so there are more than kApplyGroups passes to make:
// each then reads the cells' DOFs for more points and stores longer ranges (GRAD
// of P3^3 at 14 points, 20,001 cells: 38 us with 32 KB, 19 with 60; of 3,001 cells
// 8.0 and 11.5).
inline int apply_chunk(int64_t n, int q, int dim) {
    auto fit = [&](size_t bytes) {
        int pc = q;
        while (pc > 1 && (size_t)kBlock * apply_stage_row(pc, dim) * sizeof(double) > bytes) --pc;
        return pc;
    };
    const int64_t cells = (n + kBlock - 1) / kBlock;
    const int pc = fit(32 * 1024);
    return cells * ((q + pc - 1) / pc) > kApplyGroups ? fit(60 * 1024) : pc;
}

// Workgroups along the passes of a cell range (blockIdx.y), each with its own
// run of points.  Cells that fill the chip by themselves take one, which reads
// their DOFs once; fewer leave it to a chain of up to q passes in few workgroups
// (GRAD of P3^3 at 96 points: 255 cells 384 us against 7.7, 3,001 cells 387
// against 16; one lane per (cell, point) took 58 and 114).
inline int apply_split(int64_t n, int q, int pc) {
    const int64_t cells = (n + kBlock - 1) / kBlock, passes = (q + pc - 1) / pc;
    const int64_t want = (kApplyGroups + cells - 1) / cells;
    return (int)(want < passes ? want : passes);
}

// D: reference components per basis function (ApplyArgs::d).
template <int FEM, int D, bool MESH>
__global__ __launch_bounds__(kBlock) void apply_points_kernel(ApplyArgs a, ApplyPoints pts, int pc) {
    constexpr int NF0 = apply_nf0(FEM);
    constexpr bool VECTOR = FEM == ANIFEM_FEM_RT0 || FEM == ANIFEM_FEM_ND0;
    extern __shared__ __align__(16) double smem[];
    double* tab = smem;
    double* stage = smem + (size_t)pc * NF0 * D;
    const int dim = a.map >= 3 ? 9 : D * a.ncomp, rs = apply_stage_row(pc, dim), nf = NF0 * a.ncomp;
    const int64_t r0 = blockIdx.x * (int64_t)kBlock, r = r0 + threadIdx.x;
    const bool live = r < a.n;
    const int ncell = (int)(a.n - r0 < kBlock ? a.n - r0 : kBlock);
    double P[4][3], PSI[9], JT[9], det = 1.0;
    if (live && (a.map != 0 || a.scale != 0)) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int64_t node = MESH ? a.tetnodes[(int64_t)v * a.n + r] : 0;
#pragma unroll
            for (int c = 0; c < 3; ++c) P[v][c] = MESH ? a.coords[3 * node + c] : a.xyz[(int64_t)(3 * v + c) * a.n + r];
        }
        tet_geometry(P, PSI, det);
        tet_jacobian_t(P, JT);
    }
    const int share = ((a.q + pc - 1) / pc + gridDim.y - 1) / gridDim.y * pc;  // points of this workgroup
    const int p_end = min(a.q, (int)(blockIdx.y + 1) * share);
    for (int p0 = blockIdx.y * share; p0 < p_end; p0 += pc) {
        const int np = p_end - p0 < pc ? p_end - p0 : pc;
        if ((int)threadIdx.x < np) {
            double L[4], u[NF0 * D];
#pragma unroll
            for (int i = 0; i < 4; ++i) L[i] = pts.xyl[4 * (p0 + threadIdx.x) + i];
            if constexpr (VECTOR) vector_field(a.op, FEM, L, u);
            else if constexpr (D == 3) basis_gradients(FEM, L, u);
            else basis_values(FEM, L, u);
#pragma unroll
            for (int i = 0; i < NF0 * D; ++i) tab[threadIdx.x * (NF0 * D) + i] = u[i];
        }
        __syncthreads();
        if (live) {
            double* row = stage + threadIdx.x * rs;
            for (int c = 0; c < a.ncomp; ++c) {
                double dv[NF0];
#pragma unroll
                for (int i = 0; i < NF0; ++i) {
                    const int64_t e = r * nf + c * NF0 + i;
                    dv[i] = MESH ? a.u[a.dofmap[e]] : a.dofs[e];
                    if constexpr (VECTOR) {
                        if (MESH && a.sign) dv[i] *= (double)a.sign[e];
                        if (a.scale) dv[i] *= dof_scale(a.scale, P, det, i);
                    }
                }
                for (int p = 0; p < np; ++p) {
                    const double* T = tab + p * (NF0 * D);
                    double g[3] = {0.0, 0.0, 0.0};
#pragma unroll
                    for (int i = 0; i < NF0; ++i)
#pragma unroll
                        for (int j = 0; j < D; ++j) g[j] += T[i * D + j] * dv[i];
                    double* o = row + p * dim;
                    if (VECTOR && a.map >= 3) {  // GRAD of RT0 (vec(I) g) / ND0 (S J g): 9 components
#pragma unroll
                        for (int l = 0; l < 9; ++l) {
                            double v = 0.0;
#pragma unroll
                            for (int j = 0; j < D; ++j) v += grad9_map(a.map, JT, l, j) * g[j];
                            o[l] = v;
                        }
                    } else if (D == 3 && a.map == 1) {
#pragma unroll
                        for (int k = 0; k < 3; ++k)
                            o[k + 3 * c] = PSI[3 * k] * g[0] + PSI[1 + 3 * k] * g[1] + PSI[2 + 3 * k] * g[2];
                    } else if (D == 3 && a.map == 2) {
#pragma unroll
                        for (int k = 0; k < 3; ++k)
                            o[k + 3 * c] = JT[3 * k] * g[0] + JT[1 + 3 * k] * g[1] + JT[2 + 3 * k] * g[2];
                    } else {
#pragma unroll
                        for (int j = 0; j < D; ++j) o[j + D * c] = g[j];
                    }
                }
            }
        }
        __syncthreads();
        // the workgroup's cells in turn, np dim consecutive values each
        const int w = np * dim, total = ncell * w, dc = kBlock / w, dk = kBlock - dc * w;
        int cell = threadIdx.x / w, k = threadIdx.x - cell * w;
        double* out = a.out + r0 * dim * a.q + (int64_t)dim * p0;
        for (int i = threadIdx.x; i < total; i += kBlock) {
            out[(int64_t)cell * dim * a.q + k] = stage[cell * rs + k];
            cell += dc;
            k += dk;
            if (k >= w) {
                k -= w;
                ++cell;
            }
        }
        if (p0 + pc < p_end) __syncthreads();  // table and stage are rewritten
    }
}

// fem3DapplyX, one lane per (tet, point): Op(u)(x_n) = sum_i s_i T U_i(x_n) dof_i
// with the reference values U_i evaluated at the barycentric coordinates of the
// tet's own physical point (l_{k+1} = sum_j PSI(k, j) (x_j - P0_j),
// l_0 = 1 - l_1 - l_2 - l_3, core.inl:120-137); T = 1, PSI^T or J and s_i the
// per-DOF factor of RT0 / ND0 (component k + 3c = du_c/dx_k for GRAD of a
// vector space).  D: reference components per basis function; the U_i stay in
// registers (indexed by run-time sizes they went to scratch memory: P3^3 values
// at 2 points of 3,001 cells 17 us against 5, at 31 points of 100,003 cells 420
// against 71).
template <int FEM, int D>
__global__ __launch_bounds__(kBlock) void apply_x_kernel(ApplyArgs a) {
    constexpr int NF0 = apply_nf0(FEM);
    constexpr bool VECTOR = FEM == ANIFEM_FEM_RT0 || FEM == ANIFEM_FEM_ND0;
    const int64_t idx = blockIdx.x * (int64_t)kBlock + threadIdx.x;
    if (idx >= a.n * a.q) return;
    const int64_t r = idx / a.q;
    const int pt = (int)(idx % a.q);
    const int nf = NF0 * a.ncomp, dim = a.map >= 3 ? 9 : D * a.ncomp;
    double P[4][3], PSI[9], JT[9], det = 1.0;
    for (int v = 0; v < 4; ++v)
        for (int c = 0; c < 3; ++c) P[v][c] = a.xyz[(int64_t)(3 * v + c) * a.n + r];
    tet_geometry(P, PSI, det);
    tet_jacobian_t(P, JT);
    double T[NF0 * D];
    const double* x = a.X + (r * a.q + pt) * 3;
    const double dr[3] = {x[0] - P[0][0], x[1] - P[0][1], x[2] - P[0][2]};
    double L[4];
    for (int i = 0; i < 3; ++i) L[i + 1] = PSI[i] * dr[0] + PSI[i + 3] * dr[1] + PSI[i + 6] * dr[2];
    L[0] = 1.0 - L[1] - L[2] - L[3];
    if constexpr (VECTOR) vector_field(a.op, FEM, L, T);
    else if constexpr (D == 3) basis_gradients(FEM, L, T);
    else basis_values(FEM, L, T);
    double* o = a.out + r * dim * a.q + (int64_t)dim * pt;
    for (int c = 0; c < a.ncomp; ++c) {
        double g[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < NF0; ++i) {
            double dv = a.dofs[r * nf + c * NF0 + i];
            if constexpr (VECTOR) {
                if (a.scale) dv *= dof_scale(a.scale, P, det, i);
            }
#pragma unroll
            for (int j = 0; j < D; ++j) g[j] += T[i * D + j] * dv;
        }
        if (VECTOR && a.map >= 3) {  // GRAD of RT0 (vec(I) g) / ND0 (S J g): 9 components
#pragma unroll
            for (int l = 0; l < 9; ++l) {
                double v = 0.0;
#pragma unroll
                for (int j = 0; j < D; ++j) v += grad9_map(a.map, JT, l, j) * g[j];
                o[l] = v;
            }
        } else if (D == 3 && a.map == 1) {
#pragma unroll
            for (int k = 0; k < 3; ++k) o[k + 3 * c] = PSI[3 * k] * g[0] + PSI[1 + 3 * k] * g[1] + PSI[2 + 3 * k] * g[2];
        } else if (D == 3 && a.map == 2) {
#pragma unroll
            for (int k = 0; k < 3; ++k) o[k + 3 * c] = JT[3 * k] * g[0] + JT[1 + 3 * k] * g[1] + JT[2 + 3 * k] * g[2];
        } else {
#pragma unroll
            for (int j = 0; j < D; ++j) o[j + D * c] = g[j];
        }
    }
}

}  // namespace anifem
