// Fused assembly of the vector-valued spaces RT0 and ND0 (one operator on both
// sides, tensors constant over each cell): a geometry launch and a row-block
// launch, as for the Lagrange spaces, in place of element matrices written to
// memory and read back.
//
// The matrix entry is A(ib, ia) = s_ib s_ia sum_kk K[kk] R[ib, ia][kk] with K the
// mapped tensor (geometry_block: T = J or PSI^T) and s the per-DOF factor
// (dof_scale) times the orientation sign (assembler.inl:154-164).  A cell's row
// holds s (NF values), K (6 if symmetric, 9 or 1) and its load vector (NF): 144
// bytes for ND0, where the matrix alone takes 288 written and, row by row,
// gathered again.  The pass is bound by the chain of dependent loads of a block
// (metadata, pairs, rows), which the other resident blocks cover, and no longer
// by bytes.  Curl-curl of ND0, 196,416 cells: six launches, 102 us -> two, 40 us.
#pragma once

#include "assembly_kernels.h"

namespace anifem {

// Doubles per cell: factors, K, load vector, rows 16-byte aligned.
__host__ __device__ constexpr int piola_rowlen(int nf, int kbc) { return (2 * nf + kbc + 1) / 2 * 2; }

// The row of cell r.  D0: components of the reference field; KBC: values of K
// carried (6: packed).  K and the load vector are rounded to T, the precision of
// the contraction.
template <int D0, int KBC, int NF, typename T>
__device__ __forceinline__ void piola_row(const BlockArgs& a, int64_t r, bool live, double2* out) {
    constexpr int KB = D0 * D0, LEN = piola_rowlen(NF, KBC);
    static_assert(KBC == KB || (KBC == 6 && KB == 9), "packed K: 3 x 3");
    if (!live) return;
    double P[4][3], PSI[9], JT[9], det, Kb[KB], row[LEN];
    load_tet<true>(a.m, r, P);
    tet_geometry(P, PSI, det);
    tet_jacobian_t(P, JT);
    const double mes = fabs(det) / 6.0;
    const uint64_t sm = a.signmask[r];
    // the space's size per DOF: |face| / (|det J| / 2) (RT0) or |edge| (ND0)
    double size[NF];
#pragma unroll
    for (int i = 0; i < NF; ++i) size[i] = dof_scale(NF == 4 ? 1 : 2, P, det, i);
#pragma unroll
    for (int i = 0; i < NF; ++i) {
        const double s = a.m.scA == 0 ? 1.0 : (a.m.scA == 3 ? size[i] / det : size[i]);
        row[i] = (sm >> i) & 1 ? -s : s;
    }
    geometry_block<D0, D0, double>(a.m, r, PSI, mes, 0, 0, 0, Kb, nullptr, JT);
    if constexpr (KBC != KB) {
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int d = 0; d <= c; ++d) row[NF + sym_pack(d, c)] = (double)(T)Kb[c * 3 + d];
    } else {
#pragma unroll
        for (int i = 0; i < KB; ++i) row[NF + i] = (double)(T)Kb[i];
    }
#pragma unroll
    for (int i = NF + KBC; i < LEN; ++i) row[i] = 0.0;
    if (a.has_rhs) {
        double KF[3];
        geometry_block<1, 3, double>(a.f, r, PSI, mes, 0, 0, 0, KF, nullptr, JT);
        const T* RF = reinterpret_cast<const T*>(sizeof(T) == 8 ? (const void*)a.f.Rd : (const void*)a.f.Rf);
#pragma unroll
        for (int i = 0; i < NF; ++i) {
            T f = 0;
#pragma unroll
            for (int k = 0; k < 3; ++k) f += (T)KF[k] * RF[i * 3 + k];
            f = (T)((double)f * size[i]);  // the factor of the values (IDEN)
            row[NF + KBC + i] = (sm >> i) & 1 ? -(double)f : (double)f;
        }
    }
#pragma unroll
    for (int i = 0; i < LEN / 2; ++i) out[i] = make_double2(row[2 * i], row[2 * i + 1]);
}

template <int D0, int KBC, int NF, typename T>
__global__ __launch_bounds__(kBlock) void piola_geometry_kernel(BlockArgs a, double* __restrict__ rows, int64_t n) {
    constexpr int LEN = piola_rowlen(NF, KBC);
    // the rows leave through LDS as one range: stored lane by lane, their
    // 16-byte pieces cost more than the rest (26 us at 196,416 cells against 18.5)
    extern __shared__ __align__(16) double2 stage[];
    const int64_t r0 = blockIdx.x * (int64_t)kBlock, r = r0 + threadIdx.x;
    if (r < 4) a.status[r] = 0;  // the counts of this pass are added by the row-block launch
    piola_row<D0, KBC, NF, T>(a, r, r < n, stage + threadIdx.x * (LEN / 2));
    __syncthreads();
    const int count = (int)(n - r0 < kBlock ? n - r0 : kBlock) * (LEN / 2);
    double2* out = reinterpret_cast<double2*>(rows + r0 * LEN);
    for (int i = threadIdx.x; i < count; i += kBlock) out[i] = stage[i];
}

// One workgroup per row block (phases A and B of row_block_kernel).
template <int KBC, int NF, typename T>
__global__ __launch_bounds__(kBlock) void row_block_piola_kernel(BlockArgs a, const double* __restrict__ rows) {
    constexpr int LEN = piola_rowlen(NF, KBC);
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int lenp = pad16<T>(KBC);
    const BlockLds L = block_lds_layout(a.max_values, a.max_pairs, a.max_slots, (int)sizeof(T), NF * NF * lenp, 0);
    double* vals = reinterpret_cast<double*>(smem_raw + L.vals);
    double* fvals = reinterpret_cast<double*>(smem_raw + L.fvals);
    uint16_t* sst = reinterpret_cast<uint16_t*>(smem_raw + L.sst);
    T* R = reinterpret_cast<T*>(smem_raw + L.R);
    // each XCD takes a contiguous range of the processing order (row_block_kernel)
    const int64_t per_xcd = (a.n_blocks + 7) / 8;
    const int64_t k = (int64_t)(blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (k >= a.n_blocks) return;  // uniform over the workgroup
    const BlockMeta M = a.meta[k];
    const bool has_pair = (int)threadIdx.x < M.np;
    // the pair's records, then its cell's row, requested before the staging
    const int64_t gp = M.p0 + (has_pair ? threadIdx.x : 0);
    const int64_t tet = has_pair ? a.pair_tet[gp] : 0;
    const int ibf = has_pair ? a.pair_ib[gp] : 0;
    uint32_t pw[NF / 2];
    const uint32_t* pg = reinterpret_cast<const uint32_t*>(a.pair_pos + M.q0 + (int64_t)(has_pair ? threadIdx.x : 0) * NF);
#pragma unroll
    for (int w = 0; w < NF / 2; ++w) pw[w] = has_pair ? pg[w] : 0u;
    const int ib = ibf & 63;
    const double* row = rows + tet * LEN;
    double rv[NF + KBC + (KBC & 1)];
#pragma unroll
    for (int i = 0; i < NF + KBC + (KBC & 1); i += 2) {
        const double2 v = *reinterpret_cast<const double2*>(row + i);
        rv[i] = v.x;
        rv[i + 1] = v.y;
    }
    const double sb = row[ib], f = a.has_rhs ? row[NF + KBC + ib] : 0.0;
    pad_copy(R, reinterpret_cast<const T*>(sizeof(T) == 8 ? (const void*)a.kinds[0].Rd : (const void*)a.kinds[0].Rf),
             NF * NF, KBC, lenp);
    block_copy(sst, a.sstart + M.s0, (int)M.ns);
    __syncthreads();
    int nonfinite = 0;
    if (has_pair) {
        const bool dir = (ibf & kPairDirichlet) != 0;
#pragma unroll
        for (int ia = 0; ia < NF; ++ia) {
            const int ps = (int)((pw[ia / 2] >> (16 * (ia & 1))) & 0xFFFFu);
            if (ps == kPosDropped) continue;
            const T* Rr = R + (ib + NF * ia) * lenp;
            T acc = 0;
#pragma unroll
            for (int i = 0; i < KBC; ++i) acc += (T)rv[NF + i] * Rr[i];
            const double v = (double)(T)((double)acc * (sb * rv[ia]));
            const double x = dir ? 1.0 : v;
            nonfinite += isfinite(x) ? 0 : 1;
            vals[ps] = x;
        }
        if (a.has_rhs) {
            const double fv = dir ? 0.0 : f;
            nonfinite += isfinite(fv) ? 0 : 1;
            fvals[threadIdx.x] = fv;
        }
    }
    __syncthreads();
    row_block_finish(a, M.r0, M.nr, M.s0, M.ns, M.np, M.nv, vals, fvals, sst);
    if (nonfinite) atomicAdd(&a.status[0], nonfinite);
}

}  // namespace anifem
