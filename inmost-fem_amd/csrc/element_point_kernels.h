// Element matrices with a coefficient given at the quadrature points, on the
// matrix cores.
//
// Per component block the element matrices of a tile of tets are one product
//   C[t][e] = sum_{n, kk} K_t[n, kk] R[e][n, kk],   e = ib0 + nfB0 ia0,
// with K_t[n] = w_n |T| T_B^T D_n T_A formed per tet and point and R the table
// of basis products at the points.  The inner dimension is q KB (q points, KB
// values of K, 6 where K is symmetric): 144 for P3 with 24 points, so the
// product is bound by arithmetic, not by the matrices written.  It runs on
// v_mfma_f64_16x16x4 (FP32: v_mfma_f32_16x16x4), 16 tets x 16 entries x 4 terms
// per instruction, with the accumulation in the precision of the mode.
//
// Work split: a workgroup of four waves takes 16 MT WT tets; K of the tile is
// formed once into LDS (lane = tet, the waves share the points).  WT waves
// share the tets and 4 / WT the 16-entry tiles of R, NTW tiles per wave, all
// accumulated at once, so that R is read once per workgroup (WT = 1), from L2,
// in the lane order of the instruction's B operand (RefFragDev).  The finished
// entries go through LDS, 16 WT tets at a time, over the K tile, and are
// written as one contiguous range: stored from the accumulators, the transposed
// half of a symmetric matrix makes 8-byte writes (P3, 24 points, 93,701 tets,
// FP64: 168 us, 34 TFLOP/s, against 296 us; 25.0 ms before, with R read value
// by value in a scalar product per entry).
#pragma once

#include "element_kernels.h"

namespace anifem {

typedef double double4_t __attribute__((ext_vector_type(4)));

// Operand and accumulator types of the 16x16x4 instructions.  Lane l (j = l %
// 16, g = l / 16) holds A[row j][column g], B[row g][column j] and four values
// of D in column j: rows 4i + g (FP64) or 4g + i (FP32), i = 0..3.
template <typename T>
struct Mfma16;
template <>
struct Mfma16<double> {
    typedef double4_t acc;
    static __device__ __forceinline__ acc mul(double a, double b, acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int i, int g) { return 4 * i + g; }
};
template <>
struct Mfma16<float> {
    typedef float4_t acc;
    static __device__ __forceinline__ acc mul(float a, float b, acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int i, int g) { return 4 * g + i; }
};

// Values per tet of the K tile: an odd number of instructions, so that the
// rows of the tets of one operand start in different LDS banks.
__host__ __device__ inline int point_stride(int ks) { return 4 * (ks + 1); }

// LDS of a workgroup: the K tile, over which the staged entries (16 WT tets of
// E0) are laid afterwards, then the per-DOF factors of RT0 / ND0.
__host__ __device__ inline size_t point_scale_offset(int tile, int ks, int stage, int elem_bytes) {
    const size_t k = (size_t)tile * point_stride(ks), n = k > (size_t)stage ? k : (size_t)stage;
    return (n * elem_bytes + 15) / 16 * 16;
}
__host__ __device__ inline size_t point_lds_bytes(int tile, int ks, int stage, int elem_bytes, int n_scale) {
    return point_scale_offset(tile, ks, stage, elem_bytes) + (size_t)tile * n_scale * sizeof(double);
}

// SYM: K symmetric (one 3-dimensional operator on both sides of a scalar or
// Piola-mapped space, a NULL / SCALAR / SYMMETRIC tensor): its 6 distinct
// values against the R whose columns of K(a, b) and K(b, a) are summed, for
// the entries ib >= ia only, each stored at (ib, ia) and (ia, ib).
// a.ks: instructions along the inner dimension; a.frag, a.ent: R in operand
// order and its entries (RefFragDev), at most 16 NTW 4 / WT of them.
// Two waves per SIMD at least: the accumulators then stay in the registers the
// instruction can use directly (with one, the compiler moved them through the
// accumulation registers in every step).
template <int DA0, int DB0, typename T, bool PIOLA, bool SYM, int MT, int NTW, int WT>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2))) void element_point_kernel(ElemArgs a) {
    static_assert(!SYM || (DA0 == 3 && DB0 == 3), "packed K: 3 x 3 blocks");
    static_assert(MT == 1 || WT == 1, "the staged tets are consecutive");
    constexpr int KB = DA0 * DB0, KBC = SYM ? 6 : KB;
    constexpr int TILE = 16 * MT * WT, PARTS = kBlock / TILE, WE = kBlock / 64 / WT;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* Ks = reinterpret_cast<T*>(smem_raw);
    const int ks = a.ks, stride = point_stride(ks);
    const int E0 = a.nfA0 * a.nfB0;
    double* Ss = reinterpret_cast<double*>(smem_raw + point_scale_offset(TILE, ks, 16 * WT * E0, (int)sizeof(T)));
    const bool scaled = PIOLA && (a.scA | a.scB) != 0;
    const int ns = a.nfA0 + a.nfB0;
    const int64_t tile0 = (int64_t)blockIdx.x * TILE;
    const int ntile = (int)((a.n - tile0) < TILE ? (a.n - tile0) : TILE);

    // this lane's tet and share of the points
    const int t = threadIdx.x % TILE, part = threadIdx.x / TILE;
    const int64_t r = tile0 + t;
    const bool live = t < ntile;
    double P[4][3], PSI[9], JT[9], det = 1.0, mes = 0.0, nrm[3];
    if (live) {
        load_tet<false>(a, r, P);
        tet_geometry(P, PSI, det);
        mes = a.face < 0 ? fabs(det) / 6.0 : face_measure(P, a.face, a.dot_normal ? nrm : nullptr);
        if constexpr (PIOLA) {
            tet_jacobian_t(P, JT);
            if (scaled && part == 0) {
                double* St = Ss + t * ns;
                for (int i = 0; i < a.nfA0; ++i) St[i] = a.scA ? dof_scale(a.scA, P, det, i) : 1.0;
                for (int i = 0; i < a.nfB0; ++i) St[a.nfA0 + i] = a.scB ? dof_scale(a.scB, P, det, i) : 1.0;
            }
        }
    }
    const double* nr = a.face >= 0 && a.dot_normal ? nrm : nullptr;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), wt = w % WT, we = w / WT;
    const int l = threadIdx.x % 64, j = l % 16, g = l / 16;
    const int nt = (a.n_ent + 15) / 16;
    const int nfB = a.nfB0 * a.ncB;
    typedef typename Mfma16<T>::acc acc_t;
    // this wave's tiles (the last one again where it has fewer than NTW) and
    // the entry of each that lane column j holds
    const T* f[NTW];
    int ent[NTW];
#pragma unroll
    for (int i = 0; i < NTW; ++i) {
        const int et = we + i * WE;
        f[i] = static_cast<const T*>(a.frag) + (int64_t)(et < nt ? et : nt - 1) * ks * 64;
        ent[i] = et < nt ? a.ent[et * 16 + j] : kNoEntry;
    }

    for (int b = 0; b < a.ncA * a.ncB; ++b) {
        const int cb = b / a.ncA, ca = b % a.ncA;
        // K of the tile (zero for the tets past the end and the padding)
        T* Kt = Ks + t * stride;
        auto put = [&](int n, const double* Kb, double s) {
            if constexpr (SYM) {
#pragma unroll
                for (int c = 0; c < 3; ++c)
#pragma unroll
                    for (int d = 0; d <= c; ++d) Kt[n * KBC + sym_pack(d, c)] = (T)(s * Kb[c * 3 + d]);
            } else {
#pragma unroll
                for (int i = 0; i < KB; ++i) Kt[n * KBC + i] = (T)(s * Kb[i]);
            }
        };
        if (SYM && a.ttype == ANIFEM_TENSOR_SCALAR && a.selA <= ANIFEM_GRAD) {
            // one T^T T per tet, scaled by the points' coefficients (a single
            // derivative takes part of T only: geometry_block's selector)
            double K1[KB];
            const double* Tm = PIOLA && a.mapA ? JT : PSI;
#pragma unroll
            for (int i = 0; i < KB; ++i) {
                const int c = i / 3, d = i % 3;
                K1[i] = live ? mes * (Tm[c] * Tm[d] + Tm[c + 3] * Tm[d + 3] + Tm[c + 6] * Tm[d + 6]) : 0.0;
            }
            const double* D = a.D + (live ? r : 0);
#pragma unroll 4
            for (int n = part; n < a.q; n += PARTS) put(n, K1, a.wq[n] * D[(int64_t)n * a.coef_n]);
        } else {
            for (int n = part; n < a.q; n += PARTS) {
                double Kb[KB];
                if (live) {
                    geometry_block<DA0, DB0, double>(a, r, PSI, mes * a.wq[n], n, cb, ca, Kb, nr, PIOLA ? JT : nullptr);
                } else {
                    for (int i = 0; i < KB; ++i) Kb[i] = 0.0;
                }
                put(n, Kb, 1.0);
            }
        }
        if (part == PARTS - 1)
            for (int i = a.q * KBC; i < 4 * ks; ++i) Kt[i] = T(0);
        __syncthreads();

        // R kStep instructions at a time with the next kStep in flight
        const T* Ka = Ks + (wt * 16 * MT + j) * stride + g;
        constexpr int kStep = NTW >= 4 ? 2 : 4;
        acc_t acc[NTW][MT];
        T rn[NTW][kStep];
#pragma unroll
        for (int i = 0; i < NTW; ++i) {
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[i][m] = acc_t{0, 0, 0, 0};
#pragma unroll
            for (int u = 0; u < kStep; ++u) rn[i][u] = f[i][u * 64 + l];
        }
        for (int k = 0; k < ks; k += kStep) {
            T rb[NTW][kStep], ka[kStep][MT];
            const int kn = k + kStep < ks ? k + kStep : 0;
#pragma unroll
            for (int u = 0; u < kStep; ++u)
#pragma unroll
                for (int m = 0; m < MT; ++m) ka[u][m] = Ka[m * 16 * stride + 4 * (k + u)];
#pragma unroll
            for (int i = 0; i < NTW; ++i)
#pragma unroll
                for (int u = 0; u < kStep; ++u) {
                    rb[i][u] = rn[i][u];
                    rn[i][u] = f[i][(kn + u) * 64 + l];
                }
#pragma unroll
            for (int u = 0; u < kStep; ++u)
#pragma unroll
                for (int i = 0; i < NTW; ++i)
#pragma unroll
                    for (int m = 0; m < MT; ++m) acc[i][m] = Mfma16<T>::mul(ka[u][m], rb[i][u], acc[i][m]);
        }

        // 16 WT tets at a time through LDS to the output
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < NTW; ++i) {
                if (ent[i] == kNoEntry) continue;
                const int ib0 = ent[i] & 0xFF, ia0 = ent[i] >> 8;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int tv = 16 * wt + Mfma16<T>::row(v, g);  // row of the stage
                    T x = acc[i][m][v];
                    if constexpr (PIOLA) {
                        if (scaled) {
                            const double* St = Ss + (tv + 16 * m) * ns;  // MT = 1 or WT = 1
                            x = (T)((double)x * (St[ia0] * St[a.nfA0 + ib0]));
                        }
                    }
                    T* row = Ks + tv * E0;
                    row[ib0 + a.nfB0 * ia0] = x;
                    if constexpr (SYM) row[ia0 + a.nfB0 * ib0] = x;
                }
            }
            __syncthreads();
            const int live_tets = ntile - 16 * m < 16 * WT ? ntile - 16 * m : 16 * WT;
            T* out = static_cast<T*>(a.out) + (tile0 + 16 * m) * a.E;
            constexpr int V = 16 / (int)sizeof(T);
            if (a.ncA * a.ncB == 1 && E0 % V == 0 && (reinterpret_cast<uintptr_t>(a.out) & 15) == 0) {
                const float4* src = reinterpret_cast<const float4*>(Ks);
                float4* dst = reinterpret_cast<float4*>(out);
                for (int i = threadIdx.x; i < live_tets * (E0 / V); i += kBlock) dst[i] = src[i];
            } else {
                for (int i = threadIdx.x; i < live_tets * E0; i += kBlock) {
                    const int tv = i / E0, e0 = i - tv * E0, ia0 = e0 / a.nfB0, ib0 = e0 - ia0 * a.nfB0;
                    out[(int64_t)tv * a.E + (ib0 + a.nfB0 * cb) + nfB * (ia0 + a.nfA0 * ca)] = Ks[i];
                }
            }
        }
        if (b + 1 < a.ncA * a.ncB) __syncthreads();  // K is rewritten for the next block
    }
}

}  // namespace anifem
