// Element matrices with a tensor constant over each tet (or one point).
//
// A(ib, ia) = sum_kk K_t[kk] R[rr(ib, ia)][kk], written once: the matrices are
// nearly all of the bytes that move, so the kernel has to keep the stores
// running.  One lane per entry, reading K from LDS value by value, was bound by
// those reads (9 of 8 bytes per entry); here
//   * a lane owns VEC consecutive rows of a column (16-byte stores in FP64) and,
//     for vector spaces, two columns of every trial component, so one K block
//     read serves 2 VEC products;
//   * K blocks are 16-byte aligned in LDS and read as 16-byte words;
//   * a symmetric K (SYM) is packed to 6 values against the column-summed R;
//   * the lanes of consecutive tets store one contiguous range.
// FP64 P2 with a symmetric tensor, 1,572,864 tets: 463 us -> 364 us (4.1 TB/s; with
// 128 and 64 tets per workgroup 374 and 446 us); FP32 P2^3 elasticity, 663,552
// tets: 952 us -> 528 us (4.7 TB/s; 969 us with nontemporal stores, which leave the
// columns' shared lines unmerged).
#pragma once

#include "element_kernels.h"

namespace anifem {

// Values of a K block in LDS: padded to 16 bytes.
template <typename T>
__host__ __device__ constexpr int const_block_len(int kbc) {
    return kbc == 1 ? 1 : (kbc + 16 / (int)sizeof(T) - 1) / (16 / (int)sizeof(T)) * (16 / (int)sizeof(T));
}

// Trial columns per lane and component.
template <int NCA>
__host__ __device__ constexpr int const_columns() {
    return NCA == 3 ? 2 : 1;
}

template <int DA0, int DB0, int NCA, int NCB, typename T, bool PIOLA, bool SYM, int VEC>
__global__ __launch_bounds__(kBlock) void element_const_kernel(ElemArgs a) {
    static_assert(!SYM || (DA0 == 3 && DB0 == 3 && NCA == 1 && NCB == 1), "packed K: 3 x 3 scalar blocks");
    constexpr int KB = DA0 * DB0, KBC = SYM ? 6 : KB, KBL = const_block_len<T>(KBC), NB = NCA * NCB;
    constexpr int J = const_columns<NCA>();
    extern __shared__ __align__(16) unsigned char smem_raw[];
    T* Ks = reinterpret_cast<T*>(smem_raw);
    double* Ss = reinterpret_cast<double*>(smem_raw + element_scale_offset(a.tile, NB * KBL, (int)sizeof(T)));
    const int64_t tile0 = (int64_t)blockIdx.x * a.tile;
    const int ntile = (int)((a.n - tile0) < a.tile ? (a.n - tile0) : a.tile);
    const bool scaled = PIOLA && (a.scA | a.scB) != 0;
    const int ns = a.nfA0 + a.nfB0;

    // K: one lane per tet and share of the component blocks (a.tile and so the
    // number of shares are powers of two)
    const int t1 = threadIdx.x & (a.tile - 1), parts = kBlock / a.tile, part = threadIdx.x / a.tile;
    if (t1 < ntile && part < NB) {
        const int64_t r = tile0 + t1;
        double P[4][3], PSI[9], JT[9], det, nrm[3];
        load_tet<false>(a, r, P);
        tet_geometry(P, PSI, det);
        // volume |det|/6, or the face's area (int_face.inl:40-43, 79-84)
        const double mes = a.face < 0 ? fabs(det) / 6.0 : face_measure(P, a.face, a.dot_normal ? nrm : nullptr);
        const double* nr = a.face >= 0 && a.dot_normal ? nrm : nullptr;
        if constexpr (PIOLA) tet_jacobian_t(P, JT);
        T* Kt = Ks + t1 * (NB * KBL);
        bool lame = false;
        if constexpr (NCA == 3 && NCB == 3 && KB == 9 && !PIOLA) {
            // isotropic elasticity in closed form: with T(j, a) = PSI[a + 3 j],
            // K_(cb,ca)(b, a) = lam T(cb,b) T(ca,a) + mu (T(ca,b) T(cb,a) + d_{cb,ca} (T^T T)(b,a))
            lame = a.ttype == ANIFEM_TENSOR_LAME && a.selA == ANIFEM_GRAD && a.selB == ANIFEM_GRAD;
            if (lame) {
                const bool cst = a.storage == ANIFEM_COEF_CONST;
                const double lam = mes * (cst ? a.D[0] : a.D[r]), mu = mes * (cst ? a.D[1] : a.D[a.coef_n + r]);
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    if ((b & (parts - 1)) != part) continue;
                    const int cb = b / NCA, ca = b % NCA;
#pragma unroll
                    for (int i = 0; i < 9; ++i) {
                        const int p = i / 3, q = i % 3;
                        double v = PSI[q + 3 * cb] * PSI[p + 3 * ca];
                        if (cb == ca) v += PSI[p] * PSI[q] + PSI[p + 3] * PSI[q + 3] + PSI[p + 6] * PSI[q + 6];
                        Kt[b * KBL + i] = (T)(lam * (PSI[p + 3 * cb] * PSI[q + 3 * ca]) + mu * v);
                    }
                }
            }
        }
        if (!lame) {
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if ((b & (parts - 1)) != part) continue;
                double Kb[KB];
                geometry_block<DA0, DB0, double>(a, r, PSI, mes, 0, b / NCA, b % NCA, Kb, nr, PIOLA ? JT : nullptr);
                if constexpr (SYM) {
#pragma unroll
                    for (int c = 0; c < 3; ++c)
#pragma unroll
                        for (int d = 0; d <= c; ++d) Kt[sym_pack(d, c)] = (T)Kb[c * 3 + d];
                } else {
#pragma unroll
                    for (int i = 0; i < KB; ++i) Kt[b * KBL + i] = (T)Kb[i];
                }
            }
        }
        if (scaled && part == 0) {
            double* St = Ss + t1 * ns;
            for (int i = 0; i < a.nfA0; ++i) St[i] = a.scA ? dof_scale(a.scA, P, det, i) : 1.0;
            for (int i = 0; i < a.nfB0; ++i) St[a.nfA0 + i] = a.scB ? dof_scale(a.scB, P, det, i) : 1.0;
        }
    }
    __syncthreads();

    // a lane takes VEC rows x J columns of every component.  A matrix of more
    // than kBlock such items (P3^3: 30 x 10) goes in passes of whole columns:
    // J C of them from c0, over all tets, the tets dealt out to NG groups of lanes.
    // Passes of kBlock items, broken inside columns, left a last one of 44 lanes and
    // lines stored in two parts: P3^3 elasticity, 100,003 tets, FP64 692 -> 563 us
    // (5.1 TB/s), FP32 458 -> 378 us.  Fewer columns where a group of all of them
    // would leave a quarter of the lanes idle (P2^3 against P3^3: 150 of 256)
    const int nfB = a.nfB0 * NCB, rows = nfB / VEC;
    const T* R = reinterpret_cast<const T*>(
        sizeof(T) == 8 ? static_cast<const void*>(SYM ? a.Rds : a.Rd) : static_cast<const void*>(SYM ? a.Rfs : a.Rf));
    struct alignas(VEC * sizeof(T)) Vec {
        T v[VEC];
    };
    for (int c0 = 0, C; c0 < a.nfA0; c0 += J * C) {
        C = (a.nfA0 - c0 + J - 1) / J;
        if (C > kBlock / rows) C = kBlock / rows;
        while (C > 1 && rows * C * (kBlock / (rows * C)) < 3 * kBlock / 4) --C;
        const int L = rows * C, NG = kBlock / L, g = threadIdx.x / L, item = threadIdx.x - g * L;
        if (g >= NG) continue;
        const int c = c0 + item / rows, ib = VEC * (item % rows), cb = ib / a.nfB0, ib0 = ib - cb * a.nfB0;
        T Rr[J][VEC][KBC];
#pragma unroll
        for (int j = 0; j < J; ++j)
#pragma unroll
            for (int v = 0; v < VEC; ++v)
#pragma unroll
                for (int kk = 0; kk < KBC; ++kk) {
                    const int ia0 = c + C * j;
                    Rr[j][v][kk] = ia0 < a.nfA0 ? R[(ib0 + v + a.nfB0 * ia0) * KBC + kk] : T(0);
                }
        for (int t = g; t < ntile; t += NG) {
            T* out = static_cast<T*>(a.out) + (tile0 + t) * a.E + ib;
            const double* St = Ss + t * ns;
#pragma unroll
            for (int ca = 0; ca < NCA; ++ca) {
                T k[KBL];
                const T* Kt = static_cast<const T*>(
                    __builtin_assume_aligned(Ks + (t * NB + cb * NCA + ca) * KBL, KBC == 1 ? sizeof(T) : 16));
#pragma unroll
                for (int kk = 0; kk < KBL; ++kk) k[kk] = Kt[kk];
#pragma unroll
                for (int j = 0; j < J; ++j) {
                    const int ia0 = c + C * j;
                    if (J > 1 && ia0 >= a.nfA0) continue;
                    Vec o;
#pragma unroll
                    for (int v = 0; v < VEC; ++v) {
                        T acc = 0;
#pragma unroll
                        for (int kk = 0; kk < KBC; ++kk) acc += k[kk] * Rr[j][v][kk];
                        if constexpr (PIOLA) {
                            if (scaled) acc = (T)((double)acc * (St[ia0] * St[a.nfA0 + ib0 + v]));
                        }
                        o.v[v] = acc;
                    }
                    *reinterpret_cast<Vec*>(out + nfB * (ia0 + a.nfA0 * ca)) = o;
                }
            }
        }
    }
}

}  // namespace anifem
