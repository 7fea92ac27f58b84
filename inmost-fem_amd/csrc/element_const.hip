// Launch of the constant-tensor element kernel (element_const_kernels.h).
#include <hip/hip_runtime.h>

#include "anifem_common.h"
#include "element_const_kernels.h"

namespace anifem {

namespace {

template <int DA0, int DB0, int NCA, int NCB, typename T, bool PIOLA, bool SYM>
int launch(ElemArgs a, hipStream_t s) {
    const int kstride = NCA * NCB * const_block_len<T>(SYM ? 6 : DA0 * DB0);
    const int n_scale = (a.scA | a.scB) ? a.nfA0 + a.nfB0 : 0;
    auto lds = [&](int tile) {
        return element_scale_offset(tile, kstride, (int)sizeof(T)) + (size_t)tile * n_scale * sizeof(double);
    };
    // Cells per workgroup: 256 while five workgroups share a CU's LDS (the
    // stores of some then cover the geometry of the others); fewer for small
    // batches, whose time is the length of one workgroup's chain.
    // The Piola spaces' geometry is long and its registers let three workgroups
    // share a CU (so 48 KB each): between 384 and 768 of them, which one round
    // holds, where 512 to 1,024 ran a second, and 256 cells also where 32 KB
    // allowed 128 or 64.  RT0 IDEN, general tensor: 16,000 cells 17.1 -> 10.2 us,
    // 100,003 25.8 -> 18.6; ND0 GRAD 600,000 168 -> 122.
    const size_t lds_max = (PIOLA ? 48 : 32) * 1024;
    const int64_t least = PIOLA ? 384 : 512;
    int tile = kBlock;
    while (tile > 16 && (lds(tile) > lds_max || a.n < least * tile)) tile /= 2;
    a.tile = tile;
    const dim3 grid((unsigned)((a.n + tile - 1) / tile));
    // row pairs need an even number of rows per component and an output
    // aligned to the pair
    if (a.nfB0 % 2 == 0 && (reinterpret_cast<uintptr_t>(a.out) & (2 * sizeof(T) - 1)) == 0)
        hipLaunchKernelGGL((element_const_kernel<DA0, DB0, NCA, NCB, T, PIOLA, SYM, 2>), grid, dim3(kBlock), lds(tile),
                           s, a);
    else
        hipLaunchKernelGGL((element_const_kernel<DA0, DB0, NCA, NCB, T, PIOLA, SYM, 1>), grid, dim3(kBlock), lds(tile),
                           s, a);
    ANIFEM_HIP_CHECK(hipGetLastError());
    return ANIFEM_OK;
}

template <int DA0, int DB0, int NCA, int NCB, typename T, bool SYM = false>
int launch_map(const ElemArgs& a, hipStream_t s) {
    return (a.mapA | a.mapB | a.scA | a.scB) ? launch<DA0, DB0, NCA, NCB, T, true, SYM>(a, s)
                                             : launch<DA0, DB0, NCA, NCB, T, false, SYM>(a, s);
}

template <int DA0, int DB0, typename T>
int launch_nc(int ncA, int ncB, bool sym, const ElemArgs& a, hipStream_t s) {
    if constexpr (DA0 == 3 && DB0 == 3) {
        if (ncA == 1 && ncB == 1 && sym) return launch_map<3, 3, 1, 1, T, true>(a, s);
    }
    if (ncA == 1 && ncB == 1) return launch_map<DA0, DB0, 1, 1, T>(a, s);
    if (ncA == 3 && ncB == 3) return launch_map<DA0, DB0, 3, 3, T>(a, s);
    if (ncA == 1 && ncB == 3) return launch_map<DA0, DB0, 1, 3, T>(a, s);
    if (ncA == 3 && ncB == 1) return launch_map<DA0, DB0, 3, 1, T>(a, s);
    return ANIFEM_ERR_ARG;
}

template <typename T>
int launch_dims(const anifem_op& opA, const anifem_op& opB, bool sym, const ElemArgs& a, hipStream_t s) {
    const int dA = ref_dim(opA.op, opA.fem), dB = ref_dim(opB.op, opB.fem);
    if (dA == 3 && dB == 3) return launch_nc<3, 3, T>(opA.ncomp, opB.ncomp, sym, a, s);
    if (dA == 1 && dB == 1) return launch_nc<1, 1, T>(opA.ncomp, opB.ncomp, sym, a, s);
    if (dA == 3 && dB == 1) return launch_nc<3, 1, T>(opA.ncomp, opB.ncomp, sym, a, s);
    if (dA == 1 && dB == 3) return launch_nc<1, 3, T>(opA.ncomp, opB.ncomp, sym, a, s);
    return ANIFEM_ERR_ARG;
}

}  // namespace

// Element matrices with one carried point (a.q == 1); `sym`: K symmetric.
int launch_element_const(const anifem_op& opA, const anifem_op& opB, bool sym, bool fp64, const ElemArgs& a,
                         hipStream_t s) {
    return fp64 ? launch_dims<double>(opA, opB, sym && a.Rds, a, s) : launch_dims<float>(opA, opB, sym && a.Rfs, a, s);
}

}  // namespace anifem
