// Launch of the fused RT0 / ND0 assembly (piola_kernels.h).
#include <hip/hip_runtime.h>

#include "anifem_common.h"
#include "piola_kernels.h"

namespace anifem {

namespace {

template <int D0, int KBC, int NF, typename T>
int launch(const BlockArgs& a, double* rows, int64_t n, size_t max_lds, hipStream_t s) {
    const size_t lds = block_lds_layout(a.max_values, a.max_pairs, a.max_slots, (int)sizeof(T), NF * NF * pad16<T>(KBC),
                                        0).total;
    if (lds > max_lds) return ANIFEM_ERR_DIMS;
    hipLaunchKernelGGL((piola_geometry_kernel<D0, KBC, NF, T>), dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock),
                       kBlock * piola_rowlen(NF, KBC) * sizeof(double), s, a, rows, n);
    ANIFEM_HIP_CHECK(hipGetLastError());
    if (a.n_blocks == 0) return ANIFEM_OK;
    hipLaunchKernelGGL((row_block_piola_kernel<KBC, NF, T>), dim3((unsigned)(8 * ((a.n_blocks + 7) / 8))), dim3(kBlock),
                       lds, s, a, (const double*)rows);
    ANIFEM_HIP_CHECK(hipGetLastError());
    return ANIFEM_OK;
}

// sym: K packed, in FP64 only.
template <int NF, typename T>
int launch_dim(int d0, bool sym, const BlockArgs& a, double* rows, int64_t n, size_t max_lds, hipStream_t s) {
    if (d0 == 1) return launch<1, 1, NF, T>(a, rows, n, max_lds, s);
    if constexpr (sizeof(T) == 8) {
        if (sym) return launch<3, 6, NF, T>(a, rows, n, max_lds, s);
    }
    return launch<3, 9, NF, T>(a, rows, n, max_lds, s);
}

}  // namespace

// Bytes of the cells' rows for nf local DOFs of a d0-component reference field, in
// the longest form (K not packed): a pass in the other precision, whose rows may
// be longer, then finds room without another allocation.
size_t piola_row_bytes(int nf, int d0, int64_t n) {
    return (size_t)n * piola_rowlen(nf, d0 == 1 ? 1 : 9) * sizeof(double);
}

int launch_piola(int d0, bool sym, bool fp64, const BlockArgs& a, double* rows, int64_t n, size_t max_lds,
                 hipStream_t s) {
    const int nf = a.kinds[0].nf;
    if (nf == 4) return fp64 ? launch_dim<4, double>(d0, sym, a, rows, n, max_lds, s) : launch_dim<4, float>(d0, sym, a, rows, n, max_lds, s);
    if (nf == 6) return fp64 ? launch_dim<6, double>(d0, sym, a, rows, n, max_lds, s) : launch_dim<6, float>(d0, sym, a, rows, n, max_lds, s);
    return ANIFEM_ERR_ARG;
}

}  // namespace anifem
