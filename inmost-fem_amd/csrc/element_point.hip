// Launch of the per-point element kernel (element_point_kernels.h).
#include <hip/hip_runtime.h>

#include "anifem_common.h"
#include "element_point_kernels.h"

namespace anifem {

namespace {

// One launch shape: 16 MT WT tets per workgroup, NTW tiles of 16 entries per
// wave, WT waves along the tets.
template <int DA0, int DB0, typename T, bool PIOLA, bool SYM, int MT, int NTW, int WT>
int launch(const ElemArgs& a, hipStream_t s) {
    constexpr int TILE = 16 * MT * WT;
    const size_t lds = point_lds_bytes(TILE, a.ks, 16 * WT * a.nfA0 * a.nfB0, (int)sizeof(T),
                                       (a.scA | a.scB) ? a.nfA0 + a.nfB0 : 0);
    hipLaunchKernelGGL((element_point_kernel<DA0, DB0, T, PIOLA, SYM, MT, NTW, WT>),
                       dim3((unsigned)((a.n + TILE - 1) / TILE)), dim3(kBlock), lds, s, a);
    ANIFEM_HIP_CHECK(hipGetLastError());
    return ANIFEM_OK;
}

// The launch shape by the number of entry tiles: up to two, every wave takes
// its own 16 tets and both tiles (P1, RT0, ND0: splitting the tiles would
// leave waves without one); up to 16 the waves split the tiles over 64 tets;
// beyond (P3 with a general tensor: 25), over 32, where the accumulators of
// seven tiles still fit the registers.  16 tets per workgroup where K of more
// exceeds half a CU's LDS, or where the launch would leave workgroup slots of
// the 256 CUs empty.  False: K or the staged entries of 16 tets exceed 64 KB
// (rules beyond about 55 points of a full 3 x 3 tensor), element_kernel's case.
template <int DA0, int DB0, typename T, bool PIOLA, bool SYM>
int launch_shape(const ElemArgs& a, hipStream_t s, bool* taken) {
    const int nt = (a.n_ent + 15) / 16, E0 = a.nfA0 * a.nfB0, n_scale = (a.scA | a.scB) ? a.nfA0 + a.nfB0 : 0;
    auto lds = [&](int tile, int stage_tets) {
        return point_lds_bytes(tile, a.ks, stage_tets * E0, (int)sizeof(T), n_scale);
    };
    if (nt > 28 || lds(16, 16) > 64 * 1024) return ANIFEM_OK;
    *taken = true;
    if (nt <= 2 && lds(64, 64) <= 80 * 1024) return launch<DA0, DB0, T, PIOLA, SYM, 1, 2, 4>(a, s);
    const bool wide = a.n >= 512 * 64;
    if (nt <= 4) {
        if (wide && lds(64, 16) <= 80 * 1024) return launch<DA0, DB0, T, PIOLA, SYM, 4, 1, 1>(a, s);
        return launch<DA0, DB0, T, PIOLA, SYM, 1, 1, 1>(a, s);
    }
    if (nt <= 16) {
        if (wide && lds(64, 16) <= 80 * 1024) return launch<DA0, DB0, T, PIOLA, SYM, 4, 4, 1>(a, s);
        return launch<DA0, DB0, T, PIOLA, SYM, 1, 4, 1>(a, s);
    }
    if constexpr (!PIOLA) {  // RT0 and ND0 have at most 6 x 20 entries
        if (a.n >= 512 * 32 && lds(32, 16) <= 80 * 1024) return launch<DA0, DB0, T, false, SYM, 2, 7, 1>(a, s);
        return launch<DA0, DB0, T, false, SYM, 1, 7, 1>(a, s);
    }
    *taken = false;
    return ANIFEM_OK;
}

template <int DA0, int DB0, typename T, bool SYM>
int launch_map(const ElemArgs& a, hipStream_t s, bool* taken) {
    return (a.mapA | a.mapB | a.scA | a.scB) ? launch_shape<DA0, DB0, T, true, SYM>(a, s, taken)
                                             : launch_shape<DA0, DB0, T, false, SYM>(a, s, taken);
}

template <typename T>
int launch_dims(int dA, int dB, bool sym, const ElemArgs& a, hipStream_t s, bool* taken) {
    if (dA == 3 && dB == 3)
        return sym ? launch_map<3, 3, T, true>(a, s, taken) : launch_map<3, 3, T, false>(a, s, taken);
    if (dA == 1 && dB == 1) return launch_map<1, 1, T, false>(a, s, taken);
    if (dA == 3 && dB == 1) return launch_map<3, 1, T, false>(a, s, taken);
    if (dA == 1 && dB == 3) return launch_map<1, 3, T, false>(a, s, taken);
    return ANIFEM_OK;
}

}  // namespace

// Element matrices with a coefficient at a.q > 1 points; `sym`: K symmetric
// (6 values per point).  *taken stays false where the call is element_kernel's.
int launch_element_point(const anifem_op& opA, const anifem_op& opB, int order, bool sym, bool fp64, ElemArgs a,
                         hipStream_t s, bool* taken) {
    const int dA = ref_dim(opA.op, opA.fem), dB = ref_dim(opB.op, opB.fem);
    // element_kernel refuses a call whose K of four tets exceeds 64 KB
    const int kstride = opA.ncomp * opB.ncomp * a.q * dA * dB, es = fp64 ? 8 : 4;
    const int ns = (a.scA | a.scB) ? a.nfA0 + a.nfB0 : 0;
    if (element_scale_offset(4, kstride, es) + 4 * ns * sizeof(double) > 64 * 1024) return ANIFEM_OK;
    if (!frag_fits(frag_steps(a.q, sym ? 6 : dA * dB), es)) return ANIFEM_OK;
    RefTensorDev R;  // as prepared for the call: the table is there
    const int rc = get_ref_tensor(opA.op, opA.fem, opB.op, opB.fem, order, true, &R, a.face);
    if (rc) return rc;
    const RefFragDev& f = sym ? R.frag_sym : R.frag;
    a.frag = fp64 ? static_cast<const void*>(f.f64) : static_cast<const void*>(f.f32);
    a.ent = f.ent;
    a.ks = f.ks;
    a.n_ent = f.n_ent;
    a.ncA = opA.ncomp;
    a.ncB = opB.ncomp;
    return fp64 ? launch_dims<double>(dA, dB, sym, a, s, taken) : launch_dims<float>(dA, dB, sym, a, s, taken);
}

}  // namespace anifem
