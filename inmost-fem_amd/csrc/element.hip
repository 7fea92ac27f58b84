// Batched element matrices: anifem_fem3dtet_batch (C ABI) and the launch
// helpers shared with the fused assembly.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>
#include <vector>

#include "anifem_common.h"
#include "apply_kernels.h"
#include "element_kernels.h"

namespace anifem {

// Operator-dependent part of ElemArgs; validates the pair like the reference's
// compile-time / runtime checks (int_tet.inl:94-104, diff_tensor.h:313-315).
// Element arguments of a volume integral (face < 0) or of the integral over
// one face, plain (fem3Dface) or of (D OpA(u)) . n (fem3DfaceN, dot_normal):
// there D has 3 dimB rows, and a.dimB is that row count (the tensor's layout).
static int prepare_args(const anifem_op& opA, const anifem_op& opB, const anifem_tensor* D, int order, int face,
                        int dot_normal, ElemArgs& a) {
    if (!op_valid(opA) || !op_valid(opB) || !D) return ANIFEM_ERR_ARG;
    if (face > 3 || (face < 0 && dot_normal)) return ANIFEM_ERR_ARG;
    const double *pts, *wts;
    if ((face < 0 ? quadrature(order, &pts, &wts) : triangle_quadrature(order, &pts, &wts)) < 0) return ANIFEM_ERR_ORDER;
    a.face = face < 0 ? -1 : face;
    a.dot_normal = dot_normal ? 1 : 0;
    a.nfA0 = nf_scalar(opA.fem);
    a.nfB0 = nf_scalar(opB.fem);
    // DIV / CURL / DUDX..DUDZ run as the gradient with a signed selector in
    // the tensor (element_kernels.h: op_map); the normal form takes them on
    // the trial side only
    if (dot_normal && opB.op != ANIFEM_IDEN && opB.op != ANIFEM_GRAD) return ANIFEM_ERR_ARG;
    // RT0 / ND0: the operator is the space's own (no selector); their values
    // follow from the reference fields through space_map's map and factors
    a.selA = fem_vector(opA.fem) ? ANIFEM_IDEN : opA.op;
    a.selB = fem_vector(opB.fem) ? ANIFEM_IDEN : opB.op;
    space_map(opA.op, opA.fem, a.mapA, a.scA);
    space_map(opB.op, opB.fem, a.mapB, a.scB);
    // GRAD of RT0 / ND0 (9 components) pairs with GRAD of RT0 / ND0 only, and
    // not in the normal form
    if ((a.mapA >= 3) != (a.mapB >= 3) || (a.mapA >= 3 && dot_normal)) return ANIFEM_ERR_ARG;
    a.dimA = op_dim(opA);
    a.dimB = op_dim(opB) * (dot_normal ? 3 : 1);
    a.E = a.nfA0 * opA.ncomp * a.nfB0 * opB.ncomp;
    a.ttype = D->type;
    a.storage = D->storage;
    a.D = D->data;
    const int nfA = a.nfA0 * opA.ncomp;
    a.p0_bcast = (a.dimA != a.dimB && nfA == 1 && a.dimA == 1) ? 1 : 0;
    if ((D->type == ANIFEM_TENSOR_NULL || D->type == ANIFEM_TENSOR_SCALAR) && a.dimA != a.dimB && !a.p0_bcast)
        return ANIFEM_ERR_DIMS;
    if (tensor_ddim(D->type, a.dimA, a.dimB) < 0) return ANIFEM_ERR_ARG;
    if (D->type != ANIFEM_TENSOR_NULL && !D->data) return ANIFEM_ERR_ARG;
    if (D->storage < ANIFEM_COEF_CONST || D->storage > ANIFEM_COEF_PER_POINT) return ANIFEM_ERR_ARG;
    RefTensorDev R;
    int rc = get_ref_tensor(opA.op, opA.fem, opB.op, opB.fem, order, D->storage == ANIFEM_COEF_PER_POINT, &R, a.face);
    if (rc) return rc;
    a.q = R.q;
    a.Rd = R.r64;
    a.Rf = R.r32;
    a.Rds = R.rs64;
    a.Rfs = R.rs32;
    a.rds_sym = R.rs_sym ? 1 : 0;
    a.wq = R.w;
    a.r16 = R.r16;
    a.r16_scale = R.r16_scale;
    a.e0pad = R.e0pad;
    return ANIFEM_OK;
}

int prepare_elem_args(const anifem_op& opA, const anifem_op& opB, const anifem_tensor* D, int order, ElemArgs& a) {
    return prepare_args(opA, opB, D, order, -1, 0, a);
}

// K symmetric: the same 3-dimensional operator of one scalar or Piola-mapped
// space on both sides, a NULL / SCALAR / SYMMETRIC tensor, no normal
// contraction.
static bool symmetric_k(const anifem_op& opA, const anifem_op& opB, const ElemArgs& a) {
    return opA.op == opB.op && opA.fem == opB.fem && opA.ncomp == 1 && opB.ncomp == 1 &&
           ref_dim(opA.op, opA.fem) == 3 && a.mapA == a.mapB && a.mapA < 3 && !a.dot_normal &&
           (a.ttype == ANIFEM_TENSOR_NULL || a.ttype == ANIFEM_TENSOR_SCALAR || a.ttype == ANIFEM_TENSOR_SYMMETRIC);
}

// Tensors constant over each tet (element_const.hip).
int launch_element_const(const anifem_op& opA, const anifem_op& opB, bool sym, bool fp64, const ElemArgs& a,
                         hipStream_t s);
// Per-point kernel (element_point.hip); refuses nothing: returns false in
// *taken where element_kernel has to serve the call.
int launch_element_point(const anifem_op& opA, const anifem_op& opB, int order, bool sym, bool fp64, ElemArgs a,
                         hipStream_t s, bool* taken);

// Tets per workgroup: as many as keep the LDS geometry tensors <= 32 KiB
// (several workgroups per CU), at most `cap`.
static int choose_tile(int kstride, int elem_bytes, int cap) {
    int t = cap;
    while (t > 4 && (size_t)t * kstride * elem_bytes > 32768) t /= 2;
    return t;
}

template <int DA0, int DB0, int NCA, int NCB, typename T>
static int launch_one(ElemArgs a, int cap, hipStream_t s) {
    const bool piola = (a.mapA | a.mapB | a.scA | a.scB) != 0;
    const int kstride = NCA * NCB * a.q * DA0 * DB0;
    a.tile = choose_tile(kstride, (int)sizeof(T), cap);
    size_t lds = (size_t)a.tile * kstride * sizeof(T);
    if (a.scA | a.scB)
        lds = element_scale_offset(a.tile, kstride, (int)sizeof(T)) + (size_t)a.tile * (a.nfA0 + a.nfB0) * sizeof(double);
    if (lds > 64 * 1024) return ANIFEM_ERR_ARG;
    const int64_t blocks = (a.n + a.tile - 1) / a.tile;
    if (blocks == 0) return ANIFEM_OK;
    if (piola)
        hipLaunchKernelGGL((element_kernel<DA0, DB0, NCA, NCB, T, true>), dim3((unsigned)blocks), dim3(kBlock), lds, s,
                           a);
    else
        hipLaunchKernelGGL((element_kernel<DA0, DB0, NCA, NCB, T, false>), dim3((unsigned)blocks), dim3(kBlock), lds,
                           s, a);
    ANIFEM_HIP_CHECK(hipGetLastError());
    return ANIFEM_OK;
}

template <typename T, int DA0, int DB0>
static int launch_nc(int ncA, int ncB, const ElemArgs& a, int cap, hipStream_t s) {
    if (ncA == 1 && ncB == 1) return launch_one<DA0, DB0, 1, 1, T>(a, cap, s);
    if (ncA == 3 && ncB == 3) return launch_one<DA0, DB0, 3, 3, T>(a, cap, s);
    if (ncA == 1 && ncB == 3) return launch_one<DA0, DB0, 1, 3, T>(a, cap, s);
    if (ncA == 3 && ncB == 1) return launch_one<DA0, DB0, 3, 1, T>(a, cap, s);
    return ANIFEM_ERR_ARG;
}

template <typename T>
int launch_element(const anifem_op& opA, const anifem_op& opB, int order, const ElemArgs& a, int cap, hipStream_t s) {
    const bool sym = symmetric_k(opA, opB, a);
    if (a.q == 1) return launch_element_const(opA, opB, sym, sizeof(T) == 8, a, s);
    bool taken = false;
    const int rc = launch_element_point(opA, opB, order, sym, sizeof(T) == 8, a, s, &taken);
    if (rc || taken) return rc;
    const int dA = ref_dim(opA.op, opA.fem), dB = ref_dim(opB.op, opB.fem);
    if (dA == 3 && dB == 3) return launch_nc<T, 3, 3>(opA.ncomp, opB.ncomp, a, cap, s);
    if (dA == 1 && dB == 1) return launch_nc<T, 1, 1>(opA.ncomp, opB.ncomp, a, cap, s);
    if (dA == 3 && dB == 1) return launch_nc<T, 3, 1>(opA.ncomp, opB.ncomp, a, cap, s);
    if (dA == 1 && dB == 3) return launch_nc<T, 1, 3>(opA.ncomp, opB.ncomp, a, cap, s);
    return ANIFEM_ERR_ARG;
}

template <int DA0, int DB0, int NCA, int NCB>
static int launch_mfma_one(const ElemArgs& a, hipStream_t s) {
    if (NCA * NCB == 1) {
        const int64_t blocks = (a.n + kMfmaTets - 1) / kMfmaTets;
        hipLaunchKernelGGL((element_mfma_kernel<DA0, DB0, NCA, NCB>), dim3((unsigned)blocks), dim3(kBlock), 0, s, a);
    } else {
        const int64_t blocks = (a.n + kMfmaVecTets - 1) / kMfmaVecTets;
        hipLaunchKernelGGL((element_mfma_vec_kernel<DA0, DB0, NCA, NCB>), dim3((unsigned)blocks), dim3(kBlock), 0, s,
                           a);
    }
    ANIFEM_HIP_CHECK(hipGetLastError());
    return ANIFEM_OK;
}

template <int DA0, int DB0>
static int launch_mfma_nc(int ncA, int ncB, const ElemArgs& a, hipStream_t s) {
    if (ncA == 1 && ncB == 1) return launch_mfma_one<DA0, DB0, 1, 1>(a, s);
    if (ncA == 3 && ncB == 3) return launch_mfma_one<DA0, DB0, 3, 3>(a, s);
    if (ncA == 1 && ncB == 3) return launch_mfma_one<DA0, DB0, 1, 3>(a, s);
    if (ncA == 3 && ncB == 1) return launch_mfma_one<DA0, DB0, 3, 1>(a, s);
    return ANIFEM_ERR_ARG;
}

// FP16 hi + lo MFMA contraction: tensors constant over each tet only
int launch_element_mfma(const anifem_op& opA, const anifem_op& opB, const ElemArgs& a, hipStream_t s) {
    if (a.q != 1 || !a.r16) return ANIFEM_ERR_ARG;
    if (a.mapA | a.mapB | a.scA | a.scB) return ANIFEM_ERR_ARG;  // RT0 / ND0: FP64 and FP32 modes only
    const int dA = ref_dim(opA.op, opA.fem), dB = ref_dim(opB.op, opB.fem);
    if (dA == 3 && dB == 3) return launch_mfma_nc<3, 3>(opA.ncomp, opB.ncomp, a, s);
    if (dA == 1 && dB == 1) return launch_mfma_nc<1, 1>(opA.ncomp, opB.ncomp, a, s);
    if (dA == 3 && dB == 1) return launch_mfma_nc<3, 1>(opA.ncomp, opB.ncomp, a, s);
    if (dA == 1 && dB == 3) return launch_mfma_nc<1, 3>(opA.ncomp, opB.ncomp, a, s);
    return ANIFEM_ERR_ARG;
}

// Physical quadrature points of every tet (internalFem3DtetGeomInit_XYG,
// core.inl:250-270): X_n = P0 + sum_l lambda_{l+1,n} (P_{l+1} - P0), one lane
// per tet, stored X[(c*q + n)*n + r] (coalesced over tets; the layout of
// per-point coefficient arrays).
struct RulePoints {
    double lam[24][3];    // lambda_1..3 of each point (rules of up to 24 points)
    const double* lamd;   // the same on the device, 3 per point (larger rules), or null
    int q;
};

template <bool MESH>
__global__ __launch_bounds__(kBlock) void physical_points_kernel(ElemArgs a, RulePoints rp, double* __restrict__ X) {
    const int64_t r = blockIdx.x * (int64_t)kBlock + threadIdx.x;
    if (r >= a.n) return;
    double P[4][3];
    load_tet<MESH>(a, r, P);
    for (int n = 0; n < rp.q; ++n)
        for (int c = 0; c < 3; ++c) {
            double x = P[0][c];
            for (int l = 0; l < 3; ++l) x += (rp.lamd ? rp.lamd[3 * n + l] : rp.lam[n][l]) * (P[l + 1][c] - P[0][c]);
            X[((int64_t)c * rp.q + n) * a.n + r] = x;
        }
}

// lambda_1..3 of the points of rule `order` on the current device, uploaded
// once per device and kept until the process ends.
static const double* rule_lambda_dev(int order, int q, const double* p) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, double*> cache;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return nullptr;
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find({dev, order});
    if (it != cache.end()) return it->second;
    std::vector<double> lam((size_t)3 * q);
    for (int k = 0; k < q; ++k)
        for (int l = 0; l < 3; ++l) lam[3 * k + l] = p[4 * k + l + 1];
    double* d = nullptr;
    if (hipMalloc(&d, lam.size() * sizeof(double)) != hipSuccess) return nullptr;
    if (hipMemcpy(d, lam.data(), lam.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipFree(d);
        return nullptr;
    }
    cache[{dev, order}] = d;
    return d;
}

// Physical points of the volume rule `order` for n tets, from SoA vertices
// (xyz) or from a mesh (coords + SoA tet nodes, tets [pos0, pos0 + n)).
int launch_physical_points(int order, int64_t n, const double* xyz, const double* coords, const int32_t* tetnodes,
                           int64_t nodes_stride, double* X, hipStream_t s) {
    const double *p, *w;
    const int q = quadrature(order, &p, &w);
    if (q < 0) return ANIFEM_ERR_ORDER;
    if (n < 0 || !X || (!xyz && (!coords || !tetnodes))) return ANIFEM_ERR_ARG;
    RulePoints rp{};
    rp.q = q;
    if (q <= 24) {
        for (int k = 0; k < q; ++k)
            for (int l = 0; l < 3; ++l) rp.lam[k][l] = p[4 * k + l + 1];
    } else {
        rp.lamd = rule_lambda_dev(order, q, p);
        if (!rp.lamd) return ANIFEM_ERR_HIP;
    }
    ElemArgs a{};
    a.n = n;
    a.xyz = xyz;
    a.coords = coords;
    a.tetnodes = tetnodes;
    a.nodes_stride = nodes_stride;
    a.pos0 = 0;
    if (n == 0) return ANIFEM_OK;
    const unsigned blocks = (unsigned)((n + kBlock - 1) / kBlock);
    if (xyz)
        hipLaunchKernelGGL(physical_points_kernel<false>, dim3(blocks), dim3(kBlock), 0, s, a, rp, X);
    else
        hipLaunchKernelGGL(physical_points_kernel<true>, dim3(blocks), dim3(kBlock), 0, s, a, rp, X);
    ANIFEM_HIP_CHECK(hipGetLastError());
    return ANIFEM_OK;
}

}  // namespace anifem

extern "C" int anifem_quadrature_points_batch(int order, int64_t n_tets, const double* xyz, double* X, void* stream) {
    if (!xyz) return ANIFEM_ERR_ARG;
    return anifem::launch_physical_points(order, n_tets, xyz, nullptr, nullptr, 0, X,
                                          static_cast<hipStream_t>(stream));
}

extern "C" int anifem_fem3dtet_batch(anifem_op opA, anifem_op opB, const anifem_tensor* D, int order, int64_t n_tets,
                                     const double* xyz, int precision, void* A_out, void* stream) {
    using namespace anifem;
    if (n_tets < 0 || (n_tets > 0 && (!xyz || !A_out))) return ANIFEM_ERR_ARG;
    ElemArgs a{};
    int rc = prepare_elem_args(opA, opB, D, order, a);
    if (rc) return rc;
    if (n_tets == 0) return ANIFEM_OK;
    a.n = n_tets;
    a.coef_n = n_tets;
    a.xyz = xyz;
    a.out = A_out;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (precision == ANIFEM_PREC_FP64) return launch_element<double>(opA, opB, order, a, 256, s);
    if (precision == ANIFEM_PREC_FP32) return launch_element<float>(opA, opB, order, a, 256, s);
    if (precision == ANIFEM_PREC_FP16X3) return launch_element_mfma(opA, opB, a, s);
    return ANIFEM_ERR_ARG;
}

extern "C" int anifem_fem3dface_batch(anifem_op opA, anifem_op opB, const anifem_tensor* D, int order, int face,
                                      int dot_normal, int64_t n_tets, const double* xyz, int precision, void* A_out,
                                      void* stream) {
    using namespace anifem;
    if (n_tets < 0 || (n_tets > 0 && (!xyz || !A_out)) || face < 0 || face > 3) return ANIFEM_ERR_ARG;
    ElemArgs a{};
    int rc = prepare_args(opA, opB, D, order, face, dot_normal, a);
    if (rc) return rc;
    if (n_tets == 0) return ANIFEM_OK;
    a.n = n_tets;
    a.coef_n = n_tets;
    a.xyz = xyz;
    a.out = A_out;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (precision == ANIFEM_PREC_FP64) return launch_element<double>(opA, opB, order, a, 256, s);
    if (precision == ANIFEM_PREC_FP32) return launch_element<float>(opA, opB, order, a, 256, s);
    return ANIFEM_ERR_ARG;  // the MFMA mode computes volume integrals only
}

namespace anifem {
// Operator-dependent part of ApplyArgs: IDEN / GRAD of the scalar spaces,
// IDEN / DIV / CURL of RT0 and ND0.
static int prepare_apply(const anifem_op& op, int q, ApplyArgs& a) {
    if (!op_valid(op) || q < 1 || q > kMaxApplyPoints) return ANIFEM_ERR_ARG;
    if (!fem_vector(op.fem) && op.op != ANIFEM_IDEN && op.op != ANIFEM_GRAD) return ANIFEM_ERR_ARG;
    int m = 0, sc = 0;
    space_map(op.op, op.fem, m, sc);
    a.d = ref_dim(op.op, op.fem);
    a.map = m >= 3 ? m
                   : (m == 1 ? 2 : ((op.op == ANIFEM_GRAD || (op.fem == ANIFEM_FEM_ND0 && op.op == ANIFEM_IDEN)) ? 1 : 0));
    a.scale = sc;
    a.op = op.op;
    a.fem = op.fem;
    a.nf0 = nf_scalar(op.fem);
    a.ncomp = op.ncomp;
    a.q = q;
    return ANIFEM_OK;
}

template <int FEM, int D>
static int launch_points(const ApplyArgs& a, const ApplyPoints& pts, bool mesh, hipStream_t s) {
    const int dim = a.map >= 3 ? 9 : D * a.ncomp, pc = apply_chunk(a.n, a.q, dim);
    const size_t lds = ((size_t)pc * apply_nf0(FEM) * D + (size_t)kBlock * apply_stage_row(pc, dim)) * sizeof(double);
    const dim3 grid((unsigned)((a.n + kBlock - 1) / kBlock), (unsigned)apply_split(a.n, a.q, pc));
    if (mesh) hipLaunchKernelGGL((apply_points_kernel<FEM, D, true>), grid, dim3(kBlock), lds, s, a, pts, pc);
    else hipLaunchKernelGGL((apply_points_kernel<FEM, D, false>), grid, dim3(kBlock), lds, s, a, pts, pc);
    ANIFEM_HIP_CHECK(hipGetLastError());
    return ANIFEM_OK;
}

// f(space, reference components) with both as compile-time constants.
template <typename F>
static int for_space(int fem, int d, F f) {
    auto with = [&](auto space) {
        return d == 3 ? f(space, std::integral_constant<int, 3>{}) : f(space, std::integral_constant<int, 1>{});
    };
    switch (fem) {
        case ANIFEM_FEM_P0: return with(std::integral_constant<int, ANIFEM_FEM_P0>{});
        case ANIFEM_FEM_P1: return with(std::integral_constant<int, ANIFEM_FEM_P1>{});
        case ANIFEM_FEM_P2: return with(std::integral_constant<int, ANIFEM_FEM_P2>{});
        case ANIFEM_FEM_P3: return with(std::integral_constant<int, ANIFEM_FEM_P3>{});
        case ANIFEM_FEM_CR1: return with(std::integral_constant<int, ANIFEM_FEM_CR1>{});
        case ANIFEM_FEM_B2: return with(std::integral_constant<int, ANIFEM_FEM_B2>{});
        case ANIFEM_FEM_B4: return with(std::integral_constant<int, ANIFEM_FEM_B4>{});
        case ANIFEM_FEM_RT0: return with(std::integral_constant<int, ANIFEM_FEM_RT0>{});
        case ANIFEM_FEM_ND0: return with(std::integral_constant<int, ANIFEM_FEM_ND0>{});
    }
    return ANIFEM_ERR_ARG;
}

// op at q barycentric points xyl (host) common to all cells.
int launch_apply(const anifem_op& op, const double* xyl, int q, ApplyArgs a, bool mesh, hipStream_t s) {
    if (!xyl) return ANIFEM_ERR_ARG;
    int rc = prepare_apply(op, q, a);
    if (rc) return rc;
    if (a.n == 0) return ANIFEM_OK;
    ApplyPoints pts;
    std::copy(xyl, xyl + 4 * q, pts.xyl);
    return for_space(op.fem, a.d, [&](auto fem, auto d) { return launch_points<fem.value, d.value>(a, pts, mesh, s); });
}

// op at each cell's own physical points.
static int launch_apply_x(const anifem_op& op, const ApplyArgs& a, hipStream_t s) {
    return for_space(op.fem, a.d, [&](auto fem, auto d) {
        const int64_t blocks = (a.n * a.q + kBlock - 1) / kBlock;
        hipLaunchKernelGGL((apply_x_kernel<fem.value, d.value>), dim3((unsigned)blocks), dim3(kBlock), 0, s, a);
        ANIFEM_HIP_CHECK(hipGetLastError());
        return ANIFEM_OK;
    });
}
}  // namespace anifem

extern "C" int anifem_fem3dapplyx_batch(anifem_op op, int q, int64_t n_tets, const double* xyz, const double* X,
                                        const double* dofs, double* opU, void* stream) {
    using namespace anifem;
    if (n_tets < 0 || (n_tets > 0 && (!xyz || !X || !dofs || !opU))) return ANIFEM_ERR_ARG;
    ApplyArgs a{};
    int rc = prepare_apply(op, q, a);
    if (rc) return rc;
    if (n_tets == 0) return ANIFEM_OK;
    a.n = n_tets;
    a.xyz = xyz;
    a.X = X;
    a.dofs = dofs;
    a.out = opU;
    return launch_apply_x(op, a, static_cast<hipStream_t>(stream));
}

extern "C" int anifem_fem3dapply_batch(anifem_op op, const double* xyl, int q, int64_t n_tets, const double* xyz,
                                       const double* dofs, double* opU, void* stream) {
    using namespace anifem;
    if (n_tets < 0 || (n_tets > 0 && (!xyz || !dofs || !opU))) return ANIFEM_ERR_ARG;
    ApplyArgs a{};
    a.n = n_tets;
    a.xyz = xyz;
    a.dofs = dofs;
    a.out = opU;
    return launch_apply(op, xyl, q, a, false, static_cast<hipStream_t>(stream));
}

extern "C" int anifem_face_quadrature(int order, int face, double* p, double* w) {
    std::vector<double> pts, wts;
    const int q = anifem::rule_points(order, face, pts, wts);
    if (q < 0 || face < 0 || face > 3) return q < 0 ? ANIFEM_ERR_ORDER : ANIFEM_ERR_ARG;
    if (p) std::copy(pts.begin(), pts.end(), p);
    if (w) std::copy(wts.begin(), wts.end(), w);
    return q;
}
