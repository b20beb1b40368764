// Wigner-D bases with degrees over kLaneL, of few edges or of few columns: a thread
// per (edge, column) (lane_form tells which calls come here).
// Included by wigner_high.hip (float32) and wigner_high64.hip (float64): one
// translation unit each, which compile for minutes.
#pragma once

#include "wigner_math.h"

namespace feq {
namespace {

// Workgroup: a tile of EPB edges; thread t computes standard column c0 = t % dim
// of edge t / dim into an LDS tile of the edges' M = D[:, perm] matrices, which
// is then written with coalesced stores.
// LMAX: the largest degree the launch handles (the register footprint of the
// per-column vectors grows with it, so small representations get a small kernel).
template <int LMAX, class T>
__global__ void __launch_bounds__(256)
k_wigner(WignerArgs A, int epb, const double* __restrict__ plan, const int32_t* __restrict__ perm,
         int64_t E, const T* __restrict__ dirs, T* __restrict__ out) {
    extern __shared__ __align__(16) char sMraw[];
    T* sM = reinterpret_cast<T*>(sMraw);              // epb x dim x dim
    __shared__ EdgeFrame sFr[256];
    __shared__ int sInv[FEQ_MAX_SLOTS];
    const int dim = A.dim, dd = dim * dim;
    const int64_t e0 = static_cast<int64_t>(blockIdx.x) * epb;
    const int ne = static_cast<int>(E - e0 < epb ? E - e0 : epb);
    for (int q = threadIdx.x; q < epb * dd; q += blockDim.x) sM[q] = T(0);
    for (int j = threadIdx.x; j < dim; j += blockDim.x) sInv[perm[j]] = j;
    if (threadIdx.x < ne) {
        const EdgeFrame f = edge_frame(dirs + 3 * (e0 + threadIdx.x));
        sFr[threadIdx.x] = f;
    }
    __syncthreads();
    const int el = threadIdx.x / dim;
    if (el < ne) {
        const int c0 = threadIdx.x % dim;
        int k = 0;
        while (k + 1 < A.nirr && c0 >= A.off[k + 1]) ++k;
        const int l = A.lvals[k], base = A.off[k], c = c0 - base;
        const double* V = plan + A.plan_off[k];
        const EdgeFrame f = sFr[el];
        const Trig tr = l ? trig_of(f.phi, f.ang) : Trig{};
        T* dst = sM + el * dd + base * dim + sInv[c0];   // rows base.., column j
        switch (l) {
#define FEQ_WCASE(LL) \
    case LL:                                                                             \
        if constexpr (LL <= LMAX) column_into<LL>(V, c, tr, f.ident, dst, dim); \
        break;
            FEQ_WCASE(0) FEQ_WCASE(1) FEQ_WCASE(2) FEQ_WCASE(3) FEQ_WCASE(4) FEQ_WCASE(5)
            FEQ_WCASE(6) FEQ_WCASE(7) FEQ_WCASE(8) FEQ_WCASE(9) FEQ_WCASE(10) FEQ_WCASE(11)
            FEQ_WCASE(12) FEQ_WCASE(13) FEQ_WCASE(14) FEQ_WCASE(15) FEQ_WCASE(16)
#undef FEQ_WCASE
            default: break;
        }
    }
    __syncthreads();
    T* o = out + e0 * dd;
    for (int q = threadIdx.x; q < ne * dd; q += blockDim.x) o[q] = sM[q];
}

template <int LMAX, class T>
__global__ void __launch_bounds__(256)
k_wigner_bwd(WignerArgs A, int epb, const double* __restrict__ plan, const int32_t* __restrict__ perm,
             int64_t E, const T* __restrict__ dirs, const T* __restrict__ gM,
             T* __restrict__ gdirs) {
    extern __shared__ __align__(16) char sGraw[];
    T* sG = reinterpret_cast<T*>(sGraw);              // epb x dim x dim (dL/dM tile)
    __shared__ EdgeFrame sFr[256];
    __shared__ int sInv[FEQ_MAX_SLOTS];
    __shared__ double sT0[256], sT1[256];
    const int dim = A.dim, dd = dim * dim;
    const int64_t e0 = static_cast<int64_t>(blockIdx.x) * epb;
    const int ne = static_cast<int>(E - e0 < epb ? E - e0 : epb);
    const T* gsrc = gM + e0 * dd;
    for (int q = threadIdx.x; q < ne * dd; q += blockDim.x) sG[q] = gsrc[q];
    for (int j = threadIdx.x; j < dim; j += blockDim.x) sInv[perm[j]] = j;
    ExactFrame X{};
    if (threadIdx.x < ne) {
        X = exact_frame(dirs + 3 * (e0 + threadIdx.x));
        sFr[threadIdx.x] = X.f;
    }
    __syncthreads();
    const int el = threadIdx.x / dim;
    double t0 = 0.0, t1 = 0.0;
    if (el < ne) {
        const int c0 = threadIdx.x % dim;
        int k = 0;
        while (k + 1 < A.nirr && c0 >= A.off[k + 1]) ++k;
        const int l = A.lvals[k], base = A.off[k], c = c0 - base, n = 2 * l + 1;
        const double* V = plan + A.plan_off[k];
        const EdgeFrame f = sFr[el];
        const Trig tr = l ? trig_of(f.phi, f.ang) : Trig{};
        // column c of dL/dD is column sInv[c] of dL/dM; rows base.. of the block
        const T* gcol = sG + el * dd + base * dim + sInv[c0];
        const T* gpar = sG + el * dd + base * dim + sInv[base + n - 1 - c];
        switch (l) {
#define FEQ_WCASE(LL)                                                                    \
    case LL:                                                                             \
        if constexpr (LL <= LMAX)                                                        \
            column_grad<LL>(V, c, tr, f.ident, gcol, gpar, dim, t0, t1);                     \
        break;
            FEQ_WCASE(0) FEQ_WCASE(1) FEQ_WCASE(2) FEQ_WCASE(3) FEQ_WCASE(4) FEQ_WCASE(5)
            FEQ_WCASE(6) FEQ_WCASE(7) FEQ_WCASE(8) FEQ_WCASE(9) FEQ_WCASE(10) FEQ_WCASE(11)
            FEQ_WCASE(12) FEQ_WCASE(13) FEQ_WCASE(14) FEQ_WCASE(15) FEQ_WCASE(16)
#undef FEQ_WCASE
            default: break;
        }
    }
    sT0[threadIdx.x] = t0;
    sT1[threadIdx.x] = t1;
    __syncthreads();
    if (threadIdx.x >= ne) return;
    // per edge: sum the columns in a fixed order, then the chain rule
    double s0 = 0.0, s1 = 0.0;
    for (int q = 0; q < dim; ++q) {
        s0 += sT0[threadIdx.x * dim + q];
        s1 += sT1[threadIdx.x * dim + q];
    }
    frame_grad(X, s0, s1, dirs + 3 * (e0 + threadIdx.x), gdirs + 3 * (e0 + threadIdx.x));
}

template <class Fn>
int with_lmax(const WignerArgs& A, Fn&& f) {
    if (max_degree(A) <= 2) return f(std::integral_constant<int, 2>{});
    if (max_degree(A) <= 4) return f(std::integral_constant<int, 4>{});
    if (max_degree(A) <= kLaneL) return f(std::integral_constant<int, kLaneL>{});
    if (max_degree(A) <= 10) return f(std::integral_constant<int, 10>{});
    return f(std::integral_constant<int, 16>{});
}

}  // namespace

template <class T>
int wigner_high_fwd(const WignerArgs& A, const double* plan, const int32_t* perm, int64_t E, const T* dirs, T* out,
                    hipStream_t s) {
    const int epb = column_edges<T>(A);
    const size_t lds = sizeof(T) * static_cast<size_t>(epb) * A.dim * A.dim;
    return with_lmax(A, [&](auto LL) -> int {
        auto kern = k_wigner<decltype(LL)::value, T>;
        FEQ_LAUNCH("k_wigner", kern, dim3(ceil_div(E, epb)), dim3(256), lds, s, A, epb, plan, perm, E, dirs, out);
        return FEQ_OK;
    });
}

template <class T>
int wigner_high_bwd(const WignerArgs& A, const double* plan, const int32_t* perm, int64_t E, const T* dirs,
                    const T* grad_out, T* grad_dirs, hipStream_t s) {
    const int epb = column_edges<T>(A);
    const size_t lds = sizeof(T) * static_cast<size_t>(epb) * A.dim * A.dim;
    return with_lmax(A, [&](auto LL) -> int {
        auto kern = k_wigner_bwd<decltype(LL)::value, T>;
        FEQ_LAUNCH("k_wigner_bwd", kern, dim3(ceil_div(E, epb)), dim3(256), lds, s, A, epb, plan, perm, E, dirs,
                   grad_out, grad_dirs);
        return FEQ_OK;
    });
}

}  // namespace feq
