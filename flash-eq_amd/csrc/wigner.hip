// WignerDBasis: per-edge Wigner-D basis matrices in closed form.
//
// The reference computes D = matrix_exp(theta * (a0 G0 + a1 G1)) per edge
// (wigner.py:144-240) with axis a = (-d_y, d_x, 0)/|.| and theta = acos(d_z),
// d = v/(|v| + eps), then returns M = D[:, perm] (wigner.py:358-367).
//
// The generators obey [G0,G1] = G2 (cyclic) and G2 is m-diagonal: it couples
// only the (+m, -m) pair of every irrep.  Writing a = rho (cos phi, sin phi),
//     exp(theta rho (cos phi G0 + sin phi G1)) = Z(phi) V Z(theta rho) V^T Z(-phi)
// with Z(x) = exp(x G2) (2x2 rotations by m x on each pair) and the constant
// V = exp(pi/2 G1) (host-built in float64 per irrep).  Each thread produces
// one column j of M, i.e. column perm[j] of D, by applying the five factors
// to a unit vector: O(n^2) work per column, no matrix exponential.
//
// Plan layout per irrep (lvals order), n = 2l+1 doubles blocks:
//   V (n*n, row-major) | z (n): signed m coupling of each row | partner (n)
#include "tile_math.h"
#include "wigner_math.h"

namespace feq {
namespace {

// ---- one lane per edge ------------------------------------------------------------
// Degrees up to kLaneL.  A lane holds an edge; the workgroup's NW waves take the
// columns in turn, so every lane of a wave computes the same column of
// the same degree and the constants V are wave-uniform (scalar loads).  Finished
// (2l+1)^2 blocks go to LDS, an odd number of values from edge to edge (no bank
// conflicts), and the matrices leave in rows of consecutive addresses, zeros
// included.  FLAT: all blocks of the 64 edges fit kFlatLds and their matrices are
// one run of memory; else block by block, whose rows are one run per edge (short
// for small degrees: lvals 0..2, 640 000 edges, 121 us against 61).
// With a thread per (edge, column) a wave met every degree in turn, one branch
// after the other, and read V by lane.  Forward and backward in float32, that way
// and this: lvals 0..6, 40 000 edges 366 and 1502 us, now 97 (384 MB written, 4.0
// TB/s) and 207; lvals 0..4, 40 000 edges 74 and 259, now 36 and 63; lvals 0..2,
// 640 000 edges 133 and 296, now 61 and 150.
constexpr int kLaneEdges = 64;

constexpr size_t kFlatLds = 48 * 1024;   // three workgroups per CU
constexpr size_t kFewLds = 128 * 1024;   // one, where there is no more than one

// FLAT: place of matrix element j in an edge's staged blocks, -1 outside them.
__device__ __forceinline__ void flat_table(const WignerArgs& A, const int32_t* __restrict__ perm, int16_t* at) {
    const int dim = A.dim;
    for (int j = threadIdx.x; j < dim * dim; j += blockDim.x) {
        const int r = j / dim, col = perm[j - r * dim];
        int k = 0, off = 0;
        while (k + 1 < A.nirr && r >= A.off[k + 1]) {
            off += (2 * A.lvals[k] + 1) * (2 * A.lvals[k] + 1);
            ++k;
        }
        const int n = 2 * A.lvals[k] + 1, c = col - A.off[k];
        at[j] = static_cast<int16_t>(c >= 0 && c < n ? off + (r - A.off[k]) * n + c : -1);
    }
}

template <int LMAX, class T, bool FLAT, int NW>
__global__ void __launch_bounds__(64 * NW)
k_wigner_lane(WignerArgs A, int stride, const double* __restrict__ plan, const int32_t* __restrict__ perm,
              int64_t E, const T* __restrict__ dirs, T* __restrict__ out) {
    extern __shared__ __align__(16) char sBraw[];
    T* sB = reinterpret_cast<T*>(sBraw);              // kLaneEdges x (2l+1)^2
    __shared__ int sPerm[FEQ_MAX_SLOTS];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int dim = A.dim, dd = dim * dim;
    const int64_t e0 = static_cast<int64_t>(blockIdx.x) * kLaneEdges;
    const int ne = static_cast<int>(E - e0 < kLaneEdges ? E - e0 : kLaneEdges);
    for (int j = threadIdx.x; j < dim; j += blockDim.x) sPerm[j] = perm[j];
    const EdgeFrame f = edge_frame(dirs + 3 * (e0 + (lane < ne ? lane : ne - 1)));
    const Trig tr = trig_of(f.phi, f.ang);
    int16_t* sAt = reinterpret_cast<int16_t*>(sB + kLaneEdges * stride);
    if constexpr (FLAT) flat_table(A, perm, sAt);
    int off = 0;
    for (int k = 0, id = 0; k < A.nirr; id += 2 * A.lvals[k] + 1, ++k) {   // id: columns before
        const int l = A.lvals[k], base = A.off[k], n = 2 * l + 1;
        const double* V = plan + A.plan_off[k];
        T* mine = sB + (FLAT ? lane * stride + off : lane * n * n);
        off += n * n;
        if constexpr (!FLAT) __syncthreads();         // the previous block's copy (and sPerm)
        switch (l) {
#define FEQ_WCASE(LL)                                                                     \
    case LL:                                                                              \
        if constexpr (LL <= LMAX)                                                         \
            for (int c = (wave - id) & (NW - 1); c < n; c += NW)                          \
                column_into<LL>(V, c, tr, f.ident, mine + c, n);                          \
        break;
            FEQ_WCASE(0) FEQ_WCASE(1) FEQ_WCASE(2) FEQ_WCASE(3) FEQ_WCASE(4) FEQ_WCASE(5) FEQ_WCASE(6)
#undef FEQ_WCASE
            default: break;
        }
        if constexpr (FLAT) continue;
        __syncthreads();
        // the place in the block of each element of its rows that the lane
        // writes (the same for every edge), -1 where D has no entry
        const int row = n * dim;
        for (int q0 = 0; q0 < row; q0 += 64 * 8) {
            int at[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int q = q0 + 64 * i + lane, r = q / dim, j = q - r * dim;
                const int c = q < row ? sPerm[j] - base : -1;
                at[i] = c >= 0 && c < n ? r * n + c : -1;
            }
            for (int e = wave; e < ne; e += NW) {
                T* o = out + (e0 + e) * dd + base * dim + q0;
                const T* b = sB + e * n * n;
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (q0 + 64 * i + lane < row) o[64 * i + lane] = at[i] >= 0 ? b[at[i]] : T(0);
            }
        }
    }
    if constexpr (FLAT) {
        __syncthreads();
        const float inv = 1.0f / static_cast<float>(dd);
        T* o = out + e0 * dd;
#pragma unroll 4
        for (int q = threadIdx.x; q < ne * dd; q += 64 * NW) {
            const int e = quotient(q, inv), at = sAt[q - e * dd];
            o[q] = at >= 0 ? sB[e * stride + at] : T(0);
        }
    }
}

// One lane per edge (see k_wigner_lane): the block of dL/dM goes to LDS, every
// wave adds its columns' terms, and the first wave sums them in order.
template <int LMAX, class T, bool FLAT, int NW>
__global__ void __launch_bounds__(64 * NW)
k_wigner_lane_bwd(WignerArgs A, int stride, const double* __restrict__ plan, const int32_t* __restrict__ perm,
                  int64_t E, const T* __restrict__ dirs, const T* __restrict__ gM, T* __restrict__ gdirs) {
    extern __shared__ __align__(16) char sBraw[];
    T* sB = reinterpret_cast<T*>(sBraw);              // kLaneEdges x (2l+1)^2
    __shared__ int sInv[FEQ_MAX_SLOTS];
    __shared__ double sT0[64 * NW], sT1[64 * NW];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int dim = A.dim, dd = dim * dim;
    const int64_t e0 = static_cast<int64_t>(blockIdx.x) * kLaneEdges;
    const int ne = static_cast<int>(E - e0 < kLaneEdges ? E - e0 : kLaneEdges);
    for (int j = threadIdx.x; j < dim; j += blockDim.x) sInv[perm[j]] = j;
    const int64_t el = e0 + (lane < ne ? lane : ne - 1);
    const ExactFrame X = exact_frame(dirs + 3 * el);
    const Trig tr = trig_of(X.f.phi, X.f.ang);
    double t0 = 0.0, t1 = 0.0;
    if constexpr (FLAT) {
        int16_t* sAt = reinterpret_cast<int16_t*>(sB + kLaneEdges * stride);
        flat_table(A, perm, sAt);
        __syncthreads();
        const float inv = 1.0f / static_cast<float>(dd);
        const T* src = gM + e0 * dd;
#pragma unroll 8
        for (int q = threadIdx.x; q < ne * dd; q += 64 * NW) {
            const T v = src[q];
            const int e = quotient(q, inv), at = sAt[q - e * dd];
            if (at >= 0) sB[e * stride + at] = v;
        }
        __syncthreads();
    }
    int off = 0;
    for (int k = 0, id = 0; k < A.nirr; id += 2 * A.lvals[k] + 1, ++k) {
        const int l = A.lvals[k], base = A.off[k], n = 2 * l + 1, nn = n * n, at = off;
        off += nn;
        if (l == 0) continue;                         // D = 1 is constant
        const double* V = plan + A.plan_off[k];
        if constexpr (!FLAT) {
            __syncthreads();                          // the previous block's reads (and sInv)
            for (int q0 = 0; q0 < nn; q0 += 64) {     // a lane's element is the same in every edge
                const int q = q0 + lane, r = q / n;
                const bool ok = q < nn;
                const T* src = gM + e0 * dd + (ok ? (base + r) * dim + sInv[base + q - r * n] : 0);
#pragma unroll 4
                for (int e = wave; e < ne; e += NW) {
                    const T v = src[static_cast<int64_t>(e) * dd];
                    if (ok) sB[e * nn + q] = v;
                }
            }
            __syncthreads();
        }
        const int le = lane < ne ? lane : ne - 1;
        const T* b = sB + (FLAT ? le * stride + at : le * nn);
        switch (l) {
#define FEQ_WCASE(LL)                                                                     \
    case LL:                                                                              \
        if constexpr (LL <= LMAX)                                                         \
            for (int c = (wave - id) & (NW - 1); c < n; c += NW) {                        \
                double u0, u1;                                                            \
                column_grad<LL>(V, c, tr, X.f.ident, b + c, b + n - 1 - c, n, u0, u1);    \
                t0 += u0;                                                                 \
                t1 += u1;                                                                 \
            }                                                                             \
        break;
            FEQ_WCASE(1) FEQ_WCASE(2) FEQ_WCASE(3) FEQ_WCASE(4) FEQ_WCASE(5) FEQ_WCASE(6)
#undef FEQ_WCASE
            default: break;
        }
    }
    sT0[threadIdx.x] = t0;
    sT1[threadIdx.x] = t1;
    __syncthreads();
    if (wave || lane >= ne) return;
    double s0 = 0.0, s1 = 0.0;
    for (int w = 0; w < NW; ++w) {
        s0 += sT0[64 * w + lane];
        s1 += sT1[64 * w + lane];
    }
    frame_grad(X, s0, s1, dirs + 3 * el, gdirs + 3 * el);
}

// Calls f with std::integral_constant<int, LMAX> for the smallest compiled LMAX
// that covers every degree of A.
template <class Fn>
int with_lane_lmax(const WignerArgs& A, Fn&& f) {
    const int lmax = max_degree(A);
    if (lmax <= 2) return f(std::integral_constant<int, 2>{});
    if (lmax <= 4) return f(std::integral_constant<int, 4>{});
    return f(std::integral_constant<int, kLaneL>{});
}
// Values from edge to edge of the FLAT form, 0 where its LDS would exceed
// kFlatLds or, backward, where it would read the zeros of degrees over 2 for
// nothing (lvals 0..3, 40 000 edges: 83 us against 41).  With few edges the columns'
// latency is what counts forward: all degrees at once, kFewLds.  *lds: that of the form
// that runs (else the widest block of the edges).
template <class T>
int lane_shape(const WignerArgs& A, bool backward, bool few, size_t* lds) {
    size_t sum = 0;
    for (int i = 0; i < A.nirr; ++i) sum += (2 * A.lvals[i] + 1) * (2 * A.lvals[i] + 1);
    sum |= 1;
    const size_t flat = sizeof(T) * kLaneEdges * sum + 2 * static_cast<size_t>(A.dim) * A.dim;
    const size_t n = 2 * static_cast<size_t>(max_degree(A)) + 1;
    const bool use = backward ? flat <= kFlatLds && max_degree(A) <= 2 : flat <= (few ? kFewLds : kFlatLds);
    *lds = use ? flat : sizeof(T) * kLaneEdges * n * n;
    return use ? static_cast<int>(sum) : 0;
}
// Few workgroups: more waves share an edge's columns (16 forward, 8 backward, as the
// registers allow), up to one workgroup per CU, and up to two where the degrees give
// the waves work.  24 000 edges (375 workgroups), with and without, forward: lvals 0..2 11.1
// and 9.0 us, 0..3 18.3 and 15.8, 0..4 27.2 and 29.4, 0..6 69.5 and 71.7; backward: 0..3
// 24.6 and 17.1, 0..6 144 and 119, in float64 0..5 95 and 73, 0..6 187 and 211.
template <class T>
bool few_edges(const WignerArgs& A, int64_t E, bool backward) {
    const bool two = backward ? sizeof(T) == 8 && max_degree(A) == kLaneL : max_degree(A) > 3;
    return ceil_div(E, kLaneEdges) <= (two ? 512 : 256);
}
int set_lds(const void* fn, size_t lds) {
    if (lds > 64 * 1024)
        FEQ_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    return FEQ_OK;
}

}  // namespace
}  // namespace feq

using namespace feq;

extern "C" size_t feq_wigner_plan_doubles(const int32_t* lvals, int32_t n) {
    size_t s = 0;
    for (int i = 0; i < n; ++i) {
        const size_t d = 2 * static_cast<size_t>(lvals[i]) + 1;
        s += d * d + 2 * d;
    }
    return s;
}

namespace {
int wigner_args(const int32_t* lvals, int32_t n, WignerArgs& A) {
    if (!lvals || n < 1) return fail(FEQ_ERR_INVALID, "lvals must be non-empty");
    if (n > FEQ_MAX_IRREPS) return fail(FEQ_ERR_UNSUPPORTED, "more than %d irreps", FEQ_MAX_IRREPS);
    A = WignerArgs{};
    A.nirr = n;
    int dim = 0;
    size_t po = 0;
    for (int i = 0; i < n; ++i) {
        if (lvals[i] < 0 || lvals[i] >= FEQ_MAX_BLOCKS)
            return fail(FEQ_ERR_UNSUPPORTED, "degree %d outside [0, %d]", lvals[i], FEQ_MAX_BLOCKS - 1);
        A.lvals[i] = lvals[i];
        A.off[i] = dim;
        A.plan_off[i] = static_cast<int32_t>(po);
        const int d = 2 * lvals[i] + 1;
        dim += d;
        po += static_cast<size_t>(d) * d + 2 * d;
    }
    A.dim = dim;
    return FEQ_OK;
}

template <class T>
int wigner_fwd(const int32_t* lvals, int32_t n, const double* plan, const int32_t* perm, int64_t E,
               const T* dirs, T* out, feq_stream_t stream) {
    WignerArgs A;
    if (int rc = wigner_args(lvals, n, A)) return rc;
    if (E < 0) return fail(FEQ_ERR_INVALID, "negative edge count");
    if (E == 0) return FEQ_OK;
    if (!plan || !perm || !dirs || !out) return fail(FEQ_ERR_INVALID, "NULL pointer");
    if (int rc = check_dim<T>(A)) return rc;
    size_t lds;
    if (lane_form<T>(A, E, false))
        return with_lane_lmax(A, [&](auto LL) -> int {
            constexpr int L = decltype(LL)::value;
            const bool few = few_edges<T>(A, E, false);
            const int stride = lane_shape<T>(A, false, few, &lds);
            auto kern = few ? (stride ? k_wigner_lane<L, T, true, 16> : k_wigner_lane<L, T, false, 16>)
                            : (stride ? k_wigner_lane<L, T, true, 4> : k_wigner_lane<L, T, false, 4>);
            if (int rc = set_lds(reinterpret_cast<const void*>(kern), lds)) return rc;
            FEQ_LAUNCH("k_wigner", kern, dim3(ceil_div(E, kLaneEdges)), dim3(few ? 1024 : 256), lds, stream_of(stream),
                       A, stride, plan, perm, E, dirs, out);
            return FEQ_OK;
        });
    return wigner_high_fwd<T>(A, plan, perm, E, dirs, out, stream_of(stream));
}

template <class T>
int wigner_bwd(const int32_t* lvals, int32_t n, const double* plan, const int32_t* perm, int64_t E,
               const T* dirs, const T* grad_out, T* grad_dirs, feq_stream_t stream) {
    WignerArgs A;
    if (int rc = wigner_args(lvals, n, A)) return rc;
    if (E < 0) return fail(FEQ_ERR_INVALID, "negative edge count");
    if (E == 0) return FEQ_OK;
    if (!plan || !perm || !dirs || !grad_out || !grad_dirs) return fail(FEQ_ERR_INVALID, "NULL pointer");
    if (int rc = check_dim<T>(A)) return rc;
    size_t lds;
    if (lane_form<T>(A, E, true))
        return with_lane_lmax(A, [&](auto LL) -> int {
            constexpr int L = decltype(LL)::value;
            const bool few = few_edges<T>(A, E, true);
            const int stride = lane_shape<T>(A, true, few, &lds);
            auto kern = few ? (stride ? k_wigner_lane_bwd<L, T, true, 8> : k_wigner_lane_bwd<L, T, false, 8>)
                            : (stride ? k_wigner_lane_bwd<L, T, true, 4> : k_wigner_lane_bwd<L, T, false, 4>);
            if (int rc = set_lds(reinterpret_cast<const void*>(kern), lds)) return rc;
            FEQ_LAUNCH("k_wigner_bwd", kern, dim3(ceil_div(E, kLaneEdges)), dim3(few ? 512 : 256), lds, stream_of(stream),
                       A, stride, plan, perm, E, dirs, grad_out, grad_dirs);
            return FEQ_OK;
        });
    return wigner_high_bwd<T>(A, plan, perm, E, dirs, grad_out, grad_dirs, stream_of(stream));
}
}  // namespace

extern "C" int feq_wigner_basis(const int32_t* lvals, int32_t n, const double* plan,
                                const int32_t* perm, int64_t E, const float* dirs, float* out,
                                feq_stream_t stream) {
    return wigner_fwd<float>(lvals, n, plan, perm, E, dirs, out, stream);
}

extern "C" int feq_wigner_basis_f64(const int32_t* lvals, int32_t n, const double* plan,
                                    const int32_t* perm, int64_t E, const double* dirs, double* out,
                                    feq_stream_t stream) {
    return wigner_fwd<double>(lvals, n, plan, perm, E, dirs, out, stream);
}

extern "C" int feq_wigner_basis_bwd(const int32_t* lvals, int32_t n, const double* plan,
                                    const int32_t* perm, int64_t E, const float* dirs,
                                    const float* grad_out, float* grad_dirs, feq_stream_t stream) {
    return wigner_bwd<float>(lvals, n, plan, perm, E, dirs, grad_out, grad_dirs, stream);
}

extern "C" int feq_wigner_basis_bwd_f64(const int32_t* lvals, int32_t n, const double* plan,
                                        const int32_t* perm, int64_t E, const double* dirs,
                                        const double* grad_out, double* grad_dirs, feq_stream_t stream) {
    return wigner_bwd<double>(lvals, n, plan, perm, E, dirs, grad_out, grad_dirs, stream);
}
