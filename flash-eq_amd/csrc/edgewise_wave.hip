// Fused EquivariantEdgewiseLinear, one wave per edge, on the float32 matrix
// cores (v_mfma_f32_16x16x4_f32), for layouts without split-fp16 kernels of
// their own: any lvals whose m-blocks pack into four 16-slot blocks (lvals
// 0..6 among them), up to 64 channels each way, rank 4.
//
// Same mathematics as edgewise.hip.  The instruction's operands and its result
// let products be chained in registers: with lane l = (c = l % 16, g = l / 16),
// step r of a reduction block may take the indices 4 g + r, and the result
// holds D[4 g + r][c] in register r.  So a result's registers are, as they
// stand, the B operand (reduction over D's rows, columns kept) or the
// transposed A operand (reduction over D's rows, D's columns as rows) of a next
// product.  Every stage contracts over the rows of the one before:
//   forward   fs (ci x i) = x P,  G_k (i x co) = fs^T C_k^T,
//             m (o x co) = sum_k M_k G_k,  y^T (d x co) = Q m
//   input     gd (co x o) = gy Q,  H_k (o x ci) = gd^T C_k,
//   gradient  dfs (i x ci) = sum_k M_k^T H_k,  dx^T (d x ci) = P dfs,
//             Z_k (o x i) = H_k fs (H_k transposed through LDS) -> dF_e
//   pattern   U_k (i x co) = M_k^T gd^T,  dC_k (co x ci) += U_k^T fs^T,
//   gradient  fs^T (i x ci) = P^T x^T,  gd^T (o x co) = Q^T gy^T
// M_k (o x i) is the edge's mixing matrix, its entries s^(l_i + l_o) F_e[k, w]
// with a sign.  The m-first slots are renumbered so that every m-group lies in
// one 16-slot block (GenTab): M_k has diagonal block tiles only.  No barriers:
// each wave works alone, and x, P, Q and C go from memory to the operands.
//
// lvals 0..6 x 32 channels take 568 float32 steps (16x16x4, 32 cycles) forward, 800
// for the input gradient and 624 for the pattern gradient per edge, against 30 KB of
// memory.  At 50 000 such edges 0.68, 1.17 and 0.90 ms, of which these steps take 0.37,
// 0.52 and 0.41 with every matrix core busy: what bounds them is a wave's chain of dependent
// steps, LDS reads and scalar work between them, which the two waves per SIMD that the
// registers allow cover in part.  edgewise.hip's vector kernels (a workgroup per
// edge, every product through LDS) took 7.1 ms forward and 18.3 ms backward; at
// lvals 0..4 x 32 and 20 000 edges 0.13, 0.22 and 0.18 against 1.24 and 3.29.
// What did not carry: operands from memory without the LDS copy of the basis
// (1.5, 2.9 and 1.6 ms: requests of 4 rows x 16 scattered columns); loads under lane
// conditions (1.0, 2.0 and 1.0); Z_k summed over the channel tiles (2% faster,
// errors 5% larger: one chain instead of two).  Where an edge's values are not finite,
// its results are not either, but an infinity may come out as NaN: the tiles multiply
// positions that no weight joins by zeros.
#include "feq_internal.h"
#include "tile_math.h"

namespace feq {
namespace {

constexpr int kMaxNB = 4;       // 16-slot blocks
constexpr int kMaxCT = 4;       // 16-channel tiles
constexpr int kMaxW = 256;      // radial weights per channel pair
constexpr int kMaxDeg = 32;     // powers of s
constexpr int kRank = 4;

// The renumbered layout, built on the host and passed by value.
struct GenTab {
    int16_t code[kMaxNB][16][16];   // [block][o row][i row]: w, sign in bit 14; wd where no weight joins them
    int16_t pos0[kMaxW];            // tile position (block, o row, i row) of a weight's first entry
    int16_t pos1[kMaxW];            // and of its second (bit 14: subtracted); pos0 with bit 15 for m = 0
    int8_t deg[kMaxW];              // l_in + l_out
    int8_t in_slot[kMaxNB * 16];    // m-first slot of a position, -1 for none
    int8_t out_slot[kMaxNB * 16];
    int32_t cin, cout, din, dout, wd;
    int32_t last;                   // reduction steps that the last block needs
};

// The lane's number, opaque to the compiler: what follows from it is computed
// where it is used.  (Held in registers over the whole edge loop, the addresses
// of the staging and the tiles cost 50 to 100 of them, and spills.)
__device__ __forceinline__ int lane_id() {
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    return lane;
}

// The patterns in operand order, packed once per call by k_ewg_prep: for rank k and
// column tile c0 / 16, the reduction tiles' B operands, zero-padded to 16 channels.
// (Ragged channel counts then need no conditions in the edge loop.)
struct Patterns {
    const v4f* frag;        // [rank][column tile][reduction tile][lane]
    int ncol;               // column tiles
};
template <int CT>
struct Mixer {
    v4f q[CT];
};
template <int CT>
__device__ __forceinline__ void load_mixer(const Patterns& W, int k, int col, Mixer<CT>& M) {
    const unsigned lane = lane_id();
    const v4f* f = W.frag + (k * W.ncol + col) * CT * 64;
#pragma unroll
    for (int t = 0; t < CT; ++t) M.q[t] = f[64 * t + lane];
}
// out[b] (rows: the tiles' positions, columns: the patterns' channels) = sum over
// channels of the tiles and the patterns.  (On the fp16 matrix cores with operands split
// in two halves these products take a fourth of the cycles, 0.58 against 0.68 ms forward at
// lvals 0..6 x 32, 50 000 edges; but two halves hold 22 bits below one exponent per
// edge, and the gradients of the radial functions of a degree whose values are small
// beside the edge's largest lose theirs.)
template <int CT, int NB>
__device__ __forceinline__ void mix_channels(const v4f (&v)[CT][NB], const Mixer<CT>& M, v4f (&out)[NB]) {
#pragma unroll
    for (int b = 0; b < NB; ++b) out[b] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int b = 0; b < NB; ++b) out[b] = mfma4(v[t][b][r], M.q[t][r], out[b]);
}

// Orders a wave's LDS writes before its later reads by other lanes (LDS
// operations of one wave execute in order: only the compiler must not move them).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Rows 4 g + r of a 16-row tile at d0, as far as dim goes (p: the row of out).
__device__ __forceinline__ void store4(float* out, unsigned p, const v4f& v, int d0, int g, int dim, bool ok) {
    const int d = d0 + 4 * g;
    if (d0 + 16 <= dim) {
        if (ok) __builtin_memcpy(out + (p + d), &v, 16);
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (ok && d + r < dim) out[p + d + r] = v[r];
    }
}

// Per-wave LDS: F_e with one zero per rank (entry wd), the powers of s.
__host__ __device__ constexpr int fe_floats(int wd) { return kRank * (wd + 1) + kMaxDeg; }

// A memory request under a lane condition becomes a branch that the compiler
// does not move others across, so that a wave waits for each in turn.  The loads
// here are therefore unconditional, lanes without work repeating the last
// lane's, or under conditions that are the same for the whole wave.

// F_e[k, w] s^(l_in + l_out) of the edge, and s^l in the last kMaxDeg floats.
__device__ __forceinline__ void edge_weights(const GenTab& T, const feq_binning& B, float r,
                                             const float* __restrict__ F, float* sFe, const int (&deg)[4]) {
    const int lane = lane_id(), wd = T.wd;
    float* spow = sFe + kRank * (wd + 1);
    const EdgeBin eb = edge_bin(r, B);
    const float* flo = F + static_cast<int64_t>(__builtin_amdgcn_readfirstlane(eb.lo)) * kRank * wd;
    float lo[kMaxW / 64][kRank], hi[kMaxW / 64][kRank];
#pragma unroll
    for (int j = 0; j < kMaxW / 64; ++j)
        if (64 * j < wd) {
            const unsigned w = lane + 64 * j < wd ? lane + 64 * j : wd - 1;
#pragma unroll
            for (int k = 0; k < kRank; ++k) lo[j][k] = (flo + k * wd)[w], hi[j][k] = (flo + (kRank + k) * wd)[w];
        }
    float pw = 1.0f, base = r / (r + B.sh_scale);
#pragma unroll
    for (int bit = 0; bit < 5; ++bit) {     // as ipowf
        pw = (lane >> bit) & 1 ? pw * base : pw;
        base *= base;
    }
    wave_sync();    // the previous edge's reads
    spow[lane & (kMaxDeg - 1)] = pw;
    sFe[(lane & (kRank - 1)) * (wd + 1) + wd] = 0.0f;
    wave_sync();
#pragma unroll
    for (int j = 0; j < kMaxW / 64; ++j)
        if (64 * j < wd) {
            const int w = lane + 64 * j < wd ? lane + 64 * j : wd - 1;
            const float q = spow[deg[j]];
#pragma unroll
            for (int k = 0; k < kRank; ++k) sFe[k * (wd + 1) + w] = lerp_bins(lo[j][k], hi[j][k], eb.t) * q;
        }
    wave_sync();
}

__device__ __forceinline__ float coef(const float* sFk, const int (&code)[2], int r) {
    const unsigned q = static_cast<unsigned>(code[r >> 1]) >> (16 * (r & 1));
    return __uint_as_float(__float_as_uint(sFk[q & 0x3fff]) ^ ((q & 0x4000u) << 17));
}

// acc[b] += the mixing matrix of one rank times the tiles v: the rank's sum by itself,
// then added (one chain over the ranks' slots: errors of y and dx 2% larger, the input
// gradient 3% faster).
template <int NB>
__device__ __forceinline__ void add_mixed(const float* sFk, const int (&code)[NB][2], int last, const v4f (&v)[NB],
                                          v4f (&acc)[NB]) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        v4f one = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (b < NB - 1 || r < last) one = mfma4(coef(sFk, code[b], r), v[b][r], one);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[b][r] += one[r];
    }
}

// A basis matrix (n = dim^2 contiguous floats, 4-byte aligned) to the wave's LDS
// copy: requested by begin, written by end, so that other work stands between.
constexpr int kStage(int nb) { return nb == 1 ? 2 : nb == 2 ? 4 : nb == 3 ? 6 : 10; }   // 16-byte pieces per lane
template <int NB>
struct Staged {
    v4f v[kStage(NB)];
    float tail;
};
template <int NB>
__device__ __forceinline__ void stage_begin(const float* __restrict__ Bm, int n, Staged<NB>& st) {
    const int lane = lane_id(), n4 = n >> 2;
#pragma unroll
    for (int u = 0; u < kStage(NB); ++u)
        if (64 * u < n4) {
            const unsigned q = 64 * u + lane < n4 ? 64 * u + lane : n4 - 1;
            __builtin_memcpy(&st.v[u], Bm + 4 * q, 16);
        }
    const unsigned q = 4 * n4 + lane < n ? 4 * n4 + lane : n - 1;
    st.tail = Bm[q];
}
template <int NB>
__device__ __forceinline__ void stage_end(const float* __restrict__ Bm, int n, const Staged<NB>& st, float* sB) {
    const int lane = lane_id(), n4 = n >> 2;
    wave_sync();    // earlier reads of the copy
#pragma unroll
    for (int u = 0; u < kStage(NB); ++u)
        if (64 * u < n4) {
            const int q = 64 * u + lane;
            *reinterpret_cast<v4f*>(sB + 4 * (q < n4 ? q : n4 - 1)) = st.v[u];
        }
    const int q = 4 * n4 + lane;
    if (q < n) sB[q] = st.tail;
    for (int p = 64 * kStage(NB) + lane; p < n4; p += 64) {     // wider than the pieces
        v4f v;
        __builtin_memcpy(&v, Bm + 4 * p, 16);
        *reinterpret_cast<v4f*>(sB + 4 * p) = v;
    }
    wave_sync();
}
__host__ __device__ constexpr int basis_floats(int din, int dout) {
    return ((din > dout ? din * din : dout * dout) + 3) / 4 * 4;
}

// Per-wave LDS: the staged basis, F_e and the powers of s.
__host__ __device__ constexpr int wave_floats(int wd, int din, int dout) {
    return basis_floats(din, dout) + (fe_floats(wd) + 3) / 4 * 4;
}

template <int NB, class Fn>
__device__ __forceinline__ void stage_basis(const float* __restrict__ Bm, int dim, float* sB, Fn&& between) {
    Staged<NB> st;
    stage_begin<NB>(Bm, dim * dim, st);
    between();
    stage_end<NB>(Bm, dim * dim, st, sB);
}
// Where its registers allow, a wave requests the next edge's basis while it works
// on this one.
constexpr bool ahead(int nb) { return nb <= 2; }

// Elements 16 kb + 4 g + (0..3) of a row of dim floats; zeros past its end and
// where !ok (the row is then a valid one).
__device__ __forceinline__ v4f row4(const float* __restrict__ X, unsigned row, int kb, int dim, bool ok) {
    const int d = 16 * kb + 4 * (lane_id() >> 4);
    v4f v;
    if (16 * kb + 16 <= dim) {
        __builtin_memcpy(&v, X + (row + d), 16);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = ok ? v[r] : 0.0f;
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = X[row + (d + r < dim ? d + r : dim - 1)];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = ok && d + r < dim ? v[r] : 0.0f;
    }
    return v;
}

// acc[t][b] (16 x 16 tiles) = rows r0 + 16 t + (0..15) of X (nrow, dim) times the
// columns of the staged basis at the positions' slots; TR: the transposed tiles.
// Rows and indices outside enter as zeros; the column of an empty position is
// slot 0's, which the mixing matrix multiplies by zeros.
template <int CT, int NB, bool TR>
__device__ __forceinline__ void rotate_in(const float* __restrict__ X, int r0, int nrow, const float* sB,
                                          int dim, const int (&slot)[NB], v4f (&acc)[CT][NB]) {
    const int lane = lane_id(), c = lane & 15, g = lane >> 4;
    unsigned row[CT];
    bool rok[CT];
    v4f xa[CT], xn[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) {
        const int q = r0 + 16 * t + c;
        rok[t] = q < nrow;
        row[t] = (rok[t] ? q : 0) * dim;
        xa[t] = row4(X, row[t], 0, dim, rok[t]);
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[t][b] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const int nkb = (dim + 15) >> 4;
    for (int kb = 0; kb < nkb; ++kb) {
        if (kb + 1 < nkb) {
#pragma unroll
            for (int t = 0; t < CT; ++t) xn[t] = row4(X, row[t], kb + 1, dim, rok[t]);
        }
        const int rem = dim - 16 * kb;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (r >= rem) break;
            const int d = 16 * kb + 4 * g + r;
            const float* br = sB + (d < dim ? d : 0) * dim;
            float pb[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) pb[b] = br[slot[b]];
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int t = 0; t < CT; ++t)
                    acc[t][b] = TR ? mfma4(pb[b], xa[t][r], acc[t][b]) : mfma4(xa[t][r], pb[b], acc[t][b]);
        }
#pragma unroll
        for (int t = 0; t < CT; ++t) xa[t] = xn[t];
    }
}

// Rows 16 t + c of out (nrow, dim), t given: out[row][d] = sum over positions p
// of the staged basis [d, slot(p)] v(p, row), v's tiles as a product left them.
template <int NB>
__device__ __forceinline__ void rotate_out(const v4f (&v)[NB], const float* sB, int dim, int last,
                                           const int (&slot)[NB], float* __restrict__ out, int t, int nrow) {
    const int lane = lane_id(), c = lane & 15, g = lane >> 4;
    const unsigned row = 16 * t + c;
#pragma unroll 1
    for (int d0 = 0; d0 < dim; d0 += 16) {
        const float* br = sB + (d0 + c < dim ? d0 + c : 0) * dim;
        v4f o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (b < NB - 1 || r < last) o = mfma4(br[(slot[b] >> (8 * r)) & 0xff], v[b][r], o);
        store4(out, row * dim, o, d0, g, dim, row < static_cast<unsigned>(nrow));
    }
}

// The lane's share of the tables: the slot of column c, the slots of the
// reduction indices 4 g + r (8 bits each; 0 for an empty position, whose values
// are zero), and the mixing matrix's codes (two in a register).
template <int NB>
__device__ __forceinline__ void load_slots(const int8_t* slots, int (&col)[NB], int (&red)[NB]) {
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        col[b] = slots[16 * b + c] < 0 ? 0 : slots[16 * b + c];
        red[b] = 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int s = slots[16 * b + 4 * g + r];
            red[b] |= (s < 0 ? 0 : s) << (8 * r);
        }
    }
}
template <int NB, bool BWD>
__device__ __forceinline__ void load_codes(const GenTab& T, int (&code)[NB][2]) {
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = 4 * g + 2 * h;
            const int lo = BWD ? T.code[b][r][c] : T.code[b][c][r];
            const int hi = BWD ? T.code[b][r + 1][c] : T.code[b][c][r + 1];
            code[b][h] = lo | (hi << 16);
        }
}
__device__ __forceinline__ void load_deg(const GenTab& T, int (&deg)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int w = (threadIdx.x & 63) + 64 * j;
        deg[j] = T.deg[w < T.wd ? w : T.wd - 1];
    }
}

// C_k[co, ci] of the tile pair: B operand with columns co (reduction ci) or,
// BWD, with columns ci (reduction co); zeros outside.
template <bool BWD>
__device__ __forceinline__ v4f load_c(const float* __restrict__ Ck, int co0, int ci0, int cout, int cin) {
    const int lane = lane_id(), c = lane & 15, g = lane >> 4;
    v4f v;
    if (co0 + 16 <= cout && ci0 + 16 <= cin) {
        if constexpr (BWD) {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = (Ck + r * cin)[static_cast<unsigned>((co0 + 4 * g) * cin + ci0 + c)];
        } else {
            __builtin_memcpy(&v, Ck + static_cast<unsigned>((co0 + c) * cin + ci0 + 4 * g), 16);
        }
        return v;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int co = co0 + (BWD ? 4 * g + r : c), ci = ci0 + (BWD ? c : 4 * g + r);
        const bool ok = co < cout && ci < cin;
        const float q = Ck[static_cast<unsigned>(ok ? co * cin + ci : 0)];
        v[r] = ok ? q : 0.0f;
    }
    return v;
}

// One wave per (rank, column tile): columns co and reduction ci, or BWD the other
// way round.
template <bool BWD>
__global__ void __launch_bounds__(64)
k_ewg_prep(const float* __restrict__ C, int cout, int cin, v4f* __restrict__ frag) {
    const int k = blockIdx.x, col = blockIdx.y, ncol = gridDim.y;
    const int ct = ((BWD ? cout : cin) + 15) / 16;
    const float* Ck = C + static_cast<int64_t>(k) * cout * cin;
    for (int t = 0; t < ct; ++t)
        frag[((k * ncol + col) * ct + t) * 64 + threadIdx.x] =
            BWD ? load_c<true>(Ck, 16 * t, 16 * col, cout, cin) : load_c<false>(Ck, 16 * col, 16 * t, cout, cin);
}

// Workgroups per CU: what the registers allow without (much) spilling.  The grids
// are one such set of workgroups, each wave taking every (grid * 4)-th edge: its
// tables are read once.
constexpr int fwd_groups(int ct, int nb) { return ct * nb < 8 ? 3 : 2; }
constexpr int bwd_x_groups(int nb) { return nb == 1 ? 3 : 2; }

// ---------------------------------------------------------------------------
template <int CT, int NB>
__global__ void __launch_bounds__(256, fwd_groups(CT, NB))
k_ewg_fwd(GenTab T, feq_binning B, int64_t E, const float* __restrict__ x, const float* __restrict__ P,
          const float* __restrict__ Q, const float* __restrict__ dist, Patterns W,
          const float* __restrict__ F, float* __restrict__ y) {
    extern __shared__ float sm[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cin = T.cin, cout = T.cout, din = T.din, dout = T.dout, wd = T.wd, last = T.last;
    float* sB = sm + wave * wave_floats(wd, din, dout);
    float* sFe = sB + basis_floats(din, dout);
    int in_col[NB], in_red[NB], out_col[NB], out_red[NB], deg[4], code[NB][2];
    load_slots<NB>(T.in_slot, in_col, in_red);
    load_slots<NB>(T.out_slot, out_col, out_red);
    load_deg(T, deg);
    load_codes<NB, false>(T, code);
    const int64_t step = static_cast<int64_t>(gridDim.x) * 4, first = static_cast<int64_t>(blockIdx.x) * 4 + wave;
    Staged<ahead(NB) ? NB : 1> st;
    if constexpr (ahead(NB))
        if (first < E) stage_begin<NB>(P + first * din * din, din * din, st);
    for (int64_t e = first; e < E; e += step) {
        v4f fs[CT][NB];
        if constexpr (ahead(NB)) {
            edge_weights(T, B, dist[e], F, sFe, deg);
            stage_end<NB>(P + e * din * din, din * din, st, sB);
            stage_begin<NB>(P + (e + step < E ? e + step : e) * din * din, din * din, st);
        } else {
            stage_basis<NB>(P + e * din * din, din, sB, [&] { edge_weights(T, B, dist[e], F, sFe, deg); });
        }
        rotate_in<CT, NB, false>(x + e * cin * din, 0, cin, sB, din, in_col, fs);
        if (Q != P) stage_basis<NB>(Q + e * dout * dout, dout, sB, [] {});
        for (int co0 = 0; co0 < cout; co0 += 16) {
            v4f m[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) m[b] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            // the patterns one rank ahead: the products cover their latency
            Mixer<CT> M, next;
            load_mixer<CT>(W, 0, co0 / 16, M);
#pragma unroll 1
            for (int k = 0; k < kRank; ++k) {
                v4f G[NB];
                load_mixer<CT>(W, k + 1 < kRank ? k + 1 : k, co0 / 16, next);
                mix_channels<CT, NB>(fs, M, G);
                M = next;
                add_mixed<NB>(sFe + k * (wd + 1), code, last, G, m);
            }
            rotate_out<NB>(m, sB, dout, last, out_red, y + e * cout * dout, co0 / 16, cout);
        }
    }
}

// ---------------------------------------------------------------------------
// LDS rows of the transposed H_k tiles: 20 floats, so that the 16-byte reads
// are aligned and the writes free of bank conflicts; the Z_k tiles (rows of 17)
// reuse them.
constexpr int kTS = 20, kZS = 17;
__host__ __device__ constexpr int bwd_x_floats(int wd, int din, int dout, int nb) {
    return wave_floats(wd, din, dout) + nb * 16 * kTS;
}

template <int CT, int NB>
__global__ void __launch_bounds__(256, bwd_x_groups(NB))
k_ewg_bwd_x(GenTab T, feq_binning B, int64_t E, const float* __restrict__ gy, const float* __restrict__ x,
            const float* __restrict__ P, const float* __restrict__ Q, const float* __restrict__ dist,
            Patterns W, const float* __restrict__ F, float* __restrict__ gx,
            float* __restrict__ dFe) {
    extern __shared__ float sm[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cin = T.cin, cout = T.cout, din = T.din, dout = T.dout, wd = T.wd, last = T.last;
    float* sB = sm + wave * bwd_x_floats(wd, din, dout, NB);
    float* sFe = sB + basis_floats(din, dout);
    float* sT = sB + wave_floats(wd, din, dout);
    int pos[kMaxW / 64];                // a weight's first entry, and its second above
#pragma unroll
    for (int j = 0; j < kMaxW / 64; ++j) {
        const int w = lane + 64 * j < wd ? lane + 64 * j : wd - 1;
        pos[j] = T.pos0[w] | static_cast<int>(static_cast<unsigned>(T.pos1[w]) << 16);
    }
    int in_col[NB], in_red[NB], out_col[NB], out_red[NB], deg[4], code[NB][2];
    load_slots<NB>(T.in_slot, in_col, in_red);
    load_slots<NB>(T.out_slot, out_col, out_red);
    load_deg(T, deg);
    load_codes<NB, true>(T, code);
    const int64_t step = static_cast<int64_t>(gridDim.x) * 4, first = static_cast<int64_t>(blockIdx.x) * 4 + wave;
    Staged<ahead(NB) ? NB : 1> st;
    if constexpr (ahead(NB))
        if (first < E) stage_begin<NB>(Q + first * dout * dout, dout * dout, st);
    for (int64_t e = first; e < E; e += step) {
        v4f gd[CT][NB];
        float dF[kRank][kMaxW / 64] = {};   // of the weights lane + 64 j
        // a weight's gradient from the tiles: its one (m = 0) or two entries
        auto weights_of = [&](const v4f (&Z)[NB], float (&d)[kMaxW / 64]) {
            const int ln = lane_id(), c = ln & 15, g = ln >> 4;
            wave_sync();
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) sT[(16 * b + 4 * g + r) * kZS + c] = Z[b][r];
            wave_sync();
#pragma unroll
            for (int j = 0; j < kMaxW / 64; ++j)
                if (64 * j < wd) {
                    const float u = sT[(pos[j] >> 16) & 0x3fff];
                    float v = sT[pos[j] & 0x3fff];
                    v += pos[j] < 0 ? 0.0f : pos[j] & 0x40000000 ? -u : u;
                    d[j] += v;
                }
        };
        if constexpr (ahead(NB)) {
            edge_weights(T, B, dist[e], F, sFe, deg);
            stage_end<NB>(Q + e * dout * dout, dout * dout, st, sB);
            stage_begin<NB>(Q + (e + step < E ? e + step : e) * dout * dout, dout * dout, st);
        } else {
            stage_basis<NB>(Q + e * dout * dout, dout, sB, [&] { edge_weights(T, B, dist[e], F, sFe, deg); });
        }
        rotate_in<CT, NB, false>(gy + e * cout * dout, 0, cout, sB, dout, out_col, gd);
        if (Q != P) stage_basis<NB>(P + e * din * din, din, sB, [] {});
        for (int ci0 = 0; ci0 < cin; ci0 += 16) {
            v4f fs[1][NB], dfs[NB];
            rotate_in<1, NB, false>(x + e * cin * din, ci0, cin, sB, din, in_col, fs);
#pragma unroll
            for (int b = 0; b < NB; ++b) dfs[b] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            Mixer<CT> M, next;      // the patterns one rank ahead
            load_mixer<CT>(W, 0, ci0 / 16, M);
#pragma unroll
            for (int k = 0; k < kRank; ++k) {
                load_mixer<CT>(W, k + 1 < kRank ? k + 1 : k, ci0 / 16, next);
                const float* sFk = sFe + k * (wd + 1);
                v4f H[NB];
                v4f Z[NB];
#pragma unroll
                for (int b = 0; b < NB; ++b) Z[b] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
                mix_channels<CT, NB>(gd, M, H);
                M = next;
                const int ln = lane_id(), c = ln & 15, g = ln >> 4;
                wave_sync();    // the previous rank's reads
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r) sT[(16 * b + 4 * g + r) * kTS + c] = H[b][r];
                wave_sync();
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const v4f h = *reinterpret_cast<const v4f*>(sT + (16 * b + c) * kTS + 4 * g);
#pragma unroll
                    for (int r = 0; r < 4; ++r) Z[b] = mfma4(h[r], fs[0][b][r], Z[b]);
                }
                add_mixed<NB>(sFk, code, last, H, dfs);
                weights_of(Z, dF[k]);
            }
            rotate_out<NB>(dfs, sB, din, last, in_red, gx + e * cin * din, ci0 / 16, cin);
        }
        const float* spow = sFe + kRank * (wd + 1);
        float* de = dFe + e * kRank * wd;
        const int ln = lane_id();
#pragma unroll
        for (int j = 0; j < kMaxW / 64; ++j)
            if (64 * j < wd) {
                const unsigned w = ln + 64 * j < wd ? ln + 64 * j : wd - 1;
                const float q = spow[deg[j]];
#pragma unroll
                for (int k = 0; k < kRank; ++k) (de + k * wd)[w] = dF[k][j] * q;
            }
    }
}

// ---------------------------------------------------------------------------
// A wave owns one 16-channel tile of co for the launch; the workgroup's waves
// with the same tile take different edges, and their sums are added in order
// through LDS.  One partial (kRank, cout, cin) per workgroup.
template <int CT, int NB>
__global__ void __launch_bounds__(256, 2)
k_ewg_bwd_c(GenTab T, feq_binning B, int64_t E, int ncot, int subs, const float* __restrict__ gy,
            const float* __restrict__ x, const float* __restrict__ P, const float* __restrict__ Q,
            const float* __restrict__ dist, const float* __restrict__ F, float* __restrict__ part) {
    extern __shared__ float sm[];
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cin = T.cin, cout = T.cout, din = T.din, dout = T.dout, wd = T.wd, last = T.last;
    const int cot = wave % ncot, sub = wave / ncot;
    float* sB = sm + wave * wave_floats(wd, din, dout);
    float* sFe = sB + basis_floats(din, dout);
    int in_col[NB], in_red[NB], out_col[NB], out_red[NB], deg[4], code[NB][2];
    load_slots<NB>(T.in_slot, in_col, in_red);
    load_slots<NB>(T.out_slot, out_col, out_red);
    load_deg(T, deg);
    load_codes<NB, true>(T, code);
    v4f dC[kRank][CT];
#pragma unroll
    for (int k = 0; k < kRank; ++k)
#pragma unroll
        for (int t = 0; t < CT; ++t) dC[k][t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    const int64_t step = static_cast<int64_t>(gridDim.x) * subs, first = static_cast<int64_t>(blockIdx.x) * subs + sub;
    Staged<ahead(NB) ? NB : 1> st;
    if constexpr (ahead(NB))
        if (first < E) stage_begin<NB>(P + first * din * din, din * din, st);
    for (int64_t e = first; e < E; e += step) {
        v4f fs[CT][NB], gd[1][NB];
        if constexpr (ahead(NB)) {
            edge_weights(T, B, dist[e], F, sFe, deg);
            stage_end<NB>(P + e * din * din, din * din, st, sB);
            stage_begin<NB>(P + (e + step < E ? e + step : e) * din * din, din * din, st);
        } else {
            stage_basis<NB>(P + e * din * din, din, sB, [&] { edge_weights(T, B, dist[e], F, sFe, deg); });
        }
        rotate_in<CT, NB, true>(x + e * cin * din, 0, cin, sB, din, in_col, fs);
        if (Q != P) stage_basis<NB>(Q + e * dout * dout, dout, sB, [] {});
        rotate_in<1, NB, true>(gy + e * cout * dout, 16 * cot, cout, sB, dout, out_col, gd);
#pragma unroll
        for (int k = 0; k < kRank; ++k) {
            v4f U[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) U[b] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    if (b < NB - 1 || r < last) U[b] = mfma4(coef(sFe + k * (wd + 1), code[b], r), gd[0][b][r], U[b]);
            // the edge's product on its own, then added: a chain of additions
            // over the slots and one over the edges, not one over both
            v4f one[CT];
#pragma unroll
            for (int t = 0; t < CT; ++t) one[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (b < NB - 1 || r < last) {
#pragma unroll
                        for (int t = 0; t < CT; ++t) one[t] = mfma4(U[b][r], fs[t][b][r], one[t]);
                    }
#pragma unroll
            for (int t = 0; t < CT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) dC[k][t][r] += one[t][r];
        }
    }
    // the co tiles' sums over the workgroup's waves, in wave order
    __syncthreads();
    for (int s = 0; s < subs; ++s) {
        if (sub == s) {
#pragma unroll
            for (int k = 0; k < kRank; ++k)
#pragma unroll
                for (int t = 0; t < CT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int q = (((cot * kRank + k) * CT + t) * 4 + r) * 64 + lane;
                        sm[q] = s == 0 ? dC[k][t][r] : sm[q] + dC[k][t][r];
                    }
        }
        __syncthreads();
    }
    float* out = part + static_cast<int64_t>(blockIdx.x) * kRank * cout * cin;
    if (sub == 0) {
#pragma unroll
        for (int k = 0; k < kRank; ++k)
#pragma unroll
            for (int t = 0; t < CT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int co = 16 * cot + 4 * g + r, ci = 16 * t + c;
                    if (co < cout && ci < cin)
                        out[(static_cast<int64_t>(k) * cout + co) * cin + ci] =
                            sm[(((cot * kRank + k) * CT + t) * 4 + r) * 64 + lane];
                }
    }
}

// ---------------------------------------------------------------------------
// Packs the m-groups into blocks of 16 in and 16 out slots (first fit, widest
// group first); 0 when they do not fit kMaxNB.  Slot q of a block takes row
// 4 (q % 4) + q / 4: n slots then need ceil(n / 4) reduction steps.
int build_tab(const feq_layout& L, GenTab& T) {
    if (L.nblocks < 1 || L.nblocks > FEQ_MAX_BLOCKS || L.din < 1 || L.dout < 1 || L.cin < 1 || L.cout < 1) return 0;
    // the staged basis: four waves in a workgroup's LDS
    if (bwd_x_floats(L.wdim, L.din, L.dout, kMaxNB) > 160 * 1024 / 16) return 0;
    if (L.wdim > kMaxW || L.cin > 16 * kMaxCT || L.cout > 16 * kMaxCT || L.wdim < 1) return 0;
    T.cin = L.cin, T.cout = L.cout, T.din = L.din, T.dout = L.dout, T.wd = L.wdim;
    for (int q = 0; q < kMaxNB * 16; ++q) T.in_slot[q] = T.out_slot[q] = -1;
    for (int b = 0; b < kMaxNB; ++b)
        for (int o = 0; o < 16; ++o)
            for (int i = 0; i < 16; ++i) T.code[b][o][i] = static_cast<int16_t>(L.wdim);
    for (int w = 0; w < kMaxW; ++w) T.pos0[w] = T.pos1[w] = 0, T.deg[w] = 0;
    int order[FEQ_MAX_BLOCKS], used_in[kMaxNB] = {}, used_out[kMaxNB] = {}, nb = 0;
    auto width = [&](int k, int col) { return (L.blk[k][0] ? 2 : 1) * L.blk[k][col]; };
    for (int k = 0; k < L.nblocks; ++k) order[k] = k;
    for (int a = 1; a < L.nblocks; ++a)     // by the wider side, descending
        for (int b = a; b > 0; --b) {
            auto key = [&](int q) { return width(q, 1) > width(q, 2) ? width(q, 1) : width(q, 2); };
            if (key(order[b]) <= key(order[b - 1])) break;
            const int t = order[b];
            order[b] = order[b - 1], order[b - 1] = t;
        }
    auto row = [](int q) { return 4 * (q % 4) + q / 4; };
    for (int a = 0; a < L.nblocks; ++a) {
        const int k = order[a], wi = width(k, 1), wo = width(k, 2), z = L.blk[k][0] ? 2 : 1;
        int b = 0;
        while (b < kMaxNB && (used_in[b] + wi > 16 || used_out[b] + wo > 16)) ++b;
        if (b == kMaxNB) return 0;
        if (b + 1 > nb) nb = b + 1;
        const int i0 = used_in[b], o0 = used_out[b];
        used_in[b] += wi, used_out[b] += wo;
        for (int q = 0; q < wi; ++q) T.in_slot[16 * b + row(i0 + q)] = static_cast<int8_t>(L.blk[k][3] + q);
        for (int q = 0; q < wo; ++q) T.out_slot[16 * b + row(o0 + q)] = static_cast<int8_t>(L.blk[k][4] + q);
        auto put = [&](int o, int i, int w, int neg) {
            const int ro = row(o0 + o), ri = row(i0 + i), p = (16 * b + ro) * kZS + ri;
            T.code[b][ro][ri] = static_cast<int16_t>(w | (neg ? 0x4000 : 0));
            return p;
        };
        for (int o = 0; o < L.blk[k][2]; ++o)
            for (int i = 0; i < L.blk[k][1]; ++i) {
                const int w = L.blk[k][5] + z * (o * L.blk[k][1] + i);
                const int deg = L.lslot_in[L.blk[k][3] + z * i] + L.lslot_out[L.blk[k][4] + z * o];
                if (deg >= kMaxDeg) return 0;
                if (z == 1) {
                    T.pos0[w] = static_cast<int16_t>(put(o, i, w, 0));
                    T.pos1[w] = static_cast<int16_t>(T.pos0[w] | 0x8000);
                    T.deg[w] = static_cast<int8_t>(deg);
                    continue;
                }
                // re += a f_re + b f_im;  im += a f_im - b f_re
                T.pos0[w] = static_cast<int16_t>(put(2 * o, 2 * i, w, 0));
                T.pos1[w] = static_cast<int16_t>(put(2 * o + 1, 2 * i + 1, w, 0));
                T.pos0[w + 1] = static_cast<int16_t>(put(2 * o, 2 * i + 1, w + 1, 0));
                T.pos1[w + 1] = static_cast<int16_t>(put(2 * o + 1, 2 * i, w + 1, 1) | 0x4000);
                T.deg[w] = T.deg[w + 1] = static_cast<int8_t>(deg);
            }
    }
    const int n = used_in[nb - 1] > used_out[nb - 1] ? used_in[nb - 1] : used_out[nb - 1];
    T.last = (n + 3) / 4;
    return nb;
}

int tiles(int channels) { return (channels + 15) / 16; }

#define FEQ_EWG_NB(X, ct) X(ct, 1) X(ct, 2) X(ct, 3) X(ct, 4)
#define FEQ_EWG_SHAPES(X) FEQ_EWG_NB(X, 1) FEQ_EWG_NB(X, 2) FEQ_EWG_NB(X, 3) FEQ_EWG_NB(X, 4)

int set_lds(const void* fn, size_t bytes) {
    if (bytes > 64 * 1024)
        FEQ_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)));
    return FEQ_OK;
}

}  // namespace

bool ew_wave_supported(const feq_layout& L, int rank) {
    GenTab T;
    return rank == kRank && build_tab(L, T) > 0;
}

// Workgroups (and partials) of the pattern gradient: two per CU at most.
int ew_wave_groups(const feq_layout& L, int64_t E) {
    const int64_t n = ceil_div(E, 4 / tiles(L.cout));
    return static_cast<int>(n < 512 ? n : 512);
}

// The packed patterns.
size_t ew_wave_workspace(const feq_layout& L) {
    return kRank * tiles(L.cin) * tiles(L.cout) * 64 * sizeof(v4f) + 256;
}

template <bool BWD>
static int prep(const feq_layout& L, const float* C, void* ws, Patterns& W, hipStream_t s) {
    v4f* frag = reinterpret_cast<v4f*>(align_up(reinterpret_cast<uintptr_t>(ws), sizeof(v4f)));
    W = Patterns{frag, tiles(BWD ? L.cin : L.cout)};
    auto k = k_ewg_prep<BWD>;
    FEQ_LAUNCH("k_ewg_prep", k, dim3(kRank, W.ncol), dim3(64), 0, s, C, L.cout, L.cin, frag);
    return FEQ_OK;
}

int ew_wave_fwd(const feq_layout& L, const feq_binning& B, int rank, int64_t E, const float* x, const float* P,
                const float* Q, const float* dist, const float* C, const float* F, float* y, void* ws,
                size_t ws_bytes, hipStream_t s) {
    GenTab T;
    if (rank != kRank) return -1;
    const int nb = build_tab(L, T), ct = tiles(L.cin);
    if (!nb || !ws || ws_bytes < ew_wave_workspace(L)) return -1;
    Patterns W;
    if (int rc = prep<false>(L, C, ws, W, s)) return rc;
    void (*kern)(GenTab, feq_binning, int64_t, const float*, const float*, const float*, const float*, Patterns,
                 const float*, float*) = nullptr;
#define FEQ_PICK(c, n) if (ct == c && nb == n) kern = k_ewg_fwd<c, n>;
    FEQ_EWG_SHAPES(FEQ_PICK)
#undef FEQ_PICK
    const int64_t wgs = ceil_div(E, 4), most = 256 * fwd_groups(ct, nb);
    const dim3 grid(static_cast<unsigned>(wgs < most ? wgs : most));
    const size_t lds = 4 * sizeof(float) * wave_floats(L.wdim, L.din, L.dout);
    if (int rc = set_lds(reinterpret_cast<const void*>(kern), lds)) return rc;
    FEQ_LAUNCH("k_ewg_fwd", kern, grid, dim3(256), lds, s, T, B, E, x, P, Q, dist, W, F, y);
    return FEQ_OK;
}

int ew_wave_bwd(const feq_layout& L, const feq_binning& B, int rank, int64_t E, const float* gy, const float* x,
                const float* P, const float* Q, const float* dist, const float* C, const float* F, float* gx,
                float* dFe, float* dC_part, void* ws, hipStream_t s) {
    GenTab T;
    if (rank != kRank) return -1;
    const int nb = build_tab(L, T), cti = tiles(L.cin), cto = tiles(L.cout);
    if (!nb) return -1;
    Patterns W;
    if (int rc = prep<true>(L, C, ws, W, s)) return rc;
    void (*kx)(GenTab, feq_binning, int64_t, const float*, const float*, const float*, const float*, const float*,
               Patterns, const float*, float*, float*) = nullptr;
    void (*kc)(GenTab, feq_binning, int64_t, int, int, const float*, const float*, const float*, const float*,
               const float*, const float*, float*) = nullptr;
#define FEQ_PICK(c, n)                               \
    if (cto == c && nb == n) kx = k_ewg_bwd_x<c, n>; \
    if (cti == c && nb == n) kc = k_ewg_bwd_c<c, n>;
    FEQ_EWG_SHAPES(FEQ_PICK)
#undef FEQ_PICK
    const int64_t wgs = ceil_div(E, 4), most = 256 * bwd_x_groups(nb);
    const dim3 grid(static_cast<unsigned>(wgs < most ? wgs : most));
    const size_t lds = 4 * sizeof(float) * bwd_x_floats(L.wdim, L.din, L.dout, nb);
    if (int rc = set_lds(reinterpret_cast<const void*>(kx), lds)) return rc;
    FEQ_LAUNCH("k_ewg_bwd_x", kx, grid, dim3(256), lds, s, T, B, E, gy, x, P, Q, dist, W, F, gx, dFe);
    const int subs = 4 / cto, waves = subs * cto;
    const size_t sums = sizeof(float) * static_cast<size_t>(cto) * kRank * cti * 4 * 64;
    const size_t fe = sizeof(float) * waves * wave_floats(L.wdim, L.din, L.dout), clds = fe > sums ? fe : sums;
    if (int rc = set_lds(reinterpret_cast<const void*>(kc), clds)) return rc;
    FEQ_LAUNCH("k_ewg_bwd_c", kc, dim3(ew_wave_groups(L, E)), dim3(64 * waves), clds, s, T, B, E, cto, subs, gy, x, P,
               Q, dist, F, dC_part);
    return FEQ_OK;
}

}  // namespace feq
