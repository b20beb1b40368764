// The generic block-diagonal op in float32 as matrix products
// (v_mfma_f32_16x16x4_f32) over edges grouped by their lower bin.
//
// blockdiag.hip's per-edge kernels read both table rows of the bin for every
// edge (2 Cout Cin Wdim values: 156 KB at lvals 0..2 x 32), so the L2 bounds
// them.  Here a workgroup takes 16 edges in the order of their bins (the stable
// CSR by bin), one 16-channel tile of outputs, and reads each table row once for
// the 16:
//   forward   Y[co, e] (o)  += W_w,e[co, ci] X[ci, e] (i)
//   gradient  GX[ci, e] (i) += W_w,e[co, ci]^T G[co, e] (o)
//   table     dT_w[co, ci]  += sum over e of G[co, e] (o) X[ci, e] (i)
// with X = s^l x, G = s^l gy and W_e X = (1 - t_e) (T X) + t_e (T' X), T and T' the
// bin's row and the next one: neither term is larger than it has to be, and at either
// end of a bin its row alone counts.  Edges outside the bins, where the first and the
// last one extrapolate (|t| >> 1), take T X + t D X with the rows' difference D, which is
// well conditioned there as in the per-edge kernels; the distance gradient takes D X
// everywhere.  (T + t D for every edge: errors of y and dx 1.1 to 1.5 times the per-edge
// kernels'; the rows' mean and D: a small row beside a large one lost to it.)  The table
// is first packed into operand order (k_bdm_pack), zero-padded to 16 channels.
//
// Lane l = (c = l % 16, g = l / 16); a reduction step r takes the indices
// 4 r + g: the staged rows [slot][channel][edge] (257 floats from slot to slot)
// are then read as 64 consecutive floats.  The four waves of a workgroup share
// the staged rows and split the (m, output) pairs.  Sums run in a fixed order, the
// products of one summed index and 16 channels by themselves, then added.
//
// Lvals 0..2 x 32, 20 000 edges, 65 table rows, the per-edge kernels and these:
// forward 1163 us, now 86 + 13 (pack) + 35 (sort by bin); input and distance
// gradients 816 + 1724, now 155 + 14 (pack); table gradient 2256, now 159 + 12.
// The matrix steps alone would take 20 to 40 us each: the staging of 16 edges'
// rows, one memory latency per 16 channels, bounds these.  (Tiles dealt to the
// L2s in turn, so that each read every bin's fragments: 94 and 154 us.)
#include "blockdiag_edge.h"
#include "tile_math.h"

#include <cfloat>

namespace feq {
namespace {

constexpr int kThreads = 256;
constexpr int kSS = 257;        // floats from slot to slot of the staged rows
constexpr int kMaxSlots = 63;   // staged slots (64 KB of LDS)
constexpr int kMaxPairs = 64;
constexpr int kMaxUnits = 160;

// A pair: the z components of one index of an m-block, and the block's other side.
struct Pair {
    int8_t slot;     // first slot of the produced side
    int8_t other;    // first slot of the summed side
    int8_t n;        // indices summed over
    int8_t z;        // 1 or 2 components
    int16_t w;       // weight of the first summed index
    int16_t step;    // weights from one summed index to the next
};
struct Pairs {
    int32_t n;
    Pair p[kMaxPairs];
};
// A unit of the table gradient: the z weights of one (o, i) of an m-block.
struct Unit {
    int8_t o, i, z, pad;
    int16_t w;
};
struct Units {
    int32_t n;
    Unit u[kMaxUnits];
};

// Edge of a sorted position, with its bin state.
struct EdgeRow {
    int64_t e;
    int lo;
    float t, s, dtdr, r;
};
__device__ __forceinline__ EdgeRow edge_row(const feq_binning& B, const int32_t* __restrict__ perm,
                                            const float* __restrict__ dist, int64_t pos, int64_t E) {
    EdgeRow R;
    R.e = perm[pos < E ? pos : E - 1];
    R.r = dist[R.e];
    const EdgeBin eb = edge_bin(R.r, B);
    R.lo = eb.lo;
    R.t = eb.t;
    R.dtdr = eb.dtdr;
    R.s = R.r / (R.r + B.sh_scale);
    return R;
}

// Rows c0 .. c0 + 15 of (E, nch, dim) of the 16 edges at e[], times scale[edge][l]
// and weight[edge], to st[slot][channel][edge] (EDGE_MINOR) or
// st[slot][edge][channel]; zeros for channels outside and for edges from n on.  A
// thread requests kInFlight elements before it uses the first (four at a time took
// the table gradient 232 us instead of 154).
constexpr int kInFlight = 10;
template <bool EDGE_MINOR>
__device__ __forceinline__ void stage_rows(const float* __restrict__ x, int nch, int c0, int dim, const int64_t* e,
                                           const float* scale, int sstride, const int* deg, int n, float* st,
                                           const float* weight = nullptr) {
    const int per = 16 * dim, all = 16 * per;
    const float iper = 1.0f / static_cast<float>(per), idim = 1.0f / static_cast<float>(dim);
    for (int q0 = threadIdx.x; q0 < all; q0 += kInFlight * kThreads) {
        float v[kInFlight];
#pragma unroll
        for (int u = 0; u < kInFlight; ++u) {
            const int q = q0 + u * kThreads < all ? q0 + u * kThreads : all - 1;
            const int ed = quotient(q, iper), rest = q - ed * per, ch = quotient(rest, idim);
            const bool ok = ed < n && c0 + ch < nch;
            v[u] = x[ok ? (e[ed] * nch + c0) * dim + rest : 0];
            v[u] = ok ? v[u] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < kInFlight; ++u) {
            const int q = q0 + u * kThreads;
            if (q < all) {
                const int ed = quotient(q, iper), rest = q - ed * per, ch = quotient(rest, idim), d = rest - ch * dim;
                float sc = scale[ed * sstride + deg[d]];
                if (weight) sc *= weight[ed];
                st[d * kSS + (EDGE_MINOR ? ch * 16 + ed : ed * 16 + ch)] = v[u] * sc;
            }
        }
    }
}

__device__ __forceinline__ bool finite(float v) { return fabsf(v) <= FLT_MAX; }

constexpr int kPow = 32;        // powers of s kept per edge (+ 1: no bank conflicts)

// Operand order of the table: fragment (row b, w, row tile, reduction tile) holds for
// lane (c, g) four values r: T[co, ci] with, forward, co = 16 row + c and ci = 16 red
// + 4 r + g, and transposed (TR) with ci = 16 row + c and co = 16 red + 4 r + g.  The
// num_bins + 1 rows, then the differences D of the bins that need them: all (ALLD) or the
// first and the last.  A workgroup packs wchunk weights of the 16 x 16 channels of one
// row (all weights in turn left the chip idle: lvals 0..6 x 16, 64 bins, 155 us).
__host__ __device__ constexpr int diff_rows(int nb, bool alld) { return alld ? nb : nb < 2 ? nb : 2; }
__device__ __forceinline__ int diff_row(int bin, int nb, bool alld) { return nb + 1 + (alld ? bin : bin ? 1 : 0); }

__host__ __device__ constexpr int pack_floats(int wchunk) { return 256 * (wchunk | 1) + 16; }

// Values that a thread requests before it uses the first (one at a time: 22 us a packing
// at lvals 0..2 x 32 and 64 bins instead of 13).
constexpr int kPackAhead = 5;

template <bool TR, bool ALLD>
__global__ void __launch_bounds__(kThreads)
k_bdm_pack(const float* __restrict__ table, int nb, int cout, int cin, int wd, int wchunk, float* __restrict__ frag) {
    // T, then D: [16][16][ls], an odd number of floats from channel to channel either way
    extern __shared__ float sm[];
    const int b = blockIdx.x;
    const int nci = (cin + 15) / 16, nco = (cout + 15) / 16;
    const int cot = blockIdx.y / nci, cit = blockIdx.y % nci;
    const int row = TR ? cit : cot, red = TR ? cot : cit, nrow = TR ? nci : nco, nred = TR ? nco : nci;
    const int64_t ts = static_cast<int64_t>(cout) * cin * wd;
    const int w0 = blockIdx.z * wchunk, nw = wd - w0 < wchunk ? wd - w0 : wchunk;
    const int ls = wchunk | 1, half = pack_floats(wchunk);
    const bool diff = b < nb && (ALLD || b == 0 || b == nb - 1);
    const float inw = 1.0f / static_cast<float>(nw);
    for (int w1 = 0; w1 < nw; w1 += kPackAhead) {       // kThreads values a step, kPackAhead steps in flight
        float lo[kPackAhead], hi[kPackAhead];
        int to[kPackAhead];
#pragma unroll
        for (int u = 0; u < kPackAhead; ++u) {
            const int q = kThreads * (w1 + u < nw ? w1 + u : nw - 1) + threadIdx.x;
            const int ch = quotient(q, inw), w = q - ch * nw, co = 16 * cot + ch / 16, ci = 16 * cit + ch % 16;
            const bool ok = co < cout && ci < cin;
            const int64_t at = ok ? b * ts + (static_cast<int64_t>(co) * cin + ci) * wd + w0 + w : 0;
            lo[u] = table[at];
            hi[u] = table[ok && diff ? at + ts : at];
            lo[u] = ok ? lo[u] : 0.0f;
            hi[u] = ok ? hi[u] : 0.0f;
            to[u] = ch * ls + ch / 16 + w;
        }
#pragma unroll
        for (int u = 0; u < kPackAhead; ++u) {
            sm[to[u]] = lo[u];
            if (diff) sm[half + to[u]] = hi[u] - lo[u];
        }
    }
    __syncthreads();
    for (int q = threadIdx.x; q < (diff ? 512 : 256) * nw; q += kThreads) {
        const int d = q >= 256 * nw, w = q / 256 - d * nw, k = q & 255, l = k >> 2, r = k & 3;
        const int a = l & 15, z = 4 * r + (l >> 4);       // row and reduction channel
        const int ch = TR ? z * 16 + a : a * 16 + z;
        const int64_t fr = d ? diff_row(b, nb, ALLD) : b;
        frag[(((fr * wd + w0 + w) * nrow + row) * nred + red) * 256 + k] = sm[half * d + ch * ls + ch / 16 + w];
    }
}

// ---------------------------------------------------------------------------
// A tile's product for up to MAXP pairs per wave: acc[p] += W S, and with GD accD[p] +=
// D S, accS[p] += l (W S) (S: the staged rows, l: the degree of the summed slot; the
// distance gradient's three sums).
template <int MAXP, bool GD>
struct TileAcc {
    v4f a[MAXP][2];
    v4f d[GD ? MAXP : 1][2];
    v4f s[GD ? MAXP : 1][2];
};

// SIGN: +1 forward (re += a re + b im, im += a im - b re), -1 transposed
// (re += a re - b im, im += a im + b re).  in: whether the lane's column, an edge,
// is of this bin.  The other columns' products are formed and not taken: multiplied
// by zeros instead, a row of the table with an infinity or NaN would reach edges
// that never read it.  outer: the columns outside the bins, else those inside.
template <int MAXP, bool GD, int SIGN>
__device__ __forceinline__ void tile_product(const Pairs& PT, int wave, const float* __restrict__ frag, int bin, int nb,
                                             int wd, int nrow, int row, int nred, int red, const float* st, bool outer,
                                             bool in, float t, const int* deg, TileAcc<MAXP, GD>& A) {
    const unsigned lane = threadIdx.x & 63;
    const int64_t wstride = static_cast<int64_t>(nrow) * nred * 256, bstride = wstride * wd;
    const float* f0 = frag + (static_cast<int64_t>(row) * nred + red) * 256;
    const float* fT = f0 + bin * bstride;
    const float* fD = f0 + diff_row(bin, nb, GD) * bstride;
    const float* fB = outer ? fD : fT + bstride;
    const float ta = outer ? 1.0f : 1.0f - t;
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int p = 0; p < MAXP; ++p) {
        if (wave + 4 * p >= PT.n) break;
        const Pair P = PT.p[wave + 4 * p];
        v4f Tn[2], Bn[2], Dn[2];        // the next summed index's fragments
        auto fetch = [&](int k) {
            const int64_t at = (P.w + k * P.step) * wstride + 4 * lane;
            Tn[0] = *reinterpret_cast<const v4f*>(fT + at);
            Bn[0] = *reinterpret_cast<const v4f*>(fB + at);
            if constexpr (GD) Dn[0] = *reinterpret_cast<const v4f*>(fD + at);
            if (P.z == 2) {
                Tn[1] = *reinterpret_cast<const v4f*>(fT + at + wstride);
                Bn[1] = *reinterpret_cast<const v4f*>(fB + at + wstride);
                if constexpr (GD) Dn[1] = *reinterpret_cast<const v4f*>(fD + at + wstride);
            }
        };
        fetch(0);
        for (int k = 0; k < P.n; ++k) {
            const float* sr = st + (P.other + P.z * k) * kSS;
            const v4f T[2] = {Tn[0], Tn[1]}, T1[2] = {Bn[0], Bn[1]}, D[2] = {Dn[0], Dn[1]};
            v4f S[2];
            if (k + 1 < P.n) fetch(k + 1);
#pragma unroll
            for (int r = 0; r < 4; ++r) S[0][r] = sr[64 * r + lane];
            if (P.z == 2) {
#pragma unroll
                for (int r = 0; r < 4; ++r) S[1][r] = sr[kSS + 64 * r + lane];
            }
            // components of the product of the (a, b) fragments Q and the rows S
            auto product = [&](const v4f (&Q)[2], v4f (&out)[2]) {
                out[0] = out[1] = zero;
#pragma unroll
                for (int r = 0; r < 4; ++r) out[0] = mfma4(Q[0][r], S[0][r], out[0]);
                if (P.z == 2) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        out[1] = mfma4(Q[0][r], S[1][r], out[1]);
                        out[0] = mfma4(Q[1][r], SIGN > 0 ? S[1][r] : -S[1][r], out[0]);
                        out[1] = mfma4(Q[1][r], SIGN > 0 ? -S[0][r] : S[0][r], out[1]);
                    }
                }
            };
            v4f ts[2], bs[2], ds[2];
            product(T, ts);
            product(T1, bs);
            if constexpr (GD) product(D, ds);
            const float l = GD ? static_cast<float>(deg[P.other + P.z * k]) : 0.0f;
#pragma unroll
            for (int z = 0; z < 2; ++z)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float v = in ? fmaf(t, bs[z][r], ta * ts[z][r]) : 0.0f;
                    A.a[p][z][r] += v;
                    if constexpr (GD) {
                        A.d[p][z][r] += in ? ds[z][r] : 0.0f;
                        A.s[p][z][r] = fmaf(l, v, A.s[p][z][r]);
                    }
                }
        }
    }
}

template <int MAXP, bool GD>
__device__ __forceinline__ void clear(TileAcc<MAXP, GD>& A) {
#pragma unroll
    for (int p = 0; p < MAXP; ++p)
#pragma unroll
        for (int z = 0; z < 2; ++z) A.a[p][z] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (GD)
#pragma unroll
        for (int p = 0; p < MAXP; ++p)
#pragma unroll
            for (int z = 0; z < 2; ++z) A.d[p][z] = A.s[p][z] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
}

// Workgroup (tile of 16 sorted positions, 16-channel tile of outputs); x: the
// summed side (E, nch, din) scaled by s^l, y: the produced side (E, noch, dout).
// GD: the distance gradient's share of this channel tile to gpart[tile of
// channels][position's edge], from xo, the features on the produced side.  Edges
// whose results hold an infinity or NaN are formed again from the unpacked table,
// as the per-edge kernels form them: two infinite products are NaN where the
// interpolated weight's is not.
template <int MAXP, bool GD, int SIGN>
__global__ void __launch_bounds__(kThreads, 2)
k_bdm_apply(feq_layout L, Pairs PT, feq_binning B, int64_t E, const int32_t* __restrict__ perm,
            const float* __restrict__ dist, const float* __restrict__ x, int nch, int din, int noch, int dout, int wd,
            const float* __restrict__ table, const float* __restrict__ frag, const float* __restrict__ xo,
            float* __restrict__ y, float* __restrict__ gpart, unsigned tiles) {
    extern __shared__ float st[];
    __shared__ float sPow[16 * (kPow + 1)];
    __shared__ int64_t sE[16];
    __shared__ int sKey[16];            // 2 bin, + 1 where the edge lies outside the bins
    __shared__ float sRed[4 * 64];
    __shared__ int sBad[16];
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // the eight L2s (workgroups go to them in turn) take an eighth of the sorted
    // tiles each: a bin's fragments are then read into one or two of them
    const unsigned each = gridDim.x / 8;
    const unsigned tile = (blockIdx.x & 7) * each + (blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int64_t p0 = static_cast<int64_t>(tile) * 16;
    const int n = static_cast<int>(E - p0 < 16 ? E - p0 : 16);
    __shared__ int din_deg[kMaxSlots + 1], dout_deg[kMaxSlots + 1];
    for (int q = threadIdx.x; q < din; q += kThreads) din_deg[q] = SIGN > 0 ? L.lslot_in[q] : L.lslot_out[q];
    for (int q = threadIdx.x; q < dout; q += kThreads) dout_deg[q] = SIGN > 0 ? L.lslot_out[q] : L.lslot_in[q];
    const EdgeRow R = edge_row(B, perm, dist, p0 + (c < n ? c : n - 1), E);
    const int key = 2 * R.lo + ((R.lo == 0 && R.t < 0.0f) || (R.lo == B.num_bins - 1 && R.t > 1.0f));
    if (threadIdx.x < 16) {
        sE[c] = R.e;
        sKey[c] = key;
        sBad[c] = 0;
        float p = 1.0f;
        for (int l = 0; l < kPow; ++l) {
            sPow[c * (kPow + 1) + l] = p;
            p *= R.s;
        }
    }
    __syncthreads();
    const int row = blockIdx.y, nrow = gridDim.y, nred = (nch + 15) / 16;
    TileAcc<MAXP, GD> A;
    clear(A);
    for (int red = 0; red < nred; ++red) {
        __syncthreads();
        stage_rows<true>(x, nch, 16 * red, din, sE, sPow, kPow + 1, din_deg, n, st);
        __syncthreads();
        for (int p = 0; p < n;) {       // the tile's bins, in order
            const int bin = __builtin_amdgcn_readfirstlane(sKey[p] >> 1);
            int kinds = 0;
            while (p < n && sKey[p] >> 1 == bin) kinds |= 1 << (sKey[p++] & 1);
            kinds = __builtin_amdgcn_readfirstlane(kinds);
#pragma unroll 1
            for (int outer = 0; outer < 2; ++outer)
                if (kinds >> outer & 1)
                    tile_product<MAXP, GD, SIGN>(PT, wave, frag, bin, B.num_bins, wd, nrow, row, nred, red, st, outer,
                                                 key == 2 * bin + outer, R.t, din_deg, A);
        }
    }
    if constexpr (GD) {
        // x on the produced side: sum of x accD, and of l x acc + x accS
        __syncthreads();
        stage_rows<true>(xo, noch, 16 * row, dout, sE, sPow, kPow + 1, dout_deg, n, st);
        __syncthreads();
        float atr[4] = {}, asr[4] = {};     // four short chains of additions
#pragma unroll
        for (int p = 0; p < MAXP; ++p) {
            if (wave + 4 * p >= PT.n) break;
            const Pair P = PT.p[wave + 4 * p];
            const float l = static_cast<float>(dout_deg[P.slot]);
            for (int z = 0; z < P.z; ++z) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float q = st[(P.slot + z) * kSS + (4 * g + r) * 16 + c];
                    const v4f a = z ? A.a[p][1] : A.a[p][0], d = z ? A.d[p][1] : A.d[p][0], s = z ? A.s[p][1] : A.s[p][0];
                    atr[r] += q * d[r];
                    asr[r] += q * (l * a[r] + s[r]);
                }
            }
        }
        const float at = (atr[0] + atr[1]) + (atr[2] + atr[3]), as = (asr[0] + asr[1]) + (asr[2] + asr[3]);
        float v = at * R.dtdr;
        if (L.has_lpos) v += as * (B.sh_scale / (R.r * (R.r + B.sh_scale)));
        sRed[threadIdx.x] = v;
        __syncthreads();
        if (threadIdx.x < n) {
            float sum = 0.0f;
            for (int k = 0; k < 16; ++k) sum += sRed[16 * k + threadIdx.x];
            gpart[static_cast<int64_t>(row) * E + sE[threadIdx.x]] = sum;
            if (!finite(sum)) sBad[threadIdx.x] = 1;
        }
    }
    // the produced rows through LDS, so that they leave in whole runs
    __syncthreads();
    for (int q = threadIdx.x; q < dout * kSS; q += kThreads) st[q] = 0.0f;    // slots that no weight reaches
    __syncthreads();
#pragma unroll
    for (int p = 0; p < MAXP; ++p) {
        if (wave + 4 * p >= PT.n) break;
        const Pair P = PT.p[wave + 4 * p];
        const float sc = sPow[c * (kPow + 1) + dout_deg[P.slot]];
#pragma unroll
        for (int z = 0; z < 2; ++z)
            if (z < P.z) {
#pragma unroll
                for (int r = 0; r < 4; ++r) st[(P.slot + z) * kSS + (4 * g + r) * 16 + c] = A.a[p][z][r] * sc;
            }
    }
    __syncthreads();
    const int per = 16 * dout;
    const float iper = 1.0f / static_cast<float>(per), idim = 1.0f / static_cast<float>(dout);
    for (int q = threadIdx.x; q < n * per; q += kThreads) {
        const int ed = quotient(q, iper), rest = q - ed * per, ch = quotient(rest, idim), d = rest - ch * dout;
        if (16 * row + ch < noch) {
            const float v = st[d * kSS + ch * 16 + ed];
            y[(sE[ed] * noch + 16 * row) * dout + rest] = v;
            if (!finite(v)) sBad[ed] = 1;
        }
    }
    __syncthreads();
    const int nc = noch - 16 * row < 16 ? noch - 16 * row : 16;
    for (int ed = 0; ed < n; ++ed) {
        if (!sBad[ed]) continue;
        const int64_t e = sE[ed];
        const float r = dist[e], sw = r / (r + B.sh_scale);
        const EdgeBinT<float> eb = edge_bin_t<float>(r, B);
        const int64_t ts = static_cast<int64_t>(L.cout) * L.cin * wd;
        const float* tlo = table + eb.lo * ts;
        const float* xr = x + e * nch * din;
        float* yr = y + (e * noch + 16 * row) * dout;
        for (int q = threadIdx.x; q < nc * dout; q += kThreads)
            yr[q] = SIGN > 0 ? out_entry<float>(L, xr, 16 * row + q / dout, q % dout, tlo, tlo + ts, eb.t, sw)
                             : in_entry<float>(L, xr, 16 * row + q / dout, q % dout, tlo, tlo + ts, eb.t, sw);
        if constexpr (GD) {
            float at = 0.0f, as = 0.0f;
            for (int q = threadIdx.x; q < L.cout * nc * wd; q += kThreads) {
                const int w = q % wd, ci = 16 * row + q / wd % nc, co = q / (wd * nc);
                const float* tw = tlo + (static_cast<int64_t>(co) * L.cin + ci) * wd + w;
                dist_terms<float>(L, w, xo + (e * noch + ci) * dout, xr + co * din, tw[0], tw[ts], eb.t, sw,
                                  B.sh_scale / (r * (r + B.sh_scale)), at, as);
            }
            sRed[threadIdx.x] = at * eb.dtdr + as;
            __syncthreads();
            if (threadIdx.x == 0) {
                float sum = 0.0f;
                for (int k = 0; k < kThreads; ++k) sum += sRed[k];
                gpart[static_cast<int64_t>(row) * E + e] = sum;
            }
            __syncthreads();
        }
    }
}

// gdist[e] = the channel tiles' shares in order.
__global__ void k_bdm_dr(const float* __restrict__ part, int n, int64_t E, float* __restrict__ gdist) {
    const int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
    if (e >= E) return;
    float v = part[e];
    for (int k = 1; k < n; ++k) v += part[k * E + e];
    gdist[e] = v;
}

// ---------------------------------------------------------------------------
// Workgroup (table row b, co and ci tile, chunk of 4 kMaxU units and a split of the
// row's edges): the edges of bin b (weight 1 - t) and of bin b - 1 (weight t) in
// sorted order, 16 at a time, their indices, bins and powers 64 at a time (one
// memory latency for four tiles).  Few table rows leave the chip idle (65 rows
// and 4 tiles: 260 workgroups, 577 us, 232 with eight splits and 156 with kInFlight), so the edges
// are then split and the splits' sums added in order (k_bdm_sum).  Three workgroups
// per CU, with a few registers spilled: 190 us with two.
constexpr int kMaxU = 8;
constexpr int kHead = 64;

__global__ void __launch_bounds__(kThreads, 3)
k_bdm_table(feq_layout L, Units UT, feq_binning B, int64_t E, const int32_t* __restrict__ perm,
            const int32_t* __restrict__ offsets, const float* __restrict__ dist, const float* __restrict__ gy,
            const float* __restrict__ x, int splits, float* __restrict__ gtable) {
    extern __shared__ float st[];       // gy rows, then x rows
    __shared__ float sPow[kHead * (kPow + 1)];
    __shared__ int64_t sE[kHead];
    __shared__ float sW[kHead];
    __shared__ int sDegI[kMaxSlots + 1], sDegO[kMaxSlots + 1];
    const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int cin = L.cin, cout = L.cout, din = L.din, dout = L.dout, wd = L.wdim, nb = B.num_bins;
    const int b = blockIdx.x, nci = (cin + 15) / 16, cot = blockIdx.y / nci, cit = blockIdx.y % nci;
    const int split = blockIdx.z % splits;
    for (int q = threadIdx.x; q < din; q += kThreads) sDegI[q] = L.lslot_in[q];
    for (int q = threadIdx.x; q < dout; q += kThreads) sDegO[q] = L.lslot_out[q];
    const int u0 = (blockIdx.z / splits) * 4 * kMaxU + wave;
    float* sg = st;
    float* sx = st + dout * kSS;
    v4f acc[kMaxU][2];
#pragma unroll
    for (int u = 0; u < kMaxU; ++u) acc[u][0] = acc[u][1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    const int a0 = b < nb ? offsets[b] : 0, n_lo = b < nb ? offsets[b + 1] - a0 : 0;
    const int h0 = b > 0 ? offsets[b - 1] : 0, n_all = n_lo + (b > 0 ? offsets[b] - h0 : 0);
    const int per = ((n_all + splits - 1) / splits + 15) / 16 * 16;
    const int end = per * (split + 1) < n_all ? per * (split + 1) : n_all;
    for (int base = per * split, head = 0; base < end; base += 16, head = (head + 16) % kHead) {
        const int n = end - base < 16 ? end - base : 16;
        __syncthreads();
        if (head == 0) {
            if (threadIdx.x < kHead) {
                const int pos = base + lane < end ? base + lane : end - 1;
                const EdgeRow R = edge_row(B, perm, dist, pos < n_lo ? a0 + pos : h0 + pos - n_lo, E);
                sE[lane] = R.e;
                sW[lane] = pos < n_lo ? 1.0f - R.t : R.t;
                float p = 1.0f;
                for (int l = 0; l < kPow; ++l) {
                    sPow[lane * (kPow + 1) + l] = p;
                    p *= R.s;
                }
            }
            __syncthreads();
        }
        stage_rows<false>(gy, cout, 16 * cot, dout, sE + head, sPow + head * (kPow + 1), kPow + 1, sDegO, n, sg,
                          sW + head);
        stage_rows<false>(x, cin, 16 * cit, din, sE + head, sPow + head * (kPow + 1), kPow + 1, sDegI, n, sx);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kMaxU; ++u) {
            if (u0 + 4 * u >= UT.n) break;
            const Unit U = UT.u[u0 + 4 * u];
            const float* ga = sg + U.o * kSS;
            const float* xa = sx + U.i * kSS;
            // the 16 edges' sum by itself, then added: a short chain of additions and
            // one over the tiles, not one over all edges
            v4f one[2] = {v4f{0.0f, 0.0f, 0.0f, 0.0f}, v4f{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float gr = ga[64 * r + lane], fr = xa[64 * r + lane];
                one[0] = mfma4(gr, fr, one[0]);
                if (U.z == 2) {     // a: fr gr + fi gi, b: fi gr - fr gi
                    const float gi = ga[kSS + 64 * r + lane], fi = xa[kSS + 64 * r + lane];
                    one[0] = mfma4(gi, fi, one[0]);
                    one[1] = mfma4(gr, fi, one[1]);
                    one[1] = mfma4(gi, -fr, one[1]);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[u][0][r] += one[0][r], acc[u][1][r] += one[1][r];
        }
    }
    const int ci = 16 * cit + c;
#pragma unroll
    for (int u = 0; u < kMaxU; ++u) {
        if (u0 + 4 * u >= UT.n) break;
        const Unit U = UT.u[u0 + 4 * u];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int co = 16 * cot + 4 * g + r;
            if (co < cout && ci < cin) {
                float* o = gtable + (((static_cast<int64_t>(split) * (nb + 1) + b) * cout + co) * cin + ci) * wd + U.w;
                o[0] = acc[u][0][r];
                if (U.z == 2) o[1] = acc[u][1][r];
            }
        }
    }
}

// out[q] = the splits' sums in order.
__global__ void __launch_bounds__(kThreads)
k_bdm_sum(const float* __restrict__ part, int splits, int64_t n, float* __restrict__ out) {
    const int64_t q = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
    if (q >= n) return;
    float v = part[q];
    for (int k = 1; k < splits; ++k) v += part[k * n + q];
    out[q] = v;
}

// ---------------------------------------------------------------------------
// The pairs of the produced side, the costliest first so that the waves' shares
// are even; false when there are more than kMaxPairs.
bool build_pairs(const feq_layout& L, bool transposed, Pairs& T) {
    T.n = 0;
    for (int k = 0; k < L.nblocks; ++k) {
        const int z = L.blk[k][0] ? 2 : 1, ni = L.blk[k][1], no = L.blk[k][2];
        for (int a = 0; a < (transposed ? ni : no); ++a) {
            if (T.n == kMaxPairs) return false;
            Pair& p = T.p[T.n++];
            p.z = static_cast<int8_t>(z);
            p.n = static_cast<int8_t>(transposed ? no : ni);
            p.slot = static_cast<int8_t>((transposed ? L.blk[k][3] : L.blk[k][4]) + z * a);
            p.other = static_cast<int8_t>(transposed ? L.blk[k][4] : L.blk[k][3]);
            p.w = static_cast<int16_t>(L.blk[k][5] + z * (transposed ? a : a * ni));
            p.step = static_cast<int16_t>(transposed ? z * ni : z);
        }
    }
    auto cost = [](const Pair& p) { return p.n * p.z * p.z; };
    for (int a = 1; a < T.n; ++a)
        for (int b = a; b > 0 && cost(T.p[b]) > cost(T.p[b - 1]); --b) {
            const Pair t = T.p[b];
            T.p[b] = T.p[b - 1], T.p[b - 1] = t;
        }
    return true;
}

bool build_units(const feq_layout& L, Units& T) {
    T.n = 0;
    for (int z = 2; z >= 1; --z)        // the two-weight units first, dealt evenly
        for (int k = 0; k < L.nblocks; ++k) {
            if ((L.blk[k][0] ? 2 : 1) != z) continue;
            for (int o = 0; o < L.blk[k][2]; ++o)
                for (int i = 0; i < L.blk[k][1]; ++i) {
                    if (T.n == kMaxUnits) return false;
                    T.u[T.n++] = Unit{static_cast<int8_t>(L.blk[k][4] + z * o), static_cast<int8_t>(L.blk[k][3] + z * i),
                                      static_cast<int8_t>(z), 0,
                                      static_cast<int16_t>(L.blk[k][5] + z * (o * L.blk[k][1] + i))};
                }
        }
    return true;
}

int tiles16(int n) { return (n + 15) / 16; }
// Weights per workgroup of the packing: up to 47 KB of LDS, or 16 where they are more.
int pack_chunk(int wd) { return wd < 24 ? wd : 16; }
// alld: the differences of every bin (the distance gradient rides along).
size_t frag_floats(const feq_layout& L, const feq_binning& B, bool alld) {
    return (static_cast<size_t>(B.num_bins) + 1 + diff_rows(B.num_bins, alld)) * L.wdim * tiles16(L.cin) * tiles16(L.cout) * 256;
}
constexpr int kMaxP = 8;        // pairs per wave; 4 with the distance gradient's sums

template <bool TR, bool ALLD>
int pack(const feq_layout& L, const feq_binning& B, const float* table, float* frag, hipStream_t s) {
    auto k = k_bdm_pack<TR, ALLD>;
    const int chunk = pack_chunk(L.wdim);
    FEQ_LAUNCH("k_bdm_pack", k,
               dim3(B.num_bins + 1, tiles16(L.cin) * tiles16(L.cout), static_cast<unsigned>(ceil_div(L.wdim, chunk))),
               dim3(kThreads), sizeof(float) * 2 * pack_floats(chunk), s, table, B.num_bins, L.cout, L.cin, L.wdim, chunk, frag);
    return FEQ_OK;
}

}  // namespace

// Where the products run.  Their fixed cost is the sort by bin and two packings,
// about 60 us, against 3 to 5 ps per edge and table weight in a per-edge kernel: from
// kMinWork edges times weights on they are faster.  Around it, forward and backward in us,
// per-edge kernels and products: lvals 0..2 x 16, 8000 edges 112 and 937, 58 and 109; x 32,
// 1300 edges 98 and 434, 60 and 110; lvals 0..6 x 16, 440 edges 226 and 785, 146 and 622;
// x 8, 20 000 edges 83 and 1415, 80 and 165.
constexpr double kMinWork = 2.5e7;
// The packed table takes no more memory than this.
constexpr size_t kMaxFragBytes = size_t{4} << 30;

static bool covers(const feq_layout& L, const feq_binning& B, int64_t E) {
    Pairs P;
    Units U;
    if (L.din > kMaxSlots || L.dout > kMaxSlots || L.wdim < 1 || B.num_bins < 1) return false;
    for (int q = 0; q < L.din; ++q)
        if (L.lslot_in[q] >= kPow) return false;
    for (int q = 0; q < L.dout; ++q)
        if (L.lslot_out[q] >= kPow) return false;
    if (sizeof(float) * kSS * static_cast<size_t>(L.din + L.dout) > 128 * 1024) return false;
    if (!build_pairs(L, false, P) || P.n > 4 * kMaxP || !build_pairs(L, true, P) || P.n > 4 * kMaxP) return false;
    if (!build_units(L, U)) return false;
    return static_cast<double>(E) * L.cin * L.cout * L.wdim >= kMinWork &&
           frag_floats(L, B, true) * sizeof(float) <= kMaxFragBytes;
}

// The backward takes them wherever they are covered: it sorts in any case, and its
// per-edge distance and table gradients are slow enough that the packing of more bins
// than edges pays too (lvals 0..2 x 32, 4096 bins, 2000 edges: 1399 -> 837 us; x 1, padded
// to 16, 4096 bins, 1 400 000 edges: 12.0 -> 5.0 ms).
bool bdm_bwd_supported(const feq_layout& L, const feq_binning& B, int64_t E) { return covers(L, B, E); }

// The forward where the packing does not cost more than the per-edge kernel: 4 ps per
// packed weight (rows times weights of channels padded to 16) against 4 per edge and weight,
// or against the 2.5 ns per weight that a few edges take together.  Lvals 0..2, per-edge
// kernel and products: x 32, 4096 bins, 2000 edges 244 and 339 us, 4096 edges 456 and 361;
// 1000 bins, 1400 edges 166 and 164; x 64, 1000 bins, 700 edges 355 and 438, 1000 edges
// 453 and 440; x 16, 10 000 bins, 8000 edges 223 and 223; lvals 0..6 x 32, 100 bins, 131
// edges 829 and 775; x 128, 7 edges 8.4 and 3.1 ms.
bool bdm_fwd_supported(const feq_layout& L, const feq_binning& B, int64_t E) {
    if (!covers(L, B, E)) return false;
    const double weights = static_cast<double>(L.cin) * L.cout * L.wdim;
    const double packed = static_cast<double>(frag_floats(L, B, false));     // rows times padded weights
    return 4.0 * packed <= weights * (4.0 * static_cast<double>(E) > 2500.0 ? 4.0 * static_cast<double>(E) : 2500.0);
}

namespace {
size_t table_floats(const feq_layout& L, const feq_binning& B) {
    return static_cast<size_t>(B.num_bins + 1) * L.cout * L.cin * L.wdim;
}
// Splits of a table row's edges: enough workgroups for eight per CU, at least 32
// edges (of the 2 E / rows that a row has on average) each, at most eight.
int table_splits(const feq_layout& L, const feq_binning& B, int64_t E, int units) {
    const int64_t wgs = static_cast<int64_t>(B.num_bins + 1) * tiles16(L.cin) * tiles16(L.cout) * ceil_div(units, 4 * kMaxU);
    int64_t n = ceil_div(2048, wgs);
    const int64_t most = 2 * E / (B.num_bins + 1) / 32;
    n = n < most ? n : most;
    return static_cast<int>(n < 1 ? 1 : n > 8 ? 8 : n);
}
}  // namespace

size_t bdm_fwd_workspace(const feq_layout& L, const feq_binning& B) { return sizeof(float) * frag_floats(L, B, false); }

size_t bdm_bwd_workspace(const feq_layout& L, const feq_binning& B, int64_t E) {
    Units U;
    build_units(L, U);
    const int splits = table_splits(L, B, E, U.n);
    return sizeof(float) * (align_up(frag_floats(L, B, true), 64) + align_up(static_cast<size_t>(E) * tiles16(L.cin), 64) +
                            (splits > 1 ? splits * table_floats(L, B) : 0));
}

static int bdm_lds(const void* fn, size_t bytes) {
    if (bytes > 48 * 1024)      // with the kernels' static LDS (up to 10 KB) beyond 64 KB
        FEQ_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)));
    return FEQ_OK;
}

int bdm_fwd(const feq_layout& L, const feq_binning& B, int64_t E, const float* x, const float* table, const float* dist,
            const int32_t* perm, float* y, void* ws, hipStream_t s) {
    Pairs P;
    build_pairs(L, false, P);
    float* frag = static_cast<float*>(ws);
    if (int rc = pack<false, false>(L, B, table, frag, s)) return rc;
    auto k = P.n <= 16 ? k_bdm_apply<4, false, 1> : k_bdm_apply<kMaxP, false, 1>;
    const size_t lds = sizeof(float) * kSS * (L.din > L.dout ? L.din : L.dout);
    if (int rc = bdm_lds(reinterpret_cast<const void*>(k), lds)) return rc;
    FEQ_LAUNCH("k_bdm_fwd", k, dim3(static_cast<unsigned>(ceil_div(ceil_div(E, 16), 8) * 8), tiles16(L.cout)), dim3(kThreads), lds, s, L,
               P, B, E, perm, dist, x, L.cin, L.din, L.cout, L.dout, L.wdim, table, frag, static_cast<const float*>(nullptr), y,
               static_cast<float*>(nullptr), static_cast<unsigned>(ceil_div(E, 16)));
    return FEQ_OK;
}

int bdm_bwd(const feq_layout& L, const feq_binning& B, int64_t E, const float* gy, const float* x, const float* table,
            const float* dist, const int32_t* perm, const int32_t* offsets, float* gx, float* gtable, float* gdist,
            bool* dr_done, void* ws, hipStream_t s) {
    Pairs P;
    Units U;
    build_pairs(L, true, P);
    build_units(L, U);
    float* frag = static_cast<float*>(ws);
    float* gpart = frag + align_up(frag_floats(L, B, true), 64);
    // the distance gradient rides along where its sums fit the registers
    const bool gd = gdist && P.n <= 16;
    if (int rc = gd ? pack<true, true>(L, B, table, frag, s) : pack<true, false>(L, B, table, frag, s)) return rc;
    auto k = gd ? k_bdm_apply<4, true, -1> : P.n <= 16 ? k_bdm_apply<4, false, -1> : k_bdm_apply<kMaxP, false, -1>;
    const size_t lds = sizeof(float) * kSS * (L.din > L.dout ? L.din : L.dout);
    if (int rc = bdm_lds(reinterpret_cast<const void*>(k), lds)) return rc;
    const int nt = tiles16(L.cin);
    FEQ_LAUNCH("k_bdm_bwd_x", k, dim3(static_cast<unsigned>(ceil_div(ceil_div(E, 16), 8) * 8), nt), dim3(kThreads), lds, s,
               L, P, B, E, perm, dist, gy, L.cout, L.dout, L.cin, L.din, L.wdim, table, frag, x, gx, gpart,
               static_cast<unsigned>(ceil_div(E, 16)));
    if (gd)
        FEQ_LAUNCH("k_bdm_dr", k_bdm_dr, dim3(static_cast<unsigned>(ceil_div(E, 256))), dim3(256), 0, s, gpart, nt, E,
                   gdist);
    *dr_done = gd;
    const size_t tlds = sizeof(float) * kSS * (L.din + L.dout);
    if (int rc = bdm_lds(reinterpret_cast<const void*>(&k_bdm_table), tlds)) return rc;
    const int splits = table_splits(L, B, E, U.n);
    float* tpart = splits > 1 ? gpart + align_up(static_cast<size_t>(E) * nt, 64) : gtable;
    FEQ_LAUNCH("k_bdm_table", k_bdm_table,
               dim3(B.num_bins + 1, nt * tiles16(L.cout), static_cast<unsigned>(ceil_div(U.n, 4 * kMaxU) * splits)),
               dim3(kThreads), tlds, s, L, U, B, E, perm, offsets, dist, gy, x, splits, tpart);
    const int64_t nt_all = static_cast<int64_t>(table_floats(L, B));
    if (splits > 1)
        FEQ_LAUNCH("k_bdm_sum", k_bdm_sum, dim3(static_cast<unsigned>(ceil_div(nt_all, kThreads))), dim3(kThreads), 0, s,
                   tpart, splits, nt_all, gtable);
    return FEQ_OK;
}

}  // namespace feq
