// The block-diagonal op's terms for one edge: shared by the per-edge kernels
// (blockdiag.hip) and, for edges with infinities or NaN, by the bin-grouped ones
// (blockdiag_mm.hip).  tlo, thi: the table rows of the edge's bin, each
// (Cout, Cin, Wdim); t: the weight of thi; sw: the solid-harmonic base s.
#pragma once

#include "feq_internal.h"

namespace feq {
namespace {

struct SlotRef {
    int blk;  // m-block index, -1 when the slot has no partner block
    int o;    // index inside the block
    int c;    // 0 = +m (re) component, 1 = -m (im)
};

__device__ __forceinline__ SlotRef find_out_slot(const feq_layout& L, int slot) {
    for (int k = 0; k < L.nblocks; ++k) {
        const int m = L.blk[k][0], no = L.blk[k][2], off = L.blk[k][4];
        const int w = m == 0 ? 1 : 2;
        if (slot >= off && slot < off + w * no) {
            const int rel = slot - off;
            return {k, rel / w, rel % w};
        }
    }
    return {-1, 0, 0};
}

__device__ __forceinline__ SlotRef find_in_slot(const feq_layout& L, int slot) {
    for (int k = 0; k < L.nblocks; ++k) {
        const int m = L.blk[k][0], ni = L.blk[k][1], off = L.blk[k][3];
        const int w = m == 0 ? 1 : 2;
        if (slot >= off && slot < off + w * ni) {
            const int rel = slot - off;
            return {k, rel / w, rel % w};
        }
    }
    return {-1, 0, 0};
}

template <class T>
__device__ __forceinline__ T lerp_t(T lo, T hi, T t) {
    return lo + t * (hi - lo);
}

// Weight w's place in the layout: input slot (the +m slot of a pair), output
// slot, degree sum and the component (0: a, 1: b of the 2x2 block; m = 0: -1).
struct WeightRef {
    int is, os, lsum, comp;
};

__device__ __forceinline__ WeightRef weight_ref(const feq_layout& L, int w) {
    int k = L.nblocks - 1;
    while (k > 0 && w < L.blk[k][5]) --k;
    const int m = L.blk[k][0], ni = L.blk[k][1];
    const int in_off = L.blk[k][3], out_off = L.blk[k][4], w_off = L.blk[k][5];
    const int rel = w - w_off;
    WeightRef r;
    if (m == 0) {
        r.is = in_off + rel % ni;
        r.os = out_off + rel / ni;
        r.comp = -1;
    } else {
        const int pair = rel >> 1;
        r.is = in_off + 2 * (pair % ni);
        r.os = out_off + 2 * (pair / ni);
        r.comp = rel & 1;
    }
    r.lsum = L.lslot_in[r.is] + L.lslot_out[r.os];
    return r;
}

// d y / d T for one weight, before the solid-harmonic factor (block_diagonal.cu:514-517)
template <class T>
__device__ __forceinline__ T weight_grad(const WeightRef& r, const T* xr, const T* gr) {
    if (r.comp < 0) return xr[r.is] * gr[r.os];
    const T fr = xr[r.is], fi = xr[r.is + 1], g_r = gr[r.os], g_i = gr[r.os + 1];
    return r.comp == 0 ? fr * g_r + fi * g_i : fi * g_r - fr * g_i;
}

// y[co, slot] from the edge's features xr (Cin, Din).
template <class T>
__device__ __forceinline__ T out_entry(const feq_layout& L, const T* xr, int co, int slot, const T* tlo, const T* thi,
                                       T t, T sw) {
    const int cin = L.cin, din = L.din, wd = L.wdim;
    const SlotRef s = find_out_slot(L, slot);
    T acc = T(0);
    if (s.blk >= 0) {
        const int m = L.blk[s.blk][0], ni = L.blk[s.blk][1];
        const int in_off = L.blk[s.blk][3], w_off = L.blk[s.blk][5];
        const int lo_l = L.lslot_out[slot];
        for (int i = 0; i < ni; ++i) {
            const int islot = in_off + (m == 0 ? i : 2 * i);
            const T sc = ipow_t<T>(sw, lo_l + L.lslot_in[islot]);
            const int64_t wb = static_cast<int64_t>(co) * cin * wd;
            if (m == 0) {
                const int w = w_off + s.o * ni + i;
                for (int ci = 0; ci < cin; ++ci) {
                    const int64_t a = wb + static_cast<int64_t>(ci) * wd + w;
                    acc += lerp_t<T>(tlo[a], thi[a], t) * sc * xr[ci * din + islot];
                }
            } else {
                const int w = w_off + 2 * (s.o * ni + i);
                for (int ci = 0; ci < cin; ++ci) {
                    const int64_t a = wb + static_cast<int64_t>(ci) * wd + w;
                    const T wa = lerp_t<T>(tlo[a], thi[a], t) * sc;
                    const T wb2 = lerp_t<T>(tlo[a + 1], thi[a + 1], t) * sc;
                    const T fr = xr[ci * din + islot], fi = xr[ci * din + islot + 1];
                    acc += s.c == 0 ? (wa * fr + wb2 * fi) : (wa * fi - wb2 * fr);
                }
            }
        }
    }
    return acc;
}

// dL/dx[ci, slot] from the edge's output gradient gr (Cout, Dout).
template <class T>
__device__ __forceinline__ T in_entry(const feq_layout& L, const T* gr, int ci, int slot, const T* tlo, const T* thi,
                                      T t, T sw) {
    const int cin = L.cin, cout = L.cout, dout = L.dout, wd = L.wdim;
    const SlotRef s = find_in_slot(L, slot);
    T acc = T(0);
    if (s.blk >= 0) {
        const int m = L.blk[s.blk][0], ni = L.blk[s.blk][1], no = L.blk[s.blk][2];
        const int out_off = L.blk[s.blk][4], w_off = L.blk[s.blk][5];
        const int li = L.lslot_in[slot];
        for (int o = 0; o < no; ++o) {
            const int oslot = out_off + (m == 0 ? o : 2 * o);
            const T sc = ipow_t<T>(sw, li + L.lslot_out[oslot]);
            if (m == 0) {
                const int w = w_off + o * ni + s.o;
                for (int co = 0; co < cout; ++co) {
                    const int64_t a = (static_cast<int64_t>(co) * cin + ci) * wd + w;
                    acc += lerp_t<T>(tlo[a], thi[a], t) * sc * gr[co * dout + oslot];
                }
            } else {
                const int w = w_off + 2 * (o * ni + s.o);
                for (int co = 0; co < cout; ++co) {
                    const int64_t a = (static_cast<int64_t>(co) * cin + ci) * wd + w;
                    const T wa = lerp_t<T>(tlo[a], thi[a], t) * sc;
                    const T wb2 = lerp_t<T>(tlo[a + 1], thi[a + 1], t) * sc;
                    const T g_r = gr[co * dout + oslot], g_i = gr[co * dout + oslot + 1];
                    acc += s.c == 0 ? (wa * g_r - wb2 * g_i) : (wb2 * g_r + wa * g_i);
                }
            }
        }
    }
    return acc;
}

// Adds table weight w's share of the distance gradient for one channel pair:
// acc_t before the factor dt/dr, acc_s with deriv = sigma / (r (r + sigma)).
template <class T>
__device__ __forceinline__ void dist_terms(const feq_layout& L, int w, const T* xrow, const T* grow, T wl, T wh, T t,
                                           T sw, T deriv, T& acc_t, T& acc_s) {
    const WeightRef ref = weight_ref(L, w);
    const T u = weight_grad<T>(ref, xrow, grow);
    const T sc = ipow_t<T>(sw, ref.lsum);
    acc_t += (wh - wl) * sc * u;
    if (ref.lsum > 0) acc_s += lerp_t<T>(wl, wh, t) * u * sc * static_cast<T>(ref.lsum) * deriv;
}

}  // namespace
}  // namespace feq
