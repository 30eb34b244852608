// Epilogues of the projections' column pairs, shared by the GEMM kernels and
// the layer tail: requantization, RoPE and the cache scatter (QKV), ReGLU.
#pragma once

#include "czip_device.h"
#include "czip_kernels.h"

namespace czip {

template <bool FAST>
__device__ __forceinline__ int rq(int v, const GemmArgs& a) {
    return rq<FAST>(v, a.rq_scale, a.mult, a.shift);
}


// Chunk, position and RoPE cos/sin (columns c4 .. c4+3 of each 16-wide half)
// of one output row of the QKV projection.
struct QkvRow {
    int p, b;
    unsigned cs[2][2], sn[2][2];
};

__device__ __forceinline__ void qkv_row(const GemmArgs& a, int row, int c4, QkvRow& q) {
    row = min(row, a.M - 1);
    int b = (int)((float)row * (1.0f / (float)a.T));  // row < 2^24: within one of row / T
    if (b * a.T > row) b--;
    else if ((b + 1) * a.T <= row) b++;
    q.p = a.pos >= 0 ? a.pos : row - b * a.T;
    q.b = a.pos >= 0 ? row : b;
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const uint2 c = *(const uint2*)(a.rcos + q.p * 32 + j * 16 + c4);
        const uint2 sv = *(const uint2*)(a.rsin + q.p * 32 + j * 16 + c4);
        q.cs[j][0] = c.x; q.cs[j][1] = c.y;
        q.sn[j][0] = sv.x; q.sn[j][1] = sv.y;
    }
}

// ReGLU / QKV epilogue of one column pair: x holds columns col_base + 16 j +
// c4 .. +3 of `row`, y the columns 32 further (col_base 64-aligned: one head /
// one gate-up group; j is 0 or 1).
template <int EPI, bool FAST>
__device__ __forceinline__ void epi_pair(const GemmArgs& a, v4i x, v4i y, int row, int col_base, int j, int c4,
                                         const QkvRow& q) {
    const int i0 = j * 16 + c4;
    if (EPI == EPI_REGLU) {
        // W rows were permuted so that a 64-row group holds 32 gate rows then the
        // matching 32 up rows: output feature f = col_base/2 + j*16 + c4 + r.
        int o[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int g = rq<FAST>(x[r], a);
            const int u = rq<FAST>(y[r], a);
            const int gr = g > 0 ? g : 0;
            o[r] = clamp127(rne_shr(gr * u, 7));  // reglu.rs:20-46 (|gr * u| <= 127^2)
        }
        *(unsigned*)(a.out8 + (size_t)row * a.ldo + (col_base >> 1) + i0) = pack4i(o[0], o[1], o[2], o[3]);
        return;
    }
    // EPI_QKV: rotary pairs (i0 + r, i0 + r + 32)
    const int p = q.p, b = q.b;
    const int kcol = col_base - a.d;
    int g = 0, isv = 0;
    if (kcol >= 0) {
        if (a.kv_mode == 1) { isv = kcol >= 64 * a.G; g = (isv ? kcol - 64 * a.G : kcol) >> 6; }
        else isv = kcol >= 64;
    }
    // (selects, not an index: j is not a constant everywhere)
    const unsigned cs[2] = {j ? q.cs[1][0] : q.cs[0][0], j ? q.cs[1][1] : q.cs[0][1]};
    const unsigned sns[2] = {j ? q.sn[1][0] : q.sn[0][0], j ? q.sn[1][1] : q.sn[0][1]};
    int xq[4], yq[4], xv[4], yv[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        xv[r] = rq<FAST>(x[r], a);
        yv[r] = rq<FAST>(y[r], a);
        const int c = (int16_t)(r & 1 ? cs[r >> 1] >> 16 : cs[r >> 1] & 0xFFFFu);
        const int sn = (int16_t)(r & 1 ? sns[r >> 1] >> 16 : sns[r >> 1] & 0xFFFFu);
        const int xr = (int)((unsigned)(xv[r] * c) - (unsigned)(yv[r] * sn));
        const int yr = (int)((unsigned)(xv[r] * sn) + (unsigned)(yv[r] * c));
        if (kcol < 0) {
            // Q: attention.rs:53-83 (>>15 then NET_SHIFT=1, two roundings)
            xq[r] = clamp127(rne_shr(rne_shr(xr, 15), 1));
            yq[r] = clamp127(rne_shr(rne_shr(yr, 15), 1));
        } else {
            // K: attention.rs:29-50 (|xr|, |yr| <= 2 * 127 * 32768)
            xq[r] = clamp127(rne_shr(xr, 15));
            yq[r] = clamp127(rne_shr(yr, 15));
        }
    }
    if (kcol < 0) {
        int8_t* qo = a.out8 + (size_t)row * a.ldo + col_base;
        *(unsigned*)(qo + i0) = pack4i(xq[0], xq[1], xq[2], xq[3]);
        *(unsigned*)(qo + i0 + 32) = pack4i(yq[0], yq[1], yq[2], yq[3]);
    } else if (!isv) {
        int8_t* k = a.kc + (((size_t)b * a.KH + g) * a.T + p) * 64;
        *(unsigned*)(k + i0) = pack4i(xq[0], xq[1], xq[2], xq[3]);
        *(unsigned*)(k + i0 + 32) = pack4i(yq[0], yq[1], yq[2], yq[3]);
    } else {
        // V^T in blocks of 2^vl keys (vt_off)
        const int vl = a.vl;
        int8_t* v = a.vc + ((size_t)b * a.KH + g) * 64 * a.TP + vt_off(p, 0, vl);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            v[(i0 + r) << vl] = (int8_t)xv[r];
            v[(i0 + r + 32) << vl] = (int8_t)yv[r];
        }
    }
}

}  // namespace czip
