// Row-wise kernels: chunk preparation, embedding + RMSNorm, residual + RMSNorm,
// logits -> cumulative frequencies, and the arithmetic encoder.
#include "czip_device.h"
#include "czip_kernels.h"

namespace czip {

// ---------------------------------------------------------------------------
// Chunk preparation: inputs [BOS, t0..t_{n-2}] and targets per chunk
// (main.rs:209-226).  Padding rows get token 0 and are never read back.
// ---------------------------------------------------------------------------
__global__ void k_prep_chunks(const uint32_t* __restrict__ toks, long long n, long long chunk0, int nb, int T,
                              uint32_t* __restrict__ inp, uint32_t* __restrict__ tgt, int32_t* __restrict__ lens) {
    long long row = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (row >= (long long)nb * T) return;
    int b = (int)(row / T), p = (int)(row % T);
    long long start = (chunk0 + b) * (long long)T;
    long long len = n - start;
    if (len > T) len = T;
    if (len < 0) len = 0;
    if (p == 0) lens[b] = (int32_t)len;
    if (p < len) {
        inp[row] = p == 0 ? BOS_TOKEN : toks[start + p - 1];
        tgt[row] = toks[start + p];
    } else {
        inp[row] = 0u;
        tgt[row] = 0u;
    }
}

void launch_prep_chunks(const uint32_t* toks, int64_t n, int64_t chunk0, int nb, int T, uint32_t* inp,
                        uint32_t* tgt, int32_t* lens, hipStream_t s) {
    long long rows = (long long)nb * T;
    hipLaunchKernelGGL(k_prep_chunks, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, s, toks, (long long)n,
                       (long long)chunk0, nb, T, inp, tgt, lens);
}

// ---------------------------------------------------------------------------
// Row kernels: one wavefront per token row, d <= 1024.  Lane l owns the
// 4-element groups g = l, l + 64, ... (elements 4g .. 4g+3), so loads and
// stores are 4-byte (int8) or 16-byte (int32) vectors.
// ---------------------------------------------------------------------------
constexpr int RG = 4;  // groups per lane: d <= 64 * 4 * RG

struct RowI8 {
    int v[RG][4];
};

__device__ __forceinline__ void unpack4(unsigned w, int* o) {
    o[0] = (int)(int8_t)(w & 0xFF);
    o[1] = (int)(int8_t)((w >> 8) & 0xFF);
    o[2] = (int)(int8_t)((w >> 16) & 0xFF);
    o[3] = (int)(int8_t)(w >> 24);
}
__device__ __forceinline__ unsigned pack4(const int* v) {
    return ((unsigned)(uint8_t)(int8_t)v[0]) | ((unsigned)(uint8_t)(int8_t)v[1] << 8) |
           ((unsigned)(uint8_t)(int8_t)v[2] << 16) | ((unsigned)(uint8_t)(int8_t)v[3] << 24);
}

// rmsnorm.rs:40-75 on the wave-distributed row: y = clamp(sra_rne((x*w)*inv, 15))
__device__ __forceinline__ void rms_row(const RowI8& x, const int8_t* __restrict__ w, int d, int lane, RowI8& y) {
    const int ng = d >> 2;
    unsigned ss = 0;
#pragma unroll
    for (int j = 0; j < RG; j++)
        if (lane + 64 * j < ng)
#pragma unroll
            for (int k = 0; k < 4; k++) ss += (unsigned)(x.v[j][k] * x.v[j][k]);
    ss = wave_sum_u(ss);
    const int mean_sq = (int)(ss / (unsigned)d) + 1;  // eps_scaled = 1 (rmsnorm.rs:80-83); <= 127^2 + 1
    const int inv = inv_rms_q15_fast(mean_sq);
#pragma unroll
    for (int j = 0; j < RG; j++) {
        const int g = lane + 64 * j;
        if (g < ng) {
            int wv[4];
            unpack4(*(const unsigned*)(w + 4 * g), wv);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                int tmp = (int)((unsigned)(x.v[j][k] * wv[k]) * (unsigned)inv);
                y.v[j][k] = clamp127(sra_rne32(tmp, 15));
            }
        }
    }
}

// x = E[tok] (model.rs:372-374); xn = rmsnorm(clamp(x), w) (model.rs:384-385).
// Sixteen lanes per row, four rows per wavefront: lane s of a row owns the
// 4-element groups g = s, s + 16, ... (d <= 1024: at most 16 groups), so the
// four rows' gather -> reduce -> normalize chains overlap.
__global__ __launch_bounds__(256) void k_embed_norm(const uint32_t* __restrict__ inp, const int8_t* __restrict__ embed,
                                                    const int8_t* __restrict__ w, int M, int d,
                                                    int16_t* __restrict__ x, int8_t* __restrict__ xn) {
    constexpr int G16 = 16;  // groups per lane: d <= 16 * 4 * 16
    const int row = blockIdx.x * 16 + (threadIdx.x >> 4);
    const int sl = threadIdx.x & 15;
    const bool live = row < M;
    const int ng = d >> 2;
    const int8_t* e = embed + (size_t)(live ? inp[row] : 0u) * d;
    unsigned raw[G16];
#pragma unroll
    for (int j = 0; j < G16; j++) {
        const int g = sl + 16 * j;
        raw[j] = g < ng ? *(const unsigned*)(e + 4 * g) : 0u;
    }
    unsigned ss = 0;
#pragma unroll
    for (int j = 0; j < G16; j++) {
        int v[4];
        unpack4(raw[j], v);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int c = clamp127(v[k]);
            ss += (unsigned)(c * c);
        }
    }
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) ss += (unsigned)__shfl_xor((int)ss, o, 64);
    const int inv = inv_rms_q15_fast((int)(ss / (unsigned)d) + 1);  // eps_scaled = 1 (rmsnorm.rs:80-83)
    if (!live) return;
#pragma unroll
    for (int j = 0; j < G16; j++) {
        const int g = sl + 16 * j;
        if (g < ng) {
            int v[4], wv[4], y[4];
            unpack4(raw[j], v);
            unpack4(*(const unsigned*)(w + 4 * g), wv);
            if (x) {
                const unsigned lo = ((unsigned)v[0] & 0xFFFFu) | ((unsigned)v[1] << 16);
                const unsigned hi = ((unsigned)v[2] & 0xFFFFu) | ((unsigned)v[3] << 16);
                *(uint2*)(x + (size_t)row * d + 4 * g) = make_uint2(lo, hi);
            }
#pragma unroll
            for (int k = 0; k < 4; k++) y[k] = clamp127(rne_shr(clamp127(v[k]) * wv[k] * inv, 15));
            *(unsigned*)(xn + (size_t)row * d + 4 * g) = pack4(y);
        }
    }
}

void launch_embed_norm(const uint32_t* inp, const int8_t* embed, const int8_t* w, int M, int d, int16_t* x,
                       int8_t* xn, hipStream_t s) {
    hipLaunchKernelGGL(k_embed_norm, dim3((unsigned)((M + 15) / 16)), dim3(256), 0, s, inp, embed, w, M, d, x, xn);
}

// ---------------------------------------------------------------------------
// Epilogue of the split-K row GEMM, one wavefront per row: sum the K slices'
// int32 partials (wrapping, like the accumulator), requantize, add the
// residual (the int16 stream or the token's embedding row), both RMSNorms
// (model.rs:424-468): the same arithmetic as the fused row GEMM's epilogue.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_rn_splitk_epi(RowGemmArgs a, const int32_t* __restrict__ part, int splits) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= a.M) return;
    const int d = a.d, ng = d >> 2;
    RowI8 yi, yn, xi;
#pragma unroll
    for (int j = 0; j < RG; j++) {
        const int g = lane + 64 * j;
        if (g < ng) {
            unsigned acc[4] = {0u, 0u, 0u, 0u};
            for (int sp = 0; sp < splits; sp++) {
                const int4 v = *(const int4*)(part + ((size_t)sp * a.M + row) * d + 4 * g);
                acc[0] += (unsigned)v.x; acc[1] += (unsigned)v.y; acc[2] += (unsigned)v.z; acc[3] += (unsigned)v.w;
            }
#pragma unroll
            for (int k = 0; k < 4; k++)
                yi.v[j][k] = a.rq_fast ? clamp127(rint_fma_i32((double)(int)acc[k], a.rq_scale))
                                       : requant((int)acc[k], a.mult, a.shift);
        }
    }
    rms_row(yi, a.w1, d, lane, yn);
    const int8_t* erow = a.x_in ? nullptr : a.embed + (size_t)a.tok[row] * d;
#pragma unroll
    for (int j = 0; j < RG; j++) {
        const int g = lane + 64 * j;
        if (g < ng) {
            int xo[4];
            if (a.x_in) {
                const uint2 xv = *(const uint2*)(a.x_in + (size_t)row * d + 4 * g);
                xo[0] = (int16_t)(xv.x & 0xFFFFu); xo[1] = (int16_t)(xv.x >> 16);
                xo[2] = (int16_t)(xv.y & 0xFFFFu); xo[3] = (int16_t)(xv.y >> 16);
            } else {
                unpack4(*(const unsigned*)(erow + 4 * g), xo);
            }
            int nv[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                nv[k] = xo[k] + yn.v[j][k];
                xi.v[j][k] = clamp127(nv[k]);
            }
            if (a.x_out)
                *(uint2*)(a.x_out + (size_t)row * d + 4 * g) = make_uint2(((unsigned)nv[0] & 0xFFFFu) | ((unsigned)nv[1] << 16),
                                                                          ((unsigned)nv[2] & 0xFFFFu) | ((unsigned)nv[3] << 16));
        }
    }
    rms_row(xi, a.w2, d, lane, yn);
#pragma unroll
    for (int j = 0; j < RG; j++) {
        const int g = lane + 64 * j;
        if (g < ng) *(unsigned*)(a.xn + (size_t)row * d + 4 * g) = pack4(yn.v[j]);
    }
}

void launch_rn_splitk_epi(const RowGemmArgs& a, const int32_t* part, int splits, hipStream_t s) {
    hipLaunchKernelGGL(k_rn_splitk_epi, dim3((unsigned)((a.M + 3) / 4)), dim3(256), 0, s, a, part, splits);
}

// ---------------------------------------------------------------------------
// The same from the requantized projection (the few-row GEMM's output), one
// wavefront per row: every load is requested before the first reduction.
// ---------------------------------------------------------------------------
template <int NG>  // 4-element groups per lane: d <= 256 NG
__global__ __launch_bounds__(64) void k_rn_rows(RowGemmArgs a) {
    const int row = blockIdx.x, lane = threadIdx.x;
    const int d = a.d, ng = d >> 2;
    const int8_t* erow = a.x_in ? nullptr : a.embed + (size_t)a.tok[row] * d;
    unsigned yw[NG], w1w[NG], w2w[NG];
    uint2 xw[NG];
#pragma unroll
    for (int j = 0; j < NG; j++) {
        const int g = min(lane + 64 * j, ng - 1);
        yw[j] = *(const unsigned*)(a.y8 + (size_t)row * d + 4 * g);
        w1w[j] = *(const unsigned*)(a.w1 + 4 * g);
        w2w[j] = *(const unsigned*)(a.w2 + 4 * g);
        xw[j] = a.x_in ? *(const uint2*)(a.x_in + (size_t)row * d + 4 * g) : make_uint2(*(const unsigned*)(erow + 4 * g), 0u);
    }
    auto inv_rms = [&](unsigned ss) {
        ss = wave_sum_u(ss);
        return (double)inv_rms_q15_fast((int)(ss / (unsigned)d) + 1) * (1.0 / 32768.0);  // eps_scaled = 1 (rmsnorm.rs:80-83)
    };
    unsigned ss = 0;
#pragma unroll
    for (int j = 0; j < NG; j++) {
        int y[4];
        unpack4(yw[j], y);
#pragma unroll
        for (int k = 0; k < 4; k++) ss += lane + 64 * j < ng ? (unsigned)__mul24(y[k], y[k]) : 0u;
    }
    const double inv1 = inv_rms(ss);
    int xc[NG][4];
    ss = 0;
#pragma unroll
    for (int j = 0; j < NG; j++) {
        const int g = lane + 64 * j;
        int y[4], w1[4], xo[4];
        unpack4(yw[j], y);
        unpack4(w1w[j], w1);
        if (a.x_in) {
            xo[0] = (int16_t)(xw[j].x & 0xFFFFu); xo[1] = (int16_t)(xw[j].x >> 16);
            xo[2] = (int16_t)(xw[j].y & 0xFFFFu); xo[3] = (int16_t)(xw[j].y >> 16);
        } else {
            unpack4(xw[j].x, xo);
        }
        int nv[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            nv[k] = xo[k] + rms_el(y[k], w1[k], inv1);
            xc[j][k] = clamp127(nv[k]);
            ss += g < ng ? (unsigned)__mul24(xc[j][k], xc[j][k]) : 0u;
        }
        if (a.x_out && g < ng)
            *(uint2*)(a.x_out + (size_t)row * d + 4 * g) = make_uint2(((unsigned)nv[0] & 0xFFFFu) | ((unsigned)nv[1] << 16),
                                                                    ((unsigned)nv[2] & 0xFFFFu) | ((unsigned)nv[3] << 16));
    }
    const double inv2 = inv_rms(ss);
#pragma unroll
    for (int j = 0; j < NG; j++) {
        const int g = lane + 64 * j;
        int w2[4];
        unpack4(w2w[j], w2);
        if (g < ng)
            *(unsigned*)(a.xn + (size_t)row * d + 4 * g) =
                pack4i(rms_el(xc[j][0], w2[0], inv2), rms_el(xc[j][1], w2[1], inv2), rms_el(xc[j][2], w2[2], inv2),
                       rms_el(xc[j][3], w2[3], inv2));
    }
}

void launch_rn_rows(const RowGemmArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)a.M);
    if (a.d <= 512) hipLaunchKernelGGL(k_rn_rows<2>, grid, dim3(64), 0, s, a);
    else hipLaunchKernelGGL(k_rn_rows<4>, grid, dim3(64), 0, s, a);
}

// ---------------------------------------------------------------------------
// Layer 0's QKV from the per-token table.  One thread per (row, item): items
// 0 .. 8H-1 are query rotary groups (head i / 8, dims 4 (i % 8) .. +3 paired
// with +32), the next 8 NG key rotary groups, the last 16 NG value quads.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_qkv_table(QkvTabArgs a) {
    const int per_row = 8 * a.H + 24 * a.NG;
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= a.M * per_row) return;
    // idx / per_row from the host's 1 / per_row: the product is within 2^-21
    // of the quotient, whose fraction is 0 or >= 1 / per_row >= 2^-12, so a
    // 2^-13 bias truncates to it exactly (per_row < 2^12, idx < 2^31)
    const int row = (int)__builtin_fma((double)idx, a.inv_per_row, 0x1p-13), it = idx - row * per_row;
    const int b = a.pos >= 0 ? row : row / a.T, p = a.pos >= 0 ? a.pos : row - b * a.T;
    const int8_t* t = a.tab + (size_t)a.tok[row] * a.qkv_n;
    if (it >= 8 * a.H + 8 * a.NG) {  // V: dims 4 q .. 4 q + 3 of head g, in blocks of 2^vl keys (vt_off)
        const int v = it - 8 * a.H - 8 * a.NG, g = v >> 4, q = v & 15;
        const unsigned w = *(const unsigned*)(t + a.d + 64 * a.NG + 64 * g + 4 * q);
        const int vl = a.vl;
        int8_t* dst = a.vc + ((size_t)b * a.KH + g) * 64 * a.TP + vt_off(p, 4 * q, vl);
#pragma unroll
        for (int r = 0; r < 4; r++) dst[r << vl] = (int8_t)(w >> (8 * r));
        return;
    }
    const bool isq = it < 8 * a.H;
    // Q: >> 15 then NET_SHIFT = 1 (attention.rs:53-83); K: >> 15 (attention.rs:29-50)
    const double rm = isq ? 0.5 : 1.0, rb = isq ? ROPE_Q_BIAS : 0.0;
    const int hd = isq ? it >> 3 : (it - 8 * a.H) >> 3, i0 = 4 * (it & 7);
    const int col = isq ? 64 * hd : a.d + 64 * hd;
    const unsigned xw = *(const unsigned*)(t + col + i0), yw = *(const unsigned*)(t + col + i0 + 32);
    const uint2 cw = *(const uint2*)(a.rcos + p * 32 + i0), sw = *(const uint2*)(a.rsin + p * 32 + i0);
    int xq[4], yq[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int xv = (int8_t)(xw >> (8 * r)), yv = (int8_t)(yw >> (8 * r));
        const unsigned cc = r < 2 ? cw.x : cw.y, ss = r < 2 ? sw.x : sw.y;
        const int c = (int16_t)(r & 1 ? cc >> 16 : cc & 0xFFFFu), sn = (int16_t)(r & 1 ? ss >> 16 : ss & 0xFFFFu);
        const int xr = (int)((unsigned)(xv * c) - (unsigned)(yv * sn));
        const int yr = (int)((unsigned)(xv * sn) + (unsigned)(yv * c));
        xq[r] = clamp127(rope_round(xr, rm, rb));
        yq[r] = clamp127(rope_round(yr, rm, rb));
    }
    int8_t* dst = isq ? a.q8 + (size_t)row * a.d + 64 * hd : a.kc + (((size_t)b * a.KH + hd) * a.T + p) * 64;
    *(unsigned*)(dst + i0) = pack4(xq);
    *(unsigned*)(dst + i0 + 32) = pack4(yq);
}

// Prefill: a workgroup takes 16 consecutive positions p0 .. p0 + 15 of one
// chunk (p0 % 16 == 0), computes their Q and K rotary groups and gathers
// their V rows into LDS, then writes every output as contiguous 16-byte
// pieces: the 16 query rows (16 d bytes), each key head's 16 rows (1 KB) and
// each value head's 64 x 16-key block of the transposed cache (1 KB).  Keys
// past the chunk's T inside the last block get don't-care bytes (never
// weighted by the attention).
constexpr int QT_MAXD = 1024, QT_MAXG = 4;
__global__ __launch_bounds__(256) void k_qkv_table_blk(QkvTabArgs a) {
    __shared__ __attribute__((aligned(16))) int8_t qs[16 * QT_MAXD];
    __shared__ __attribute__((aligned(16))) int8_t ks[QT_MAXG * 16 * 64];
    __shared__ __attribute__((aligned(16))) int8_t vs[QT_MAXG * 16 * 64];
    __shared__ uint32_t tk[16];
    const int tid = threadIdx.x;
    const int nkb = (a.T + 15) / 16;
    const int b = blockIdx.x / nkb, p0 = (blockIdx.x - b * nkb) * 16;
    const int nrows = min(16, a.T - p0);
    const int row0 = b * a.T + p0;
    if (tid < 16) tk[tid] = tid < nrows ? a.tok[row0 + tid] : 0u;
    __syncthreads();
    // Q and K rotary groups: item = (row k, group i): group < 8H query, else key
    const int per_row = 8 * a.H + 8 * a.NG;
    // item idx = (row k, group it), advanced by 256 per pass: one division per thread
    const int kstep = 256 / per_row, istep = 256 - kstep * per_row;
    int k = tid / per_row, it = tid - k * per_row;
    for (int idx = tid; idx < 16 * per_row; idx += 256, k += kstep, it += istep) {
        if (it >= per_row) {
            it -= per_row;
            k++;
        }
        const int8_t* t = a.tab + (size_t)tk[k] * a.qkv_n;
        const bool isq = it < 8 * a.H;
        // Q: >> 15 then NET_SHIFT = 1 (attention.rs:53-83); K: >> 15 (attention.rs:29-50)
        const double rm = isq ? 0.5 : 1.0, rb = isq ? ROPE_Q_BIAS : 0.0;
        const int hd = isq ? it >> 3 : (it - 8 * a.H) >> 3, i0 = 4 * (it & 7);
        const int col = isq ? 64 * hd : a.d + 64 * hd;
        const unsigned xw = *(const unsigned*)(t + col + i0), yw = *(const unsigned*)(t + col + i0 + 32);
        const int p = min(p0 + k, a.T - 1);
        const uint2 cw = *(const uint2*)(a.rcos + p * 32 + i0), sw = *(const uint2*)(a.rsin + p * 32 + i0);
        int xq[4], yq[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int xv = (int8_t)(xw >> (8 * r)), yv = (int8_t)(yw >> (8 * r));
            const unsigned cc = r < 2 ? cw.x : cw.y, ss = r < 2 ? sw.x : sw.y;
            const int c = (int16_t)(r & 1 ? cc >> 16 : cc & 0xFFFFu), sn = (int16_t)(r & 1 ? ss >> 16 : ss & 0xFFFFu);
            const int xr = (int)((unsigned)(xv * c) - (unsigned)(yv * sn));
            const int yr = (int)((unsigned)(xv * sn) + (unsigned)(yv * c));
            xq[r] = clamp127(rope_round(xr, rm, rb));
            yq[r] = clamp127(rope_round(yr, rm, rb));
        }
        int8_t* dst = isq ? qs + k * a.d + 64 * hd : ks + (hd * 16 + k) * 64;
        *(unsigned*)(dst + i0) = pack4(xq);
        *(unsigned*)(dst + i0 + 32) = pack4(yq);
    }
    // V rows (16 bytes per item)
    for (int idx = tid; idx < 16 * a.NG * 4; idx += 256) {
        const int k = idx / (4 * a.NG), r = idx - k * 4 * a.NG, g = r >> 2, c = r & 3;
        *(uint4*)(vs + (g * 16 + k) * 64 + 16 * c) =
            *(const uint4*)(a.tab + (size_t)tk[k] * a.qkv_n + a.d + 64 * a.NG + 64 * g + 16 * c);
    }
    __syncthreads();
    // query rows: nrows * d contiguous bytes
    const int qn = nrows * a.d / 16;
    for (int i = tid; i < qn; i += 256) *(uint4*)(a.q8 + (size_t)row0 * a.d + 16 * i) = *(const uint4*)(qs + 16 * i);
    // key rows of each head: nrows * 64 contiguous bytes
    for (int i = tid; i < a.NG * nrows * 4; i += 256) {
        const int g = i / (nrows * 4), c = i - g * nrows * 4;
        *(uint4*)(a.kc + (((size_t)b * a.KH + g) * a.T + p0) * 64 + 16 * c) = *(const uint4*)(ks + g * 1024 + 16 * c);
    }
    // value blocks: dim j of head g -> the 16 keys' bytes
    for (int i = tid; i < a.NG * 64; i += 256) {
        const int g = i >> 6, j = i & 63;
        unsigned w[4];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int8_t* v = vs + (g * 16 + 4 * q) * 64 + j;
            w[q] = (unsigned)(uint8_t)v[0] | ((unsigned)(uint8_t)v[64] << 8) | ((unsigned)(uint8_t)v[128] << 16) |
                   ((unsigned)(uint8_t)v[192] << 24);
        }
        *(uint4*)(a.vc + ((size_t)b * a.KH + g) * 64 * a.TP + (size_t)(p0 >> 4) * 1024 + 16 * j) =
            make_uint4(w[0], w[1], w[2], w[3]);
    }
}

void launch_qkv_table(const QkvTabArgs& a, hipStream_t s) {
    if (a.pos < 0 && a.d <= QT_MAXD && a.NG <= QT_MAXG) {
        const int nb = a.M / a.T, nkb = (a.T + 15) / 16;
        hipLaunchKernelGGL(k_qkv_table_blk, dim3((unsigned)(nb * nkb)), dim3(256), 0, s, a);
        return;
    }
    const int per_row = 8 * a.H + 24 * a.NG;
    const long long n = (long long)a.M * per_row;
    // n < 2^31 (the caller takes the table path only then) and per_row <= 512 (d <= 1024)
    QkvTabArgs g = a;
    g.inv_per_row = 1.0 / per_row;
    hipLaunchKernelGGL(k_qkv_table, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, g);
}

// x += rmsnorm(y8, w1) (model.rs:429-434 / 463-468);
// xn = rmsnorm(clamp(x), w2) (model.rs:438-439, next layer 384-385, final 473-474)
__global__ __launch_bounds__(256) void k_resid_norm(int16_t* __restrict__ x, const int8_t* __restrict__ y8,
                                                    const int8_t* __restrict__ w1, const int8_t* __restrict__ w2,
                                                    int M, int d, int8_t* __restrict__ xn) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= M) return;
    const int ng = d >> 2;
    RowI8 yi, yn, xi;
#pragma unroll
    for (int j = 0; j < RG; j++) {
        const int g = lane + 64 * j;
        if (g < ng) unpack4(*(const unsigned*)(y8 + (size_t)row * d + 4 * g), yi.v[j]);
    }
    rms_row(yi, w1, d, lane, yn);
#pragma unroll
    for (int j = 0; j < RG; j++) {
        const int g = lane + 64 * j;
        if (g < ng) {
            // |x| <= 127 * (2 * n_layers + 1) < 2^15: the i32 sums of the reference fit int16
            uint2* px = (uint2*)(x + (size_t)row * d + 4 * g);
            const uint2 xv = *px;
            const int nv[4] = {(int16_t)(xv.x & 0xFFFFu) + yn.v[j][0], (int16_t)(xv.x >> 16) + yn.v[j][1],
                               (int16_t)(xv.y & 0xFFFFu) + yn.v[j][2], (int16_t)(xv.y >> 16) + yn.v[j][3]};
            *px = make_uint2(((unsigned)nv[0] & 0xFFFFu) | ((unsigned)nv[1] << 16),
                             ((unsigned)nv[2] & 0xFFFFu) | ((unsigned)nv[3] << 16));
#pragma unroll
            for (int k = 0; k < 4; k++) xi.v[j][k] = clamp127(nv[k]);
        }
    }
    rms_row(xi, w2, d, lane, yn);
#pragma unroll
    for (int j = 0; j < RG; j++) {
        const int g = lane + 64 * j;
        if (g < ng) *(unsigned*)(xn + (size_t)row * d + 4 * g) = pack4(yn.v[j]);
    }
}

void launch_resid_norm(int16_t* x, const int8_t* y8, const int8_t* w1, const int8_t* w2, int M, int d, int8_t* xn,
                       hipStream_t s) {
    hipLaunchKernelGGL(k_resid_norm, dim3((unsigned)((M + 3) / 4)), dim3(256), 0, s, x, y8, w1, w2, M, d, xn);
}

// ---------------------------------------------------------------------------
// Logits -> cumulative frequencies (softmax_cdf.rs:85-139).
// WPR wavefronts per row, EPL consecutive logits per lane (V <= 64*WPR*EPL).
// The frequency f = 1 + floor(e * R / S) (R = total - V) is formed exactly as
// f = 1 + e*Q + floor(e*Rm / S) with Q = R / S, Rm = R % S: e*Q < 2^31
// because S >= 65535 (the max logit weighs 65535), and the small quotient is
// an f32 estimate corrected by one exact 64-bit remainder test.
// mode 0: write (cum_lo, cum_hi) of the row's target; mode 1: write the full
// inclusive table; mode 2: targets holds the row's decoder value (the
// ((code - low + 1) * total - 1) / range of arith_coder.rs:199-203) and the
// row gets (sym, cum_lo, cum_hi) with sym the first index whose inclusive
// cumulative frequency exceeds the value, clamped to V - 1
// (bisect_cumfreqs, arith_coder.rs:225-241).
// ---------------------------------------------------------------------------
template <int WPR, int EPL>
__global__ __launch_bounds__(64 * WPR) void k_cdf(const int32_t* __restrict__ logits, int V,
                                                  const uint32_t* __restrict__ targets,
                                                  const int32_t* __restrict__ lens, int T,
                                                  const uint16_t* __restrict__ glut, unsigned coef, unsigned total,
                                                  int mode, uint32_t* __restrict__ out, long long out_row0) {
    __shared__ uint16_t lut[256];
    __shared__ int red_i[WPR];
    __shared__ unsigned red_u[WPR];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = blockIdx.x;
    for (int i = tid; i < 256; i += 64 * WPR) lut[i] = glut[i];
    if (lens && (row % T) >= lens[row / T]) return;  // uniform per block
    __syncthreads();
    const int i0 = tid * EPL;
    const int32_t* L = logits + (size_t)row * V;
    int lv[EPL];
    if (i0 + EPL <= V) {
#pragma unroll
        for (int k = 0; k < EPL; k += 4) {
            int4 v = *(const int4*)(L + i0 + k);
            lv[k] = v.x; lv[k + 1] = v.y; lv[k + 2] = v.z; lv[k + 3] = v.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < EPL; k++) lv[k] = (i0 + k < V) ? L[i0 + k] : INT32_MIN;
    }
    auto bmax = [&](int v) {
        v = wave_max_i(v);
        if (WPR == 1) return v;
        if (lane == 0) red_i[wave] = v;
        __syncthreads();
        int r = red_i[0];
        for (int w = 1; w < WPR; w++) r = max(r, red_i[w]);
        __syncthreads();
        return r;
    };
    auto bmin = [&](int v) {
        v = wave_min_i(v);
        if (WPR == 1) return v;
        if (lane == 0) red_i[wave] = v;
        __syncthreads();
        int r = red_i[0];
        for (int w = 1; w < WPR; w++) r = min(r, red_i[w]);
        __syncthreads();
        return r;
    };
    auto bsum = [&](unsigned v) {
        v = wave_sum_u(v);
        if (WPR == 1) return v;
        if (lane == 0) red_u[wave] = v;
        __syncthreads();
        unsigned r = 0;
        for (int w = 0; w < WPR; w++) r += red_u[w];
        __syncthreads();
        return r;
    };
    int mx = INT32_MIN;
#pragma unroll
    for (int k = 0; k < EPL; k++) mx = max(mx, lv[k]);
    mx = bmax(mx);
    int am = 0x7FFFFFFF;
#pragma unroll
    for (int k = EPL - 1; k >= 0; k--)
        if (i0 + k < V && lv[k] == mx) am = i0 + k;
    am = bmin(am);
    unsigned e[EPL];
    unsigned ls = 0;
#pragma unroll
    for (int k = 0; k < EPL; k++) {
        e[k] = (i0 + k < V) ? exp_q16((int)((unsigned)lv[k] - (unsigned)mx), lut, coef) : 0u;
        ls += e[k];
    }
    const unsigned S = bsum(ls);  // <= 8192 * 65535 < 2^32
    const unsigned R = total - (unsigned)V;
    const unsigned Q = R / S, Rm = R - Q * S;
    const float rf = (float)Rm / (float)S;
    unsigned fl = 0;
#pragma unroll
    for (int k = 0; k < EPL; k++) {
        unsigned f = 0;
        if (i0 + k < V) {
            unsigned q = (unsigned)((float)e[k] * rf);
            const unsigned long long t = (unsigned long long)e[k] * Rm, u = (unsigned long long)q * S;
            if (t < u) q -= 1;
            else if (t - u >= S) q += 1;
            f = 1u + e[k] * Q + q;
        }
        e[k] = f;
        fl += f;
    }
    const unsigned rem = total - bsum(fl);
    if (mode == 0) {
        const int tok = (int)targets[row];
        unsigned lo = 0, ft = 0;
#pragma unroll
        for (int k = 0; k < EPL; k++) {
            lo += (i0 + k < tok) ? e[k] : 0u;
            ft += (i0 + k == tok) ? e[k] : 0u;
        }
        lo = bsum(lo);
        ft = bsum(ft);
        if (am < tok) lo += rem;
        if (am == tok) ft += rem;
        if (tid == 0) {
            out[(size_t)(out_row0 + row) * 2] = lo;
            out[(size_t)(out_row0 + row) * 2 + 1] = lo + ft;
        }
    } else {
        // exclusive scan of lane sums across the row
        unsigned incl = fl;
        for (int o = 1; o < 64; o <<= 1) {
            unsigned v = (unsigned)__shfl_up((int)incl, o, 64);
            if (lane >= o) incl += v;
        }
        unsigned excl = incl - fl;
        if (WPR > 1) {
            if (lane == 63) red_u[wave] = incl;
            __syncthreads();
            for (int w = 0; w < wave; w++) excl += red_u[w];
        }
        unsigned run = excl + (am < i0 ? rem : 0u);
        if (mode == 1) {
            uint32_t* o = out + (size_t)(out_row0 + row) * V;
#pragma unroll
            for (int k = 0; k < EPL; k++) {
                if (i0 + k < V) {
                    run += e[k] + (i0 + k == am ? rem : 0u);
                    o[i0 + k] = run;
                }
            }
        } else {
            const unsigned value = targets[row];
            int cand = 0x7FFFFFFF;
            unsigned clo = 0, chi = 0;
#pragma unroll
            for (int k = 0; k < EPL; k++) {
                if (i0 + k < V) {
                    const unsigned before = run;
                    run += e[k] + (i0 + k == am ? rem : 0u);
                    // the last symbol also takes a value at or past the total (the clamp)
                    if (cand == 0x7FFFFFFF && (value < run || i0 + k == V - 1)) {
                        cand = i0 + k;
                        clo = before;
                        chi = run;
                    }
                }
            }
            const int sym = bmin(cand);
            if (cand == sym) {
                uint32_t* o = out + (size_t)(out_row0 + row) * 3;
                o[0] = (uint32_t)sym;
                o[1] = clo;
                o[2] = chi;
            }
        }
    }
}

void launch_cdf(const int32_t* logits, int M, int V, const uint32_t* targets, const int32_t* lens, int T,
                const uint16_t* lut, unsigned coef, unsigned total, int mode, uint32_t* out, int64_t out_row0,
                hipStream_t s) {
#define CZIP_CDF(W, E)                                                                                             \
    hipLaunchKernelGGL((k_cdf<W, E>), dim3((unsigned)M), dim3(64 * W), 0, s, logits, V, targets, lens, T, lut, coef, \
                       total, mode, out, (long long)out_row0)
    const bool few = M <= CDF_FEW_ROWS * (V <= 1024 || V > 4096 ? 2 : 1);
    if (V <= 1024) { if (few) CZIP_CDF(4, 4); else CZIP_CDF(1, 16); }
    else if (V <= 4096) { if (few) CZIP_CDF(16, 4); else CZIP_CDF(4, 16); }
    else { if (few) CZIP_CDF(16, 8); else CZIP_CDF(4, 32); }
#undef CZIP_CDF
}

// ---------------------------------------------------------------------------
// Rows of a [B, T] block of coder targets for the prefill (main.rs:220-226):
// the input of row (b, p) is BOS at p = 0, else target (b, p - 1); lens are
// clamped to [0, T]; rows past a chunk's length get zeros, and so does their
// (cum_lo, cum_hi) in out (the head writes only live rows).  A live target
// >= V sets *err and reads as 0.  One thread per row.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_prep_rows(const uint32_t* __restrict__ targets,
                                                   const int32_t* __restrict__ lens_in, int B, int T, unsigned V,
                                                   uint32_t* __restrict__ inp, uint32_t* __restrict__ tgt,
                                                   int32_t* __restrict__ lens, uint32_t* __restrict__ out,
                                                   int32_t* __restrict__ err) {
    const long long r = (long long)blockIdx.x * 256 + threadIdx.x;
    if (r >= (long long)B * T) return;
    const int b = (int)(r / T), p = (int)(r - (long long)b * T);
    const int n = min(max(lens_in[b], 0), T);
    if (p == 0) lens[b] = n;
    uint32_t t = 0, prev = 0;
    if (p < n) {
        t = targets[r];
        if (t >= V) {
            atomicOr(err, 1);
            t = 0;
        }
        prev = p == 0 ? BOS_TOKEN : targets[r - 1];
        prev = prev < V ? prev : 0u;
    }
    inp[r] = prev;
    tgt[r] = t;
    *(uint2*)(out + 2 * r) = make_uint2(0u, 0u);
}

__global__ void k_zero_i32(int32_t* p) { *p = 0; }

void launch_prep_rows(const uint32_t* targets, const int32_t* lens_in, int B, int T, int V, uint32_t* inp,
                      uint32_t* tgt, int32_t* lens, uint32_t* out, int32_t* err, hipStream_t s) {
    const long long M = (long long)B * T;
    hipLaunchKernelGGL(k_zero_i32, dim3(1), dim3(1), 0, s, err);
    if (M > 0)
        hipLaunchKernelGGL(k_prep_rows, dim3((unsigned)((M + 255) / 256)), dim3(256), 0, s, targets, lens_in, B, T,
                           (unsigned)V, inp, tgt, lens, out, err);
}

// ---------------------------------------------------------------------------
// Coded chunks from their fixed-size slots to one back-to-back buffer (the
// chunk data layout of the container, file_format.rs:324-331), so that only
// the coded bytes cross PCIe.  One workgroup per chunk; lens[c] <= slot.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_pack_chunks(const uint8_t* __restrict__ src, long long slot,
                                                     const int32_t* __restrict__ lens,
                                                     const long long* __restrict__ offs, uint8_t* __restrict__ dst) {
    const int c = blockIdx.x;
    const uint8_t* s = src + (size_t)c * slot;
    uint8_t* d = dst + offs[c];
    const int n = lens[c];
    for (int i = threadIdx.x; i < n; i += 256) d[i] = s[i];
}

void launch_pack_chunks(const uint8_t* src, int64_t slot, const int32_t* lens, const int64_t* offs, int n,
                        uint8_t* dst, hipStream_t s) {
    if (n > 0)
        hipLaunchKernelGGL(k_pack_chunks, dim3((unsigned)n), dim3(256), 0, s, src, (long long)slot, lens,
                           (const long long*)offs, dst);
}

// ---------------------------------------------------------------------------
// Arithmetic encoder (arith_coder.rs:26-136), one thread per chunk.  A chunk
// is one chain of dependent steps, so the kernel is bound by that chain's
// latency whatever the number of chunks.  A step takes its shifts in closed
// form: after the k = clz(low ^ high) shifts that settle a leading bit (32 of
// them when low == high), the leading bits differ, and the u following ones
// of low & ~high behind them are the E3 shifts; an E3 shift leaves the leading
// bits different, so no settled bit follows.  The divisions are one f64
// estimate each (x / total formed ahead of the chain) with a branch-free
// integer correction, the intervals are loaded ENC_AHEAD tokens ahead, and the
// bits leave as whole words, a symbol's settled and pending bits in one append.
// Measured against a loop per shift, pending bit and correction: 11 chunks of
// 64 tokens 179 -> 27 us, 49 of 4096 16.3 -> 1.4 ms (4.0 -> 0.34 us a token), 38
// thousand of 512 2.19 -> 0.22 ms.
// ---------------------------------------------------------------------------
constexpr int ENC_AHEAD = 8;  // intervals in flight per thread

struct BitOut {
    uint8_t* buf;  // 4-byte aligned
    long long cap, len;
    unsigned long long acc;  // the low nacc bits are pending, the oldest on top
    int nacc;                // < 32 between calls
    int overflow;
    // whole words leave in stream order (the most significant bit first)
    __device__ __forceinline__ void flush_word() {
        const unsigned w = (unsigned)(acc >> (nacc - 32));
        if (len + 4 <= cap) {
            *(unsigned*)(buf + len) = __builtin_bswap32(w);
        } else {
            for (int i = 0; i < 4; i++)
                if (len + i < cap) buf[len + i] = (uint8_t)(w >> (24 - 8 * i));
                else overflow = 1;
        }
        len += 4;
        nacc -= 32;
    }
    // the low n bits of v, n <= 32
    __device__ __forceinline__ void bits(unsigned v, int n) {
        acc = (acc << n) | (n < 32 ? v & ((1u << n) - 1u) : v);
        nacc += n;
        if (nacc >= 32) flush_word();
    }
    __device__ __forceinline__ void bit(unsigned b) { bits(b, 1); }
    __device__ __forceinline__ void run(unsigned b, unsigned n) {  // n copies of b
        const unsigned v = b ? 0xFFFFFFFFu : 0u;
        for (; n > 32; n -= 32) bits(v, 32);
        bits(v, (int)n);
    }
    __device__ __forceinline__ void finish() {  // the partial word's bytes, zero-padded
        while (nacc > 0) {
            const unsigned b = nacc >= 8 ? (unsigned)(acc >> (nacc - 8)) : (unsigned)(acc << (8 - nacc));
            if (len < cap) buf[len] = (uint8_t)b;
            else overflow = 1;
            len++;
            nacc -= 8;
        }
    }
};

__global__ __launch_bounds__(64) void k_encode(const uint32_t* __restrict__ lohi, const int32_t* __restrict__ lens,
                                               int nb, int T, unsigned total, uint8_t* __restrict__ out,
                                               long long slot, int32_t* __restrict__ out_lens,
                                               int32_t* __restrict__ err) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= nb) return;
    const unsigned long long MASK = 0xFFFFFFFFull, HALF = 1ull << 31, QUART = 1ull << 30;
    unsigned low = 0, high = 0xFFFFFFFFu;
    unsigned underflow = 0;
    BitOut o{out + (size_t)c * slot, slot, 0, 0ull, 0, 0};
    const double invT = 1.0 / (double)total;
    const int n = lens[c];
    const uint2* lh = (const uint2*)(lohi + (size_t)c * T * 2);
    bool stuck = false;
    auto step = [&](uint2 cur) {
        if (stuck) return;
        const unsigned rm1 = high - low;
        const double range = (double)rm1 + 1.0;
        const unsigned long long ql = coder_div(cur.x, (double)cur.x * invT, rm1, range, total);
        const unsigned long long qh = coder_div(cur.y, (double)cur.y * invT, rm1, range, total);
        const unsigned nl = low + (unsigned)ql, nh = low + (unsigned)qh - 1u;
        if (ql < qh) {
            const int k = __clz((int)(nl ^ nh));  // 32 when they are equal
            if (k > 0) {
                // the first settled bit b, the pending bits (each 1 - b), the k - 1
                // bits behind: b and n pending ones are the number 2^n - 1 + b
                const unsigned b = nl >> 31;
                if (underflow + (unsigned)k <= 32u) {
                    const unsigned head = ((1u << underflow) - 1u + b) << (k - 1);
                    o.bits(head | ((nl >> (32 - k)) & ((1u << (k - 1)) - 1u)), (int)underflow + k);
                } else {
                    o.bit(b);
                    o.run(b ^ 1u, underflow);
                    if (k > 1) o.bits(nl >> (32 - k), k - 1);
                }
                underflow = 0;
            }
            const unsigned l1 = k < 32 ? nl << k : 0u;
            const unsigned h1 = k < 32 ? (nh << k) | ((1u << k) - 1u) : 0xFFFFFFFFu;
            // E3: bits 30, 29, .. of low & ~high
            const int u = __clz((int)~((l1 & ~h1) << 1));
            underflow += (unsigned)u;
            low = (l1 << u) & 0x7FFFFFFFu;
            high = (h1 << u) | ((1u << u) - 1u) | 0x80000000u;
        } else {
            // an empty interval (a total beyond the coder's range): the
            // reference's shifts one by one; its range is 0 from here on, and
            // no later symbol shifts anything
            unsigned long long l = nl, h = nh;
            stuck = true;
            if (low + (unsigned)qh == 0u) return;  // high wrapped below 0: nothing to shift
            for (;;) {
                if (((l ^ h) & HALF) == 0) {
                    const unsigned b = (unsigned)((l >> 31) & 1);
                    o.bit(b);
                    o.run(b ^ 1u, underflow);
                    underflow = 0;
                    l = (l << 1) & MASK;
                    h = ((h << 1) & MASK) | 1;
                } else if ((l & ~h & QUART) != 0) {
                    underflow += 1;
                    l = ((l << 1) ^ HALF) & MASK;
                    h = (((h ^ HALF) << 1) | HALF | 1) & MASK;
                } else {
                    break;
                }
            }
        }
    };
    uint2 cur[ENC_AHEAD], nxt[ENC_AHEAD];
    auto load = [&](uint2* d, int i0) {
#pragma unroll
        for (int j = 0; j < ENC_AHEAD; j++) d[j] = lh[min(i0 + j, n - 1)];
    };
    if (n > 0) load(cur, 0);
    for (int i0 = 0; i0 < n; i0 += ENC_AHEAD) {
        load(nxt, i0 + ENC_AHEAD);
#pragma unroll
        for (int j = 0; j < ENC_AHEAD; j++)
            if (i0 + j < n) step(cur[j]);
#pragma unroll
        for (int j = 0; j < ENC_AHEAD; j++) cur[j] = nxt[j];
    }
    o.bit(1u);  // finish(): terminating bit, then flush the partial byte
    o.finish();
    out_lens[c] = (int32_t)o.len;
    if (o.overflow) atomicOr(err, 1);
}

void launch_encode(const uint32_t* lohi, const int32_t* lens, int nb, int T, unsigned total, uint8_t* out,
                   int64_t slot, int32_t* out_lens, int32_t* err, hipStream_t s) {
    hipLaunchKernelGGL(k_encode, dim3((unsigned)((nb + 63) / 64)), dim3(64), 0, s, lohi, lens, nb, T, total, out,
                       (long long)slot, out_lens, err);
}

}  // namespace czip
