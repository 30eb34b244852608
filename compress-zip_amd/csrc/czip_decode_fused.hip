// Whole-stream decode of one-layer models in one launch: every step of the
// chunk loop of main.rs:377-396 (forward, frequency table, symbol, decoder
// step) for the 1 to 16 streams of a workgroup.
//
// A step of a few streams is a chain of small dependent products.  As
// launches (six to eight a step, 3-8 us each) the chain is bound by launch
// and drain latency; streams are independent, so a workgroup that owns its
// streams needs no other workgroup at any step and the whole decode is one
// kernel, its phases separated by workgroup barriers.  What bounds it then is
// the weights (1.7 MB for the shipped model), streamed from the XCD's L2 by
// every workgroup at every step (135-150 GB/s a CU: 12 us), which is why only
// models whose weights stay in an L2 take it, and the latency of the
// attention.  The 16 MFMA columns are the workgroup's streams.
//
// Wave r owns stream r: its decoder (in registers), its layer 0 Q/K/V from
// the per-token table, its row norms and residual, and its symbol search; the
// products and the (stream, head) attention rows are spread over all waves.
// A phase's first weights are requested before the barrier that opens it, so
// the barriers order LDS only; the one that publishes the step's K and V also
// waits for those stores.
//
// Measured (shipped model, 512 steps, step kernels -> here): 1 stream 21.8 ->
// 12.1 ms, 115 26.4 -> 12.2, 512 30.8 -> 14.5, 1024 36.8 -> 17.6, 2048 41.9 ->
// 25.7 ms, 3500 42.6 -> 37.0; 115 streams of 64 steps 3.4 -> 1.3 ms.
#include <algorithm>

#include "czip_attn_row.h"
#include "czip_device.h"
#include "czip_head.h"
#include "czip_kernels.h"

namespace czip {

namespace {

constexpr int FNW = 16;       // waves
constexpr int FMAXF = 1024;   // widest feed-forward
constexpr int FV = 1024;      // vocabulary
constexpr int FPAD = 16;      // row padding (words) of the int32 rows in LDS: 16 rows of 16-byte pieces in four passes

__device__ __forceinline__ unsigned wave_total(unsigned x) {
    return (unsigned)__builtin_amdgcn_readlane((int)wave_scan(x, 0u, [](unsigned a, unsigned b) { return a + b; }), 63);
}

// A stream's arithmetic decoder (arith_coder.rs:139-264), uniform over its
// wave.  bit: stream bits taken; w: the three words of the chunk buffer from
// that bit's (clamped) byte on, requested as soon as the position is known.
struct RowDecoder {
    const uint8_t* data;  // all chunk bytes (16 bytes of padding behind them)
    long long off;        // the chunk's first byte
    unsigned len;
    unsigned low, high, code;
    unsigned bit;
    unsigned w0, w1, w2;

    __device__ __forceinline__ void request() {
        const long long base = (off + min(bit >> 3, len)) & ~3ll;
        const unsigned* w = (const unsigned*)(data + base);
        w0 = w[0];
        w1 = w[1];
        w2 = w[2];
    }
    // kept in scalar registers between the steps
    __device__ __forceinline__ void settle() {
        low = uni(low);
        high = uni(high);
        code = uni(code);
        bit = uni(bit);
    }
    // the stream's next 57 or more bits, left-aligned; 0 past the chunk's end
    __device__ __forceinline__ unsigned long long window() const {
        const unsigned by = min(bit >> 3, len);
        const int sh = (int)((off + by) & 3ll) * 8;
        const unsigned long long lo = ((unsigned long long)w1 << 32) | w0;
        unsigned long long v = sh ? (lo >> sh) | ((unsigned long long)w2 << (64 - sh)) : lo;
        const unsigned nv = len - by;  // bytes left
        if (nv < 8) v &= (1ull << (8 * nv)) - 1ull;
        return __builtin_bswap64(v) << (bit & 7u);
    }
    __device__ __forceinline__ void begin() {
        bit = 0;
        request();
        code = (unsigned)(window() >> 32);
        low = 0u;
        high = 0xFFFFFFFFu;
        bit = 32;
        settle();
        request();
    }
    // ((code - low + 1) * total - 1) / range, clamped to total - 1 (arith_coder.rs:199-203, 225-241)
    __device__ __forceinline__ unsigned value(unsigned total) const {
        const unsigned long long range = (unsigned long long)(high - low) + 1;
        const unsigned long long a = ((unsigned long long)(code - low) + 1) * total - 1;
        unsigned long long q = (unsigned long long)((double)a / (double)range);
        const long long r = (long long)(a - q * range);
        q += r >= (long long)range ? 1ull : 0ull;
        q -= r < 0 ? 1ull : 0ull;
        return (unsigned)min(q, (unsigned long long)total - 1);
    }
    // the step of a symbol with interval [lo, hi), lo < hi, total <= 2^30: the
    // shifts in closed form (as the encoder: k settled bits, then u E3 shifts,
    // at most 32 in all)
    __device__ __forceinline__ void advance(unsigned lo, unsigned hi, unsigned total, double inv_total) {
        const unsigned rm1 = high - low;
        const double range = (double)rm1 + 1.0;
        const unsigned nl = low + (unsigned)coder_div(lo, (double)lo * inv_total, rm1, range, total);
        const unsigned nh = low + (unsigned)coder_div(hi, (double)hi * inv_total, rm1, range, total) - 1u;
        const int k = nl == nh ? 32 : __clz((int)(nl ^ nh));
        const unsigned l1 = k < 32 ? nl << k : 0u;
        const unsigned h1 = k < 32 ? (nh << k) | ((1u << k) - 1u) : 0xFFFFFFFFu;
        const int u = __clz((int)~((l1 & ~h1) << 1));
        low = (l1 << u) & 0x7FFFFFFFu;
        high = (h1 << u) | ((1u << u) - 1u) | 0x80000000u;
        const unsigned long long win = window();
        const unsigned long long c1 = ((unsigned long long)code << 32 | (unsigned)(win >> 32)) << k;  // k <= 32
        const unsigned cd = (unsigned)(c1 >> 32);
        // E3 keeps the leading bit and shifts the others
        const unsigned long long c2 = ((unsigned long long)cd << 32 | (unsigned)((win << k) >> 32)) << u;
        code = (cd & 0x80000000u) | ((unsigned)(c2 >> 32) & 0x7FFFFFFFu);
        bit += (unsigned)(k + u);
        settle();
        request();
    }
};

}  // namespace

// KS: K steps of 64 of the model width (d = 64 KS = 64 heads)
template <int KS, bool GEN>
__global__ __launch_bounds__(64 * FNW) void k_decode_fused(FusedDecArgs a) {
    constexpr int D = 64 * KS, H = KS, YS = D + FPAD, LS = FV + FPAD;
    constexpr int HK = KS / 2;               // K steps of half an output projection
    constexpr int NT = KS * 8 / FNW;         // (column tile, K half) units of an output projection per wave
    constexpr int NG = (D + 255) / 256;      // 4-element groups per lane of a row
    constexpr int FK = FMAXF / 128;          // K steps of half a down projection (zeros past F)
    constexpr int YB = 2 * 16 * YS * 4, LB = 16 * LS * 4;
    __shared__ __attribute__((aligned(16))) int8_t As[KS][1024];  // attention rows, then normalized rows (lds64 rows)
    __shared__ __attribute__((aligned(16))) int8_t qs[16][D];
    // the projections' partial sums [2][16][YS], then the logits [16][LS]
    __shared__ __attribute__((aligned(16))) int8_t big[YB > LB ? YB : LB];
    __shared__ __attribute__((aligned(16))) int8_t r8[FMAXF / 64 * 1024];  // ReGLU rows (lds64), zero from F on
    __shared__ short xs[16][D];  // residual streams
    __shared__ __attribute__((aligned(16))) uint16_t etb[ETB_PAD];
    __shared__ unsigned hetab[ETAB_N];
    __shared__ __attribute__((aligned(16))) AttnRowLds wl[FNW];
    __shared__ __attribute__((aligned(16))) int8_t nw[4][D];  // norms: ffn, post_attn, post_ffn, final
    __shared__ int nt[16];
    int(*ys)[16][YS] = (int(*)[16][YS])big;
    int(*lg)[LS] = (int(*)[LS])big;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b0 = (int)blockIdx.x * a.R;
    const int rows = min(a.R, a.S - b0);
    for (int i = tid; i < ETB_PAD / 8; i += 64 * FNW) ((uint4*)etb)[i] = ((const uint4*)a.etab)[i];
    for (int t = tid; t < ETAB_N; t += 64 * FNW) hetab[t] = head_etab_entry(t, a.lut);
    for (int i = tid; i < 4 * D; i += 64 * FNW) {
        const int8_t* w = i < D ? a.w_ffn : i < 2 * D ? a.w_post_attn : i < 3 * D ? a.w_post_ffn : a.w_final;
        ((int8_t*)nw)[i] = w[i % D];
    }
    for (int i = tid + a.F; i < FMAXF; i += 64 * FNW) *(v4i*)(r8 + i * 16) = (v4i){0, 0, 0, 0};
    if (tid < 16) nt[tid] = tid < rows ? a.ds.ntok[b0 + tid] : 0;
    __syncthreads();
    int steps = 0;
    for (int r = 0; r < 16; r++) steps = max(steps, nt[r]);
    steps = __builtin_amdgcn_readfirstlane(steps);
    const int n = __builtin_amdgcn_readfirstlane(nt[wave]);  // this wave's stream: n tokens (0: none)
    const int b = b0 + min(wave, rows - 1);
    const double inv_total = 1.0 / (double)a.total;
    RowDecoder dec;
    dec.data = a.ds.data;
    dec.off = a.ds.offs[b];
    dec.len = (unsigned)a.ds.blen[b];
    uint32_t* tok_out = a.ds.tokens + a.ds.tok_offs[b];
    if (n > 0) dec.begin();
    unsigned tok = BOS_TOKEN;
    const size_t skv = (size_t)a.KH * a.TP * 64;  // a stream's K (and V) bytes
    const int half = wave & 1, tile0 = wave >> 1;  // (tile, K half) units: tiles tile0 + 8 i

    // the row norms of an output projection: x += rmsnorm(requant(y), w1),
    // normalized rows rmsnorm(clamp(x), w2) into As (model.rs:424-439, 459-474)
    auto row_norms = [&](double scale, const int8_t* w1, const int8_t* w2) {
        const int lane = opaque_tid() & 63;
        int y[NG][4], x[NG][4];
        unsigned ss = 0;
#pragma unroll
        for (int j = 0; j < NG; j++) {
            const int g = lane + 64 * j;
            if (g < D / 4) {
                const v4i p0 = *(const v4i*)&ys[0][wave][4 * g], p1 = *(const v4i*)&ys[1][wave][4 * g];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    y[j][k] = clamp127(rint_fma_i32((double)(int)((unsigned)p0[k] + (unsigned)p1[k]), scale));
                    ss += (unsigned)__mul24(y[j][k], y[j][k]);
                }
            }
        }
        // eps_scaled = 1 (rmsnorm.rs:80-83)
        double inv = (double)inv_rms_q15_fast((int)(wave_total(ss) / (unsigned)D) + 1) * (1.0 / 32768.0);
        ss = 0;
#pragma unroll
        for (int j = 0; j < NG; j++) {
            const int g = lane + 64 * j;
            if (g < D / 4) {
                int w[4];
                unpack4s(*(const unsigned*)(w1 + 4 * g), w);
                const uint2 xw = *(const uint2*)&xs[wave][4 * g];
                x[j][0] = (int16_t)(xw.x & 0xFFFFu); x[j][1] = (int16_t)(xw.x >> 16);
                x[j][2] = (int16_t)(xw.y & 0xFFFFu); x[j][3] = (int16_t)(xw.y >> 16);
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    x[j][k] += rms_el(y[j][k], w[k], inv);
                    const int c = clamp127(x[j][k]);
                    ss += (unsigned)__mul24(c, c);
                }
                *(uint2*)&xs[wave][4 * g] = make_uint2(((unsigned)x[j][0] & 0xFFFFu) | ((unsigned)x[j][1] << 16),
                                                       ((unsigned)x[j][2] & 0xFFFFu) | ((unsigned)x[j][3] << 16));
            }
        }
        inv = (double)inv_rms_q15_fast((int)(wave_total(ss) / (unsigned)D) + 1) * (1.0 / 32768.0);
#pragma unroll
        for (int j = 0; j < NG; j++) {
            const int g = lane + 64 * j;
            if (g < D / 4) {
                int w[4], o[4];
                unpack4s(*(const unsigned*)(w2 + 4 * g), w);
#pragma unroll
                for (int k = 0; k < 4; k++) o[k] = rms_el(clamp127(x[j][k]), w[k], inv);
                *(unsigned*)(As[g >> 4] + lds64(wave, (g >> 2) & 3) + (g & 3) * 4) = pack4i(o[0], o[1], o[2], o[3]);
            }
        }
    };

    const __amdgpu_buffer_rsrc_t r_out = weights_rsrc(a.out_wf, D * D), r_up = weights_rsrc(a.up_wf, 2 * a.F * D),
                                 r_down = weights_rsrc(a.down_wf, a.F * D), r_head = weights_rsrc(a.head_wf, FV * D);
    for (int p = 0; p < steps; p++) {
        // each phase forms its lane-dependent addresses anew (opaque_tid): held
        // across the step, they take registers from the attention
        const bool own = p < n;
        unsigned value = 0;
        if (own) {
            const int lane = opaque_tid() & 63;
            // residual input and layer 0's Q/K/V of the stream's token (k_qkv_table's arithmetic)
            const int8_t* t = a.tab + (size_t)tok * a.qkv_n;
#pragma unroll
            for (int j = 0; j < NG; j++) {
                const int g = lane + 64 * j;
                if (g < D / 4) {
                    int e[4];
                    unpack4s(*(const unsigned*)(a.embed + (size_t)tok * D + 4 * g), e);
                    *(uint2*)&xs[wave][4 * g] = make_uint2(((unsigned)e[0] & 0xFFFFu) | ((unsigned)e[1] << 16),
                                                           ((unsigned)e[2] & 0xFFFFu) | ((unsigned)e[3] << 16));
                }
            }
            for (int it = lane; it < 8 * H + 24 * a.NKV; it += 64) {
                if (it >= 8 * H + 8 * a.NKV) {  // V: dims 4 q .. +3 of head g
                    const int v = it - 8 * H - 8 * a.NKV, g = v >> 4, q = v & 15;
                    const unsigned w = *(const unsigned*)(t + D + 64 * a.NKV + 64 * g + 4 * q);
                    int8_t* dst = a.vc + (size_t)b * skv + (size_t)g * 64 * a.TP + vt_off(p, 4 * q, 2);
#pragma unroll
                    for (int r = 0; r < 4; r++) dst[r << 2] = (int8_t)(w >> (8 * r));
                    continue;
                }
                const bool isq = it < 8 * H;
                const double rm = isq ? 0.5 : 1.0, rb = isq ? ROPE_Q_BIAS : 0.0;
                const int hd = isq ? it >> 3 : (it - 8 * H) >> 3, i0 = 4 * (it & 7);
                const int col = isq ? 64 * hd : D + 64 * hd;
                const unsigned xw = *(const unsigned*)(t + col + i0), yw = *(const unsigned*)(t + col + i0 + 32);
                const uint2 cw = *(const uint2*)(a.rcos + p * 32 + i0), sw = *(const uint2*)(a.rsin + p * 32 + i0);
                int xq[4], yq[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int xv = (int8_t)(xw >> (8 * r)), yv = (int8_t)(yw >> (8 * r));
                    const unsigned cc = r < 2 ? cw.x : cw.y, sc = r < 2 ? sw.x : sw.y;
                    const int c = (int16_t)(r & 1 ? cc >> 16 : cc & 0xFFFFu), sn = (int16_t)(r & 1 ? sc >> 16 : sc & 0xFFFFu);
                    xq[r] = clamp127(rope_round((int)((unsigned)(xv * c) - (unsigned)(yv * sn)), rm, rb));
                    yq[r] = clamp127(rope_round((int)((unsigned)(xv * sn) + (unsigned)(yv * c)), rm, rb));
                }
                int8_t* dst = isq ? &qs[wave][64 * hd] : a.kc + (size_t)b * skv + ((size_t)hd * a.TP + p) * 64;
                *(unsigned*)(dst + i0) = pack4i(xq[0], xq[1], xq[2], xq[3]);
                *(unsigned*)(dst + i0 + 32) = pack4i(yq[0], yq[1], yq[2], yq[3]);
            }
            value = uni(dec.value(a.total));
        }
        __syncthreads();  // queries in LDS, the step's K and V in the caches
        for (int it = wave; it < rows * H; it += FNW) {
            const int lane = opaque_tid() & 63;
            const int r = it / H, h = it - r * H;
            if (p >= __builtin_amdgcn_readfirstlane(nt[r])) continue;
            const int g = a.kv_mode == 1 ? h * a.G / H : 0;
            const size_t base = (size_t)(b0 + r) * skv + (size_t)g * a.TP * 64;
            const int8_t* kb = a.kc + base + lane * 64;
            const int* vb = (const int*)(a.vc + base) + lane;
            v4i k[4];
            int v[16], q[16];
            auto load = [&](int t0) {
#pragma unroll
                for (int i = 0; i < 4; i++) k[i] = *(const v4i*)(kb + t0 * 64 + i * 16);
#pragma unroll
                for (int i = 0; i < 16; i++) v[i] = vb[(t0 / 4 + i) * 64];
            };
            load(0);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const v4i w = *(const v4i*)&qs[r][h * 64 + i * 16];
#pragma unroll
                for (int j = 0; j < 4; j++) q[4 * i + j] = __builtin_amdgcn_readfirstlane(w[j]);
            }
            const double mscale = (double)a.score_mult[h] * (1.0 / 32768.0);
            AttnRow st = attn_row_begin<GEN>(q, a.sink, mscale);
            for (int t0 = 0; t0 <= p; t0 += 64) {
                v4i kc[4];
                int vc[16];
#pragma unroll
                for (int i = 0; i < 4; i++) kc[i] = k[i];
#pragma unroll
                for (int i = 0; i < 16; i++) vc[i] = v[i];
                if (t0 + 64 <= p) load(t0 + 64);
                attn_row_tile<GEN>(q, kc, vc, mscale, min(p + 1 - t0, 64), etb, wl[wave], st);
            }
            As[h][lds64(r, lane >> 4) + (lane & 15)] = attn_row_out(st);
        }

        // output projection: half the K steps of NT column tiles per wave
        {
            const int lane = opaque_tid() & 63, lr = lane & 15, grp = lane >> 4, c4 = grp * 4;
            v4i w[NT][HK];
#pragma unroll
            for (int i = 0; i < NT; i++) load_ops(w[i], r_out, (tile0 + 8 * i) * KS + half * HK, lane);
            lds_barrier();
#pragma unroll
            for (int i = 0; i < NT; i++) {
                v4i acc = {0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < HK; s++)
                    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                        w[i][s], *(const v4i*)(As[half * HK + s] + lds64(lr, grp)), acc, 0, 0, 0);
                if (lr < rows) *(v4i*)&ys[half][lr][(tile0 + 8 * i) * 16 + c4] = acc;
            }
        }
        lds_barrier();
        if (own) row_norms(a.o_scale, nw[0], nw[1]);

        // up projection + ReGLU: 16 gate and the matching 16 up columns at a time
        {
            const int lane = opaque_tid() & 63, lr = lane & 15, grp = lane >> 4, c4 = grp * 4;
            const int np = a.F / 16;
            v4i wg[KS], wu[KS], xf[KS];
            auto gate = [&](int g) { return ((g >> 1) * 4 + (g & 1)) * KS; };
            if (wave < np) load_ops(wg, r_up, gate(wave), lane);
            lds_barrier();
#pragma unroll
            for (int s = 0; s < KS; s++) xf[s] = *(const v4i*)(As[s] + lds64(lr, grp));
            for (int g = wave; g < np; g += FNW) {
                load_ops(wu, r_up, gate(g) + 2 * KS, lane);
                v4i ag = {0, 0, 0, 0}, au = {0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < KS; s++) ag = __builtin_amdgcn_mfma_i32_16x16x64_i8(wg[s], xf[s], ag, 0, 0, 0);
                if (g + FNW < np) load_ops(wg, r_up, gate(g + FNW), lane);
#pragma unroll
                for (int s = 0; s < KS; s++) au = __builtin_amdgcn_mfma_i32_16x16x64_i8(wu[s], xf[s], au, 0, 0, 0);
                int o[4];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int gv = max(clamp127(rint_fma_i32((double)ag[r], a.up_scale)), 0);
                    o[r] = clamp127(rne_shr(gv * clamp127(rint_fma_i32((double)au[r], a.up_scale)), 7));  // reglu.rs:20-46
                }
                *(unsigned*)(r8 + (g >> 2) * 1024 + lds64(lr, g & 3) + c4) = pack4i(o[0], o[1], o[2], o[3]);
            }
        }
        // down projection: half the K steps of NT column tiles per wave
        {
            const int lane = opaque_tid() & 63, lr = lane & 15, grp = lane >> 4, c4 = grp * 4;
            const int nk = a.F / 64;
            v4i w[2][FK];
            auto load = [&](v4i (&d)[FK], int tile) {  // past the last K step: the last one, times zeros
#pragma unroll
                for (int s = 0; s < FK; s++)
                    d[s] = __builtin_amdgcn_raw_buffer_load_b128(r_down, lane * 16, (tile * nk + min(half * FK + s, nk - 1)) * 1024, 0);
            };
            load(w[0], tile0);
            lds_barrier();
#pragma unroll
            for (int i = 0; i < NT; i++) {
                if (i + 1 < NT) load(w[(i + 1) & 1], tile0 + 8 * (i + 1));
                v4i acc = {0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < FK; s++)
                    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                        w[i & 1][s], *(const v4i*)(r8 + (half * FK + s) * 1024 + lds64(lr, grp)), acc, 0, 0, 0);
                if (lr < rows) *(v4i*)&ys[half][lr][(tile0 + 8 * i) * 16 + c4] = acc;
            }
        }
        lds_barrier();
        if (own) row_norms(a.dn_scale, nw[2], nw[3]);

        // LM head: 4 column tiles per wave
        {
            constexpr int HT = FV / 16 / FNW;
            const int lane = opaque_tid() & 63, lr = lane & 15, grp = lane >> 4, c4 = grp * 4;
            v4i w[2][KS], xf[KS];
            load_ops(w[0], r_head, wave * KS, lane);
            lds_barrier();
#pragma unroll
            for (int s = 0; s < KS; s++) xf[s] = *(const v4i*)(As[s] + lds64(lr, grp));
#pragma unroll
            for (int i = 0; i < HT; i++) {
                if (i + 1 < HT) load_ops(w[(i + 1) & 1], r_head, (wave + FNW * (i + 1)) * KS, lane);
                v4i acc = {0, 0, 0, 0};
#pragma unroll
                for (int s = 0; s < KS; s++) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[i & 1][s], xf[s], acc, 0, 0, 0);
                if (lr < rows) *(v4i*)&lg[lr][(wave + FNW * i) * 16 + c4] = acc;
            }
        }
        lds_barrier();
        if (own) {
            // frequencies (head_freqs' arithmetic) of the lane's 16 columns, and the symbol
            const int lane = opaque_tid() & 63;
            int l[16];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const v4i t = *(const v4i*)&lg[wave][lane * 16 + 4 * i];
#pragma unroll
                for (int k = 0; k < 4; k++) l[4 * i + k] = t[k];
            }
            int mx = l[0];
#pragma unroll
            for (int i = 1; i < 16; i++) mx = max(mx, l[i]);
            mx = __builtin_amdgcn_readlane(
                (int)wave_scan((unsigned)mx, 0x80000000u, [](unsigned u, unsigned v) { return (unsigned)max((int)u, (int)v); }), 63);
            const long long kr = (long long)mx * (long long)(a.coef << 8) + 0x80000000ll;
            const int negc = -(int)(a.coef << 8);
            int ak = 16;
            unsigned f[16], s = 0;
#pragma unroll
            for (int i = 15; i >= 0; i--) {
                ak = l[i] == mx ? i : ak;
                const unsigned st = min((unsigned)((unsigned long long)((long long)l[i] * (long long)negc + kr) >> 32), 4096u);
                f[i] = hetab[l[i] == mx ? ETAB_N - 1 : (int)st];
                s += f[i];
            }
            const unsigned long long hold_max = __builtin_amdgcn_ballot_w64(ak < 16);
            const int am_lane = __builtin_ctzll(hold_max);  // the first lane (columns ascend with the lane)
            const unsigned S = wave_total(s);
            const unsigned Rt = a.total - (unsigned)FV, Q = Rt / S;
            const double yq = (double)(Rt - Q * S) / (double)S;
            unsigned fs = 0;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                f[i] = __umul24(f[i], Q) + (unsigned)__builtin_fma((double)f[i], yq, 1.0 + 0x1p-30);
                fs += f[i];
            }
            const unsigned rem = a.total - wave_total(fs);
            const bool has_am = lane == am_lane;
            fs += has_am ? rem : 0u;
            const unsigned base = wave_scan(fs, 0u, [](unsigned u, unsigned v) { return u + v; }) - fs;
            // the lane whose range holds the value, then its column
            const unsigned long long hold = __builtin_amdgcn_ballot_w64(value - base < fs);
            const int hl = __builtin_ctzll(hold);
            unsigned run = base, lo = base, hi = 0u;
            int kc = 0;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const unsigned nx = run + f[i] + (has_am && ak == i ? rem : 0u);
                const bool here = value >= run;  // columns up to the symbol's
                lo = here ? run : lo;
                hi = here ? nx : hi;
                kc = here ? i : kc;
                run = nx;
            }
            tok = (unsigned)__builtin_amdgcn_readlane(hl * 16 + kc, hl);
            const unsigned slo = (unsigned)__builtin_amdgcn_readlane((int)lo, hl), shi = (unsigned)__builtin_amdgcn_readlane((int)hi, hl);
            if (lane == 0) tok_out[p] = tok;
            dec.advance(slo, shi, a.total, inv_total);
        }
    }
}

// Streams per workgroup: one while they fit the CUs (the weights' stream per
// step is the same for 1 and 16, the attention is not), 16 at most.
int decode_fused_rows(int S) { return std::max(1, (S + 255) / 256); }

// Its row-wise attention is no match for the step kernels' tiles once there are
// many rows and many keys, the sooner the more query heads share a KV head (the
// tiles share their keys; with one or two they have no more to share).  The line
// is rows^2 T, where both sides meet, in ms, steps -> here: shipped model, 1024
// tokens 2560 streams 105.6 -> 87.7, 3072 107 -> 105, 4096 117 -> 142, 512 tokens
// 4096 44.2 -> 41.2; d512, 4 heads a KV head, 512 tokens 2048 42.6 -> 39.3, 3072
// 50.1 -> 51.3, 1024 tokens 2048 122 -> 118, 4096 175 -> 211; 8 heads a KV head, 512
// tokens 2048 39.4 -> 36.5, 3072 42.6 -> 45.6, 1024 tokens 1536 90 -> 84, 2048 96 ->
// 102, 64 tokens 4096 4.5 -> 3.9; 2 heads, 1024 tokens 4096 294 -> 284.
int decode_fused_streams(int d, int H, int G, int T) {
    const int share = H / G;
    if (share <= 2) return DECODE_FUSED_MAX_STREAMS;
    const double line = d >= 512 && share > 4 ? 1.6e11 : 2.9e11;
    return std::min(DECODE_FUSED_MAX_STREAMS, (int)(__builtin_sqrt(line / (T < 1 ? 1 : T)) / H));
}

bool decode_fused_supported(int d, int F, int V) {
    return (d == 256 || d == 384 || d == 512) && F % 64 == 0 && F <= FMAXF && V == FV;
}

void launch_decode_fused(const FusedDecArgs& a, int d, bool general, hipStream_t s) {
    FusedDecArgs g = a;
    g.R = decode_fused_rows(a.S);
    const dim3 grid((unsigned)((a.S + g.R - 1) / g.R));
#define CZIP_DF(KS)                                                                                   \
    do {                                                                                              \
        if (general) hipLaunchKernelGGL((k_decode_fused<KS, true>), grid, dim3(64 * FNW), 0, s, g);   \
        else hipLaunchKernelGGL((k_decode_fused<KS, false>), grid, dim3(64 * FNW), 0, s, g);          \
    } while (0)
    if (d == 256) CZIP_DF(4);
    else if (d == 384) CZIP_DF(6);
    else CZIP_DF(8);
#undef CZIP_DF
}

}  // namespace czip
