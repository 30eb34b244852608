// One wavefront's exact decode attention for ONE query row (a stream and a
// head, attention.rs:162-289), for steps with few rows in flight.
//
// attn_tile (czip_attn_tile.h) fills a wave with 8 to 16 rows and walks a
// stream's keys tile by tile: about 900 VALU instructions a tile for all its
// rows, but one wave's serial chain of ~5 us a tile however few streams there
// are.  Here a wave has one row, so that everything the records decide is
// uniform and sits in scalar registers:
//  - scores, running max, weights: lane = key of the 64-key tile (dot
//    products by sdot4, the running max by a DPP scan, one table read);
//  - value sums: lane = head dim; V^T in 4-key blocks gives a lane four keys
//    of its dim in one word, and a block takes three sdot4 (the weights' high
//    and low offset bytes and ones, see WOFF), a split block one masked pair
//    more per record;
//  - the records' rescales of the weight sum are scalar arithmetic.
// About 180 VALU a tile and row: two to three times the MFMA tile's work per
// row, a fraction of its latency.  Attention of a 512-step decode, MFMA tile ->
// one row a wave: v001 12 rows 12.3 -> 5.1 ms, 690 14.6 -> 5.4, 3072 15.3 ->
// 7.5, 12288 16.7 -> 18.3; d512 (8 layers) 4096 rows 118 -> 64 ms, 16384 131 ->
// 180; d768 (12 layers, 256 steps) 708 rows 55 -> 26 ms, 3072 60 -> 38, 12288
// 81 -> 91.
#pragma once

#include "czip_attn_tile.h"

namespace czip {

// DPP moves of the wave64 scans: lanes whose source is out of range, and rows
// outside the row mask, read `old`
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned dpp_mov(unsigned old, unsigned x) {
    return (unsigned)__builtin_amdgcn_update_dpp((int)old, (int)x, CTRL, ROWS, 0xF, false);
}
constexpr int DPP_ROW_SHR = 0x110, DPP_WAVE_SHR1 = 0x138, DPP_BCAST15 = 0x142, DPP_BCAST31 = 0x143;

// inclusive scan over the 64 lanes; id: the operation's identity
template <class Op>
__device__ __forceinline__ unsigned wave_scan(unsigned x, unsigned id, Op op) {
    x = op(x, dpp_mov<DPP_ROW_SHR + 1, 0xF>(id, x));
    x = op(x, dpp_mov<DPP_ROW_SHR + 2, 0xF>(id, x));
    x = op(x, dpp_mov<DPP_ROW_SHR + 4, 0xF>(id, x));
    x = op(x, dpp_mov<DPP_ROW_SHR + 8, 0xF>(id, x));
    x = op(x, dpp_mov<DPP_BCAST15, 0xA>(id, x));
    x = op(x, dpp_mov<DPP_BCAST31, 0xC>(id, x));
    return x;
}

struct AttnRowLds {
    unsigned hi[16], lo[16];  // the tile's weights as offset bytes (^ WB), byte k of word b = key 4 b + k
};

// The row's state: everything but vacc is uniform over the wave.
struct AttnRow {
    unsigned m;     // running max (attn_m_empty / the tile's representation)
    unsigned S;     // weight sum
    unsigned vacc;  // lane = head dim
};

__device__ __forceinline__ unsigned uni(unsigned x) { return (unsigned)__builtin_amdgcn_readfirstlane((int)x); }

// q . k of 64 int8 as 16 words each (two chains)
__device__ __forceinline__ int dot64(const int* q, const v4i* k) {
    int a = 0, b = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        a = __builtin_amdgcn_sdot4(q[4 * i], k[i][0], a, false);
        b = __builtin_amdgcn_sdot4(q[4 * i + 1], k[i][1], b, false);
        a = __builtin_amdgcn_sdot4(q[4 * i + 2], k[i][2], a, false);
        b = __builtin_amdgcn_sdot4(q[4 * i + 3], k[i][3], b, false);
    }
    return a + b;
}

// The row before its first key (sink: the row's sink key, or nullptr).
template <bool GEN>
__device__ __forceinline__ AttnRow attn_row_begin(const int* q, const int8_t* sink, double mscale) {
    AttnRow r{(unsigned)attn_m_empty<GEN>(), 0u, 0u};
    if (sink) {  // attention.rs:211-224: the sink's score is the initial max, its weight E(0) = 65535
        v4i k[4];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) k[i][j] = ((const int*)sink)[4 * i + j];
        r.m = uni((unsigned)attn_sink_m<GEN>(dot64(q, k), mscale));
        r.S = 65535u;
    }
    return r;
}

// One tile of 64 keys, the first nkeys (1..64, uniform) of them visible.
// q: the query's 16 words.  k: the lane's key (64 bytes).  v[b]: keys 4 b ..
// 4 b + 3 of head dim `lane`.
template <bool GEN>
__device__ __forceinline__ void attn_row_tile(const int* q, const v4i (&k)[4], const int (&v)[16], double mscale, int nkeys,
                                              const uint16_t* etb, AttnRowLds& W, AttnRow& st) {
    const int lane = threadIdx.x & 63;
    const bool vis = lane < nkeys;
    const unsigned none = (unsigned)attn_m_empty<GEN>();
    const int dot = dot64(q, k);
    unsigned s = GEN ? (unsigned)score_g(dot, mscale) : score_u(dot, mscale * 0.25, score_bias_u(mscale));
    s = vis ? s : none;  // never a record; its weight is 0 below
    auto vmax = [](unsigned a, unsigned b) { return GEN ? (unsigned)max((int)a, (int)b) : max(a, b); };
    const unsigned incl = wave_scan(s, none, vmax);
    const unsigned M = vmax(st.m, dpp_mov<DPP_WAVE_SHR1, 0xF>(none, incl));  // max before the lane's key
    const bool rec = GEN ? (int)s > (int)M : s > M;
    unsigned x;  // E(-|s - M|): the weight, or at a record the rescale factor
    if (GEN) {
        const int d = (int)(rec ? M - s : s - M);  // i32 wrap, as the reference
        const unsigned e = (unsigned)etb[exp_step_g(0u - (unsigned)d)] ^ WB;
        x = d >= 0 ? 65535u : e;
    } else {
        x = (unsigned)etb[exp_step_u(s > M ? s - M : M - s)] ^ WB;
    }
    const unsigned w = !vis ? 0u : (rec ? 65535u : x);
    // segments split at the records that rescale (one over "nothing seen" does not)
    const unsigned long long spl = __builtin_amdgcn_ballot_w64(rec && M != none);
    st.m = vmax(st.m, (unsigned)__builtin_amdgcn_readlane((int)incl, 63));
    ((uint8_t*)W.hi)[lane] = (uint8_t)((w ^ WB) >> 8);
    ((uint8_t*)W.lo)[lane] = (uint8_t)(w ^ WB);
    const unsigned wsum = wave_scan(w, 0u, [](unsigned a, unsigned b) { return a + b; });
    wave_lds_fence();
    unsigned hi[16], lo[16];
#pragma unroll
    for (int b = 0; b < 4; b++) {
        const uint4 h = ((const uint4*)W.hi)[b], l = ((const uint4*)W.lo)[b];
        hi[4 * b] = h.x; hi[4 * b + 1] = h.y; hi[4 * b + 2] = h.z; hi[4 * b + 3] = h.w;
        lo[4 * b] = l.x; lo[4 * b + 1] = l.y; lo[4 * b + 2] = l.z; lo[4 * b + 3] = l.w;
    }
    // the segment being summed: sums of hi v, lo v and v over its blocks (a
    // block's keys outside the segment carry w = 0, bytes -128), and the
    // weight sum before it
    int ah = 0, al = 0, vs = 0;
    unsigned before = 0u;
#pragma unroll
    for (int b = 0; b < 16; b++) {
        if (4 * b >= nkeys) break;
        unsigned nib = (unsigned)(spl >> (4 * b)) & 15u;
        unsigned h = hi[b], l = lo[b];
        const int bs = __builtin_amdgcn_sdot4(v[b], 0x01010101, 0, false);
        while (nib) {  // a record at key kk of the block: its earlier keys end the segment
            const int kk = __builtin_ctz(nib), key = 4 * b + kk;
            nib &= nib - 1u;
            const unsigned msk = (1u << (8 * kk)) - 1u;
            ah = __builtin_amdgcn_sdot4(v[b], (int)pick(msk, h, 0x80808080u), ah, false);
            al = __builtin_amdgcn_sdot4(v[b], (int)pick(msk, l, 0x80808080u), al, false);
            h = pick(msk, 0x80808080u, h);
            l = pick(msk, 0x80808080u, l);
            const unsigned e = (unsigned)__builtin_amdgcn_readlane((int)x, key);
            const unsigned ws = key > 0 ? (unsigned)__builtin_amdgcn_readlane((int)wsum, key - 1) : 0u;
            st.vacc = rescale_v(st.vacc + ((unsigned)ah << 8) + (unsigned)al + (unsigned)(vs + bs) * WOFF, e);
            st.S = rescale_s(st.S + (ws - before), e);
            before = ws;
            ah = al = vs = 0;
        }
        ah = __builtin_amdgcn_sdot4(v[b], (int)h, ah, false);
        al = __builtin_amdgcn_sdot4(v[b], (int)l, al, false);
        vs += bs;
    }
    st.vacc += ((unsigned)ah << 8) + (unsigned)al + (unsigned)vs * WOFF;
    st.S += (unsigned)__builtin_amdgcn_readlane((int)wsum, 63) - before;
}

// attn_normalize for the lane's head dim
__device__ __forceinline__ int8_t attn_row_out(const AttnRow& st) {
    const double den = (double)max(st.S, 1u);
    const double nf = (double)(int)st.vacc;
    const double q = __builtin_rint(nf * (1.0 / den));
    const double r2 = 2.0 * __builtin_fma(-q, den, nf);
    const int qi = (int)q;
    const int qt = __builtin_fabs(r2) == den ? (qi + (r2 > 0.0 ? 1 : 0)) & ~1 : qi;
    return (int8_t)clamp127(qt);
}

}  // namespace czip
