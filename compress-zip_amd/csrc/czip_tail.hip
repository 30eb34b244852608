// The rest of a layer after its attention in one launch (model.rs:423-468):
// output projection, residual + norms, up projection, ReGLU, down projection,
// residual + norms, and for decode steps the next layer's Q/K/V.
//
// As five launches a step of a few thousand rows is bound by each launch's own
// start: its weights arrive from the memory behind the L2 at the latency of
// what one CU has in flight, and the rows go out and come back in between.
// Here a workgroup takes 16 or 32 rows through all of it: only the attention
// output and the residual come in, only the residual (and the next layer's
// Q/K/V or the normalized rows) go out.  Every workgroup streams all of the
// layer's weights (3.7 MB for d512, 1.3 MB for the shipped model) from its
// XCD's L2 at 135 GB/s, which is what bounds it; the first workgroups touch a
// share of them each as they start, so that they are in the L2 before they are
// streamed (streaming them cold, in step, a workgroup gets 69 GB/s).  So it
// pays where a layer's weights fit an L2, between the few rows at which
// spreading the columns over the chip is faster and the many at which the
// strip-wise kernels reuse each weight for more rows.
//
// Eight waves; wave w owns output columns [w d/8, (w+1) d/8) of both d-wide
// projections, so that the residual stays in its registers in between.  A phase's
// first weights are requested before the norms or the barrier in front of it.
// d512, 4096 rows: 48 us a launch (events included) for the 66 of the four
// kernels it replaces, 28 of them the weights' stream at 135 GB/s a CU.
#include <algorithm>

#include "czip_device.h"
#include "czip_gemm_epi.h"
#include "czip_kernels.h"

namespace czip {

namespace {

constexpr int TNW = 8;
constexpr int TAIL_R8_BYTES = 64 << 10;  // ReGLU rows in LDS: 16 RT F bytes

// one 128-byte line of share `s` of `ns` of a weight array (past its end: nothing is read)
__device__ __forceinline__ int touch(__amdgpu_buffer_rsrc_t r, int u, int s, int ns, int tid) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, ((u * ns + s) * 64 * TNW + tid) << 7, 0, 0);
}

}  // namespace

// KS: K steps of 64 of the model width d; RT: row tiles of 16; QKV: the next layer's projection follows
template <int KS, int RT, bool QKV>
__global__ __launch_bounds__(64 * TNW) void k_layer_tail(TailArgs a) {
    constexpr int D = 64 * KS, CT = KS / 2, R = 16 * RT;
    constexpr int P = CT <= 3 ? 5 : 4;  // K steps of the down projection's weights in flight
    __shared__ __attribute__((aligned(16))) int8_t As[KS][R * 64];  // attention rows, then normalized rows (lds64 rows)
    __shared__ __attribute__((aligned(16))) int8_t r8[TAIL_R8_BYTES / 16 / R * 16 * R];
    __shared__ unsigned red[2][TNW][R];  // the two norms' row sums (a norm's reads end before the one after next writes)
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, grp = lane >> 4, c4 = grp * 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m0 = (int)blockIdx.x * R;
    const int nb = wave * CT * 16;
    const int nk = a.F / 64;
    const __amdgpu_buffer_rsrc_t r_out = weights_rsrc(a.out_wf, D * D), r_up = weights_rsrc(a.up_wf, 2 * a.F * D),
                                 r_down = weights_rsrc(a.down_wf, a.F * D);

    // the rows' attention output, the output projection's weights, the residual and the norm weights
    {
        const __amdgpu_buffer_rsrc_t rA =
            __builtin_amdgcn_make_buffer_rsrc((void*)(a.attn + (size_t)m0 * D), (short)0, min(a.M - m0, R) * D, BUF_DWORD3);
        // piece c: row c / (4 KS), 16-byte piece c % (4 KS) of it (rows past M read 0)
        for (int c = tid; c < R * 4 * KS; c += 64 * TNW) {
            const int row = c / (4 * KS), pc = c - row * 4 * KS;
            const v4i x = __builtin_amdgcn_raw_buffer_load_b128(rA, row * D + pc * 16, 0, 0);
            *(v4i*)(As[pc >> 2] + lds64(row, pc & 3)) = x;
        }
    }
    v4i wo[CT][KS];
#pragma unroll
    for (int t = 0; t < CT; t++) load_ops(wo[t], r_out, (wave * CT + t) * KS, lane);
    int x[RT][CT][4];
    unsigned w1[2][CT], w2[2][CT];
    {
        uint2 xr[RT][CT];
#pragma unroll
        for (int i = 0; i < RT; i++) {
            const int row = min(m0 + i * 16 + lr, a.M - 1);
            const int8_t* erow = a.x_in ? nullptr : a.embed + (size_t)a.tok[row] * D;
#pragma unroll
            for (int t = 0; t < CT; t++) {
                const int n = nb + t * 16 + c4;
                xr[i][t] = a.x_in ? *(const uint2*)(a.x_in + (size_t)row * D + n) : make_uint2(*(const unsigned*)(erow + n), 0u);
            }
        }
#pragma unroll
        for (int t = 0; t < CT; t++) {
            const int n = nb + t * 16 + c4;
            w1[0][t] = *(const unsigned*)(a.w_ffn + n);
            w2[0][t] = *(const unsigned*)(a.w_post_attn + n);
            w1[1][t] = *(const unsigned*)(a.w_post_ffn + n);
            w2[1][t] = *(const unsigned*)(a.w_next + n);
        }
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int t = 0; t < CT; t++) {
                if (a.x_in) {
                    x[i][t][0] = (int16_t)(xr[i][t].x & 0xFFFFu); x[i][t][1] = (int16_t)(xr[i][t].x >> 16);
                    x[i][t][2] = (int16_t)(xr[i][t].y & 0xFFFFu); x[i][t][3] = (int16_t)(xr[i][t].y >> 16);
                } else {
                    unpack4s(xr[i][t].x, x[i][t]);
                }
            }
    }
    // a share of the weights ahead of their streaming, 64 KB a workgroup and
    // request: with 32 workgroups an XCD up to 4 MB of the up rows (the second
    // request lies past those of most models), 2 MB each of the others
    int touched[4] = {0, 0, 0, 0};
    const int tns = min((int)gridDim.x, 256) >> 3, ts = (int)blockIdx.x >> 3;
    if (ts < tns) {
        touched[0] = touch(r_up, 0, ts, tns, tid);
        touched[1] = touch(r_up, 1, ts, tns, tid);
        touched[2] = touch(r_down, 0, ts, tns, tid);
        if (QKV) touched[3] = touch(weights_rsrc(a.qkv.Wf, a.qkv.N * D), 0, ts, tns, tid);
    }

    // x += rmsnorm(requant(acc), w1); rmsnorm(clamp(x), w2) into As and, with
    // `out`, to the rows of out (the epilogue of the row GEMMs)
    auto norms = [&](v4i (&acc)[RT][CT], double scale, const unsigned (&wa)[CT], const unsigned (&wb)[CT], int8_t* out) {
        // every wave forms its rows' inverse RMS itself: one barrier a norm
        auto row_inv = [&](int which, double (&inv)[RT]) {
            lds_barrier();
#pragma unroll
            for (int i = 0; i < RT; i++) {
                unsigned s = 0;
#pragma unroll
                for (int w = 0; w < TNW; w++) s += red[which][w][i * 16 + lr];
                inv[i] = (double)inv_rms_q15_fast((int)(s / (unsigned)D) + 1) * (1.0 / 32768.0);  // eps_scaled = 1 (rmsnorm.rs:80-83)
            }
        };
        auto row_sum = [&](int which, int i, unsigned ss) {
            ss += (unsigned)__shfl_xor((int)ss, 16, 64);
            ss += (unsigned)__shfl_xor((int)ss, 32, 64);
            if (lane < 16) red[which][wave][i * 16 + lane] = ss;
        };
        double inv[RT];
#pragma unroll
        for (int i = 0; i < RT; i++) {
            unsigned ss = 0;
#pragma unroll
            for (int t = 0; t < CT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int y = clamp127(rint_fma_i32((double)acc[i][t][r], scale));
                    acc[i][t][r] = y;
                    ss += (unsigned)__mul24(y, y);
                }
            row_sum(0, i, ss);
        }
        row_inv(0, inv);
#pragma unroll
        for (int i = 0; i < RT; i++) {
            unsigned ss = 0;
#pragma unroll
            for (int t = 0; t < CT; t++) {
                int w[4];
                unpack4s(wa[t], w);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    x[i][t][r] += rms_el(acc[i][t][r], w[r], inv[i]);
                    const int c = clamp127(x[i][t][r]);
                    ss += (unsigned)__mul24(c, c);
                }
            }
            row_sum(1, i, ss);
        }
        row_inv(1, inv);
#pragma unroll
        for (int i = 0; i < RT; i++) {
            const int row = m0 + i * 16 + lr;
#pragma unroll
            for (int t = 0; t < CT; t++) {
                const int n = nb + t * 16 + c4;
                int w[4], o[4];
                unpack4s(wb[t], w);
#pragma unroll
                for (int r = 0; r < 4; r++) o[r] = rms_el(clamp127(x[i][t][r]), w[r], inv[i]);
                const unsigned v = pack4i(o[0], o[1], o[2], o[3]);
                *(unsigned*)(As[n >> 6] + lds64(i * 16 + lr, (n >> 4) & 3) + (n & 15)) = v;
                if (out && row < a.M) *(unsigned*)(out + (size_t)row * D + n) = v;
            }
        }
    };

    // column pairs (16 columns and the 16 that lie 32 further) of a projection
    // of the normalized rows, the pair after next requested ahead
    auto pair_mma = [&](const v4i (&wa)[KS], const v4i (&wb)[KS], v4i (&ya)[RT], v4i (&yb)[RT]) {
#pragma unroll
        for (int i = 0; i < RT; i++) {
            ya[i] = yb[i] = (v4i){0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const v4i af = *(const v4i*)(As[s] + lds64(i * 16 + lr, grp));
                ya[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa[s], af, ya[i], 0, 0, 0);
                yb[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wb[s], af, yb[i], 0, 0, 0);
            }
        }
    };
    auto load_pair = [&](v4i (&wa)[KS], v4i (&wb)[KS], __amdgpu_buffer_rsrc_t rw, int g, int np) {
        g = min(g, np - 1);  // past the last pair: the last one, unused
        const int pc = ((g >> 1) * 4 + (g & 1)) * KS;
        load_ops(wa, rw, pc, lane);
        load_ops(wb, rw, pc + 2 * KS, lane);
    };
    v4i wa[2][KS], wb[2][KS];  // the wave's first pair is requested by the caller
    auto pairs = [&](__amdgpu_buffer_rsrc_t rw, int np, auto emit) {
        auto load = [&](int u, int g) { load_pair(wa[u], wb[u], rw, g, np); };
        lds_barrier();
        for (int g = wave; g < np; g += 2 * TNW) {
            v4i ya[RT], yb[RT];
            load(1, g + TNW);
            pair_mma(wa[0], wb[0], ya, yb);
            emit(g, ya, yb);
            if (g + TNW >= np) break;
            load(0, g + 2 * TNW);
            pair_mma(wa[1], wb[1], ya, yb);
            emit(g + TNW, ya, yb);
        }
    };
    __syncthreads();
    {
        v4i acc[RT][CT];
#pragma unroll
        for (int i = 0; i < RT; i++) {
#pragma unroll
            for (int t = 0; t < CT; t++) acc[i][t] = (v4i){0, 0, 0, 0};
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const v4i af = *(const v4i*)(As[s] + lds64(i * 16 + lr, grp));
#pragma unroll
                for (int t = 0; t < CT; t++) acc[i][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wo[t][s], af, acc[i][t], 0, 0, 0);
            }
        }
        load_pair(wa[0], wb[0], r_up, wave, a.F / 16);  // in flight during the norms
        norms(acc, a.o_scale, w1[0], w2[0], nullptr);
    }

    pairs(r_up, a.F / 16, [&](int g, const v4i (&ya)[RT], const v4i (&yb)[RT]) {
#pragma unroll
        for (int i = 0; i < RT; i++) {
            int o[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int gv = max(clamp127(rint_fma_i32((double)ya[i][r], a.up_scale)), 0);
                o[r] = clamp127(rne_shr(gv * clamp127(rint_fma_i32((double)yb[i][r], a.up_scale)), 7));  // reglu.rs:20-46
            }
            *(unsigned*)(r8 + (g >> 2) * R * 64 + lds64(i * 16 + lr, g & 3) + c4) = pack4i(o[0], o[1], o[2], o[3]);
        }
    });

    // down projection: P K steps of the wave's columns in flight
    {
        v4i acc[RT][CT], w[P][CT];
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
            for (int t = 0; t < CT; t++) acc[i][t] = (v4i){0, 0, 0, 0};
        auto load = [&](v4i (&d)[CT], int kt) {
            kt = min(kt, nk - 1);  // past the last step: the last one, unused
#pragma unroll
            for (int t = 0; t < CT; t++)
                d[t] = __builtin_amdgcn_raw_buffer_load_b128(r_down, lane * 16, ((wave * CT + t) * nk + kt) * 1024, 0);
        };
#pragma unroll
        for (int u = 0; u < P - 1; u++) load(w[u], u);
        lds_barrier();
        for (int k0 = 0; k0 < nk; k0 += P) {
#pragma unroll
            for (int u = 0; u < P; u++) {
                const int kt = k0 + u;
                if (kt >= nk) break;
                load(w[(u + P - 1) % P], kt + P - 1);
#pragma unroll
                for (int i = 0; i < RT; i++) {
                    const v4i af = *(const v4i*)(r8 + kt * R * 64 + lds64(i * 16 + lr, grp));
#pragma unroll
                    for (int t = 0; t < CT; t++) acc[i][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[u][t], af, acc[i][t], 0, 0, 0);
                }
            }
        }
        if (QKV) load_pair(wa[0], wb[0], weights_rsrc(a.qkv.Wf, a.qkv.N * D), wave, a.qkv.N / 32);
        norms(acc, a.dn_scale, w1[1], w2[1], a.xn);
    }
    if (a.x_out) {
#pragma unroll
        for (int i = 0; i < RT; i++) {
            const int row = m0 + i * 16 + lr;
            if (row < a.M)
#pragma unroll
                for (int t = 0; t < CT; t++)
                    *(uint2*)(a.x_out + (size_t)row * D + nb + t * 16 + c4) =
                        make_uint2(((unsigned)x[i][t][0] & 0xFFFFu) | ((unsigned)x[i][t][1] << 16),
                                   ((unsigned)x[i][t][2] & 0xFFFFu) | ((unsigned)x[i][t][3] << 16));
        }
    }
    if constexpr (QKV) {
        QkvRow qr[RT];
#pragma unroll
        for (int i = 0; i < RT; i++) qkv_row(a.qkv, m0 + i * 16 + lr, c4, qr[i]);
        pairs(weights_rsrc(a.qkv.Wf, a.qkv.N * D), a.qkv.N / 32, [&](int g, const v4i (&ya)[RT], const v4i (&yb)[RT]) {
#pragma unroll
            for (int i = 0; i < RT; i++) {
                const int row = m0 + i * 16 + lr;
                if (row < a.M) epi_pair<EPI_QKV, true>(a.qkv, ya[i], yb[i], row, (g >> 1) * 64, g & 1, c4, qr[i]);
            }
        });
    }
    // the touched lines' loads have a use
    asm volatile("" ::"v"(touched[0]), "v"(touched[1]), "v"(touched[2]), "v"(touched[3]));
}

static int tail_rt(int M, int F) { return M > 16 * 256 && 32 * F <= TAIL_R8_BYTES ? 2 : 1; }

bool tail_supported(int d, int F) { return (d == 256 || d == 384 || d == 512) && F % 64 == 0 && 16 * F <= TAIL_R8_BYTES; }

// A workgroup's time is the weights' stream whatever its rows, so past one round
// of the 256 CUs the tail loses where the next round is nearly empty, the more
// the larger the weights.  Rows of a round: 8192, or 4096 where a feed-forward
// past 2048 leaves LDS for 16 rows a workgroup only.  4 to 8 layers, separate
// kernels -> tail:
//  - 16 rows only: up to one round and the fuller half of the second.  d384 / F =
//    3072 prefill 4096 rows 462 -> 438 us, 4200 510 -> 583, 6400 625 -> 596, 8192 647
//    -> 622, 8400 665 -> 770; 32 decode steps 4200 10.7 -> 13.2 ms, 6400 14.3 -> 13.5,
//    8400 15.7 -> 19.1; d256 / 4096 prefill 12288 570 -> 587, 20480 791 -> 862
//  - more than 3 MB (d512 / 2048): prefills up to one round (8192 rows 1.28 -> 1.08
//    ms, 8320 1.30 -> 1.43, 12288 1.48 -> 1.55, 18432 2.17 -> 2.15); decode steps
//    not in the emptier half of the second (8200 33.8 -> 35.0 ms, 11000 37.4 ->
//    37.7, 13300 40.9 -> 39.6, 16500 57.5 -> 56.5)
//  - 2 to 3 MB: prefills likewise without that half (d512 / 1536 8320 rows 739 ->
//    769 us, 12288 831 -> 834, 16640 1093 -> 1058; d384 / 2048 8200 596 -> 605, 13300
//    662 -> 646), decode steps all (d512 / 1024 8200 14.4 -> 13.8 ms)
//  - less: all (shipped model 8200 rows 253 -> 243 us, 16500 306 -> 295)
// Beside other decode lanes, whose kernels fill the separate ones' last rounds,
// only with weights of up to 2 MB (32 steps of 40 thousand streams in two lanes:
// d512 / 2048, 8 layers 91.1 -> 97.5 ms, d384 / 2048 37.8 -> 40.8, d512 / 1024 38.9 ->
// 40.0; shipped model 7.69 -> 7.42, d256 / 1024 21.3 -> 20.8).
static constexpr size_t TAIL_WEIGHTS_LARGE = (size_t)3 << 20, TAIL_WEIGHTS_MEDIUM = (size_t)2 << 20;
bool tail_rounds_pay(int64_t M, int F, size_t weights, bool decode, bool lanes) {
    if (lanes && weights > TAIL_WEIGHTS_MEDIUM) return false;
    if (F > 2048) return M <= 4096 || (M >= 6144 && M <= 8192);
    if (M <= 8192 || weights <= TAIL_WEIGHTS_MEDIUM) return true;
    if (weights <= TAIL_WEIGHTS_LARGE) return decode || M >= 12288;
    return decode && M >= 12288;
}

template <int KS>
static void launch_tail(const TailArgs& a, hipStream_t s) {
    const int rt = tail_rt(a.M, a.F);
    const dim3 grid((unsigned)((a.M + 16 * rt - 1) / (16 * rt)));
    const bool qkv = a.qkv.Wf != nullptr;
    if (rt == 1 && qkv) hipLaunchKernelGGL((k_layer_tail<KS, 1, true>), grid, dim3(64 * TNW), 0, s, a);
    else if (rt == 1) hipLaunchKernelGGL((k_layer_tail<KS, 1, false>), grid, dim3(64 * TNW), 0, s, a);
    else if (qkv) hipLaunchKernelGGL((k_layer_tail<KS, 2, true>), grid, dim3(64 * TNW), 0, s, a);
    else hipLaunchKernelGGL((k_layer_tail<KS, 2, false>), grid, dim3(64 * TNW), 0, s, a);
}

void launch_layer_tail(const TailArgs& a, int d, hipStream_t s) {
    if (a.M <= 0) return;
    if (d == 256) launch_tail<4>(a, s);
    else if (d == 384) launch_tail<6>(a, s);
    else launch_tail<8>(a, s);
}

}  // namespace czip
