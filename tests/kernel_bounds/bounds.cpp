// Runs the GEMM, layer tail, whole-stream decode and prefill attention
// launches on the CPU with every buffer access checked (hip/hip_runtime.h of
// this folder).  The .hip sources are copies with their inline asm taken out.
#include <vector>

#include "czip_gemm.hip"
#include "czip_tail.hip"
#include "czip_decode_fused.hip"
#include "czip_attention.hip"

namespace czip {  // kernels that are not looked at here
void launch_rn_rows(const RowGemmArgs&, hipStream_t) {}
void launch_rn_splitk_epi(const RowGemmArgs&, const int32_t*, int, hipStream_t) {}
}  // namespace czip
using namespace czip;

namespace {
int8_t* const mem = (int8_t*)std::calloc(192, 1 << 20);  // plain loads and stores land here
int8_t* at(size_t mb) { return mem + (mb << 20); }

GemmArgs gemm_args(int M, int N, int K, int T) {
    GemmArgs g{};
    g.A = at(0); g.W = at(8); g.Wf = at(8); g.M = M; g.N = N; g.K = K; g.out32 = (int32_t*)at(64); g.out8 = at(64); g.ldo = N;
    g.rq_scale = 1.0; g.rq_fast = 1; g.d = K; g.T = T; g.TP = (T + 63) & ~63; g.kc = at(96); g.vc = at(112);
    g.vl = 4; g.kv_mode = 1; g.G = 1; g.KH = 1; g.pos = -1; g.rcos = (int16_t*)at(128); g.rsin = (int16_t*)at(130);
    return g;
}

// every projection of a layer of width d, by the kernel that the limits choose
void gemms(int M, int d, int F, int T, int skinny, int wide) {
    for (int epi : {EPI_QKV, EPI_REGLU, EPI_RAW, EPI_REQ}) {
        GemmArgs g = gemm_args(M, epi == EPI_QKV ? d + 128 : epi == EPI_REGLU ? 2 * F : epi == EPI_RAW ? 1088 : d, d, T);
        if (epi == EPI_QKV) g.ldo = d;
        g.skinny_rows = skinny; g.wide_rows = wide;
        launch_gemm(g, epi, nullptr);
    }
    for (int K : {d, F}) {
        RowGemmArgs a{};
        a.A = at(0); a.W = at(8); a.Wf = at(8); a.M = M; a.K = K; a.d = d; a.rq_scale = 1.0; a.rq_fast = 1;
        a.w1 = a.w2 = at(60); a.x_in = a.x_out = (int16_t*)at(64); a.xn = at(96); a.y8 = at(112); a.ws = nullptr;
        a.skinny_rows = skinny; a.wide_rows = wide;
        launch_gemm_rn(a, nullptr);
    }
}

void tail(int M, int d, int F, bool qkv) {
    TailArgs t{};
    t.attn = at(0); t.M = M; t.F = F; t.out_wf = at(8); t.up_wf = at(8); t.down_wf = at(8);
    t.o_scale = t.up_scale = t.dn_scale = 1.0;
    t.w_ffn = t.w_post_attn = t.w_post_ffn = t.w_next = at(60);
    t.x_in = t.x_out = (int16_t*)at(64);
    if (qkv) {
        t.qkv = gemm_args(M, d + 128, d, 64);
        t.qkv.pos = 3; t.qkv.vl = 2; t.qkv.ldo = d;
    } else {
        t.xn = at(112);
    }
    launch_layer_tail(t, d, nullptr);
}

void fused(int S, int d, int F) {
    FusedDecArgs f{};
    std::vector<int64_t> zero((size_t)S, 0);
    std::vector<int32_t> len((size_t)S, 8), ntok((size_t)S, 3);
    f.ds = DecStreams{(const uint8_t*)at(60), zero.data(), len.data(), ntok.data(), (uint32_t*)at(160), zero.data()};
    f.S = S; f.TP = 64; f.KH = 1; f.NKV = 1; f.kv_mode = 1; f.G = 1; f.qkv_n = d + 128; f.F = F;
    f.tab = at(0); f.embed = at(0); f.rcos = (int16_t*)at(128); f.rsin = (int16_t*)at(130); f.kc = at(96); f.vc = at(112);
    f.score_mult = (const int32_t*)at(60); f.etab = (const uint16_t*)at(61); f.lut = (const uint16_t*)at(62);
    f.out_wf = f.up_wf = f.down_wf = f.head_wf = at(8);
    f.o_scale = f.up_scale = f.dn_scale = 1.0;
    f.w_ffn = f.w_post_attn = f.w_post_ffn = f.w_final = at(60);
    f.coef = 378194u; f.total = 1u << 24;
    launch_decode_fused(f, d, false, nullptr);
}

void attention(int B, int T, int H) {
    std::vector<int32_t> lens((size_t)B, T);
    AttnArgs a{};
    a.q = at(0); a.kc = at(96); a.vc = at(112); a.TP = (T + 63) & ~63; a.lens = lens.data(); a.score_mult = (const int32_t*)at(60);
    a.etab = (const uint16_t*)at(61); a.out = at(64); a.M = B * T; a.T = T; a.H = H; a.G = 1; a.KH = 1; a.kv_mode = 1; a.coef = 378194u;
    launch_attention(a, B, nullptr);
}
}  // namespace

int main(int argc, char** argv) {
    if (argc < 2) return 2;
    std::vector<int> v;
    for (int i = 2; i < argc; i++) v.push_back(std::atoi(argv[i]));
    v.resize(6);
    if (!std::strcmp(argv[1], "gemms")) gemms(v[0], v[1], v[2], v[3], v[4], v[5]);
    else if (!std::strcmp(argv[1], "tail")) tail(v[0], v[1], v[2], v[3] != 0);
    else if (!std::strcmp(argv[1], "fused")) fused(v[0], v[1], v[2]);
    else if (!std::strcmp(argv[1], "attention")) attention(v[0], v[1], v[2]);
    else if (!std::strcmp(argv[1], "tail_rounds")) return std::printf("%d\n", tail_rounds_pay(v[0], v[1], (size_t)v[2], v[3], v[4])) < 0;
    else return 2;
    std::printf("%ld accesses, %ld bad\n", bounds::accesses, bounds::bad);
    return bounds::bad ? 1 : 0;
}
