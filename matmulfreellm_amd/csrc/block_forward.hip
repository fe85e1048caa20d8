// One HGRNBit block (mmfreelm/models/hgrn_bit/modeling_hgrn_bit.py:97-111) over B sequences of T tokens as ONE host call: the
// launches of the module path, in its order, with every elementwise op folded into the BitLinear next to it.
//
// Host code only.  Short prompts are bound by what it costs to issue a launch: through nn.Module calls, output allocations and
// one foreign-function call per kernel a 24-layer forward of 77 tokens spent 8.9 ms on the host and 1.6 ms on the GPU.  Here a
// layer costs one foreign-function call, and its buffers are offsets into one workspace.
#include "mmf_common.h"

namespace {

constexpr int64_t kGemvRows = 8;      // rows up to which every workgroup of a BitLinear redoes the row's prologue (one launch)

// prologue / epilogue ids of mmf_bitlinear_gemv_fused and mmf_rmsnorm_quant_fused
enum { G_PLAIN = 0, G_NORM = 1, G_RESNORM = 2, G_GATEDNORM = 3, E_PLAIN = 0, E_STEP = 1, E_SWIGLU = 2 };
enum { Q_PLAIN = 0, Q_NORM = 1, Q_RESNORM = 2, Q_STEP_GATE = 3, Q_SWIGLU = 4, Q_GATEDNORM = 5 };

int64_t esize(const mmf_block* p) { return p->dtype == MMF_F32 ? 4 : 2; }
bool few_rows(const mmf_block* p, int64_t M) {
    const int64_t k = p->H > p->I ? p->H : p->I;
    return M <= kGemvRows && (k > p->D ? k : p->D) <= mmf_bitlinear_gemv_max_k();
}

// The quantisers of middle-sized prompts bring the weights behind them (the packed bytes of [n, k], n a multiple of 32) into the last-level
// cache: a contraction that finds them in memory waits for each of its first k-blocks.  us a launch at the 1.3B shape, weights in memory and in the
// cache: 459 rows, i/f/g 13.4 and 12.4, o 7.0 and 6.2, gate/up 19.9 and 18.5, down 13.0 and 11.9; 1377 rows 25.8 / 25.0, 13.2 / 11.7, 33.4 / 32.8,
// 23.6 / 20.5.  The quantiser, 8 to 9 us of 1377 rows, takes 0.1 to 0.5 us more, memory's time for the weights.  Forwards: 3 x 459 tokens 3630 -> 3530 us, 2 x 1001 with logits 4406 -> 4285,
// 270 tokens 1603 -> 1576, 2 x 2000 6398 -> 6320; 370M shape, 4 x 700 2781 -> 2754.  With fewer rows the quantiser is as short as memory's answer (a
// decode step of 64 rows 0.5 to 5 % longer, however the touches were spread over its launches); with 8192 and 16384, rounds of tiles hide
// the start and the touches only delay the rows (1 to 2 % of a forward).
constexpr int64_t kAheadMinRows = 256, kAheadMaxRows = 5120;
struct Ahead { const void* p; int64_t bytes; };
Ahead ahead(const void* packed, int64_t n, int64_t k, int64_t M) {
    return M > kAheadMinRows && M <= kAheadMaxRows ? Ahead{packed, n * mmf_round_up(k, 128) / 4} : Ahead{nullptr, 0};
}

// What the i/f/g projections contract: codes of x under the block norm and their inner norm(s), q [1 or 3], deq, qsum.
int project_ifg(const mmf_block* p, const void* x, int64_t M, int8_t* q, float* deq, int* qsum, void* ifg, void* stream) {
    const int64_t H = p->H, D = p->D;
    const int dt = p->dtype, wt = p->weight_dtype;
    const Ahead w = ahead(p->ifg_packed, 3 * D, H, M);
    if (p->f_norm) {
        if (const int rc = mmf_rmsnorm_quant_multi_ahead(x, H, p->attn_norm, p->attn_eps, p->i_norm, p->f_norm, p->g_proj_norm, p->ifg_eps, q,
                                                         deq, qsum, M, H, w.p, w.bytes, dt, wt, stream))
            return rc;
        return mmf_bitlinear_mfma_multi(q, mmf_codes_bytes(M, H, 1), deq, qsum, p->ifg_packed, p->ifg_wdeq, D, ifg, 3 * D, M, H, 3 * D, dt,
                                        -1, stream);
    }
    if (const int rc = mmf_rmsnorm_quant_fused_ahead(Q_NORM, x, H, nullptr, 0, nullptr, 0, nullptr, p->attn_norm, p->attn_eps, p->i_norm,
                                                     p->ifg_eps, nullptr, nullptr, q, deq, qsum, M, H, w.p, w.bytes, dt, wt, stream))
        return rc;
    return mmf_bitlinear_mfma(q, deq, qsum, p->ifg_packed, p->ifg_wdeq, D, nullptr, nullptr, ifg, 3 * D, M, H, 3 * D, dt, -1, stream);
}

// Offsets of the intermediates in the workspace (each 256-byte aligned).
struct Layout {
    int64_t ifg = 0, o = 0, attn = 0, res, big = 0, q, deq, qsum, bytes = 0;
    Layout(const mmf_block* p, int64_t M, bool train) {
        const int64_t e = esize(p);
        auto take = [&](int64_t n) {
            const int64_t at = bytes;
            bytes += mmf_round_up(n, 256);
            return at;
        };
        res = take(M * p->H * e);
        if (!train) {                                            // training keeps these in tensors of the caller's
            attn = take(M * p->H * e);
            ifg = take(M * 3 * p->D * e);
            o = take(M * p->D * e);
            big = take(M * p->I * e);                            // the MLP's activation
        }
        int64_t codes = 3 * mmf_codes_bytes(M, p->H, 1);
        for (int64_t k : {(int64_t)p->D, (int64_t)p->I})
            if (mmf_codes_bytes(M, k, 1) > codes) codes = mmf_codes_bytes(M, k, 1);
        q = take(codes);
        deq = take(3 * M * 4);
        qsum = take(3 * M * 4);
    }
};

}  // namespace

extern "C" {

int64_t mmf_block_struct_bytes(void) { return (int64_t)sizeof(mmf_block); }

int64_t mmf_block_workspace_bytes(const mmf_block* p, int64_t rows) {
    if (!p || rows <= 0) return 0;
    return Layout(p, rows, false).bytes;
}

int64_t mmf_block_train_workspace_bytes(const mmf_block* p, int64_t rows) {
    if (!p || rows <= 0) return 0;
    return Layout(p, rows, true).bytes;
}

int mmf_block_train_forward(const mmf_block* p, const void* x, void* out, void* ifg, void* xg, void* o, void* attn, void* y, int64_t B,
                            int64_t T, const float* lower_bound, const uint8_t* mask, void* workspace, void* stream) {
    if (!p || B < 0 || T < 0 || p->H <= 0 || p->D <= 0 || p->I <= 0 || p->D % 32 || p->I % 32) return MMF_ERR_ARG;
    const int64_t M = B * T, H = p->H, D = p->D, I = p->I, e = esize(p);
    if (M == 0) return 0;
    if (!x || !out || !ifg || !xg || !o || !attn || !y || !workspace) return MMF_ERR_ARG;
    if (reinterpret_cast<uintptr_t>(workspace) & 255u) return MMF_ERR_ALIGN;
    const Layout L(p, M, true);
    char* w = static_cast<char*>(workspace);
    void* res = w + L.res;
    int8_t* q = reinterpret_cast<int8_t*>(w + L.q);
    float* deq = reinterpret_cast<float*>(w + L.deq);
    int* qsum = reinterpret_cast<int*>(w + L.qsum);
    char *i = static_cast<char*>(ifg), *f = i + D * e, *g = i + 2 * D * e, *gs = static_cast<char*>(xg) + M * D * e;
    char* up = static_cast<char*>(y) + I * e;
    const int dt = p->dtype, wt = p->weight_dtype;
    const Ahead o_w = ahead(p->o_packed, H, D, M), gate_w = ahead(p->gate_packed, 2 * I, H, M), down_w = ahead(p->down_packed, H, I, M);
    int rc = 0;
#define MMF_DO(call)                \
    do {                            \
        if ((rc = (call))) return rc; \
    } while (0)
    MMF_DO(project_ifg(p, x, M, q, deq, qsum, ifg, stream));
    MMF_DO(mmf_hgrn_gate(i, 3 * D, f, 3 * D, lower_bound, mask, xg, gs, M, D, dt, stream));
    MMF_DO(mmf_hgrn_recurrent(xg, gs, nullptr, o, nullptr, B, T, D, dt, stream));
    MMF_DO(mmf_rmsnorm_quant_fused_ahead(Q_GATEDNORM, g, 3 * D, o, D, nullptr, 0, nullptr, p->g_norm, p->g_eps, p->o_norm, p->o_eps, nullptr,
                                         nullptr, q, deq, qsum, M, D, o_w.p, o_w.bytes, dt, wt, stream));
    MMF_DO(mmf_bitlinear_mfma(q, deq, qsum, p->o_packed, p->o_wdeq, p->o_seg_rows, nullptr, nullptr, attn, H, M, D, H, dt, -1, stream));
    MMF_DO(mmf_rmsnorm_quant_fused_ahead(Q_RESNORM, attn, H, x, H, nullptr, 0, res, p->mlp_norm, p->mlp_eps, p->gate_norm, p->gate_eps, nullptr,
                                         nullptr, q, deq, qsum, M, H, gate_w.p, gate_w.bytes, dt, wt, stream));
    MMF_DO(mmf_bitlinear_mfma(q, deq, qsum, p->gate_packed, p->gate_wdeq, p->gate_seg_rows, nullptr, nullptr, y, 2 * I, M, H, 2 * I, dt, -1,
                              stream));
    MMF_DO(mmf_rmsnorm_quant_fused_ahead(Q_SWIGLU, y, 2 * I, up, 2 * I, nullptr, 0, nullptr, nullptr, 0.0f, p->down_norm, p->down_eps, nullptr,
                                         nullptr, q, deq, qsum, M, I, down_w.p, down_w.bytes, dt, wt, stream));
    MMF_DO(mmf_bitlinear_mfma(q, deq, qsum, p->down_packed, p->down_wdeq, p->down_seg_rows, nullptr, res, out, H, M, I, H, dt, -1, stream));
#undef MMF_DO
    return 0;
}

int mmf_block_forward(const mmf_block* p, const void* x, void* out, int64_t B, int64_t T, const float* lower_bound,
                      const uint8_t* mask, const float* h0, float* ht, void* workspace, void* stream) {
    if (!p || B < 0 || T < 0 || p->H <= 0 || p->D <= 0 || p->I <= 0 || p->D % 32 || p->I % 32) return MMF_ERR_ARG;
    const int64_t M = B * T, H = p->H, D = p->D, I = p->I, e = esize(p);
    if (M == 0) return 0;
    if (!x || !out || x == out || !workspace) return MMF_ERR_ARG;
    if (reinterpret_cast<uintptr_t>(workspace) & 255u) return MMF_ERR_ALIGN;
    const Layout L(p, M, false);
    char* w = static_cast<char*>(workspace);
    char* ifg = w + L.ifg;
    char *i = ifg, *f = ifg + D * e, *g = ifg + 2 * D * e;     // columns of the stacked projection, row stride 3 D
    void *o = w + L.o, *attn = w + L.attn, *res = w + L.res;
    char* big = w + L.big;
    int8_t* q = reinterpret_cast<int8_t*>(w + L.q);
    float* deq = reinterpret_cast<float*>(w + L.deq);
    int* qsum = reinterpret_cast<int*>(w + L.qsum);
    const int dt = p->dtype, wt = p->weight_dtype;
    const bool multi = p->f_norm != nullptr;                   // i, f and g have inner norms of their own
    const bool step = T == 1 && h0 && h0 == ht;                // one token on a kept state: gate math + recurrence step in one kernel
    const Ahead o_w = ahead(p->o_packed, H, D, M), gate_w = ahead(p->gate_packed, 2 * I, H, M), down_w = ahead(p->down_packed, H, I, M);
    int rc = 0;
#define MMF_DO(call)                \
    do {                            \
        if ((rc = (call))) return rc; \
    } while (0)
    auto scan = [&]() -> int {                                 // gate math, then the recurrence: o [M, D] contiguous
        if (step) return mmf_hgrn_step(i, 3 * D, f, 3 * D, lower_bound, mask, ht, o, M, D, dt, stream);
        return mmf_hgrn_gate_scan(i, 3 * D, f, 3 * D, lower_bound, mask, h0, o, ht, B, T, D, dt, stream);
    };
    if (few_rows(p, M)) {
        const int epi = step && !mask ? E_STEP : E_PLAIN;
        void* first = epi == E_STEP ? o : ifg;
        void* g_row = epi == E_STEP ? ifg : (void*)g;           // the raw g projection, row stride D or 3 D
        if (multi)
            MMF_DO(mmf_bitlinear_gemv_multi(epi, x, H, p->attn_norm, p->attn_eps, p->i_norm, p->f_norm, p->g_proj_norm, p->ifg_eps,
                                            p->ifg_packed, p->ifg_wdeq, D, first, ifg, lower_bound, ht, M, H, 3 * D, dt, wt,
                                            stream));
        else
            MMF_DO(mmf_bitlinear_gemv_fused(G_NORM, epi, x, H, nullptr, 0, nullptr, p->attn_norm, p->attn_eps, p->i_norm, p->ifg_eps,
                                            p->ifg_packed, p->ifg_wdeq, D, nullptr, nullptr, first, ifg, lower_bound, ht, M, H,
                                            3 * D, dt, wt, stream));
        if (epi != E_STEP) MMF_DO(scan());
        MMF_DO(mmf_bitlinear_gemv_fused(G_GATEDNORM, E_PLAIN, g_row, epi == E_STEP ? D : 3 * D, o, D, nullptr, p->g_norm, p->g_eps,
                                        p->o_norm, p->o_eps, p->o_packed, p->o_wdeq, p->o_seg_rows, nullptr, nullptr, attn, nullptr,
                                        nullptr, nullptr, M, D, H, dt, wt, stream));
        MMF_DO(mmf_bitlinear_gemv_fused(G_RESNORM, E_SWIGLU, attn, H, x, H, res, p->mlp_norm, p->mlp_eps, p->gate_norm, p->gate_eps,
                                        p->gate_packed, p->gate_wdeq, p->gate_seg_rows, nullptr, nullptr, big, nullptr, nullptr,
                                        nullptr, M, H, 2 * I, dt, wt, stream));
        MMF_DO(mmf_bitlinear_gemv_fused(G_PLAIN, E_PLAIN, big, I, nullptr, 0, nullptr, nullptr, 0.0f, p->down_norm, p->down_eps,
                                        p->down_packed, p->down_wdeq, p->down_seg_rows, nullptr, res, out, nullptr, nullptr, nullptr,
                                        M, I, H, dt, wt, stream));
        return 0;
    }
    MMF_DO(project_ifg(p, x, M, q, deq, qsum, ifg, stream));
    if (step && !mask) {
        MMF_DO(mmf_rmsnorm_quant_fused(Q_STEP_GATE, i, 3 * D, f, 3 * D, g, 3 * D, nullptr, p->g_norm, p->g_eps, p->o_norm, p->o_eps,
                                       lower_bound, ht, q, deq, qsum, M, D, dt, wt, stream));
    } else {
        MMF_DO(scan());
        MMF_DO(mmf_rmsnorm_quant_fused_ahead(Q_GATEDNORM, g, 3 * D, o, D, nullptr, 0, nullptr, p->g_norm, p->g_eps, p->o_norm, p->o_eps,
                                             nullptr, nullptr, q, deq, qsum, M, D, o_w.p, o_w.bytes, dt, wt, stream));
    }
    MMF_DO(mmf_bitlinear_mfma(q, deq, qsum, p->o_packed, p->o_wdeq, p->o_seg_rows, nullptr, nullptr, attn, H, M, D, H, dt, -1, stream));
    MMF_DO(mmf_rmsnorm_quant_fused_ahead(Q_RESNORM, attn, H, x, H, nullptr, 0, res, p->mlp_norm, p->mlp_eps, p->gate_norm, p->gate_eps, nullptr,
                                         nullptr, q, deq, qsum, M, H, gate_w.p, gate_w.bytes, dt, wt, stream));
    MMF_DO(mmf_bitlinear_mfma_swiglu(q, deq, qsum, p->gate_packed, p->gate_wdeq, p->gate_seg_rows, big, I, M, H, 2 * I, dt, stream));
    MMF_DO(mmf_rmsnorm_quant_fused_ahead(Q_PLAIN, big, I, nullptr, 0, nullptr, 0, nullptr, nullptr, 0.0f, p->down_norm, p->down_eps, nullptr,
                                         nullptr, q, deq, qsum, M, I, down_w.p, down_w.bytes, dt, wt, stream));
    MMF_DO(mmf_bitlinear_mfma(q, deq, qsum, p->down_packed, p->down_wdeq, p->down_seg_rows, nullptr, res, out, H, M, I, H, dt, -1, stream));
#undef MMF_DO
    return 0;
}

}  // extern "C"
