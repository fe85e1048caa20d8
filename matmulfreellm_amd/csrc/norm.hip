// One-pass row kernels: RMSNorm, RMSNorm * swish-gate, RMSNorm + int8 quantiser, swiglu.
//
// One workgroup of 256 threads owns one row; the row lives in registers (8-element
// vectors, up to NV per thread), sums of squares are reduced in fp64 with a wave64
// butterfly plus a 4-entry LDS exchange, so HBM sees each input once and each output
// once.  Replaces the Triton row kernels at mmfreelm/modules/layernorm.py:104-165,
// mmfreelm/modules/fused_norm_gate.py:68-131, mmfreelm/ops/fusedbitnet.py:63-131 and
// the jiterator kernel at mmfreelm/modules/activations.py:115-119.
#include "mmf_common.h"
#include <type_traits>
#include "../../include/mmf.h"

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;

enum RowMode : int { ROW_NORM = 0, ROW_GATE = 1, ROW_QUANT = 2 };

struct RowArgs {
    const void* x;          // [M, K]
    const void* residual;   // [M, K] or null            (dtype TR)
    const void* gate;       // [M, K] or null            (ROW_GATE, dtype T)
    const void* weight;     // [K] or null               (dtype TW)
    const void* bias;       // [K] or null: added after the weight (dtype TW)
    int center;             // LayerNorm: subtract the row mean before the variance (else RMSNorm)
    void* y;                // [M, K] T                  (ROW_NORM / ROW_GATE)
    void* residual_out;     // [M, K] TR or null
    int8_t* q;              // codes                     (ROW_QUANT)
    float* deq;             // [M]
    int* qsum;              // [M]
    int64_t M, K, Kp, ldx;   // ldx: row stride of x in elements
    double inv_K;            // RN(1 / K)
    float eps;
    int q_tiled;            // 0: row-major [M, Kp]; 1: [ceil32(M)/32][Kp/16][32][16]
};

template <typename T, typename TR, typename TW, int MODE, int NV>
__global__ __launch_bounds__(kThreads) void row_kernel(RowArgs a) {
    __shared__ double red_d[kWaves];
    __shared__ float red_f[kWaves];
    __shared__ int red_i[kWaves];

    const int64_t row = blockIdx.x;
    const int64_t K = a.K;
    const bool vec_ok = (K % 8) == 0;
    const T* x = static_cast<const T*>(a.x) + row * a.ldx;
    const TR* res = a.residual ? static_cast<const TR*>(a.residual) + row * K : nullptr;
    TR* res_out = a.residual_out ? static_cast<TR*>(a.residual_out) + row * K : nullptr;
    const TW* w = static_cast<const TW*>(a.weight);

    // Every global load of the row is issued up front (x, residual, norm weight, gate) so
    // their latencies overlap; the reductions below then run on registers only.
    float xv[NV][8];
    float wv[NV][8];
    float ov[MODE == ROW_GATE ? NV : 1][8];
    double ss = 0.0;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int64_t k0 = ((int64_t)v * kThreads + threadIdx.x) * 8;
        if (k0 < K) {
            if (w) mmf_load8<TW>(w, k0, K, vec_ok, wv[v]);
            if constexpr (MODE == ROW_GATE)
                mmf_load8<T>(static_cast<const T*>(a.gate) + row * K, k0, K, vec_ok, ov[v]);
        }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int64_t k0 = ((int64_t)v * kThreads + threadIdx.x) * 8;
        if (k0 < K) {
            mmf_load8<T>(x, k0, K, vec_ok, xv[v]);
            if (res) {
                float rv[8];
                mmf_load8<TR>(res, k0, K, vec_ok, rv);
#pragma unroll
                for (int i = 0; i < 8; ++i) xv[v][i] = __fadd_rn(xv[v][i], rv[i]);
            }
            if (res_out) mmf_store8<TR>(res_out, k0, K, vec_ok, xv[v]);
#pragma unroll
            for (int i = 0; i < 8; ++i) ss = mmf_add_square(ss, xv[v][i]);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) xv[v][i] = 0.0f;
        }
    }
    if (a.center) {
        // LayerNorm: mean = fp32(sum / K) with the sum in fp64; the variance is that of the fp32 differences
        double sx = 0.0;
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int i = 0; i < 8; ++i) sx += (double)xv[v][i];
        sx = mmf_block_sum<kWaves>(sx, red_d);
        const float mean = (float)mmf_quotient_by_count(sx, K, a.inv_K);
        ss = 0.0;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int64_t k0 = ((int64_t)v * kThreads + threadIdx.x) * 8;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                xv[v][i] = k0 + i < K ? __fsub_rn(xv[v][i], mean) : 0.0f;
                ss = mmf_add_square(ss, xv[v][i]);
            }
        }
    }
    ss = mmf_block_sum<kWaves>(ss, red_d);
    const float rstd = mmf_rstd(ss, K, a.inv_K, a.eps);

    float amax = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int64_t k0 = ((int64_t)v * kThreads + threadIdx.x) * 8;
        if (k0 < K) {
            float bv[8];
            if (a.bias) mmf_load8<TW>(static_cast<const TW*>(a.bias), k0, K, vec_ok, bv);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                float y = __fmul_rn(xv[v][i], rstd);
                if (w) y = __fmul_rn(y, wv[v][i]);
                if (a.bias) y = k0 + i < K ? __fadd_rn(y, bv[i]) : 0.0f;
                xv[v][i] = y;
                amax = fmaxf(amax, fabsf(y));
            }
            if constexpr (MODE == ROW_GATE) {
                float y[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) y[i] = xv[v][i];
                // fp16 falls back in most waves of 512 elements: rows of one vector a thread keep the definition (64 x 2048 3.8 us, near 5.4; 16384 x 2048
                // 51 and 63), longer ones where there are more rows than CUs (2002 x 2560 12.1 near, 13.2 exact; 64 x 2560 4.4 and 4.2)
                if (!std::is_same<T, f16_t>::value || (NV > 1 && gridDim.x > 256)) mmf_swish_gate_n<T, 8, !std::is_same<T, f16_t>::value || (NV > 1)>(y, ov[v], xv[v]);
                else mmf_swish_gate_n<T, 8, false>(y, ov[v], xv[v]);
            }
            if constexpr (MODE != ROW_QUANT)
                mmf_store8<T>(static_cast<T*>(a.y) + row * K, k0, K, vec_ok, xv[v]);
        }
    }
    if constexpr (MODE != ROW_QUANT) return;

    amax = mmf_block_max<kWaves>(amax, red_f);
    const float amaxc = fmaxf(amax, 1e-5f);
    const float scale = mmf_127_over(amaxc);
    int qs = 0;
    const int64_t Kp = a.Kp;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int64_t k0 = ((int64_t)v * kThreads + threadIdx.x) * 8;
        if (k0 < Kp) {
            float y[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) y[i] = k0 + i < K ? xv[v][i] : 0.0f;
            const uint32_t lo = mmf_code4({y[0], y[1], y[2], y[3]}, scale), hi = mmf_code4({y[4], y[5], y[6], y[7]}, scale);
            qs = mmf_code4_sum(hi, mmf_code4_sum(lo, qs));
            int64_t off;
            if (a.q_tiled)
                off = ((row >> 5) * (Kp >> 4) + (k0 >> 4)) * 512 + (row & 31) * 16 + (k0 & 15);
            else
                off = row * Kp + k0;
            *reinterpret_cast<uint2*>(a.q + off) = make_uint2(lo, hi);
        }
    }
    qs = mmf_block_sum<kWaves>(qs, red_i);
    if (threadIdx.x == 0) {
        a.deq[row] = mmf_rcp_pos(scale);
        a.qsum[row] = qs;
    }
}

template <typename T, typename TR, typename TW, int MODE>
int launch_row(const RowArgs& a, hipStream_t s) {
    if (a.M == 0) return 0;
    const int64_t width = (MODE == ROW_QUANT) ? a.Kp : a.K;   // the quantiser also zero-fills the padding
    const int64_t nv = mmf_ceil_div(width, (int64_t)kThreads * 8);
    dim3 grid((unsigned)a.M), block(kThreads);
    if (nv <= 1) row_kernel<T, TR, TW, MODE, 1><<<grid, block, 0, s>>>(a);
    else if (nv <= 2) row_kernel<T, TR, TW, MODE, 2><<<grid, block, 0, s>>>(a);
    else if (nv <= 4) row_kernel<T, TR, TW, MODE, 4><<<grid, block, 0, s>>>(a);
    else if (nv <= 8) row_kernel<T, TR, TW, MODE, 8><<<grid, block, 0, s>>>(a);
    else return MMF_ERR_WIDE;
    MMF_CHECK_LAUNCH();
    return 0;
}

template <typename T, typename TR, int MODE>
int dispatch_w(const RowArgs& a, int x_dtype, int w_dtype, hipStream_t s) {
    // The norm weight is either fp32 or the activation dtype.
    if (w_dtype == MMF_F32) return launch_row<T, TR, float, MODE>(a, s);
    if (w_dtype == x_dtype) return launch_row<T, TR, T, MODE>(a, s);
    return MMF_ERR_ARG;
}

template <typename T, int MODE>
int dispatch_r(const RowArgs& a, int x_dtype, int r_dtype, int w_dtype, hipStream_t s) {
    // The residual stream is either the activation dtype or fp32 (residual_in_fp32).
    if (r_dtype == MMF_F32) return dispatch_w<T, float, MODE>(a, x_dtype, w_dtype, s);
    return dispatch_w<T, T, MODE>(a, x_dtype, w_dtype, s);
}

template <int MODE>
int dispatch_x(const RowArgs& a, int x_dtype, int r_dtype, int w_dtype, hipStream_t s) {
    const bool uses_res = a.residual || a.residual_out;
    if (uses_res && r_dtype != MMF_F32 && r_dtype != x_dtype) return MMF_ERR_ARG;
    if (!uses_res) r_dtype = x_dtype;
    if (!a.weight) w_dtype = MMF_F32;
    switch (x_dtype) {
        case MMF_F32: return dispatch_r<float, MODE>(a, x_dtype, r_dtype, w_dtype, s);
        case MMF_BF16: return dispatch_r<bf16_t, MODE>(a, x_dtype, r_dtype, w_dtype, s);
        case MMF_F16: return dispatch_r<f16_t, MODE>(a, x_dtype, r_dtype, w_dtype, s);
    }
    return MMF_ERR_ARG;
}

// ---------------------------------------------------------------- fused prologue + quantiser
// The int8 quantiser with the elementwise op that precedes each BitLinear of a decode step
// folded in (batch sizes that go to the matrix cores, where the codes must exist in memory):
//   QPRO_PLAIN      v = x                                                  (nothing in front: many-row form of ROW_QUANT)
//   QPRO_NORM       v = T(RMSNorm(x; w1, eps1))                            (block norm)
//   QPRO_RESNORM    s = x + aux; res_out = s; v = T(RMSNorm(s; w1, eps1))  (fused residual norm)
//   QPRO_STEP_GATE  i = x, f = aux, g = aux2 (raw projections of one token): gate math, one recurrence
//                   step on the fp32 state (in place), o = T(h); v = T(RMSNorm(g; w1, eps1) * o * sigmoid(o))
//   QPRO_SWIGLU     v = T((x * aux) / (1 + exp(-x)))                       (MLP activation)
//   QPRO_GATEDNORM  v = T(RMSNorm(x; w1, eps1) * aux * sigmoid(aux))       (g_norm in front of o_proj, any T)
// then  y = RMSNorm(v; norm_w, eps),  q = int8 absmax codes of y  (tiled operand layout).
enum QPro : int { QPRO_PLAIN = 0, QPRO_NORM = 1, QPRO_RESNORM = 2, QPRO_STEP_GATE = 3, QPRO_SWIGLU = 4, QPRO_GATEDNORM = 5 };

struct FusedQuantArgs {
    const void* x; const void* aux; const void* aux2;
    int64_t ldx, ldaux, ldaux2;
    void* res_out;
    const void* w1; const void* norm_w;
    const void* norm_w2; const void* norm_w3;   // NN = 3: the second and third norm weight
    int64_t q_stride;                           // NN = 3: bytes from one norm's codes to the next's (deq, qsum: M entries)
    const float* lb; float* state;
    int8_t* q; float* deq; int* qsum;
    int64_t M, K, Kp;
    double inv_K;            // RN(1 / K)
    float eps1, eps;
    MmfAhead ahead;          // the packed weights that the next launch contracts
};

constexpr int kQWaves = 8, kQThreads = kQWaves * 64;

// RPW rows per workgroup, 512 / RPW threads per row, NV passes of (512 / RPW) * 4 elements.
//   RPW = 1 : a decode batch has few rows and each launch is a step of a dependent chain, so all
//             8 waves share one row (shortest latency);
//   RPW = 2, 4, 8 : prefill has hundreds to thousands of rows and the kernel should stream: few waves per row, whose
//             reductions cost little, and many elements per thread.
// Bound by HBM and the vector units about equally (a row of 2048 quantised three times: ~1100 issue slots a wave against 16 KiB of
// traffic), so what does not depend on the data is kept out: no bounds test in passes known to lie in the row, codes rounded and
// packed four at a time.  8192 x 2048 bf16, three norms: 37 -> 28 us; residual norm: 33 -> 22.  The gated form takes its sigmoids near
// (16384 x 2048: 56 -> 52 us, 2002 x 2048 10.6 -> 9.8), and so does the step form (64 x 2048: 5.5 -> 4.9); with a row a workgroup, or one
// vector a thread, the gated form keeps the exact ones (64 x 2048: 4.1 against 4.3; 320 x 1024 fp16 4.7 against 5.1).
// With several rows a workgroup the codes go out through LDS: a thread's four are 4 bytes of a 16-byte piece, pieces of a row lie 512 bytes apart,
// and written as they come every store touched 16 lines for 256 bytes; the caches' write requests, not the bytes, set the pace.  From LDS a
// store writes 16 pieces of all the workgroup's rows (64 bytes for four), and neighbouring workgroups share an XCD, so that whole lines leave its L2.
// 16384 rows bf16: 5632 wide 73.5 -> 53.3 us (5.2 TB/s; 57.6 without the sharing, 64.8 with it alone), residual norm of 2048 60.4 -> 46.9, gated
// norm 53.3 -> 44.0, norm 30.0 -> 29.8 (bound by the vector units); 2002 rows the same to 6 % faster.
// VEC: K, the strides and every pointer allow 4-element accesses (the entry points ask for codes at 16 bytes).
// NN = 3: the row is normalised once and quantised under three norm weights (the projections of a trained layer share their
// input, not their inner norm): one read of the row and one rstd instead of three, the three maxima in one exchange.
template <typename T, typename TW, int NV, int PRO, bool VEC, int RPW, int NN = 1>
__global__ __launch_bounds__(kQThreads) void row_quant_fused_kernel(FusedQuantArgs a) {
    constexpr int TPR = kQThreads / RPW, WPR = TPR / 64;        // threads / waves per row
    __shared__ double red_a[kQWaves], red_b[kQWaves];
    __shared__ float red_f[NN][kQWaves];
    __shared__ int red_i[NN][kQWaves];
    constexpr bool STAGED = VEC && RPW > 1;                     // the codes go out through LDS, as [group of 16 inputs][row][16 bytes]
    __shared__ __align__(16) uint32_t stage[STAGED ? NN : 1][STAGED ? NV * kQThreads : 1];
    constexpr bool HAS_AUX = PRO >= QPRO_RESNORM, STEP = PRO == QPRO_STEP_GATE, HAS_W1 = PRO != QPRO_SWIGLU && PRO != QPRO_PLAIN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int w0 = (wave / WPR) * WPR;                          // first wave of this row
    const int tr = (int)threadIdx.x % TPR;                      // thread within the row
    // XCD: workgroups are dealt round-robin to the 8 XCDs; of every 64 in turn each takes 8 neighbours, so the rows of a 32-row code block meet in
    // one L2 and leave it as whole lines
    const uint32_t in64 = blockIdx.x & 63, wg = RPW > 1 && (blockIdx.x | 63) < gridDim.x ? blockIdx.x - in64 + (in64 & 7) * 8 + (in64 >> 3) : blockIdx.x;
    const int64_t row0 = (int64_t)wg * RPW, row_raw = row0 + (int)threadIdx.x / TPR;
    const bool live = row_raw < a.M;                            // rows past M compute on row M-1 and store nothing
    const int64_t row = live ? row_raw : a.M - 1;
    const int K = (int)a.K, Kp = (int)a.Kp;
    // the first FULL passes lie inside the row whatever K this instance is launched for (the next smaller one would take it otherwise)
    constexpr int FULL = !VEC ? 0 : NV <= 4 ? NV - 1 : NV == 6 ? 4 : NV == 8 ? 6 : 8;
    // element k0 + i of pass v of the row exists; with vector accesses (K a multiple of 4) a thread's 4 elements stand or fall together
    auto inb = [&](int v, int k0, int i) __attribute__((always_inline)) { return v < FULL || (VEC ? k0 < K : k0 + i < K); };
    // a pass's four elements of a row of E
    auto ld = [&](auto* p, int v, int k0) __attribute__((always_inline)) {
        using E = std::remove_const_t<std::remove_pointer_t<decltype(p)>>;
        if (v < FULL) return Raw4<E>{*reinterpret_cast<const decltype(Raw4<E>::v)*>(p + k0)};
        return raw4_load<E, VEC>(static_cast<const E*>(p), k0, K);
    };
    const T* x = static_cast<const T*>(a.x) + row * a.ldx;
    const T* aux = static_cast<const T*>(a.aux) + row * a.ldaux;
    const T* aux2 = static_cast<const T*>(a.aux2) + row * a.ldaux2;
    const TW* w1 = static_cast<const TW*>(a.w1);
    const TW* const nws[3] = {static_cast<const TW*>(a.norm_w), static_cast<const TW*>(a.norm_w2), static_cast<const TW*>(a.norm_w3)};
    const TW* nw = nws[0];
    float* st = a.state + row * K;

    // every load of the kernel first, raw; conversions only after the last one is issued
    Raw4<T> xraw[NV], araw[HAS_AUX ? NV : 1], graw[STEP ? NV : 1];
    Raw4<float> straw[STEP ? NV : 1], lbraw[STEP ? NV : 1];
    Raw4<TW> w1raw[HAS_W1 ? NV : 1], nwraw[NN][NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int k0 = (v * TPR + tr) * 4;
        xraw[v] = ld(x, v, k0);
        if constexpr (HAS_AUX) araw[v] = ld(aux, v, k0);
        if constexpr (STEP) {
            graw[v] = ld(aux2, v, k0);
            straw[v] = ld(st, v, k0);
            if (a.lb) lbraw[v] = ld(a.lb, v, k0);
        }
        if constexpr (HAS_W1) w1raw[v] = ld(w1, v, k0);
        if (NN > 1 || nw) {
#pragma unroll
            for (int j = 0; j < NN; ++j) nwraw[j][v] = ld(nws[j], v, k0);
        }
    }
    uint32_t touched = 0;
    if constexpr (RPW > 1) touched = mmf_touch(a.ahead, (uint32_t)wave * (((uint32_t)a.M + RPW - 1) / RPW) + blockIdx.x);   // (a row a workgroup: decode, no longer than the touch would take)
    float xv[NV][4], av[HAS_AUX ? NV : 1][4];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int k0 = (v * TPR + tr) * 4;
        raw4_unpack<T>(xraw[v], xv[v]);
        if constexpr (HAS_AUX) raw4_unpack<T>(araw[v], av[v]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (!inb(v, k0, i)) xv[v][i] = 0.0f;
    }
    if constexpr (PRO == QPRO_RESNORM) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int k0 = (v * TPR + tr) * 4;
#pragma unroll
            for (int i = 0; i < 4; ++i) xv[v][i] = inb(v, k0, i) ? __fadd_rn(xv[v][i], av[v][i]) : 0.0f;
            if (a.res_out && live) raw4_store<T, VEC>(static_cast<T*>(a.res_out) + row * K, k0, K, xv[v]);
        }
    }
    if constexpr (STEP) {
        // gate math + one recurrence step per channel; xv becomes the raw g projection, av the new o
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int k0 = (v * TPR + tr) * 4;
            float gv[4], stv[4], lbv[4] = {0.0f, 0.0f, 0.0f, 0.0f}, xo[4], go[4];
            raw4_unpack<T>(graw[v], gv);
            raw4_unpack<float>(straw[v], stv);
            if (a.lb) raw4_unpack<float>(lbraw[v], lbv);
            mmf_gate_n<T, 4>(xv[v], av[v], lbv, xo, go);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float h = __fadd_rn(__fmul_rn(go[i], stv[i]), xo[i]);
                stv[i] = h;
                av[v][i] = mmf_round_to<T>(h);          // o, the swish gate of the gated norm
                xv[v][i] = inb(v, k0, i) ? gv[i] : 0.0f;   // the gated norm normalises the g projection
            }
            if (live) raw4_store<float, VEC>(st, k0, K, stv);
        }
    }
    if constexpr (HAS_W1) {
        double s1 = 0.0;
#pragma unroll
        for (int v = 0; v < NV; ++v)
#pragma unroll
            for (int i = 0; i < 4; ++i) s1 = mmf_add_square(s1, xv[v][i]);
        s1 = mmf_wave_sum(s1);
        if constexpr (WPR > 1) {
            if ((threadIdx.x & 63) == 0) red_a[wave] = s1;
            __syncthreads();
            s1 = red_a[w0];
#pragma unroll
            for (int w = 1; w < WPR; ++w) s1 += red_a[w0 + w];
        }
        const float rstd1 = mmf_rstd(s1, K, a.inv_K, a.eps1);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int k0 = (v * TPR + tr) * 4;
            float w1v[4], y[4];
            raw4_unpack<TW>(w1raw[v], w1v);
#pragma unroll
            for (int i = 0; i < 4; ++i) y[i] = __fmul_rn(__fmul_rn(xv[v][i], rstd1), w1v[i]);
            if constexpr (STEP || PRO == QPRO_GATEDNORM) mmf_swish_gate_n<T, 4, STEP || (RPW > 1 && NV > 1)>(y, av[v], xv[v]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (!(STEP || PRO == QPRO_GATEDNORM)) xv[v][i] = mmf_round_to<T>(y[i]);
                if (!inb(v, k0, i)) xv[v][i] = 0.0f;
            }
        }
    } else if constexpr (PRO == QPRO_SWIGLU) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int k0 = (v * TPR + tr) * 4;
            float z[4];
            mmf_swiglu_n<T, 4>(xv[v], av[v], z);
#pragma unroll
            for (int i = 0; i < 4; ++i) xv[v][i] = inb(v, k0, i) ? z[i] : 0.0f;
        }
    }
    // BitLinear's own norm + absmax codes
    double ss = 0.0;
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int i = 0; i < 4; ++i) ss = mmf_add_square(ss, xv[v][i]);
    ss = mmf_wave_sum(ss);
    if constexpr (WPR > 1) {
        if ((threadIdx.x & 63) == 0) red_b[wave] = ss;
        __syncthreads();
        ss = red_b[w0];
#pragma unroll
        for (int w = 1; w < WPR; ++w) ss += red_b[w0 + w];
    }
    const float rstd = mmf_rstd(ss, K, a.inv_K, a.eps);
    float amax[NN];
#pragma unroll
    for (int j = 0; j < NN; ++j) amax[j] = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
#pragma unroll
        for (int i = 0; i < 4; ++i) xv[v][i] = __fmul_rn(xv[v][i], rstd);   // elements past K are exact zeros and stay so
#pragma unroll
        for (int j = 0; j < NN; ++j) {
            float wv[4];
            if (NN > 1 || nw) raw4_unpack<TW>(nwraw[j][v], wv);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float y = xv[v][i];
                if (NN > 1 || nw) y = __fmul_rn(y, wv[i]);
                if constexpr (NN == 1) xv[v][i] = y;
                amax[j] = fmaxf(amax[j], fabsf(y));
            }
        }
    }
#pragma unroll
    for (int j = 0; j < NN; ++j) amax[j] = mmf_wave_max(amax[j]);
    if constexpr (WPR > 1) {
#pragma unroll
        for (int j = 0; j < NN; ++j)
            if ((threadIdx.x & 63) == 0) red_f[j][wave] = amax[j];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NN; ++j) {
            amax[j] = red_f[j][w0];
#pragma unroll
            for (int w = 1; w < WPR; ++w) amax[j] = fmaxf(amax[j], red_f[j][w0 + w]);
        }
    }
    float scale[NN];
    int qs[NN];
#pragma unroll
    for (int j = 0; j < NN; ++j) {
        scale[j] = mmf_127_over(fmaxf(amax[j], 1e-5f));
        qs[j] = 0;
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int k0 = (v * TPR + tr) * 4;
        if (v < FULL || k0 < Kp) {
            const int64_t off = ((row >> 5) * (Kp >> 4) + (k0 >> 4)) * 512 + (row & 31) * 16 + (k0 & 15);
#pragma unroll
            for (int j = 0; j < NN; ++j) {
                float wv[4];
                if constexpr (NN > 1) raw4_unpack<TW>(nwraw[j][v], wv);
                float y[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) y[i] = NN > 1 && (VEC || inb(v, k0, i)) ? __fmul_rn(xv[v][i], wv[i]) : xv[v][i];   // zeros past K
                uint32_t packed4 = mmf_code4(y, scale[j]);
                if (VEC && !inb(v, k0, 0)) packed4 = 0;
                qs[j] = mmf_code4_sum(packed4, qs[j]);
                if constexpr (STAGED) stage[j][((k0 >> 4) * RPW + (int)threadIdx.x / TPR) * 4 + ((k0 & 15) >> 2)] = packed4;
                else if (live) *reinterpret_cast<uint32_t*>(a.q + j * a.q_stride + off) = packed4;
            }
        }
    }
#pragma unroll
    for (int j = 0; j < NN; ++j) qs[j] = mmf_wave_sum(qs[j]);
    if constexpr (WPR > 1) {
#pragma unroll
        for (int j = 0; j < NN; ++j)
            if ((threadIdx.x & 63) == 0) red_i[j][wave] = qs[j];
    }
    if constexpr (WPR > 1 || STAGED) __syncthreads();
    if constexpr (WPR > 1) {
#pragma unroll
        for (int j = 0; j < NN; ++j) {
            qs[j] = 0;
#pragma unroll
            for (int w = 0; w < WPR; ++w) qs[j] += red_i[j][w0 + w];
        }
    }
    if constexpr (STAGED) {
        // the workgroup's rows lie in one 32-row block (RPW divides 32): RPW * 16 contiguous bytes per group
        const int chunks = (Kp >> 4) * RPW;
        const int64_t base = (row0 >> 5) * (Kp >> 4) * 512 + (row0 & 31) * 16;
#pragma unroll
        for (int v = 0; v < mmf_ceil_div(NV, 4); ++v) {
            const int c = v * kQThreads + (int)threadIdx.x, r = c % RPW;
            if (c < chunks && row0 + r < a.M) {
#pragma unroll
                for (int j = 0; j < NN; ++j)
                    *reinterpret_cast<uint4*>(a.q + j * a.q_stride + base + (int64_t)(c / RPW) * 512 + r * 16) = *reinterpret_cast<const uint4*>(&stage[j][c * 4]);
            }
        }
    }
    if (tr == 0 && live) {
#pragma unroll
        for (int j = 0; j < NN; ++j) {
            a.deq[j * a.M + row] = mmf_rcp_pos(scale[j]);
            a.qsum[j * a.M + row] = qs[j];
        }
    }
    if constexpr (RPW > 1) mmf_touched(touched);
}

template <typename T, typename TW, int PRO, int RPW, int NN>
int launch_fused_quant_rpw(const FusedQuantArgs& a, hipStream_t s) {
    constexpr int TPR = kQThreads / RPW;
    const int64_t nv = mmf_ceil_div(a.Kp, (int64_t)TPR * 4);
    dim3 grid((unsigned)mmf_ceil_div(a.M, (int64_t)RPW)), block(kQThreads);
    if (nv <= 1) row_quant_fused_kernel<T, TW, 1, PRO, true, RPW, NN><<<grid, block, 0, s>>>(a);
    else if (nv <= 2) row_quant_fused_kernel<T, TW, 2, PRO, true, RPW, NN><<<grid, block, 0, s>>>(a);
    else if (nv <= 3) row_quant_fused_kernel<T, TW, 3, PRO, true, RPW, NN><<<grid, block, 0, s>>>(a);
    else if (nv <= 4) row_quant_fused_kernel<T, TW, 4, PRO, true, RPW, NN><<<grid, block, 0, s>>>(a);
    else if constexpr (RPW < 8) {
        if (nv <= 6) row_quant_fused_kernel<T, TW, 6, PRO, true, RPW, NN><<<grid, block, 0, s>>>(a);
        else if (nv <= 8) row_quant_fused_kernel<T, TW, 8, PRO, true, RPW, NN><<<grid, block, 0, s>>>(a);
        else if constexpr (PRO == QPRO_PLAIN && RPW == 4) {
            if (nv > 12) return MMF_ERR_WIDE;
            row_quant_fused_kernel<T, TW, 12, PRO, true, RPW, NN><<<grid, block, 0, s>>>(a);
        } else return MMF_ERR_WIDE;
    } else return MMF_ERR_WIDE;
    MMF_CHECK_LAUNCH();
    return 0;
}

template <typename T, typename TW, int PRO, int NN = 1>
int launch_fused_quant(const FusedQuantArgs& a, bool vec, hipStream_t s) {
    if (mmf_ceil_div(a.Kp, (int64_t)kQThreads * 4) > 8) return MMF_ERR_WIDE;
    if (!vec) {                                                 // ragged rows: one generic build
        row_quant_fused_kernel<T, TW, 8, PRO, false, 1, NN><<<dim3((unsigned)a.M), dim3(kQThreads), 0, s>>>(a);
        MMF_CHECK_LAUNCH();
        return 0;
    }
    // The recurrence-step prologue exists for decode only: one token per row, latency.
    if constexpr (PRO != QPRO_STEP_GATE) {
        // Thousands of rows: 16 to 24 elements a thread (8192 x 2048: four rows a workgroup 22 to 28 us where eight, with 32 elements
        // a thread, took 23 to 31; 8192 x 1024: eight 13 to 17, four 14 to 19).  Fewer rows: as few rows a workgroup as reach every
        // CU about once (320 x 2048: two rows 5.0 to 5.9 us, one 5.5 to 7.0, eight 7.4 to 9.7; 1024 x 2048: four 6.5 to 7.9, one 8.5
        // to 10.7).  Wide rows with nothing folded in (5632, in front of down_proj) need few registers and take 48 elements.  Just past a workgroup a CU (four rows: 1024)
        // the few CUs with a second one set the time: 1025 to 1536 rows take two a workgroup, at most three a CU (1377 rows, four / two: 2048 wide, three norms
        // 9.6 / 9.3 us, residual norm 8.2 / 7.7, gated 8.8 / 8.1, 5632 plain 9.2 / 8.5, 2560 wide three norms 11.7 / 10.8; 1700 rows 10.0 / 10.9, 8.7 / 9.1, 8.8 / 9.4,
        // 9.5 / 9.9, 12.3 / 12.7), narrow rows eight (1200 x 1024: 6.8 / 6.3, 5.9 / 5.5; 1001 5.4 / 6.2, 5.0 / 5.5).
        if (a.M > 1024 && a.Kp <= 1024) return launch_fused_quant_rpw<T, TW, PRO, 8, NN>(a, s);
        const bool second = a.M > 1024 && a.M <= 1536;
        if (a.M > 512 && !second && a.Kp <= (PRO == QPRO_PLAIN ? 6144 : 3072)) return launch_fused_quant_rpw<T, TW, PRO, 4, NN>(a, s);
        if (a.M > 192 && a.Kp <= 8192) return launch_fused_quant_rpw<T, TW, PRO, 2, NN>(a, s);
    }
    return launch_fused_quant_rpw<T, TW, PRO, 1, NN>(a, s);
}

template <typename T, typename TW>
int dispatch_fused_quant(const FusedQuantArgs& a, int pro, bool vec, hipStream_t s) {
    switch (pro) {
        case QPRO_PLAIN: return launch_fused_quant<T, TW, QPRO_PLAIN>(a, vec, s);
        case QPRO_NORM:
            return a.norm_w2 ? launch_fused_quant<T, TW, QPRO_NORM, 3>(a, vec, s) : launch_fused_quant<T, TW, QPRO_NORM>(a, vec, s);
        case QPRO_RESNORM: return launch_fused_quant<T, TW, QPRO_RESNORM>(a, vec, s);
        case QPRO_STEP_GATE: return launch_fused_quant<T, TW, QPRO_STEP_GATE>(a, vec, s);
        case QPRO_SWIGLU: return launch_fused_quant<T, TW, QPRO_SWIGLU>(a, vec, s);
        case QPRO_GATEDNORM: return launch_fused_quant<T, TW, QPRO_GATEDNORM>(a, vec, s);
    }
    return MMF_ERR_ARG;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Checks the accesses the kernel will make and picks the instance for the types.
int run_fused_quant(const FusedQuantArgs& a, int prologue, int x_dtype, int weight_dtype, hipStream_t stream) {
    const uintptr_t xa = 4 * (x_dtype == MMF_F32 ? 4 : 2), wa = 4 * (weight_dtype == MMF_F32 ? 4 : 2);
    auto al = [](const void* ptr, uintptr_t n) { return (reinterpret_cast<uintptr_t>(ptr) % n) == 0; };
    const bool vec = a.K % 4 == 0 && a.ldx % 4 == 0 && a.ldaux % 4 == 0 && a.ldaux2 % 4 == 0;
    if (vec && !(al(a.x, xa) && al(a.aux, xa) && al(a.aux2, xa) && al(a.res_out, xa) && al(a.w1, wa) && al(a.norm_w, wa) && al(a.norm_w2, wa) && al(a.norm_w3, wa) &&
                 al(a.lb, 16) && al(a.state, 16)))
        return MMF_ERR_ALIGN;
    const bool wf32 = weight_dtype == MMF_F32;
    if (!wf32 && weight_dtype != x_dtype) return MMF_ERR_ARG;
    switch (x_dtype) {
        case MMF_F32: return dispatch_fused_quant<float, float>(a, prologue, vec, stream);
        case MMF_BF16: return wf32 ? dispatch_fused_quant<bf16_t, float>(a, prologue, vec, stream)
                                   : dispatch_fused_quant<bf16_t, bf16_t>(a, prologue, vec, stream);
        case MMF_F16: return wf32 ? dispatch_fused_quant<f16_t, float>(a, prologue, vec, stream)
                                  : dispatch_fused_quant<f16_t, f16_t>(a, prologue, vec, stream);
    }
    return MMF_ERR_ARG;
}

// ---------------------------------------------------------------- swiglu (elementwise)
template <typename T>
__global__ __launch_bounds__(256) void swiglu_kernel(const T* __restrict__ x, int64_t ldx, const T* __restrict__ y,
                                                     int64_t ldy, T* __restrict__ out, int64_t rows, int64_t cols) {
    // cols % 8 == 0; one 8-vector per thread.
    const int64_t vpr = cols / 8;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= rows * vpr) return;
    const int64_t r = idx / vpr, c0 = (idx % vpr) * 8;
    float xv[8], yv[8], z[8];
    mmf_load8<T>(x + r * ldx, c0, cols, true, xv);
    mmf_load8<T>(y + r * ldy, c0, cols, true, yv);
    // fp16 near only with more workgroups than CUs: fewer run as long as their slowest wave (64 x 2048 3.2 us, near 3.4)
    if (!std::is_same<T, f16_t>::value || gridDim.x > 256) mmf_swiglu_n<T, 8>(xv, yv, z);
    else mmf_swiglu_n<T, 8, false>(xv, yv, z);
    mmf_store8<T>(out + r * cols, c0, cols, true, z);
}

template <typename T>
__global__ __launch_bounds__(256) void swiglu_scalar_kernel(const T* __restrict__ x, int64_t ldx, const T* __restrict__ y,
                                                            int64_t ldy, T* __restrict__ out, int64_t rows, int64_t cols) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= rows * cols) return;
    const int64_t r = idx / cols, c = idx % cols;
    const float xv = mmf_to_float(x[r * ldx + c]), yv = mmf_to_float(y[r * ldy + c]);
    out[r * cols + c] = mmf_from_float<T>(mmf_swiglu_definition(xv, yv));
}

template <typename T>
int launch_swiglu(const void* x, int64_t ldx, const void* y, int64_t ldy, void* out, int64_t rows, int64_t cols,
                  hipStream_t s) {
    if (rows == 0 || cols == 0) return 0;
    const int esz = sizeof(T);
    const bool vec = cols % 8 == 0 && ldx % 8 == 0 && ldy % 8 == 0 && aligned16(x) && aligned16(y) && aligned16(out);
    (void)esz;
    if (vec) {
        const int64_t n = rows * (cols / 8);
        swiglu_kernel<T><<<(unsigned)mmf_ceil_div(n, 256), 256, 0, s>>>(static_cast<const T*>(x), ldx,
                                                                       static_cast<const T*>(y), ldy,
                                                                       static_cast<T*>(out), rows, cols);
    } else {
        const int64_t n = rows * cols;
        swiglu_scalar_kernel<T><<<(unsigned)mmf_ceil_div(n, 256), 256, 0, s>>>(static_cast<const T*>(x), ldx,
                                                                              static_cast<const T*>(y), ldy,
                                                                              static_cast<T*>(out), rows, cols);
    }
    MMF_CHECK_LAUNCH();
    return 0;
}

}  // namespace

extern "C" {

int mmf_rmsnorm(const void* x, const void* residual, const void* weight, void* y, void* residual_out, int64_t M,
                int64_t K, float eps, int x_dtype, int residual_dtype, int weight_dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (M < 0 || K <= 0 || (M > 0 && (!x || !y))) return MMF_ERR_ARG;
    if (K % 8 == 0 && !(aligned16(x) && aligned16(y) && aligned16(residual) && aligned16(residual_out) && aligned16(weight)))
        return MMF_ERR_ALIGN;
    RowArgs a{};
    a.x = x; a.residual = residual; a.weight = weight; a.y = y; a.residual_out = residual_out;
    a.M = M; a.K = K; a.inv_K = 1.0 / (double)K; a.Kp = K; a.ldx = K; a.eps = eps;
    return dispatch_x<ROW_NORM>(a, x_dtype, residual_dtype, weight_dtype, stream);
}

int mmf_rmsnorm_swishgate(const void* x, int64_t ldx, const void* gate, const void* residual, const void* weight, void* y,
                          void* residual_out, int64_t M, int64_t K, float eps, int x_dtype, int residual_dtype,
                          int weight_dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (M < 0 || K <= 0 || ldx < K || (M > 0 && (!x || !y || !gate))) return MMF_ERR_ARG;
    if (K % 8 == 0 && ldx % 8 != 0) return MMF_ERR_ALIGN;
    if (K % 8 == 0 && !(aligned16(x) && aligned16(y) && aligned16(gate) && aligned16(residual) &&
                        aligned16(residual_out) && aligned16(weight)))
        return MMF_ERR_ALIGN;
    RowArgs a{};
    a.x = x; a.gate = gate; a.residual = residual; a.weight = weight; a.y = y; a.residual_out = residual_out;
    a.M = M; a.K = K; a.inv_K = 1.0 / (double)K; a.Kp = K; a.ldx = ldx; a.eps = eps;
    return dispatch_x<ROW_GATE>(a, x_dtype, residual_dtype, weight_dtype, stream);
}

int64_t mmf_codes_bytes(int64_t M, int64_t K, int tiled) {
    const int64_t Kp = mmf_round_up(K, 128);
    return (tiled ? mmf_round_up(M, 32) : M) * Kp;
}

int mmf_rmsnorm_quant(const void* x, const void* residual, const void* weight, int8_t* q, float* deq, int* qsum,
                      void* residual_out, int64_t M, int64_t K, float eps, int x_dtype, int residual_dtype,
                      int weight_dtype, int tiled, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (M < 0 || K <= 0 || (M > 0 && (!x || !q || !deq || !qsum))) return MMF_ERR_ARG;
    if (!aligned16(q)) return MMF_ERR_ALIGN;
    if (K % 8 == 0 && !(aligned16(x) && aligned16(residual) && aligned16(residual_out) && aligned16(weight)))
        return MMF_ERR_ALIGN;
    // nothing but the norm in front: the fused kernel's plain form, whose rows per workgroup follow their number
    if (tiled && !residual && !residual_out && K % 8 == 0 && K <= 16384)
        return mmf_rmsnorm_quant_fused(QPRO_PLAIN, x, K, nullptr, 0, nullptr, 0, nullptr, nullptr, 0.0f, weight, eps, nullptr, nullptr, q, deq,
                                       qsum, M, K, x_dtype, weight_dtype, stream_);
    RowArgs a{};
    a.x = x; a.residual = residual; a.weight = weight; a.residual_out = residual_out;
    a.q = q; a.deq = deq; a.qsum = qsum;
    a.M = M; a.K = K; a.inv_K = 1.0 / (double)K; a.Kp = mmf_round_up(K, 128); a.ldx = K; a.eps = eps; a.q_tiled = tiled;
    return dispatch_x<ROW_QUANT>(a, x_dtype, residual_dtype, weight_dtype, stream);
}

int mmf_layernorm_quant(const void* x, const void* residual, const void* weight, const void* bias, int8_t* q, float* deq,
                        int* qsum, void* residual_out, int64_t M, int64_t K, float eps, int x_dtype, int residual_dtype,
                        int weight_dtype, int tiled, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (M < 0 || K <= 0 || (M > 0 && (!x || !q || !deq || !qsum))) return MMF_ERR_ARG;
    if (bias && !weight) return MMF_ERR_ARG;                     // the bias shares the weight's dtype
    if (!aligned16(q)) return MMF_ERR_ALIGN;
    if (K % 8 == 0 && !(aligned16(x) && aligned16(residual) && aligned16(residual_out) && aligned16(weight) && aligned16(bias)))
        return MMF_ERR_ALIGN;
    RowArgs a{};
    a.x = x; a.residual = residual; a.weight = weight; a.bias = bias; a.center = 1; a.residual_out = residual_out;
    a.q = q; a.deq = deq; a.qsum = qsum;
    a.M = M; a.K = K; a.inv_K = 1.0 / (double)K; a.Kp = mmf_round_up(K, 128); a.ldx = K; a.eps = eps; a.q_tiled = tiled;
    return dispatch_x<ROW_QUANT>(a, x_dtype, residual_dtype, weight_dtype, stream);
}

int mmf_rmsnorm_quant_fused(int prologue, const void* x, int64_t ldx, const void* aux, int64_t ldaux, const void* aux2,
                            int64_t ldaux2, void* res_out, const void* w1, float eps1, const void* norm_weight, float eps,
                            const float* lower_bound, float* state, int8_t* q, float* deq, int* qsum, int64_t M, int64_t K,
                            int x_dtype, int weight_dtype, void* stream_) {
    return mmf_rmsnorm_quant_fused_ahead(prologue, x, ldx, aux, ldaux, aux2, ldaux2, res_out, w1, eps1, norm_weight, eps, lower_bound, state, q,
                                         deq, qsum, M, K, nullptr, 0, x_dtype, weight_dtype, stream_);
}

int mmf_rmsnorm_quant_fused_ahead(int prologue, const void* x, int64_t ldx, const void* aux, int64_t ldaux, const void* aux2,
                                  int64_t ldaux2, void* res_out, const void* w1, float eps1, const void* norm_weight, float eps,
                                  const float* lower_bound, float* state, int8_t* q, float* deq, int* qsum, int64_t M, int64_t K,
                                  const void* ahead, int64_t ahead_bytes, int x_dtype, int weight_dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (M < 0 || K <= 0 || ldx < K) return MMF_ERR_ARG;
    if (M == 0) return 0;
    if (!x || !q || !deq || !qsum) return MMF_ERR_ARG;
    if (prologue < QPRO_PLAIN || prologue > QPRO_GATEDNORM) return MMF_ERR_ARG;
    if (prologue >= QPRO_RESNORM && (!aux || ldaux < K)) return MMF_ERR_ARG;
    if (prologue == QPRO_STEP_GATE && (!aux2 || ldaux2 < K || !state)) return MMF_ERR_ARG;
    if (prologue != QPRO_SWIGLU && prologue != QPRO_PLAIN && !w1) return MMF_ERR_ARG;
    FusedQuantArgs a{};
    a.x = x; a.aux = aux ? aux : x; a.aux2 = aux2 ? aux2 : x; a.ldx = ldx; a.ldaux = aux ? ldaux : ldx;
    a.ldaux2 = aux2 ? ldaux2 : ldx; a.res_out = res_out; a.w1 = w1; a.norm_w = norm_weight; a.lb = lower_bound; a.state = state;
    a.q = q; a.deq = deq; a.qsum = qsum; a.M = M; a.K = K; a.inv_K = 1.0 / (double)K; a.Kp = mmf_round_up(K, 128); a.eps1 = eps1; a.eps = eps;
    if (const int rc = mmf_set_ahead(a.ahead, ahead, ahead_bytes)) return rc;
    if (!aligned16(q)) return MMF_ERR_ALIGN;
    if (!norm_weight && !w1) weight_dtype = MMF_F32;
    return run_fused_quant(a, prologue, x_dtype, weight_dtype, stream);
}

int mmf_rmsnorm_quant_multi(const void* x, int64_t ldx, const void* w1, float eps1, const void* norm_weight0, const void* norm_weight1,
                            const void* norm_weight2, float eps, int8_t* q, float* deq, int* qsum, int64_t M, int64_t K, int x_dtype,
                            int weight_dtype, void* stream_) {
    return mmf_rmsnorm_quant_multi_ahead(x, ldx, w1, eps1, norm_weight0, norm_weight1, norm_weight2, eps, q, deq, qsum, M, K, nullptr, 0, x_dtype,
                                         weight_dtype, stream_);
}

int mmf_rmsnorm_quant_multi_ahead(const void* x, int64_t ldx, const void* w1, float eps1, const void* norm_weight0,
                                  const void* norm_weight1, const void* norm_weight2, float eps, int8_t* q, float* deq, int* qsum, int64_t M,
                                  int64_t K, const void* ahead, int64_t ahead_bytes, int x_dtype, int weight_dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (M < 0 || K <= 0 || ldx < K) return MMF_ERR_ARG;
    if (M == 0) return 0;
    if (!x || !w1 || !norm_weight0 || !norm_weight1 || !norm_weight2 || !q || !deq || !qsum) return MMF_ERR_ARG;
    if (!aligned16(q)) return MMF_ERR_ALIGN;
    FusedQuantArgs a{};
    a.x = a.aux = a.aux2 = x; a.ldx = a.ldaux = a.ldaux2 = ldx; a.w1 = w1; a.norm_w = norm_weight0; a.norm_w2 = norm_weight1;
    a.norm_w3 = norm_weight2; a.q_stride = mmf_codes_bytes(M, K, 1); a.q = q; a.deq = deq; a.qsum = qsum; a.M = M; a.K = K;
    a.inv_K = 1.0 / (double)K; a.Kp = mmf_round_up(K, 128); a.eps1 = eps1; a.eps = eps;
    if (const int rc = mmf_set_ahead(a.ahead, ahead, ahead_bytes)) return rc;
    return run_fused_quant(a, QPRO_NORM, x_dtype, weight_dtype, stream);
}

int mmf_swiglu(const void* x, int64_t ldx, const void* y, int64_t ldy, void* out, int64_t rows, int64_t cols,
               int dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (rows < 0 || cols < 0 || (rows * cols > 0 && (!x || !y || !out))) return MMF_ERR_ARG;
    switch (dtype) {
        case MMF_F32: return launch_swiglu<float>(x, ldx, y, ldy, out, rows, cols, stream);
        case MMF_BF16: return launch_swiglu<bf16_t>(x, ldx, y, ldy, out, rows, cols, stream);
        case MMF_F16: return launch_swiglu<f16_t>(x, ldx, y, ldy, out, rows, cols, stream);
    }
    return MMF_ERR_ARG;
}

}  // extern "C"
