// Backward of an HGRNBit block between its dense products: the row kernels that carry a gradient through a BitLinear's norm
// AND the elementwise op in front of it in one pass, and the ternary weights as a dense matrix.
//
//   mmf_chain_bwd        CHAIN_NORM    norm(x; w1) -> 1 or 3 BitLinears' norms (block norm in front of i/f/g, norm in front of the head)
//                        CHAIN_RESNORM norm(x + a; w1) -> a BitLinear's norm (residual and mlp_norm in front of gate/up)
//                        CHAIN_GATED   norm(x; w1) * a * sigmoid(a) -> a BitLinear's norm (g_norm in front of o_proj)
//                        CHAIN_SWIGLU  swiglu(x, a) -> a BitLinear's norm (the MLP activation in front of down_proj)
//     i.e. mmfreelm/ops/fusedbitnet.py:209-317 followed by mmfreelm/modules/layernorm.py:245-330,
//     mmfreelm/modules/fused_norm_gate.py:210-300 or mmfreelm/modules/activations.py:121-126.
//   mmf_unpack_dequant   the de-quantised weight of fusedbitnet.py:456-458 for the product dout @ W_q; mmf_unpack_dequant_t stores it
//     with the contraction contiguous.
//
// HBM is the bound: a step read and wrote every row of gradient between these ops (norm behind norm, three norms and two
// additions behind i/f/g); here the row stays in registers from the products' output to the next products' input.  The
// quantised activations that the weight gradient contracts with are recomputed in the forward's arithmetic, bit for bit;
// gradients are fp32 between the stages.
#include "mmf_common.h"
#include "column_sum.h"

namespace {

enum Chain : int { CHAIN_NORM = 0, CHAIN_GATED = 1, CHAIN_SWIGLU = 2, CHAIN_RESNORM = 3 };

struct ChainArgs {
    const void* x; const void* aux;     // the op's inputs, row strides ldx, ldaux
    const void* w1;                     // all but SWIGLU: weight of the norm in front
    const void* w2[3];                  // the BitLinears' norm weights
    const void* dy[3];                  // gradients of their normalised inputs (dout @ W_q), row stride lddy
    const void* dres;                   // NORM, RESNORM: null, or a gradient that joins dx (the residual branch), row stride K
    void* dx; void* daux;               // gradients of x and aux, row strides lddx, lddaux
    void* y;                            // [NN][M, K]: the de-quantised codes of the BitLinears' inputs
    float* part;                        // [gridDim.x][W1 + NN][K]: sums for w1, then for the w2
    int64_t M, ldx, ldaux, lddy, lddx, lddaux;
    int K;
    float eps1, eps2;
    double inv_K;
};

// One row per workgroup and turn, 4 elements per thread and pass, the next row's loads in flight under this row's arithmetic;
// four exchanges of per-wave partials a row, each with slots of its own and one barrier.
// The vector units are the bound next to HBM: a wave spends ~300 instructions a row whatever it carries (addresses, exchanges, the
// roots) on top of ~45 to 100 an element, so rows go to few waves with 8 elements a thread, as long as the registers still leave
// two rows on a CU.  8192 rows of 2048 in bf16: 4 waves with 8 elements 45 us (norm) and 57 us (gated) where 8 waves with 4 took
// 52 and 70; three norms keep 8 waves (194 registers otherwise).  5632 wide (swiglu): 12 waves with 8, 153 us; 8 waves with 12,
// one to two on a SIMD, 159 us.
template <typename T, typename TW, int KT, int NV, int ST, int NN>
__global__ __launch_bounds__(KT) void chain_bwd_kernel(ChainArgs a) {
    // RESNORM adds its operands again instead of reading their rounded sum: the forward normalised the unrounded one, and from the rounded
    // one 4.5 % of the bf16 codes come out as others (8192 x 2048), which put gate_proj's weight gradient 8.7e-3 from the exact one
    // where it is 3.3e-3 now.  The second operand's load hides: 54 us with either (column sums included).
    constexpr bool W1 = ST != CHAIN_SWIGLU, AUX = ST != CHAIN_NORM, ADD = ST == CHAIN_RESNORM, RES = ST == CHAIN_NORM || ADD;
    constexpr int kW = KT / 64;
    __shared__ double s_sum1[kW], s_sum2[kW];
    __shared__ float s_max[NN][kW], s_dot2[kW], s_dot1[kW];
    const int K = a.K, lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    float acc1[W1 ? NV : 1][4], acc2[NN][NV][4];
    Raw4<TW> w1r[W1 ? NV : 1], w2r[NN][NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int k0 = (v * KT + (int)threadIdx.x) * 4;
        if constexpr (W1) w1r[v] = raw4_load<TW, true>(static_cast<const TW*>(a.w1), k0, K);
#pragma unroll
        for (int n = 0; n < NN; ++n) w2r[n][v] = raw4_load<TW, true>(static_cast<const TW*>(a.w2[n]), k0, K);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (W1) acc1[v][i] = 0.0f;
#pragma unroll
            for (int n = 0; n < NN; ++n) acc2[n][v][i] = 0.0f;
        }
    }
    Raw4<T> xr[NV], ar[AUX ? NV : 1], rr[RES ? NV : 1], dr[NN][NV];
    auto load = [&](int64_t row) __attribute__((always_inline)) {
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int k0 = (v * KT + (int)threadIdx.x) * 4;
            xr[v] = raw4_load<T, true>(static_cast<const T*>(a.x) + row * a.ldx, k0, K);
            if constexpr (AUX) ar[v] = raw4_load<T, true>(static_cast<const T*>(a.aux) + row * a.ldaux, k0, K);
#pragma unroll
            for (int n = 0; n < NN; ++n) dr[n][v] = raw4_load<T, true>(static_cast<const T*>(a.dy[n]) + row * a.lddy, k0, K);
            if constexpr (RES) {
                if (a.dres) rr[v] = raw4_load<T, true>(static_cast<const T*>(a.dres) + row * (int64_t)K, k0, K);
            }
        }
    };
    auto fold = [&](float v) __attribute__((always_inline)) {
        v += mmf_dpp<kDppXor1>(v);
        v += mmf_dpp<kDppXor2>(v);
        v += mmf_dpp<kDppHalfMirror>(v);
        v += mmf_dpp<kDppMirror>(v);
        return (mmf_readlane(v, 0) + mmf_readlane(v, 16)) + (mmf_readlane(v, 32) + mmf_readlane(v, 48));
    };
    auto total = [&](const float* s) __attribute__((always_inline)) {
        float t = s[0];
#pragma unroll
        for (int w = 1; w < kW; ++w) t += s[w];
        return t;
    };
    auto in_row = [&](int v) __attribute__((always_inline)) { return (v * KT + (int)threadIdx.x) * 4 < K; };   // K is a multiple of 4

    load((int64_t)blockIdx.x < a.M ? blockIdx.x : 0);
    for (int64_t row = blockIdx.x; row < a.M; row += gridDim.x) {
        float x[NV][4], av[AUX ? NV : 1][4], res[RES ? NV : 1][4], dy[NN][NV][4];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            raw4_unpack<T>(xr[v], x[v]);
            if constexpr (AUX) raw4_unpack<T>(ar[v], av[v]);
#pragma unroll
            for (int n = 0; n < NN; ++n) raw4_unpack<T>(dr[n][v], dy[n][v]);
            if constexpr (RES) raw4_unpack<T>(rr[v], res[v]);
            const bool in = in_row(v);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (ADD) x[v][i] = __fadd_rn(x[v][i], av[v][i]);
                x[v][i] = in ? x[v][i] : 0.0f;
                if constexpr (AUX) av[v][i] = in ? av[v][i] : 0.0f;
#pragma unroll
                for (int n = 0; n < NN; ++n) dy[n][v][i] = in ? dy[n][v][i] : 0.0f;
                if constexpr (RES) res[v][i] = a.dres ? res[v][i] : 0.0f;
            }
        }
        load(row + gridDim.x < a.M ? row + gridDim.x : row);

        // ---- the op in front, as the forward rounds it: s = what the BitLinear saw
        float s[NV][4], sg[AUX ? NV : 1][4];
        float rstd1 = 0.0f;
        if constexpr (W1) {
            double q = 0.0;
#pragma unroll
            for (int v = 0; v < NV; ++v)
#pragma unroll
                for (int i = 0; i < 4; ++i) q = mmf_add_square(q, x[v][i]);
            rstd1 = mmf_rstd(mmf_block_sum_once<kW>(q, s_sum1), K, a.inv_K, a.eps1);
        }
        double q2 = 0.0;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            float w1[4];
            if constexpr (W1) raw4_unpack<TW>(w1r[v], w1);
            // The gradients take the sigmoid of the definition, in 16-bit rows too: nothing decides there, as the rounding of s does in the
            // forward, and mmf_sigmoid_near is up to 30 units of 2^-24 off at arguments near -30 where this is up to 2.7.  8192 rows in bf16
            // 54.5 us (gated, 2048 wide) and 145 (swiglu, 5632), with the near form 49.7 and 128.
            if constexpr (ST == CHAIN_GATED) mmf_sigmoid_n<4>(av[v], sg[v]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (ST == CHAIN_SWIGLU) {
                    const float e = __fadd_rn(1.0f, mmf_exp(-x[v][i]));
                    s[v][i] = mmf_round_to<T>(__fdiv_rn(__fmul_rn(x[v][i], av[v][i]), e));
                    sg[v][i] = __builtin_amdgcn_rcpf(e);
                } else {
                    float y = __fmul_rn(__fmul_rn(x[v][i], rstd1), w1[i]);
                    if constexpr (ST == CHAIN_GATED) y = __fmul_rn(__fmul_rn(y, av[v][i]), sg[v][i]);
                    s[v][i] = mmf_round_to<T>(y);
                }
                if (!in_row(v)) s[v][i] = 0.0f;
                q2 = mmf_add_square(q2, s[v][i]);
            }
        }
        // ---- the BitLinears' norms: codes, and the gradient through them
        const float rstd2 = mmf_rstd(mmf_block_sum_once<kW>(q2, s_sum2), K, a.inv_K, a.eps2);
        float amax[NN], dot2 = 0.0f, wd[NV][4];
#pragma unroll
        for (int n = 0; n < NN; ++n) amax[n] = 0.0f;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                s[v][i] = __fmul_rn(s[v][i], rstd2);
                wd[v][i] = 0.0f;
            }
#pragma unroll
            for (int n = 0; n < NN; ++n) {
                float w2[4];
                raw4_unpack<TW>(w2r[n][v], w2);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    amax[n] = fmaxf(amax[n], fabsf(__fmul_rn(s[v][i], w2[i])));
                    wd[v][i] += w2[i] * dy[n][v][i];
                    acc2[n][v][i] += dy[n][v][i] * s[v][i];
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) dot2 += s[v][i] * wd[v][i];
        }
        dot2 = fold(dot2);
#pragma unroll
        for (int n = 0; n < NN; ++n) {
            amax[n] = mmf_wave_max(amax[n]);
            if (lane == 0) s_max[n][wave] = amax[n];
        }
        if (lane == 0) s_dot2[wave] = dot2;
        __syncthreads();
        const float c2 = total(s_dot2) / (float)K;
        float scale[NN], deq[NN];
#pragma unroll
        for (int n = 0; n < NN; ++n) {
            amax[n] = s_max[n][0];
#pragma unroll
            for (int w = 1; w < kW; ++w) amax[n] = fmaxf(amax[n], s_max[n][w]);
            scale[n] = mmf_127_over(fmaxf(amax[n], 1e-5f));
            deq[n] = mmf_rcp_pos(scale[n]);
        }
        float dot1 = 0.0f;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int k0 = (v * KT + (int)threadIdx.x) * 4;
#pragma unroll
            for (int n = 0; n < NN; ++n) {
                float w2[4], o[4];
                raw4_unpack<TW>(w2r[n][v], w2);
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = __fmul_rn(mmf_code_f(__fmul_rn(s[v][i], w2[i]), scale[n]), deq[n]);
                raw4_store<T, true>(static_cast<T*>(a.y) + ((int64_t)n * a.M + row) * K, k0, K, o);
            }
            float w1[4], o[4];
            if constexpr (W1) raw4_unpack<TW>(w1r[v], w1);
            // ---- back through the op in front: wd = gradient of s
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float d = (wd[v][i] - s[v][i] * c2) * rstd2;
                if constexpr (ST == CHAIN_SWIGLU) {
                    const float g = x[v][i];
                    o[i] = d * g * sg[v][i];
                    x[v][i] = sg[v][i] * (1.0f + g * (1.0f - sg[v][i])) * d * av[v][i];
                } else {
                    const float xh = x[v][i] * rstd1;
                    if constexpr (ST == CHAIN_GATED) {
                        o[i] = d * xh * w1[i] * sg[v][i] * (1.0f + av[v][i] * (1.0f - sg[v][i]));
                        d *= av[v][i] * sg[v][i];
                    }
                    acc1[v][i] += d * xh;
                    wd[v][i] = d * w1[i];
                    x[v][i] = xh;
                    dot1 += xh * wd[v][i];
                }
            }
            if constexpr (AUX && !ADD) raw4_store<T, true>(static_cast<T*>(a.daux) + row * a.lddaux, k0, K, o);
            if constexpr (ST == CHAIN_SWIGLU) raw4_store<T, true>(static_cast<T*>(a.dx) + row * a.lddx, k0, K, x[v]);
        }
        if constexpr (W1) {
            dot1 = fold(dot1);
            if (lane == 0) s_dot1[wave] = dot1;
            __syncthreads();
            const float c1 = total(s_dot1) / (float)K;
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                float o[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = (wd[v][i] - x[v][i] * c1) * rstd1 + (RES ? res[v][i] : 0.0f);
                raw4_store<T, true>(static_cast<T*>(a.dx) + row * a.lddx, (v * KT + (int)threadIdx.x) * 4, K, o);
            }
        } else {
            __syncthreads();                                     // the slots are free for the next row
        }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int k0 = (v * KT + (int)threadIdx.x) * 4;
        float* p = a.part + (int64_t)blockIdx.x * ((W1 ? 1 : 0) + NN) * K;
        if constexpr (W1) raw4_store<float, true>(p, k0, K, acc1[v]);
#pragma unroll
        for (int n = 0; n < NN; ++n) raw4_store<float, true>(p + (int64_t)((W1 ? 1 : 0) + n) * K, k0, K, acc2[n][v]);
    }
}

template <typename T, typename TW, int ST, int NN>
int launch_chain(const ChainArgs& a, int groups, void* dw, hipStream_t s) {
    if (a.K <= 1024) chain_bwd_kernel<T, TW, 256, 1, ST, NN><<<groups, 256, 0, s>>>(a);
    else if (a.K <= 2048) {
        if constexpr (NN == 1) chain_bwd_kernel<T, TW, 256, 2, ST, NN><<<groups, 256, 0, s>>>(a);
        else chain_bwd_kernel<T, TW, 512, 1, ST, NN><<<groups, 512, 0, s>>>(a);
    }
    else if (a.K <= 4096) chain_bwd_kernel<T, TW, 512, 2, ST, NN><<<groups, 512, 0, s>>>(a);
    else if constexpr (NN == 1) {                                // (three norms: a wider row would not fit the registers)
        if (a.K <= 6144) chain_bwd_kernel<T, TW, 768, 2, ST, NN><<<groups, 768, 0, s>>>(a);
        else chain_bwd_kernel<T, TW, 512, 4, ST, NN><<<groups, 512, 0, s>>>(a);
    } else return MMF_ERR_WIDE;
    MMF_CHECK_LAUNCH();
    const int cols = ((ST != CHAIN_SWIGLU ? 1 : 0) + NN) * a.K;
    launch_colsum(a.part, groups, cols, static_cast<TW*>(dw), s);
    MMF_CHECK_LAUNCH();
    return 0;
}
template <typename T, typename TW>
int dispatch_chain(const ChainArgs& a, int kind, int n, int groups, void* dw, hipStream_t s) {
    switch (kind) {
        case CHAIN_NORM: return n == 3 ? launch_chain<T, TW, CHAIN_NORM, 3>(a, groups, dw, s) : launch_chain<T, TW, CHAIN_NORM, 1>(a, groups, dw, s);
        case CHAIN_RESNORM: return launch_chain<T, TW, CHAIN_RESNORM, 1>(a, groups, dw, s);
        case CHAIN_GATED: return launch_chain<T, TW, CHAIN_GATED, 1>(a, groups, dw, s);
        case CHAIN_SWIGLU: return launch_chain<T, TW, CHAIN_SWIGLU, 1>(a, groups, dw, s);
    }
    return MMF_ERR_ARG;
}

// ------------------------------------------------------------------------------------------ weights
// Bound by the write, 2 (4) bytes a weight.  A thread owns one 16-byte vector of kUdRows consecutive rows, so a wave's store is 1 KiB
// of one row and the rows of a workgroup use up the lines of the packed blocks (a row's codes of 128 inputs are two 16-byte pieces
// 512 bytes apart, the next row's follow each).  The 32000 x 2048 head in bf16: one thread per dword of codes, 64-byte strides
// between the lanes' stores and a 64-bit division took 44 us.
constexpr int kUdRows = 8;
template <typename T>
__global__ __launch_bounds__(256) void unpack_dequant_kernel(const uint32_t* __restrict__ packed, const float* __restrict__ wdeq,
                                                             uint32_t seg_rows, int N, int K, int KB, bool whole, T* __restrict__ out) {
    constexpr int VE = 16 / (int)sizeof(T);
    const int k0 = ((int)blockIdx.y * 256 + (int)threadIdx.x) * VE;
    if (k0 >= K) return;
    const int n0 = (int)blockIdx.x * kUdRows, part = (k0 & 15) >> 2;     // VE is 4 or 8: one or two groups of 4 codes
    const uint32_t* src = packed + ((((int64_t)(n0 >> 5) * KB + (k0 >> 7)) * 64 + ((k0 >> 4) & 1) * 32 + (n0 & 31)) * 4 + ((k0 >> 5) & 3));
    uint32_t code[kUdRows];
#pragma unroll
    for (int r = 0; r < kUdRows; ++r) code[r] = src[r * 4];              // (rows are padded to 32 there)
#pragma unroll
    for (int r = 0; r < kUdRows; ++r) {
        if (n0 + r >= N) break;
        const float wd = wdeq[(uint32_t)(n0 + r) / seg_rows];
        float e[VE];
#pragma unroll
        for (int j = 0; j < VE; ++j) e[j] = (float)((int)((code[r] >> (8 * (j & 3) + 2 * (part + (j >> 2)))) & 3u) - 1) * wd;
        T* row = out + (int64_t)(n0 + r) * K + k0;
        if (whole) {
            if constexpr (VE == 8) mmf_store8<T>(row, 0, VE, true, e);
            else *reinterpret_cast<float4*>(row) = make_float4(e[0], e[1], e[2], e[3]);
        } else {
            for (int j = 0; j < VE; ++j)
                if (k0 + j < K) row[j] = mmf_from_float<T>(e[j]);
        }
    }
}

// The same matrix stored [K, N]: the product dout @ W_q contracts over N, and the library's kernels run fastest where both
// operands are contiguous along the contraction.  8192 rows in bf16 on random data, [N, K] against [K, N]: 32000 x 2048 798 / 657 us,
// 11264 x 2048 300 / 242, 2048 x 5632 158 / 161; inside a training step of three layers the 19 products take 2797 / 2501 us (the step 10739 /
// 10544).  fp32 products take either in the same time (666 and 2002 rows, 1024 to 32000 outputs), so fp32
// weights are stored [N, K], 23 against 27 us at 32000 x 1024.  A thread owns one dword of codes (16 inputs) of VE neighbouring output rows, so a wave's store is 1 KiB of one input's row.
template <typename T>
__global__ __launch_bounds__(256) void unpack_dequant_t_kernel(const uint32_t* __restrict__ packed, const float* __restrict__ wdeq,
                                                               uint32_t seg_rows, int N, int K, int KB, bool whole, T* __restrict__ out) {
    constexpr int VE = 16 / (int)sizeof(T);
    const int n0 = ((int)blockIdx.x * 256 + (int)threadIdx.x) * VE;      // VE divides 32: one packed block
    if (n0 >= N) return;
    const int kb = (int)blockIdx.y >> 3, s = ((int)blockIdx.y >> 1) & 3, half = (int)blockIdx.y & 1;
    const int k0 = kb * 128 + s * 32 + half * 16;
    if (k0 >= K) return;
    const uint32_t* src = packed + (((int64_t)(n0 >> 5) * KB + kb) * 64 + half * 32 + (n0 & 31)) * 4 + s;
    uint32_t code[VE];
    float wd[VE];
#pragma unroll
    for (int r = 0; r < VE; ++r) code[r] = src[r * 4];                   // (rows are padded to 32 there)
    const uint32_t last = (uint32_t)(n0 + VE <= N ? n0 + VE : N) - 1, seg = (uint32_t)n0 / seg_rows;
    const bool one = last / seg_rows == seg;
#pragma unroll
    for (int r = 0; r < VE; ++r) wd[r] = one ? wdeq[seg] : wdeq[((uint32_t)n0 + r < last ? (uint32_t)n0 + r : last) / seg_rows];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        if (k0 + i >= K) break;
        float e[VE];
#pragma unroll
        for (int r = 0; r < VE; ++r) e[r] = (float)((int)((code[r] >> (8 * (i & 3) + 2 * (i >> 2))) & 3u) - 1) * wd[r];
        T* row = out + (int64_t)(k0 + i) * N + n0;
        if (whole) {
            if constexpr (VE == 8) mmf_store8<T>(row, 0, VE, true, e);
            else *reinterpret_cast<float4*>(row) = make_float4(e[0], e[1], e[2], e[3]);
        } else {
            for (int r = 0; r < VE; ++r)
                if (n0 + r < N) row[r] = mmf_from_float<T>(e[r]);
        }
    }
}

// out [cols, rows] = x [rows, cols] of 16-bit elements.  Bound by its 4 bytes an element (8192 x 2048: 12.6 us, 5.3 TB/s; the library's strided copy
// 74): a 64 x 64 tile passes through LDS, whole 128-byte lines in and
// out, 16 bytes a thread.  Rows of 33 dwords: the eight elements a thread gathers for its store, and its neighbours', fall on different banks.
template <bool VEC>
__global__ __launch_bounds__(256) void transpose16_kernel(const uint16_t* __restrict__ x, int rows, int cols, uint16_t* __restrict__ out) {
    __shared__ uint32_t tile[64][33];
    const int r0 = (int)blockIdx.y * 64, c0 = (int)blockIdx.x * 64, at = (int)threadIdx.x & 7, line = (int)threadIdx.x >> 3;
    uint4 v[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int r = r0 + line + 32 * h, c = c0 + at * 8;
        const uint16_t* p = x + (int64_t)r * cols + c;
        if constexpr (VEC) {
            if (r < rows && c < cols) v[h] = *reinterpret_cast<const uint4*>(p);
        } else {
            uint16_t e[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) e[i] = r < rows && c + i < cols ? p[i] : (uint16_t)0;
            __builtin_memcpy(&v[h], e, 16);
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t* t = &tile[line + 32 * h][at * 4];
        t[0] = v[h].x; t[1] = v[h].y; t[2] = v[h].z; t[3] = v[h].w;
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int cl = line + 32 * h, c = c0 + cl, r = r0 + at * 8;
        uint16_t e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = (uint16_t)(tile[at * 8 + i][cl >> 1] >> (16 * (cl & 1)));
        uint16_t* p = out + (int64_t)c * rows + r;
        if constexpr (VEC) {
            if (r < rows && c < cols) __builtin_memcpy(p, e, 16);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (r + i < rows && c < cols) p[i] = e[i];
        }
    }
}

}  // namespace

extern "C" {

int mmf_chain_bwd_groups(int64_t rows) { return (int)(rows < 1 ? 1 : rows < 1024 ? rows : 1024); }

int mmf_chain_bwd(int kind, const void* x, int64_t ldx, const void* aux, int64_t ldaux, const void* w1, float eps1, int norms,
                  const void* const* w2, float eps2, const void* const* dy, int64_t lddy, const void* dres, void* dx, int64_t lddx,
                  void* daux, int64_t lddaux, void* y, float* part, void* dweights, int64_t M, int64_t K, int x_dtype, int weight_dtype,
                  void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (kind < CHAIN_NORM || kind > CHAIN_RESNORM || M < 0 || K <= 0 || ldx < K || lddy < K || lddx < K) return MMF_ERR_ARG;
    if (M == 0) return 0;
    if (!(norms == 1 || (norms == 3 && kind == CHAIN_NORM)) || !x || !w2 || !dy || !dx || !y || !part || !dweights) return MMF_ERR_ARG;
    if (kind != CHAIN_SWIGLU && !w1) return MMF_ERR_ARG;
    if (kind != CHAIN_NORM && (!aux || ldaux < K)) return MMF_ERR_ARG;
    const bool two = kind == CHAIN_GATED || kind == CHAIN_SWIGLU;             // gradients of both operands
    if (two && (!daux || lddaux < K || dres)) return MMF_ERR_ARG;
    if (K % 4 != 0 || K > 8192) return MMF_ERR_WIDE;
    ChainArgs a{};
    a.x = x; a.aux = aux; a.w1 = w1; a.dres = dres; a.dx = dx; a.daux = daux; a.y = y; a.part = part;
    for (int n = 0; n < norms; ++n) {
        if (!w2[n] || !dy[n]) return MMF_ERR_ARG;
        a.w2[n] = w2[n];
        a.dy[n] = dy[n];
    }
    a.M = M; a.ldx = ldx; a.ldaux = ldaux; a.lddy = lddy; a.lddx = lddx; a.lddaux = lddaux; a.K = (int)K;
    a.eps1 = eps1; a.eps2 = eps2; a.inv_K = 1.0 / (double)K;
    const uintptr_t xm = 4 * (x_dtype == MMF_F32 ? 4 : 2) - 1, wm = 4 * (weight_dtype == MMF_F32 ? 4 : 2) - 1;
    auto off = [](const void* p, uintptr_t m) { return (reinterpret_cast<uintptr_t>(p) & m) != 0; };
    for (int64_t ld : {ldx, kind != CHAIN_NORM ? ldaux : 0, lddy, lddx, two ? lddaux : 0})
        if (ld % 4 != 0) return MMF_ERR_ALIGN;
    for (const void* p : {x, aux, dres, (const void*)dx, (const void*)daux, (const void*)y, a.dy[0], a.dy[1], a.dy[2]})
        if (off(p, xm)) return MMF_ERR_ALIGN;
    for (const void* p : {w1, a.w2[0], a.w2[1], a.w2[2]})
        if (off(p, wm)) return MMF_ERR_ALIGN;
    if (off(part, 15)) return MMF_ERR_ALIGN;
    const bool wf32 = weight_dtype == MMF_F32;
    if (!wf32 && weight_dtype != x_dtype) return MMF_ERR_ARG;
    const int groups = mmf_chain_bwd_groups(M);
    switch (x_dtype) {
        case MMF_F32: return dispatch_chain<float, float>(a, kind, norms, groups, dweights, stream);
        case MMF_BF16: return wf32 ? dispatch_chain<bf16_t, float>(a, kind, norms, groups, dweights, stream)
                                   : dispatch_chain<bf16_t, bf16_t>(a, kind, norms, groups, dweights, stream);
        case MMF_F16: return wf32 ? dispatch_chain<f16_t, float>(a, kind, norms, groups, dweights, stream)
                                  : dispatch_chain<f16_t, f16_t>(a, kind, norms, groups, dweights, stream);
    }
    return MMF_ERR_ARG;
}

int mmf_unpack_dequant(const void* packed, const float* wdeq, int64_t seg_rows, int64_t N, int64_t K, void* out, int dtype,
                       void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (N <= 0 || K <= 0 || seg_rows <= 0 || !packed || !wdeq || !out) return MMF_ERR_ARG;
    if (K % 8 == 0 && (reinterpret_cast<uintptr_t>(out) & 15u)) return MMF_ERR_ALIGN;
    if (N > 0x7fffffff || K > 0x7fffffff || seg_rows > 0x7fffffff) return MMF_ERR_WIDE;
    const int64_t KB = mmf_ceil_div(K, 128), columns = mmf_ceil_div(K, 256 * (dtype == MMF_F32 ? 4 : 8));
    if (columns > 65535) return MMF_ERR_WIDE;
    const bool whole = K % (dtype == MMF_F32 ? 4 : 8) == 0 && (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
#define MMF_UD(T) unpack_dequant_kernel<T><<<dim3((unsigned)mmf_ceil_div(N, kUdRows), (unsigned)columns), 256, 0, stream>>>( \
        static_cast<const uint32_t*>(packed), wdeq, (uint32_t)seg_rows, (int)N, (int)K, (int)KB, whole, static_cast<T*>(out))
    switch (dtype) {
        case MMF_F32: MMF_UD(float); break;
        case MMF_BF16: MMF_UD(bf16_t); break;
        case MMF_F16: MMF_UD(f16_t); break;
        default: return MMF_ERR_ARG;
    }
#undef MMF_UD
    MMF_CHECK_LAUNCH();
    return 0;
}

int mmf_unpack_dequant_t(const void* packed, const float* wdeq, int64_t seg_rows, int64_t N, int64_t K, void* out, int dtype,
                         void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (N <= 0 || K <= 0 || seg_rows <= 0 || !packed || !wdeq || !out) return MMF_ERR_ARG;
    if (N > 0x7fffffff - 2048 || K > 0x7fffffff || seg_rows > 0x7fffffff) return MMF_ERR_WIDE;
    const int ve = dtype == MMF_F32 ? 4 : 8;
    const int64_t KB = mmf_ceil_div(K, 128);
    if (KB * 8 > 65535) return MMF_ERR_WIDE;
    const bool whole = N % ve == 0 && (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
#define MMF_UD(T) unpack_dequant_t_kernel<T><<<dim3((unsigned)mmf_ceil_div(N, 256 * ve), (unsigned)(KB * 8)), 256, 0, stream>>>( \
        static_cast<const uint32_t*>(packed), wdeq, (uint32_t)seg_rows, (int)N, (int)K, (int)KB, whole, static_cast<T*>(out))
    switch (dtype) {
        case MMF_F32: MMF_UD(float); break;
        case MMF_BF16: MMF_UD(bf16_t); break;
        case MMF_F16: MMF_UD(f16_t); break;
        default: return MMF_ERR_ARG;
    }
#undef MMF_UD
    MMF_CHECK_LAUNCH();
    return 0;
}

int mmf_transpose16(const void* x, int64_t rows, int64_t cols, void* out, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (rows < 0 || cols < 0 || (rows * cols > 0 && (!x || !out))) return MMF_ERR_ARG;
    if (rows * cols == 0) return 0;
    if (rows > 65535 * 64 || cols > 0x7fffffff) return MMF_ERR_WIDE;
    const bool vec = rows % 8 == 0 && cols % 8 == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0;
    const dim3 grid((unsigned)mmf_ceil_div(cols, 64), (unsigned)mmf_ceil_div(rows, 64));
    auto kern = vec ? transpose16_kernel<true> : transpose16_kernel<false>;
    kern<<<grid, 256, 0, stream>>>(static_cast<const uint16_t*>(x), (int)rows, (int)cols, static_cast<uint16_t*>(out));
    MMF_CHECK_LAUNCH();
    return 0;
}

}  // extern "C"
