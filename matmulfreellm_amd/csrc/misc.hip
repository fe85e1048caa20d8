// Embedding row gather and greedy argmax: the two ends of a decode step, kept as plain
// kernels so the whole step can be captured into one HIP graph without library calls.
//
// mmf_embedding replaces nn.Embedding.forward at mmfreelm/models/hgrn_bit/modeling_hgrn_bit.py:212;
// mmf_argmax replaces the argmax over the vocabulary that greedy decoding performs on the
// logits of HGRNBitForCausalLM.forward (modeling_hgrn_bit.py:386).  Ties go to the lowest
// index (BitLinear logits are integer accumulators times two scalars, so exact ties happen).
#include "mmf_common.h"

namespace {

template <typename T>
__global__ __launch_bounds__(256) void embedding_kernel(const T* __restrict__ table, const int64_t* __restrict__ ids,
                                                        T* __restrict__ out, int64_t rows, int64_t H, int64_t vocab,
                                                        int64_t* __restrict__ history, int* __restrict__ pos, int cap) {
    const int64_t r = blockIdx.x;
    int64_t id = ids[r];
    if (history && threadIdx.x == 0) {   // a decode loop's record of what it fed: row r counts its own steps
        const int at = pos[r];
        history[(int64_t)at * rows + r] = id;
        pos[r] = at + 1 < cap ? at + 1 : 0;
    }
    if (id < 0 || id >= vocab) id = 0;   // out-of-range ids read row 0 instead of faulting
    const T* src = table + id * H;
    T* dst = out + r * H;
    constexpr int PER = 16 / (int)sizeof(T);
    if (H % PER == 0 && ((reinterpret_cast<uintptr_t>(table) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0) {
        // 16 bytes per thread: a 2048-wide 16-bit row is one load and one store per thread
        const uint4* s4 = reinterpret_cast<const uint4*>(src);
        uint4* d4 = reinterpret_cast<uint4*>(dst);
        for (int64_t c = threadIdx.x; c < H / PER; c += 256) d4[c] = s4[c];
    } else {
        for (int64_t c = threadIdx.x; c < H; c += 256) dst[c] = src[c];
    }
}

// One workgroup of 1024 threads per row, four vectors of 8 elements a thread requested before the first is looked at, so that a 32000-wide row costs one
// memory round trip.  First the largest value (one operation an element), then the lowest index that holds it, which only the
// threads whose own maximum it is look for: with an index carried beside every comparison a row took 8.5 us.  us, then and now: bf16 1 row 8.0 and 4.1, 64 rows 8.4
// and 4.6, 64 rows of 128000 22.6 and 8.7; fp32 64 rows 19.3 and 16.9.
// NaNs never win; a row of nothing else gives 0.
template <typename T>
__global__ __launch_bounds__(1024) void argmax_kernel(const T* __restrict__ logits, int64_t ld, int64_t V, int64_t* __restrict__ out) {
    constexpr int VECS = 4;
    __shared__ float top[16];
    __shared__ unsigned long long lowest;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const T* row = logits + (int64_t)blockIdx.x * ld;
    const bool vec_ok = (V % 8) == 0 && (ld % 8) == 0 && (reinterpret_cast<uintptr_t>(logits) & 15u) == 0;
    constexpr int64_t kPass = VECS * 1024 * 8;
    Raw8<T> raw[VECS];
    auto load = [&](int64_t at) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < VECS; ++c) raw[c] = mmf_load8_raw<T>(row, at + (c * 1024 + t) * 8, V, vec_ok);
    };
    float best = __builtin_nanf("");                            // NaN: nothing yet (fmaxf takes the other)
    int64_t where = 0, last = 0;                                // the pass this thread's maximum was first seen in, the pass in its registers
    for (int64_t at = 0; at < V; at += kPass) {
        load(at);
        last = at;
        float most = __builtin_nanf("");
#pragma unroll
        for (int c = 0; c < VECS; ++c) {
            float v[8];
            mmf_unpack8<T>(raw[c], v);
            const int64_t c0 = at + (c * 1024 + t) * 8;
            if (c0 + 8 <= V) {
#pragma unroll
                for (int i = 0; i < 8; ++i) most = fmaxf(most, v[i]);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) most = c0 + i < V ? fmaxf(most, v[i]) : most;
            }
        }
        if (most > best || (best != best && most == most)) { best = most; where = at; }
    }
    const float mine = mmf_wave_max(best);
    if (lane == 0) top[wave] = mine;
    if (t == 0) lowest = (unsigned long long)V;
    __syncthreads();
    float mx = top[0];
#pragma unroll
    for (int w = 1; w < 16; ++w) mx = fmaxf(mx, top[w]);
    if (best == mx) {
        if (where != last) load(where);
        unsigned long long idx = (unsigned long long)V;
#pragma unroll
        for (int c = VECS - 1; c >= 0; --c) {
            float v[8];
            mmf_unpack8<T>(raw[c], v);
            const int64_t c0 = where + (c * 1024 + t) * 8;
#pragma unroll
            for (int i = 7; i >= 0; --i)
                if (c0 + i < V && v[i] == mx) idx = (unsigned long long)(c0 + i);
        }
        atomicMin(&lowest, idx);
    }
    __syncthreads();
    if (t == 0) out[blockIdx.x] = lowest < (unsigned long long)V ? (int64_t)lowest : 0;
}


// Every float through the kernels' short forms of exp, the sigmoid, the reciprocal, the square root and 127 / a,
// against the sequences that define them.  counts[0..4]: arguments on which mmf_exp / mmf_sigmoid / mmf_rcp_pos /
// mmf_sqrt_pos / mmf_127_over differ from mmf_exp_definition / mmf_sigmoid_definition / __fdiv_rn(1, x) / sqrtf(x) /
// __fdiv_rn(127, x) (two NaNs count as equal); counts[5]: arguments seen; counts[6]: arguments that pass
// mmf_sigmoid_mid_ok and on which mmf_sigmoid_mid differs from the definition.  A grid-stride walk over all 2^32 bit patterns.
__global__ __launch_bounds__(256) void exact_forms_kernel(unsigned long long* counts) {
    unsigned long long bad[5] = {0, 0, 0, 0, 0}, seen = 0, bad_mid = 0;
    auto same = [](float a, float b) { return (a != a && b != b) || __float_as_uint(a) == __float_as_uint(b); };
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < (1ull << 32); i += stride) {
        const float x = __uint_as_float((uint32_t)i);
        ++seen;
        if (!same(mmf_exp(x), mmf_exp_definition(x))) ++bad[0];
        if (!same(mmf_sigmoid(x), mmf_sigmoid_definition(x))) ++bad[1];
        if (!same(mmf_rcp_pos(x), __fdiv_rn(1.0f, x))) ++bad[2];
        if (!same(mmf_sqrt_pos(x), sqrtf(x))) ++bad[3];
        if (!same(mmf_127_over(x), __fdiv_rn(127.0f, x))) ++bad[4];
        if (mmf_sigmoid_mid_ok(x) && !same(mmf_sigmoid_mid(x), mmf_sigmoid_definition(x))) ++bad_mid;
    }
#pragma unroll
    for (int j = 0; j < 5; ++j)
        if (bad[j]) atomicAdd(&counts[j], bad[j]);
    atomicAdd(&counts[5], seen);
    if (bad_mid) atomicAdd(&counts[6], bad_mid);
}

// counts[0]: floats x >= -87 where mmf_sigmoid_near(x) is further from 1 / (1 + exp(-x)) than mmf_near_slack allows it.
__global__ __launch_bounds__(256) void near_sigmoid_kernel(unsigned long long* counts) {
    unsigned long long bad = 0;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < (1ull << 32); i += stride) {
        const float x = __uint_as_float((uint32_t)i);
        if (!mmf_near_ok(x)) continue;
        const double d = (double)__fadd_rn(1.0f, mmf_exp(-x));
        if (x < 1e30f && fabs((double)mmf_sigmoid_near(x) * d - 1.0) > (3.0 + 1.25 * fabs((double)x)) * 0x1p-24) ++bad;
        if (x >= 1e30f && mmf_sigmoid_near(x) != 1.0f) ++bad;
    }
    if (bad) atomicAdd(&counts[0], bad);
}
// Each of the 65536 values of T as the argument of the activations, against `partners` values for the other operands: results whose
// bits differ from the definitions' (two NaNs count as equal).  counts[1..4]: swiglu, swish gate, gate math's g and x.
template <typename T>
__global__ __launch_bounds__(256) void near_forms_kernel(int partners, unsigned long long* counts) {
    unsigned long long bad[4] = {0, 0, 0, 0};
    const float a = mmf_to_float(mmf_from_bits16<T>((uint16_t)(blockIdx.x * 256 + threadIdx.x)));
    auto same = [](float p, float q) { return (p != p && q != q) || __float_as_uint(p) == __float_as_uint(q); };
    auto mix = [](uint32_t x) { x ^= x >> 16; x *= 0x7feb352du; x ^= x >> 15; x *= 0x846ca68bu; x ^= x >> 16; return x; };
    for (int j = blockIdx.y; j < partners; j += gridDim.y) {
        const uint32_t h = mix(blockIdx.x * 256 + threadIdx.x + 65536u * (uint32_t)j), h2 = mix(h + 0x9e3779b9u);
        // operands of every magnitude for a quarter of the partners, of an activation's for the rest
        const float wild = mmf_to_float(mmf_from_bits16<T>((uint16_t)h)), tame = ((float)(int)h2) * 0x1p-29f;
        const float u[1] = {mmf_round_to<T>((j & 3) == 0 ? wild : tame)}, y[1] = {(j & 3) == 0 ? __uint_as_float(h) : tame}, av[1] = {a};
        const float lb[1] = {(j & 1) == 0 ? 0.0f : (j & 7) == 1 ? wild : (float)(h2 >> 8) * 0x1p-24f};
        float o[1], x[1], g[1];
        mmf_swiglu_n<T, 1>(av, u, o);
        bad[0] += !same(o[0], mmf_round_to<T>(mmf_swiglu_definition(a, u[0])));
        mmf_swish_gate_n<T, 1>(y, av, o);
        bad[1] += !same(o[0], mmf_round_to<T>(__fmul_rn(__fmul_rn(y[0], a), mmf_sigmoid_definition(a))));
        mmf_gate_n<T, 1>(u, av, lb, x, g);
        const float gd = mmf_round_to<T>(mmf_gate_definition(mmf_sigmoid_definition(a), lb[0]));
        bad[2] += !same(g[0], gd);
        bad[3] += !same(x[0], mmf_round_to<T>(mmf_swiglu_definition(u[0], __fsub_rn(1.0f, gd))));
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (bad[j]) atomicAdd(&counts[1 + j], bad[j]);
}

}  // namespace

extern "C" {

int mmf_embedding_record(const void* table, const int64_t* ids, void* out, int64_t rows, int64_t H, int64_t vocab, int64_t* history,
                         int* pos, int cap, int dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (rows < 0 || H <= 0 || vocab <= 0 || (history && (!pos || cap <= 0))) return MMF_ERR_ARG;
    if (rows == 0) return 0;
    if (!table || !ids || !out) return MMF_ERR_ARG;
#define MMF_EM(T) embedding_kernel<T><<<(unsigned)rows, 256, 0, stream>>>(static_cast<const T*>(table), ids, static_cast<T*>(out), rows, H, \
                                                                         vocab, history, pos, cap)
    switch (dtype) {
        case MMF_F32: MMF_EM(float); break;
        case MMF_BF16: MMF_EM(bf16_t); break;
        case MMF_F16: MMF_EM(f16_t); break;
        default: return MMF_ERR_ARG;
    }
#undef MMF_EM
    MMF_CHECK_LAUNCH();
    return 0;
}

int mmf_embedding(const void* table, const int64_t* ids, void* out, int64_t rows, int64_t H, int64_t vocab, int dtype, void* stream) {
    return mmf_embedding_record(table, ids, out, rows, H, vocab, nullptr, nullptr, 0, dtype, stream);
}

int mmf_argmax(const void* logits, int64_t ld, int64_t rows, int64_t V, int64_t* out, int dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (rows < 0 || V <= 0 || ld < V) return MMF_ERR_ARG;
    if (rows == 0) return 0;
    if (!logits || !out) return MMF_ERR_ARG;
    switch (dtype) {
        case MMF_F32: argmax_kernel<float><<<(unsigned)rows, 1024, 0, stream>>>(static_cast<const float*>(logits), ld, V, out); break;
        case MMF_BF16: argmax_kernel<bf16_t><<<(unsigned)rows, 1024, 0, stream>>>(static_cast<const bf16_t*>(logits), ld, V, out); break;
        case MMF_F16: argmax_kernel<f16_t><<<(unsigned)rows, 1024, 0, stream>>>(static_cast<const f16_t*>(logits), ld, V, out); break;
        default: return MMF_ERR_ARG;
    }
    MMF_CHECK_LAUNCH();
    return 0;
}

int mmf_diag_check_exact_forms(unsigned long long* counts, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (!counts) return MMF_ERR_ARG;
    exact_forms_kernel<<<4096, 256, 0, stream>>>(counts);
    MMF_CHECK_LAUNCH();
    return 0;
}

int mmf_diag_check_near_forms(int partners, unsigned long long* counts, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (!counts || partners < 1 || partners > (1 << 16)) return MMF_ERR_ARG;
    near_sigmoid_kernel<<<4096, 256, 0, stream>>>(counts);
    MMF_CHECK_LAUNCH();
    near_forms_kernel<bf16_t><<<dim3(256, 16), 256, 0, stream>>>(partners, counts);
    MMF_CHECK_LAUNCH();
    near_forms_kernel<f16_t><<<dim3(256, 16), 256, 0, stream>>>(partners, counts + 4);   // its results go to [5..8]
    MMF_CHECK_LAUNCH();
    return 0;
}

}  // extern "C"
