// HGRN recurrence  h_t = g_t * h_{t-1} + x_t  and the gate math in front of it.
//
//   mmf_hgrn_recurrent : g is the decay itself (linear domain); strictly sequential
//                        arithmetic (multiply, round, add, round) like
//                        mmfreelm/ops/hgrn/recurrent_fuse.py:32-68 / ops/hgrn/naive.py:8-31.
//   mmf_hgrn_gate      : sigmoid / lower bound / swiglu / mask of
//                        mmfreelm/layers/hgrn_bit.py:113-120 as one elementwise pass.
//   mmf_hgrn_step      : the same gate math fused with one recurrence step (decode, T = 1).
//   mmf_hgrn_gate_scan : gate math and recurrence of whole sequences in one launch (prompts).
//
// Layout: x, g, o are [BH, T, D] contiguous; a lane owns one channel d, a wave 64
// consecutive channels (128 B per time step in bf16), a workgroup of 8 waves one
// 64-channel column of one (b, h).  Time is cut into chunks of 64 steps; a wave holds a
// whole chunk of x and g in registers, and the waves take turns ("baton" = running state
// in LDS): on its turn a wave runs its 64 dependent steps from registers and hands the
// state on, so the serial chain sees no memory latency while the other waves' loads and
// stores are in flight.
#include <type_traits>
#include "mmf_common.h"
#include "../../include/mmf.h"

namespace {

constexpr int kCH = 64;   // time steps per register-resident chunk

// -------------------------------------------------------------------------- recurrence
// A wave's memory work is spread over the rounds between its turns.  Issuing a chunk's 64
// stores and the next chunk's 128 loads in one go overruns the 64-deep vector-memory queue and
// puts a full memory round trip inside every round; here each of the four rounds after a turn
// issues 16 stores and 32 loads, so a round lasts as long as one wave's 64 dependent steps and
// the waiting waves keep ~40 KiB in flight.
//
// Every wave runs the same straight-line iteration (turn, four memory rounds, three idle
// rounds: eight barriers), entered `wave` barriers late, so the register arrays are never
// assigned under a branch and stay where they are.  Memory goes through buffer instructions:
// the resource holds the chunk base, the lane's byte offset sits in one VGPR and the row offset
// in one SGPR.  What must not happen is switched off without a branch: a resource of zero
// records turns the loads past the last chunk into zeros and drops the stores of the padding
// chunks, lanes past D carry an out-of-range offset, the tail chunk clamps its row index for
// loads and feeds the missing steps (g, x) = (1, -0), which leaves the state bit for bit.
template <typename R>
__device__ __forceinline__ R buf_load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    if constexpr (sizeof(R) == 4) return __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
    else return (R)__builtin_amdgcn_raw_buffer_load_b16(r, voff, soff, 0);
}
template <typename T>
__device__ __forceinline__ void buf_store(float v, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    if constexpr (sizeof(T) == 4) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, voff, soff, 0);
    } else {
        T t = mmf_from_float<T>(v);
        __builtin_amdgcn_raw_buffer_store_b16(mmf_bits16(t), r, voff, soff, 0);
    }
}
template <typename T, typename R>
__device__ __forceinline__ float raw_get(R v) {
    if constexpr (sizeof(T) == 4) return v;
    else return mmf_to_float(mmf_from_bits16<T>((uint16_t)v));
}

// Compile-time loop: the body sees its index as a constant from the front end on, so the
// register arrays below are split into scalars before any pass can turn a 16-bit array into
// packed pairs (packing would make every load wait for its neighbour inside the memory rounds).
template <int V> struct IntC { static constexpr int value = V; };
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) { f(IntC<B>{}); static_for<B + 1, E>(f); }
}

// Requires (checked by the launcher): 64 rows of D elements span < 2^31 bytes, Tlen / 64 < 2^30.
// NW waves per workgroup: 8 for long sequences (the schedule above); 4 or 2 when the sequence has
// at most 4 or 2 chunks, where more waves would only idle through the barriers - the memory
// rounds then carry two or all four quarters each.
template <typename T, int NW>
__global__ __launch_bounds__(64 * NW) void hgrn_recurrent_pipelined_kernel(const T* __restrict__ x, const T* __restrict__ g,
                                                                       const float* __restrict__ h0, T* __restrict__ o,
                                                                       float* __restrict__ ht, int64_t Tlen, int64_t D) {
    using R = typename std::conditional<sizeof(T) == 4, float, uint16_t>::type;
    constexpr int MR = NW >= 8 ? 4 : NW / 2;                    // memory rounds per iteration
    constexpr int QPR = 4 / MR;                                 // quarters per memory round
    constexpr int kRsrcFlags = 0x00020000;                      // raw buffer, 32-bit data format, no swizzle
    constexpr int kAll = 0x7fffffff;
    __shared__ float baton[64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t bh = blockIdx.y;
    const uint32_t d = blockIdx.x * 64u + lane;
    const bool active = d < D;
    const uint32_t voff = active ? d * (uint32_t)sizeof(T) : 0x80000000u;   // lanes past D: always out of range
    const int NC = (int)((Tlen + kCH - 1) / kCH);
    const int iters = (NC + NW - 1) / NW;
    const uint32_t rowb = (uint32_t)D * (uint32_t)sizeof(T);
    const int64_t chunkb = (int64_t)kCH * rowb;
    const char* xb = reinterpret_cast<const char*>(x + bh * Tlen * D);
    const char* gb = reinterpret_cast<const char*>(g + bh * Tlen * D);
    char* ob = reinterpret_cast<char*>(o + bh * Tlen * D);

    R xr[kCH], gr[kCH];
    float hs[kCH];

    auto rem_of = [&](int c) {                                  // steps of chunk c inside the sequence, as a scalar int
        return __builtin_amdgcn_readfirstlane((int)max((int64_t)0, min((int64_t)kCH, Tlen - (int64_t)c * kCH)));
    };

#define MMF_LOAD_QUARTER(c_, q_)                                                                                       \
    {                                                                                                                  \
        const int cc = (c_);                                                                                           \
        const int rem = rem_of(cc);                                                                                    \
        const int recs = cc < NC ? kAll : 0;                                                                           \
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)(xb + cc * chunkb), 0, recs, kRsrcFlags); \
        const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc((void*)(gb + cc * chunkb), 0, recs, kRsrcFlags); \
        static_for<16 * (q_), 16 * (q_) + 16>([&](auto I) __attribute__((always_inline)) {                             \
            constexpr int t = decltype(I)::value;                                                                      \
            const uint32_t so = (uint32_t)max(0, min(t, rem - 1)) * rowb; /* rows past the end re-read the last one */ \
            xr[t] = buf_load<R>(rx, voff, so);                                                                         \
            gr[t] = buf_load<R>(rg, voff, so);                                                                         \
        });                                                                                                            \
    }
#define MMF_STORE_QUARTER(c_, q_)                                                                                      \
    {                                                                                                                  \
        const int cc = (c_);                                                                                           \
        const int rem = rem_of(cc);                                                                                    \
        const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc((void*)(ob + cc * chunkb), 0, cc < NC ? kAll : 0, kRsrcFlags); \
        static_for<16 * (q_), 16 * (q_) + 16>([&](auto I) __attribute__((always_inline)) {                             \
            constexpr int t = decltype(I)::value;                                                                      \
            if (t < rem) buf_store<T>(hs[t], ro, voff, (uint32_t)t * rowb);                                            \
        });                                                                                                            \
    }

    if (wave == 0) baton[lane] = (h0 && active) ? h0[bh * D + d] : 0.0f;
    MMF_LOAD_QUARTER(wave, 0) MMF_LOAD_QUARTER(wave, 1) MMF_LOAD_QUARTER(wave, 2) MMF_LOAD_QUARTER(wave, 3)
    __syncthreads();
    for (int i = 0; i < wave; ++i) __syncthreads();              // wave w takes its first turn in round w

    for (int it = 0; it < iters; ++it) {
        const int c = it * NW + wave;
        {                                                        // my turn: chunk c, 64 dependent steps
            const int rem = rem_of(c);
            float h = baton[lane];
            if (rem == kCH) {                                    // full chunk: no selects on the serial chain's inputs
                static_for<0, kCH>([&](auto I) __attribute__((always_inline)) {
                    constexpr int t = decltype(I)::value;
                    const float gl = raw_get<T, R>(gr[t]);
                    h = __fadd_rn(__fmul_rn(gl, h), raw_get<T, R>(xr[t]));
                    hs[t] = h;
                });
            } else {
                static_for<0, kCH>([&](auto I) __attribute__((always_inline)) {
                    constexpr int t = decltype(I)::value;
                    const float gl = raw_get<T, R>(gr[t]);
                    const float gv = t < rem ? gl : 1.0f;
                    const float xv = t < rem ? raw_get<T, R>(xr[t]) : -0.0f;
                    h = __fadd_rn(__fmul_rn(gv, h), xv);
                    hs[t] = h;
                });
            }
            baton[lane] = h;
        }
        __syncthreads();
        static_for<0, MR>([&](auto RI) __attribute__((always_inline)) {
            static_for<0, QPR>([&](auto QI) __attribute__((always_inline)) {
                constexpr int q = decltype(RI)::value * QPR + decltype(QI)::value;
                MMF_STORE_QUARTER(c, q) MMF_LOAD_QUARTER(c + NW, q)
            });
            __syncthreads();
        });
#pragma unroll
        for (int i = 0; i < NW - 1 - MR; ++i) __syncthreads();   // idle rounds
    }
    for (int i = wave; i < NW - 1; ++i) __syncthreads();         // every wave passes the same number of barriers
    __syncthreads();
    if (ht && wave == 0 && active) ht[bh * D + d] = baton[lane];
#undef MMF_LOAD_QUARTER
#undef MMF_STORE_QUARTER
}

// -------------------------------------------------------------------------- gate math
// mmf_gate_n gives g_out and x_out, x_out zeroed where mask == 0.

// -------------------------------------------------------------------------- gate math and recurrence of a prompt in one launch
// o = scan of the gated (x, g), x and g never leaving the CU.  A workgroup owns CPW channels of one sequence; wave 0 runs the
// recurrence, the other 15 feed it: they load raw i and f two tiles ahead, do the gate math of the next tile into LDS (float2 per
// step and channel) and round and store the outputs of the tile before, while wave 0 walks the current tile -- per step one LDS
// read, multiply, add, LDS write -- at raised priority.  One LDS-only barrier per tile (a full one would wait for the loads ahead).
// HBM and the vector units bound it about equally (the gate math is ~55 issue slots an element, which a wave walking time alone
// would put behind the recurrence); with 16-channel workgroups even one sequence reaches 64 to 128 CUs.  CPW is the narrowest that
// leaves at most two workgroups per CU (wider blocks have longer rows to load, 32 bytes at 16 channels; the four blocks that share
// a 128-byte line run on one XCD).  A turn requests and stores the same number of vectors whatever the tile, past the sequence's
// ends through resources without records: the compiler then waits for one set of loads by count, where a store or load under a
// branch made it wait for everything in flight, a trip to memory in every turn.  Wave 0 reads its steps a group ahead into two
// sets of registers in turn, without copies between them.  bf16 in us, against branches, copies and the exact gate math, operands in the last-level
// cache: 8 x 2048 x 2048 95 -> 63, 16 x 900 x 1024 42 -> 28, 2 x 1001 x 2048 24 -> 17, 3 x 459 x 2048 16 -> 12, 64 x 32 x 2048 23 -> 17, 4 x 300 x 1024
// 9.5 -> 7.1, 1 x 77 x 1024 5.1 -> 4.7; in memory 8 x 2048 x 2048 takes 74 to 79.  With few columns time is wave 0's own, 12 ns a step (1 x 2048 x 1024
// 40 -> 28; half as many channels a workgroup: 28).  hgrn_gate_scan_kernel takes single channels (odd widths and strides, rows beyond 256 KiB), the kernel behind it pairs.
struct GateScanArgs {
    const void* i; const void* f;       // rows [B * T, D], row strides ldi, ldf
    const float* lb; const uint8_t* mask;
    const float* h0; float* ht;         // [B, D]
    void* o;                            // [B * T, D]
    int64_t ldi, ldf, D;
    int T;
    int span;                           // pairs: tiles between two shifts of the bases
};
__device__ __forceinline__ void lds_only_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Wave 0: time, tile after tile.  gx, hb: two tiles of (gate, input) and of states.
template <int CPW, int TT, int U>
__device__ __forceinline__ void walk_time(const GateScanArgs& a, const float2* gx, float* hb, int64_t d, bool active, int turns) {
    static_assert(TT % (2 * U) == 0, "the recurrence walks a full tile in pairs of groups");
    const int lane = threadIdx.x & 63, c = lane & (CPW - 1);
    const int64_t dd = active ? d : 0;
    __builtin_amdgcn_s_setprio(3);
    float h = a.h0 && active ? a.h0[(int64_t)blockIdx.y * a.D + dd] : 0.0f;
    lds_only_barrier();                                     // tile 0 is there
    for (int k = 0; k < turns; ++k) {
        const int n = a.T - k * TT < TT ? a.T - k * TT : TT;   // (<= 0 in the turn that evens their number)
        const float2* src = gx + (k & 1) * (TT * CPW) + c;
        float* dst = hb + (k & 1) * (TT * CPW) + c;
        float2 va[U], vb[U];                                // groups of steps, read one ahead
        auto read = [&](float2 (&v)[U], int j) __attribute__((always_inline)) {
            const float2* p = src + (j <= TT - U ? j : TT - U) * CPW;
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = p[u * CPW];
            __builtin_amdgcn_sched_barrier(0);              // in front of the group walked meanwhile, not behind it (2 x 1001: 17.7 -> 16.8 us)
        };
        auto walk = [&](const float2 (&v)[U], int j) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                h = __fadd_rn(__fmul_rn(v[u].x, h), v[u].y);
                dst[(j + u) * CPW] = h;
            }
        };
        auto walk_tail = [&](const float2 (&v)[U], int j) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (j + u < n) {
                    h = __fadd_rn(__fmul_rn(v[u].x, h), v[u].y);
                    dst[(j + u) * CPW] = h;
                }
            }
        };
        if (lane < CPW) {
            read(va, 0);
            int j = 0;
            for (; j + 2 * U <= n; j += 2 * U) {
                read(vb, j + U);
                walk(va, j);
                __builtin_amdgcn_sched_barrier(0);
                read(va, j + 2 * U);
                walk(vb, j + U);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (j + U <= n) {                               // what is left of the last tile
                read(vb, j + U);
                walk(va, j);
                walk_tail(vb, j + U);
            } else if (j < n) {
                walk_tail(va, j);
            }
        }
        lds_only_barrier();
    }
    if (a.ht && active && lane < CPW) a.ht[(int64_t)blockIdx.y * a.D + d] = h;
}

template <typename T, int CPW, int PASS, bool MASK>
__global__ __launch_bounds__(1024) void hgrn_gate_scan_kernel(GateScanArgs a) {
    constexpr int NP = 15, SPW = 64 / CPW, TT = NP * SPW * PASS, U = TT >= 60 ? 10 : 5;   // steps of a tile: 120 (60), 60 or 30
    __shared__ float2 gx[2][TT * CPW];
    __shared__ float hb[2][TT * CPW];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    unsigned cb = blockIdx.x;
    if (CPW == 16 && gridDim.x % 32 == 0) cb = (cb & ~31u) + (cb & 7u) * 4 + ((cb >> 3) & 3u);
    if (CPW == 32 && gridDim.x % 16 == 0) cb = (cb & ~15u) + (cb & 7u) * 2 + ((cb >> 3) & 1u);
    const int c = lane & (CPW - 1), sub = lane / CPW;
    const int64_t d = (int64_t)cb * CPW + c;
    const bool active = d < a.D;
    const int64_t dd = active ? d : 0, r0 = (int64_t)blockIdx.y * a.T;
    const int NT = (a.T + TT - 1) / TT, turns = NT + NT % 2;

    if (wave == 0) {
        walk_time<CPW, TT, U>(a, &gx[0][0], &hb[0][0], d, active, turns);
        return;
    }

    using R = typename std::conditional<sizeof(T) == 4, float, uint16_t>::type;
    constexpr int e = (int)sizeof(T), kRsrcFlags = 0x00020000;
    const int p = wave - 1;
    const float lb = a.lb ? a.lb[dd] : 0.0f;
    R ir[2][PASS], fr[2][PASS];
    uint8_t mr[2][PASS];
    auto at = [&](int q) __attribute__((always_inline)) { return (q * NP + p) * SPW + sub; };   // step of a tile
    const int ldi = (int)a.ldi * e, ldf = (int)a.ldf * e, ldo = (int)a.D * e;   // bytes; the launcher: a tile of rows fits 31 bits
    uint32_t oi[PASS], of[PASS], oo[PASS];                      // byte offsets into a tile's rows
#pragma unroll
    for (int q = 0; q < PASS; ++q) {
        oi[q] = (uint32_t)at(q) * (uint32_t)ldi + (uint32_t)dd * e;
        of[q] = (uint32_t)at(q) * (uint32_t)ldf + (uint32_t)dd * e;
        oo[q] = active ? (uint32_t)at(q) * (uint32_t)ldo + (uint32_t)dd * e : 0x80000000u;   // lanes past D store nothing
    }
    // the tile to load next and the tile to store next: bases, and the sequence's rows from there on (loads past them give zeros,
    // stores are dropped: a resource of no records)
    const char* ip = static_cast<const char*>(a.i) + r0 * ldi;
    const char* fp = static_cast<const char*>(a.f) + r0 * ldf;
    const uint8_t* mp = MASK ? a.mask + r0 : nullptr;
    char* op = static_cast<char*>(a.o) + r0 * ldo;
    int rows_in = a.T, rows_out = a.T;
    auto rsrc = [&](const void* base, int rows, int ld) __attribute__((always_inline)) {
        // (uniform values, which the compiler has to be told of pointers carried round the loop: it looped over lanes otherwise)
        const uint64_t b = (uint64_t)base;
        const uint32_t lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
        return __builtin_amdgcn_make_buffer_rsrc((void*)((uint64_t)hi << 32 | lo), 0,
                                                 __builtin_amdgcn_readfirstlane((rows < 0 ? 0 : rows < TT ? rows : TT) * ld), kRsrcFlags);
    };
    auto load = [&](auto S) __attribute__((always_inline)) {
        constexpr int s = decltype(S)::value;
        const __amdgpu_buffer_rsrc_t ti = rsrc(ip, rows_in, ldi), tf = rsrc(fp, rows_in, ldf);
#pragma unroll
        for (int q = 0; q < PASS; ++q) {
            ir[s][q] = buf_load<R>(ti, oi[q], 0);
            fr[s][q] = buf_load<R>(tf, of[q], 0);
        }
        if constexpr (MASK) {
            const __amdgpu_buffer_rsrc_t tm = rsrc(mp, rows_in, 1);
#pragma unroll
            for (int q = 0; q < PASS; ++q) mr[s][q] = (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(tm, (uint32_t)at(q), 0, 0);
            mp += TT;
        }
        ip += (int64_t)TT * ldi;
        fp += (int64_t)TT * ldf;
        rows_in -= TT;
    };
    auto gates = [&](int k, auto S) __attribute__((always_inline)) {
        constexpr int s = decltype(S)::value;
        float iv[PASS], fv[PASS], lbv[PASS], xo[PASS], go[PASS];
#pragma unroll
        for (int q = 0; q < PASS; ++q) {
            iv[q] = raw_get<T, R>(ir[s][q]);
            fv[q] = raw_get<T, R>(fr[s][q]);
            lbv[q] = lb;
        }
        mmf_gate_n<T, PASS>(iv, fv, lbv, xo, go);
#pragma unroll
        for (int q = 0; q < PASS; ++q) {
            if constexpr (MASK) xo[q] = mr[s][q] == 0 ? 0.0f : xo[q];
            gx[k & 1][(q * NP + p) * 64 + lane] = make_float2(go[q], xo[q]);
        }
    };
    float hv[PASS];                                             // outputs on their way from LDS to memory
    auto fetch = [&](int k) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < PASS; ++q) hv[q] = hb[k & 1][(q * NP + p) * 64 + lane];
    };
    auto put = [&](int rows) __attribute__((always_inline)) {
        const __amdgpu_buffer_rsrc_t to = rsrc(op, rows, ldo);
#pragma unroll
        for (int q = 0; q < PASS; ++q) buf_store<T>(hv[q], to, oo[q], 0);
    };
    fetch(0);
    load(IntC<0>{});
    load(IntC<1>{});
    put(0);                                                     // nothing: the count of a turn
    gates(0, IntC<0>{});
    load(IntC<0>{});
    put(0);
    lds_only_barrier();
    // wave 0 walks tile k: store tile k - 1, whose outputs are read first and arrive under the arithmetic; prepare tile k + 1 (set S)
    auto turn = [&](int k, auto S) __attribute__((always_inline)) {
        fetch(k - 1);
        if (k + 1 < NT) gates(k + 1, S);
        load(S);
        put(k > 0 ? rows_out : 0);
        op += k > 0 ? (int64_t)TT * ldo : 0;
        rows_out -= k > 0 ? TT : 0;
        lds_only_barrier();
    };
    for (int k = 0; k < NT; k += 2) {                           // (an odd number of tiles: one more turn, of nothing but the last store)
        turn(k, IntC<1>{});
        turn(k + 1, IntC<0>{});
    }
    if (NT % 2 == 0) {
        fetch(NT - 1);
        put(rows_out);
    }
}

// The same where rows and pointers allow two channels at once: a lane takes a pair of channels of one step, so a turn is one request each for i, f
// and the store, and one LDS vector each way, instead of two, and the resources stand for the whole sequence: offsets advance by a vector add where the
// bases of every tile took some 70 scalar operations a turn.  NP waves feed the one that walks: 15, or 8 for up to 512 steps in 16-channel workgroups,
// whose tiles of 64 are sooner ready.  us, single channels / pairs, operands in memory (four sets in turn) and in the last-level cache: 8 x 2048 x 2048 bf16 79.2 / 58.0
// (3.5 TB/s) and 56.4 / 47.7, 16 x 1000 x 1024 36.1 / 30.5 and 26.6 / 25.4; about the same in both: 8 x 512 x 2048 16.8 / 15.8, 64 x 32 x 2048 16.6 / 14.5, 3 x 459 x 2048
// fp16 12.4 / 10.9, 1 x 77 x 1024 5.6 / 5.0; 1 x 2000 x 1024 27.6 / 27.4, the walk itself: 12.5 ns a step, two dependent operations and one LDS access.
// Boxes differ by up to 17 % (8 x 2048 x 2048 in memory 73.9 / 67.8 on another).  Where there are many columns the vector units bound it: there, with
// neither the test of the near forms nor their fall-back it took 42 us, without gate math 38.
template <typename T, int CPW, int NP, bool MASK>
__global__ __launch_bounds__(64 * (NP + 1)) void hgrn_gate_scan_pair_kernel(GateScanArgs a) {
    constexpr int CP = CPW / 2, SPW = 64 / CP, TT = NP * SPW, U = TT % 20 == 0 ? 10 : TT % 16 == 0 ? 8 : 5, e = (int)sizeof(T), kRsrcFlags = 0x00020000;
    __shared__ __align__(16) float2 gx[2][TT * CPW];
    __shared__ __align__(16) float hb[2][TT * CPW];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned cbs = ((unsigned)a.D + CPW - 1) / CPW;       // workgroups of a sequence
    unsigned cb = blockIdx.x;
    if (CPW == 16 && cbs % 32 == 0) cb = (cb & ~31u) + (cb & 7u) * 4 + ((cb >> 3) & 3u);
    if (CPW == 32 && cbs % 16 == 0) cb = (cb & ~15u) + (cb & 7u) * 2 + ((cb >> 3) & 1u);
    const int64_t r0 = (int64_t)blockIdx.y * a.T;
    const int NT = (a.T + TT - 1) / TT, turns = NT + NT % 2;
    if (wave == 0) {
        const int64_t d = (int64_t)cb * CPW + (lane & (CPW - 1));
        walk_time<CPW, TT, U>(a, &gx[0][0], &hb[0][0], d, d < a.D, turns);
        return;
    }
    using V = typename std::conditional<sizeof(T) == 4, uint2, uint32_t>::type;   // a pair as loaded
    const int p = wave - 1, D = (int)a.D;
    const int d = (int)cb * CPW + 2 * (lane % CP), dd = d < D ? d : 0;            // (D is even)
    const int step = p * SPW + lane / CP;
    const float lb0 = a.lb ? a.lb[dd] : 0.0f, lb1 = a.lb ? a.lb[dd + 1] : 0.0f;
    const int ldi = (int)a.ldi * e, ldf = (int)a.ldf * e, ldo = D * e;            // bytes
    const int tile_i = TT * ldi, tile_f = TT * ldf, tile_o = TT * ldo;
    const char* ip = static_cast<const char*>(a.i) + r0 * ldi;
    const char* fp = static_cast<const char*>(a.f) + r0 * ldf;
    const uint8_t* mp = MASK ? a.mask + r0 : nullptr;
    char* op = static_cast<char*>(a.o) + r0 * ldo;
    // Steps past the sequence load zeros and store nothing: their offsets lie past the resource's records.  So do those of the three stores in
    // front of the first tile's (unsigned, they wrap) and, by 2^31, those of lanes past D.
    uint32_t oi = (uint32_t)(step * ldi + dd * e), of = (uint32_t)(step * ldf + dd * e), om = (uint32_t)step;
    uint32_t oo = (d < D ? (uint32_t)(step * ldo + d * e) : 0x80000000u) - 3u * (uint32_t)tile_o;
    int rows = a.T, base = 0;                                   // of the sequence, from tile `base` on, where the bases stand
    auto records = [&](int ld) { return (rows < (a.span + 8) * TT ? rows : (a.span + 8) * TT) * ld; };
    auto rsrc = [&](const void* ptr, int ld) __attribute__((always_inline)) {
        const uint64_t b = (uint64_t)ptr;
        const uint32_t lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
        return __builtin_amdgcn_make_buffer_rsrc((void*)((uint64_t)hi << 32 | lo), 0, __builtin_amdgcn_readfirstlane(records(ld)), kRsrcFlags);
    };
    __amdgpu_buffer_rsrc_t ti = rsrc(ip, ldi), tf = rsrc(fp, ldf), to = rsrc(op, ldo), tm = rsrc(MASK ? (const void*)mp : ip, 1);
    V ir[2], fr[2];
    uint8_t mr[2];
    auto ld2 = [](__amdgpu_buffer_rsrc_t r, uint32_t off) __attribute__((always_inline)) {
        if constexpr (sizeof(T) == 4) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
            return make_uint2(v[0], v[1]);
        } else return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
    };
    auto load = [&](auto S) __attribute__((always_inline)) {
        constexpr int s = decltype(S)::value;
        ir[s] = ld2(ti, oi);
        fr[s] = ld2(tf, of);
        if constexpr (MASK) mr[s] = (uint8_t)__builtin_amdgcn_raw_buffer_load_b8(tm, om, 0, 0);
        oi += (uint32_t)tile_i;
        of += (uint32_t)tile_f;
        om += TT;
    };
    auto floats_of = [](V v, float (&f)[2]) __attribute__((always_inline)) {
        if constexpr (sizeof(T) == 4) { f[0] = __uint_as_float(v.x); f[1] = __uint_as_float(v.y); }
        else { f[0] = mmf_to_float(mmf_from_bits16<T>((uint16_t)v)); f[1] = mmf_to_float(mmf_from_bits16<T>((uint16_t)(v >> 16))); }
    };
    auto gates = [&](int k, auto S) __attribute__((always_inline)) {
        constexpr int s = decltype(S)::value;
        float iv[2], fv[2], xo[2], go[2];
        const float lbv[2] = {lb0, lb1};
        floats_of(ir[s], iv);
        floats_of(fr[s], fv);
        mmf_gate_n<T, 2>(iv, fv, lbv, xo, go);
        if constexpr (MASK) {
            xo[0] = mr[s] == 0 ? 0.0f : xo[0];
            xo[1] = mr[s] == 0 ? 0.0f : xo[1];
        }
        *reinterpret_cast<float4*>(&gx[k & 1][(p * 64 + lane) * 2]) = make_float4(go[0], xo[0], go[1], xo[1]);
    };
    float2 hv;                                                  // outputs on their way from LDS to memory
    auto fetch = [&](int k) __attribute__((always_inline)) { hv = *reinterpret_cast<const float2*>(&hb[k & 1][(p * 64 + lane) * 2]); };
    auto put = [&]() __attribute__((always_inline)) {
        if constexpr (sizeof(T) == 4) {
            typedef unsigned u2 __attribute__((ext_vector_type(2)));
            __builtin_amdgcn_raw_buffer_store_b64(u2{__float_as_uint(hv.x), __float_as_uint(hv.y)}, to, oo, 0, 0);
        } else {
            const uint32_t w = (uint32_t)mmf_bits16(mmf_from_float<T>(hv.x)) | (uint32_t)mmf_bits16(mmf_from_float<T>(hv.y)) << 16;
            __builtin_amdgcn_raw_buffer_store_b32(w, to, oo, 0, 0);
        }
        oo += (uint32_t)tile_o;
    };
    fetch(0);
    load(IntC<0>{});
    load(IntC<1>{});
    put();                                                      // nothing: the count of a turn
    gates(0, IntC<0>{});
    load(IntC<0>{});
    put();
    lds_only_barrier();
    // wave 0 walks tile k: store tile k - 1, whose outputs are read first and arrive under the arithmetic; prepare tile k + 1 (set S)
    auto turn = [&](int k, auto S) __attribute__((always_inline)) {
        if (k - base > a.span) {                                // offsets stay below 2^30: the bases move to tile k - 1
            const int n = k - 1 - base;
            base += n;
            rows -= n * TT;
            ip += (int64_t)n * tile_i; fp += (int64_t)n * tile_f; op += (int64_t)n * tile_o;
            oi -= (uint32_t)n * (uint32_t)tile_i; of -= (uint32_t)n * (uint32_t)tile_f; oo -= (uint32_t)n * (uint32_t)tile_o;
            ti = rsrc(ip, ldi); tf = rsrc(fp, ldf); to = rsrc(op, ldo);
            if constexpr (MASK) {
                mp += n * TT;
                om -= (uint32_t)(n * TT);
                tm = rsrc(mp, 1);
            }
        }
        fetch(k - 1);
        if (k + 1 < NT) gates(k + 1, S);
        load(S);
        put();
        lds_only_barrier();
    };
    for (int k = 0; k < NT; k += 2) {                           // (an odd number of tiles: one more turn, of nothing but the last store)
        turn(k, IntC<1>{});
        turn(k + 1, IntC<0>{});
    }
    if (NT % 2 == 0) {
        fetch(NT - 1);
        put();
    }
}

template <typename T, bool MASK>
int launch_gate_scan_masked(GateScanArgs a, int64_t B, hipStream_t s) {
    const int64_t D = a.D;
    auto grid = [&](int64_t cpw) { return dim3((unsigned)mmf_ceil_div(D, cpw), (unsigned)B); };
    auto even = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % (2 * sizeof(T)) == 0; };
    const int64_t row = (a.ldi > a.ldf ? a.ldi : a.ldf) * (int64_t)sizeof(T);   // (the outputs' rows, D, are no longer)
    // pairs of channels: faster at every size (hgrn_gate_scan_pair_kernel has the times); 2^18 bytes a row keep 16 tiles within 2^29
    if (D % 2 == 0 && a.ldi % 2 == 0 && a.ldf % 2 == 0 && even(a.i) && even(a.f) && even(a.o) && row <= (1 << 18)) {
        a.span = (int)((1 << 29) / (128 * row));                // at least 16; offsets reach (span + 8) tiles
        if (a.span > (1 << 20)) a.span = 1 << 20;
        if (B * mmf_ceil_div(D, (int64_t)16) <= 512) {
            if (a.T <= 512) hgrn_gate_scan_pair_kernel<T, 16, 8, MASK><<<grid(16), 64 * (8 + 1), 0, s>>>(a);
            else hgrn_gate_scan_pair_kernel<T, 16, 15, MASK><<<grid(16), 1024, 0, s>>>(a);
        } else if (B * mmf_ceil_div(D, (int64_t)32) <= 512) hgrn_gate_scan_pair_kernel<T, 32, 15, MASK><<<grid(32), 1024, 0, s>>>(a);
        else hgrn_gate_scan_pair_kernel<T, 64, 15, MASK><<<grid(64), 1024, 0, s>>>(a);
        MMF_CHECK_LAUNCH();
        return 0;
    }
    if (B * mmf_ceil_div(D, (int64_t)16) <= 512) {
        // short sequences: half the steps a tile, so that the recurrence starts sooner
        if (a.T <= 512) hgrn_gate_scan_kernel<T, 16, 1, MASK><<<grid(16), 1024, 0, s>>>(a);
        else hgrn_gate_scan_kernel<T, 16, 2, MASK><<<grid(16), 1024, 0, s>>>(a);
    } else if (B * mmf_ceil_div(D, (int64_t)32) <= 512) hgrn_gate_scan_kernel<T, 32, 2, MASK><<<grid(32), 1024, 0, s>>>(a);
    else hgrn_gate_scan_kernel<T, 64, 2, MASK><<<grid(64), 1024, 0, s>>>(a);
    MMF_CHECK_LAUNCH();
    return 0;
}
template <typename T>
int launch_gate_scan(const GateScanArgs& a, int64_t B, hipStream_t s) {
    return a.mask ? launch_gate_scan_masked<T, true>(a, B, s) : launch_gate_scan_masked<T, false>(a, B, s);
}

// One kernel for both forms: STEP = false writes (x, g); STEP = true runs one recurrence step on the
// fp32 state in place and writes o.  grid = (ceil(D / 1024), rows): a thread owns 4 consecutive
// channels of one row, so there is no index division and the loads are 8- / 16-byte vectors
// (VEC: D, the row strides and every pointer allow that; otherwise element accesses).
template <typename T, bool STEP, bool VEC>
__global__ __launch_bounds__(256) void hgrn_gate_kernel(const T* __restrict__ i_in, int64_t ldi, const T* __restrict__ f_in,
                                                        int64_t ldf, const float* __restrict__ lb,
                                                        const uint8_t* __restrict__ mask, float* __restrict__ state,
                                                        T* __restrict__ x_out, T* __restrict__ g_out, int D) {
    const int64_t r = blockIdx.y;
    const int d0 = ((int)blockIdx.x * 256 + (int)threadIdx.x) * 4;
    if (d0 >= D) return;
    const Raw4<T> iraw = raw4_load<T, VEC>(i_in + r * ldi, d0, D);
    const Raw4<T> fraw = raw4_load<T, VEC>(f_in + r * ldf, d0, D);
    Raw4<float> lbraw, straw;
    if (lb) lbraw = raw4_load<float, VEC>(lb, d0, D);
    if constexpr (STEP) straw = raw4_load<float, VEC>(state + r * D, d0, D);
    const bool keep = !(mask && mask[r] == 0);
    float iv[4], fv[4], lbv[4] = {0.0f, 0.0f, 0.0f, 0.0f}, stv[4], xo[4], go[4];
    raw4_unpack<T>(iraw, iv);
    raw4_unpack<T>(fraw, fv);
    if (lb) raw4_unpack<float>(lbraw, lbv);
    if constexpr (STEP) raw4_unpack<float>(straw, stv);
    // with no more workgroups than CUs the slowest wave counts, and the definition is the shorter chain: 64 x 2048 fp16 2.9 us, near 3.1
    if (gridDim.x * gridDim.y > 256) mmf_gate_n<T, 4>(iv, fv, lbv, xo, go);
    else mmf_gate_n<T, 4, false>(iv, fv, lbv, xo, go);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (!keep) xo[e] = 0.0f;
        if constexpr (STEP) {
            stv[e] = __fadd_rn(__fmul_rn(go[e], stv[e]), xo[e]);
            xo[e] = stv[e];                                     // o = T(h)
        }
    }
    if constexpr (STEP) raw4_store<float, VEC>(state + r * D, d0, D, stv);
    raw4_store<T, VEC>(x_out + r * D, d0, D, xo);
    if constexpr (!STEP) raw4_store<T, VEC>(g_out + r * D, d0, D, go);
}

// ht = h0 (or zeros) for an empty sequence; a kernel, not a memset, so it can be graph captured.
__global__ __launch_bounds__(256) void state_init_kernel(const float* __restrict__ h0, float* __restrict__ ht, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) ht[i] = h0 ? h0[i] : 0.0f;
}

// The kernel addresses a 64-step chunk with 32-bit offsets and counts chunks in an int.
template <typename T>
bool scan_fits(int64_t Tlen, int64_t D) {
    return mmf_ceil_div(Tlen, (int64_t)kCH) < (1 << 30) && (int64_t)kCH * D * (int64_t)sizeof(T) < (1ll << 31);
}

template <typename T>
int launch_scan(const void* x, const void* g, const float* h0, void* o, float* ht, int64_t BH, int64_t Tlen, int64_t D,
                hipStream_t s) {
    if (!scan_fits<T>(Tlen, D)) return MMF_ERR_WIDE;
    dim3 grid((unsigned)mmf_ceil_div(D, 64), (unsigned)BH);
    const int64_t NC = mmf_ceil_div(Tlen, (int64_t)kCH);
    const T* xp = static_cast<const T*>(x);
    const T* gp = static_cast<const T*>(g);
    T* op = static_cast<T*>(o);
    if (NC <= 2) hgrn_recurrent_pipelined_kernel<T, 2><<<grid, 128, 0, s>>>(xp, gp, h0, op, ht, Tlen, D);
    else if (NC <= 4) hgrn_recurrent_pipelined_kernel<T, 4><<<grid, 256, 0, s>>>(xp, gp, h0, op, ht, Tlen, D);
    else hgrn_recurrent_pipelined_kernel<T, 8><<<grid, 512, 0, s>>>(xp, gp, h0, op, ht, Tlen, D);
    MMF_CHECK_LAUNCH();
    return 0;
}

template <typename T>
int launch_gate(const void* i_in, int64_t ldi, const void* f_in, int64_t ldf, const float* lb, const uint8_t* mask,
                void* x_out, void* g_out, float* state, int64_t rows, int64_t D, bool step, hipStream_t s) {
    if (rows * D == 0) return 0;
    if (rows > 65535 * (int64_t)32768 || D > INT32_MAX - 4) return MMF_ERR_WIDE;
    auto al = [](const void* p, uintptr_t n) { return (reinterpret_cast<uintptr_t>(p) % n) == 0; };
    const uintptr_t ea = 4 * sizeof(T);
    const bool vec = D % 4 == 0 && ldi % 4 == 0 && ldf % 4 == 0 && al(i_in, ea) && al(f_in, ea) && al(x_out, ea) &&
                     al(g_out, ea) && al(lb, 16) && al(state, 16);
    const T* ip = static_cast<const T*>(i_in);
    const T* fp = static_cast<const T*>(f_in);
    T* xp = static_cast<T*>(x_out);
    T* gp = static_cast<T*>(g_out);
    const unsigned gx = (unsigned)mmf_ceil_div(D, (int64_t)1024);
    // rows go on grid.y (<= 65535 per launch)
    for (int64_t r0 = 0; r0 < rows; r0 += 65535) {
        const int64_t nr = rows - r0 < 65535 ? rows - r0 : 65535;
        dim3 grid(gx, (unsigned)nr);
        const T* ipr = ip + r0 * ldi;
        const T* fpr = fp + r0 * ldf;
        const uint8_t* mk = mask ? mask + r0 : nullptr;
        float* st = state ? state + r0 * D : nullptr;
        T* xpr = xp + r0 * D;
        T* gpr = gp ? gp + r0 * D : nullptr;
        if (step) {
            if (vec) hgrn_gate_kernel<T, true, true><<<grid, 256, 0, s>>>(ipr, ldi, fpr, ldf, lb, mk, st, xpr, gpr, (int)D);
            else hgrn_gate_kernel<T, true, false><<<grid, 256, 0, s>>>(ipr, ldi, fpr, ldf, lb, mk, st, xpr, gpr, (int)D);
        } else {
            if (vec) hgrn_gate_kernel<T, false, true><<<grid, 256, 0, s>>>(ipr, ldi, fpr, ldf, lb, mk, st, xpr, gpr, (int)D);
            else hgrn_gate_kernel<T, false, false><<<grid, 256, 0, s>>>(ipr, ldi, fpr, ldf, lb, mk, st, xpr, gpr, (int)D);
        }
        MMF_CHECK_LAUNCH();
    }
    return 0;
}

}  // namespace

extern "C" {

int mmf_hgrn_recurrent(const void* x, const void* g, const float* h0, void* o, float* ht, int64_t BH, int64_t T,
                       int64_t D, int dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (BH < 0 || T < 0 || D <= 0 || BH > 65535) return MMF_ERR_ARG;
    if (BH == 0) return 0;
    if (T == 0) {   // nothing to scan: the final state is the initial one
        if (ht) {
            state_init_kernel<<<(unsigned)mmf_ceil_div(BH * D, 256), 256, 0, stream>>>(h0, ht, BH * D);
            MMF_CHECK_LAUNCH();
        }
        return 0;
    }
    if (!x || !g || !o) return MMF_ERR_ARG;
    switch (dtype) {
        case MMF_F32: return launch_scan<float>(x, g, h0, o, ht, BH, T, D, stream);
        case MMF_BF16: return launch_scan<bf16_t>(x, g, h0, o, ht, BH, T, D, stream);
        case MMF_F16: return launch_scan<f16_t>(x, g, h0, o, ht, BH, T, D, stream);
    }
    return MMF_ERR_ARG;
}

int mmf_hgrn_gate_scan(const void* i_in, int64_t ldi, const void* f_in, int64_t ldf, const float* lower_bound, const uint8_t* mask,
                       const float* h0, void* o, float* ht, int64_t B, int64_t T, int64_t D, int dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (B < 0 || T < 0 || D <= 0 || ldi < D || ldf < D || B > 65535) return MMF_ERR_ARG;
    if (B == 0 || T == 0) return 0;
    if (!i_in || !f_in || !o) return MMF_ERR_ARG;
    if (T > (1 << 30) || ldi > (1 << 22) || ldf > (1 << 22)) return MMF_ERR_WIDE;   // a tile of 120 rows within 32-bit offsets
    GateScanArgs a{};
    a.i = i_in; a.f = f_in; a.lb = lower_bound; a.mask = mask; a.h0 = h0; a.ht = ht; a.o = o; a.ldi = ldi; a.ldf = ldf; a.D = D; a.T = (int)T;
    switch (dtype) {
        case MMF_F32: return launch_gate_scan<float>(a, B, stream);
        case MMF_BF16: return launch_gate_scan<bf16_t>(a, B, stream);
        case MMF_F16: return launch_gate_scan<f16_t>(a, B, stream);
    }
    return MMF_ERR_ARG;
}

int mmf_hgrn_gate(const void* i_in, int64_t ldi, const void* f_in, int64_t ldf, const float* lower_bound,
                  const uint8_t* mask, void* x_out, void* g_out, int64_t rows, int64_t D, int dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (rows < 0 || D <= 0 || ldi < D || ldf < D) return MMF_ERR_ARG;
    if (rows > 0 && (!i_in || !f_in || !x_out || !g_out)) return MMF_ERR_ARG;
    switch (dtype) {
        case MMF_F32: return launch_gate<float>(i_in, ldi, f_in, ldf, lower_bound, mask, x_out, g_out, nullptr, rows, D, false, stream);
        case MMF_BF16: return launch_gate<bf16_t>(i_in, ldi, f_in, ldf, lower_bound, mask, x_out, g_out, nullptr, rows, D, false, stream);
        case MMF_F16: return launch_gate<f16_t>(i_in, ldi, f_in, ldf, lower_bound, mask, x_out, g_out, nullptr, rows, D, false, stream);
    }
    return MMF_ERR_ARG;
}

int mmf_hgrn_step(const void* i_in, int64_t ldi, const void* f_in, int64_t ldf, const float* lower_bound,
                  const uint8_t* mask, float* state, void* o, int64_t rows, int64_t D, int dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (rows < 0 || D <= 0 || ldi < D || ldf < D) return MMF_ERR_ARG;
    if (rows > 0 && (!i_in || !f_in || !state || !o)) return MMF_ERR_ARG;
    switch (dtype) {
        case MMF_F32: return launch_gate<float>(i_in, ldi, f_in, ldf, lower_bound, mask, o, nullptr, state, rows, D, true, stream);
        case MMF_BF16: return launch_gate<bf16_t>(i_in, ldi, f_in, ldf, lower_bound, mask, o, nullptr, state, rows, D, true, stream);
        case MMF_F16: return launch_gate<f16_t>(i_in, ldi, f_in, ldf, lower_bound, mask, o, nullptr, state, rows, D, true, stream);
    }
    return MMF_ERR_ARG;
}

}  // extern "C"
