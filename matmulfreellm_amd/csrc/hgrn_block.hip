// The HGRN recurrence evaluated in register blocks, where the order of the additions is free: the forward on log gates and
// the backward of both forms.
//
//   mmf_hgrn_chunk          mmfreelm/ops/hgrn/chunk.py:49-116, 223-254:  h_t = exp(g_t) * h_{t-1} + x_t
//   mmf_hgrn_recurrent_bwd  mmfreelm/ops/hgrn/recurrent_fuse.py:89-133 (with log gates the gradient that chunk.py:137-220
//                           computes chunk-wise): time runs backwards, dh += do_t; dx_t = dh; dg_t = dh * h_{t-1}
//                           (* exp(g_t) for log gates); dh *= g_t (exp(g_t))
//
// HBM is the bound: three streams of [BH, T, D] pass through the forward once, five through the backward.  A lane owns a
// channel, a workgroup 64 channels of one sequence (or of one time segment of it), a wave register blocks of 24 steps
// (forward: 28):
//   1. it loads its block (the backward g, do and the outputs one step earlier; 56 or 72 loads in flight per lane, none
//      behind a branch);
//   2. local pass from zero: l = the block's own contribution to what leaves it, P = product of its gates;
//   3. its turn (blocks in order; the carry sits in LDS): ONE dependent step, carry = l + P * carry;
//   4. the recurrence once more, from the carry that entered, stores.
// The waves run steps 1, 2 and 4 concurrently; what is serial across blocks is step 3, a handful of instructions.
// Step 4 takes as many operations as l_t + P_t * carry per step would, in the same registers, and rounds each step once, as a
// sequential kernel with fused multiply-adds does.  Distance from 64 bits in fp32, relative to the sequential kernels (two roundings a
// step) that stood here before: 0.74 to 0.99 times.  With l_t + P_t * carry it was 1.03 to 1.13 times theirs, the final state up to 1.4 times.
// LS = 2: a workgroup owns 32 channels and the halves of a wave two consecutive runs of steps, for twice the workgroups.
// When there are still too few, a first launch (AGG) runs steps 1-3 only and leaves per time segment the pair (P, l); the
// second enters segment s with the fold carry = l_j + P_j * carry over the segments before (backward: behind) it.
// Measured, bf16, backward: 8 x 1024 x 2048 145 -> 40 us (4.1 TB/s), 64 x 16384 x 128 with log gates 2290 -> 369 us
// (3.6 TB/s), against a kernel that loaded under a branch per step, so one load after the other, and read g and do twice.
// 16 to 28 steps a block and 8 or 16 waves a workgroup lie within 10 % of each other.  Forward, bf16:
// 64 x 16384 x 128 317 -> 214 us (3.8 TB/s), 4 x 2048 x 2048 61 -> 28 us, against 64-step blocks that took a second exp per step
// for P_t and cut these shapes in time, two launches over x and g.
#include <type_traits>
#include "mmf_common.h"

namespace {

constexpr int kMaxWaves = 8, kFwdBlk = 28, kBwdBlk = 24;

template <typename T>
__device__ __forceinline__ uint32_t buf_bits(__amdgpu_buffer_rsrc_t r, uint32_t vo, uint32_t so) {   // a register per value: no packing of pairs
    if constexpr (sizeof(T) == 2) return (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, vo, so, 0);
    else return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, vo, so, 0);
}
template <typename T>
__device__ __forceinline__ void buf_put(__amdgpu_buffer_rsrc_t r, uint32_t vo, uint32_t so, float v) {
    if constexpr (sizeof(T) == 2) __builtin_amdgcn_raw_buffer_store_b16(mmf_bits16(mmf_from_float<T>(v)), r, vo, so, 0);
    else __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, vo, so, 0);
}
template <typename T>
__device__ __forceinline__ float bits_val(uint32_t v) {
    if constexpr (sizeof(T) == 2) return mmf_to_float(mmf_from_bits16<T>((uint16_t)v));
    else return __uint_as_float(v);
}
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const T* p) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0x7fffffff, 0x00020000);
}
// LS = 2: the two halves of a 128-byte row go to workgroups 8 apart, which run on one XCD and share its L2.
template <int LS>
__device__ __forceinline__ unsigned column_block() {
    return LS == 2 && gridDim.x % 16 == 0 ? (blockIdx.x & ~15u) + (blockIdx.x & 7u) * 2 + ((blockIdx.x >> 3) & 1u) : blockIdx.x;
}
__device__ __forceinline__ void wait_turn(int& turn, int n) {
    while (__hip_atomic_load(&turn, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) != n) __builtin_amdgcn_s_sleep(1);
}
// What the carry c makes of a run of steps with the product P and the own contribution l.  (A zero carry stays zero also where
// a product of gates beyond one has overflowed.)
__device__ __forceinline__ float fold(float l, float P, float c) { return c == 0.0f ? l : fmaf(P, c, l); }
// The parts of a wave's block in the order the scan takes them, k = 0 .. LS - 1 in lanes part(k): (lin, Pin) composes the parts
// in front of this lane's, (lb, Pb) all of them.
template <int LS, bool REVERSE>
__device__ __forceinline__ void compose_parts(float l, float P, int u, int ch, float& lin, float& Pin, float& lb, float& Pb) {
    lb = 0.0f;
    Pb = 1.0f;
#pragma unroll
    for (int i = 0; i < LS; ++i) {
        const int k = REVERSE ? LS - 1 - i : i;
        if (u == k) {
            lin = lb;
            Pin = Pb;
        }
        const float lk = LS > 1 ? __shfl(l, k * (64 / LS) + ch, 64) : l, Pk = LS > 1 ? __shfl(P, k * (64 / LS) + ch, 64) : P;
        lb = fold(lk, Pk, lb);
        Pb *= Pk;
    }
}

// -------------------------------------------------------------------------- forward, log gates
template <typename T, bool AGG, int LS>
__global__ __launch_bounds__(64 * kMaxWaves) void hgrn_scan_fwd_kernel(const T* __restrict__ x, const T* __restrict__ g,
                                                                       const float* __restrict__ h0, T* __restrict__ o,
                                                                       float* __restrict__ ht, float* __restrict__ agg,
                                                                       int64_t Tlen, int64_t D, int64_t seg_len, int NS) {
    constexpr int CH = 64 / LS, kBlk = kFwdBlk, kStep = LS * kBlk;      // channels of a workgroup, steps of a wave's block
    __shared__ float carry_h[CH], carry_p[CH];
    __shared__ int turn;
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), nw = (int)blockDim.x >> 6;
    const int ch = lane % CH, u = lane / CH;                            // channel, and which kBlk steps of the wave's block
    const int64_t bh = blockIdx.y;
    const int seg = (int)blockIdx.z;                                    // AGG: nobody folds the pair of the last segment
    const int64_t d = (int64_t)column_block<LS>() * CH + ch;
    const bool active = d < D;
    const int64_t dl = active ? d : D - 1;
    const uint32_t rowb = (uint32_t)D * (uint32_t)sizeof(T);
    const uint32_t cho = active ? (uint32_t)d * (uint32_t)sizeof(T) : 0x80000000u;    // lanes past D: out of range, nothing stored
    const uint32_t voff = cho + (uint32_t)(u * kBlk) * rowb;
    const int64_t t0 = (int64_t)seg * seg_len, t1 = t0 + seg_len < Tlen ? t0 + seg_len : Tlen;
    const int nblk = (int)((t1 - t0 + kStep - 1) / kStep);
    if (wave == 0) {
        float c = h0 && (!AGG || seg == 0) ? h0[bh * D + dl] : 0.0f;    // h0 enters the fold through segment 0's pair
        if constexpr (!AGG) {
            if (seg > 0) c = 0.0f;
            for (int j = 0; j < seg; ++j) {
                const float* ag = agg + (bh * NS + j) * 2 * D + dl;
                c = fold(ag[D], ag[0], c);
            }
        }
        carry_h[ch] = c;
        carry_p[ch] = 1.0f;
        if (lane == 0) turn = 0;
    }
    __syncthreads();
    // One block; FULL: it has all its steps (no tests), otherwise the tail of the segment.
    auto block = [&](int n, int64_t tb, int rem, auto full) __attribute__((always_inline)) {
        constexpr bool FULL = decltype(full)::value;
        const int64_t row0 = (bh * Tlen + tb) * D;
        const __amdgpu_buffer_rsrc_t rg = rsrc(g + row0), rx = rsrc(x + row0);
        const int remu = rem - u * kBlk;                                // steps of this lane's part
        uint32_t gr[kBlk], xr[kBlk];
#pragma unroll
        for (int t = 0; t < kBlk; ++t) {
            if constexpr (FULL) {
                gr[t] = buf_bits<T>(rg, voff, (uint32_t)t * rowb);
                xr[t] = buf_bits<T>(rx, voff, (uint32_t)t * rowb);
            } else {                                                     // rows past the end re-read the last one
                const int row = u * kBlk + t < rem ? u * kBlk + t : rem - 1;
                gr[t] = buf_bits<T>(rg, cho + (uint32_t)row * rowb, 0);
                xr[t] = buf_bits<T>(rx, cho + (uint32_t)row * rowb, 0);
            }
        }
        float l = 0.0f, P = 1.0f;
#pragma unroll
        for (int t = 0; t < kBlk; ++t) {
            float gl = __expf(bits_val<T>(gr[t])), xv = bits_val<T>(xr[t]);
            if constexpr (!FULL) {                                       // steps past the end: (g, x) = (1, 0) change nothing
                gl = t < remu ? gl : 1.0f;
                xv = t < remu ? xv : 0.0f;
            }
            l = fmaf(l, gl, xv);
            P *= gl;
            if constexpr (!AGG) {
                xr[t] = __float_as_uint(xv);
                gr[t] = __float_as_uint(gl);
            }
        }
        float lin, Pin, lb, Pb;
        compose_parts<LS, false>(l, P, u, ch, lin, Pin, lb, Pb);
        wait_turn(turn, n);
        const float cb = carry_h[ch];
        carry_h[ch] = fold(lb, Pb, cb);                                 // (the parts of a channel write the same value)
        if constexpr (AGG) carry_p[ch] *= Pb;
        __hip_atomic_store(&turn, n + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        if constexpr (!AGG) {
            const __amdgpu_buffer_rsrc_t ro = rsrc(o + row0);
            float h = fold(lin, Pin, cb);
#pragma unroll
            for (int t = 0; t < kBlk; ++t) {
                h = fmaf(h, __uint_as_float(gr[t]), __uint_as_float(xr[t]));
                if (FULL || t < remu) buf_put<T>(ro, voff, (uint32_t)t * rowb, h);
            }
            // (steps past the end have left h alone; the part that holds the last step knows the state)
            if (ht && seg == NS - 1 && n == nblk - 1 && active && u == (rem - 1) / kBlk) ht[bh * D + d] = h;
        }
    };
    for (int n = wave; n < nblk; n += nw) {
        const int64_t tb = t0 + (int64_t)n * kStep;
        const int rem = __builtin_amdgcn_readfirstlane((int)((t1 - tb) < (int64_t)kStep ? (t1 - tb) : (int64_t)kStep));
        if (rem == kStep) block(n, tb, rem, std::true_type{});
        else block(n, tb, rem, std::false_type{});
    }
    if constexpr (AGG) {
        if (wave == 0) {
            wait_turn(turn, nblk);
            if (active) {
                float* ag = agg + (bh * NS + seg) * 2 * D;
                ag[d] = carry_p[ch];
                ag[D + d] = carry_h[ch];
            }
        }
    }
}

// -------------------------------------------------------------------------- backward
template <typename T, bool LOG, bool AGG, int LS>
__global__ __launch_bounds__(64 * kMaxWaves) void hgrn_scan_bwd_kernel(const T* __restrict__ g, const T* __restrict__ o,
                                                                       const T* __restrict__ dout, const float* __restrict__ h0,
                                                                       T* __restrict__ dx, T* __restrict__ dg,
                                                                       float* __restrict__ agg, int64_t Tlen, int64_t D,
                                                                       int64_t seg_len, int NS) {
    constexpr int CH = 64 / LS, kBlk = kBwdBlk, kStep = LS * kBlk;                      // channels of a workgroup, steps of a wave's block
    __shared__ float carry_l[CH], carry_p[CH];
    __shared__ int turn;
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), nw = (int)blockDim.x >> 6;
    const int ch = lane % CH, u = lane / CH;                            // channel, and which kBlk steps of the wave's block
    const int64_t bh = blockIdx.y;
    const int seg = AGG ? (int)blockIdx.z + 1 : (int)blockIdx.z;       // nobody folds the pair of segment 0
    const int64_t d = (int64_t)column_block<LS>() * CH + ch;
    const bool active = d < D;
    const int64_t dl = active ? d : D - 1;
    const uint32_t rowb = (uint32_t)D * (uint32_t)sizeof(T);
    const uint32_t cho = active ? (uint32_t)d * (uint32_t)sizeof(T) : 0x80000000u;    // lanes past D: out of range, nothing stored
    const uint32_t voff = cho + (uint32_t)(u * kBlk) * rowb;
    const int64_t t0 = (int64_t)seg * seg_len, t1 = t0 + seg_len < Tlen ? t0 + seg_len : Tlen;
    const int nblk = (int)((t1 - t0 + kStep - 1) / kStep);
    const float hinit = !AGG && h0 ? h0[bh * D + dl] : 0.0f;
    if (wave == 0) {
        float c = 0.0f;
        if constexpr (!AGG) {
            for (int j = NS - 1; j > seg; --j) {
                const float* ag = agg + (bh * NS + j) * 2 * D + dl;
                c = fold(ag[D], ag[0], c);
            }
        }
        carry_l[ch] = c;
        carry_p[ch] = 1.0f;
        if (lane == 0) turn = 0;
    }
    __syncthreads();
    // One block; FULL: it has all its steps (no tests), otherwise the tail of the segment.
    auto block = [&](int n, int64_t tb, int rem, auto full) __attribute__((always_inline)) {
        constexpr bool FULL = decltype(full)::value;
        const int64_t row0 = (bh * Tlen + tb) * D;
        const __amdgpu_buffer_rsrc_t rg = rsrc(g + row0), rd = rsrc(dout + row0);
        const int back = tb > 0 ? 1 : 0;                                // h_{t-1}: the outputs one row earlier
        const __amdgpu_buffer_rsrc_t ro = rsrc(o + row0 - (int64_t)back * D);
        const uint32_t first = back ? rowb : 0u;                        // where the block's second step finds its h
        const int remu = rem - u * kBlk;                                // steps of this lane's part
        uint32_t gr[kBlk], dr[kBlk], hr[kBlk];
#pragma unroll
        for (int t = kBlk - 1; t >= 0; --t) {
            if constexpr (FULL) {
                gr[t] = buf_bits<T>(rg, voff, (uint32_t)t * rowb);
                dr[t] = buf_bits<T>(rd, voff, (uint32_t)t * rowb);
                if constexpr (!AGG) {
                    if (t > 0) hr[t] = buf_bits<T>(ro, voff, (uint32_t)(t - 1) * rowb + first);
                    else hr[t] = buf_bits<T>(ro, back || u == 0 ? voff : voff - rowb, 0);
                }
            } else {                                                     // rows past the end re-read the last one
                const int row = u * kBlk + t < rem ? u * kBlk + t : rem - 1, prev = row - 1 + back;
                gr[t] = buf_bits<T>(rg, cho + (uint32_t)row * rowb, 0);
                dr[t] = buf_bits<T>(rd, cho + (uint32_t)row * rowb, 0);
                if constexpr (!AGG) hr[t] = buf_bits<T>(ro, cho + (uint32_t)(prev > 0 ? prev : 0) * rowb, 0);
            }
        }
        float last = 0.0f, glast = 1.0f, P = 1.0f;                      // the step after t: its dh from zero, its gate
#pragma unroll
        for (int t = kBlk - 1; t >= 0; --t) {
            float gl = bits_val<T>(gr[t]), a = bits_val<T>(dr[t]);
            if constexpr (LOG) gl = __expf(gl);
            if constexpr (!FULL) {                                       // steps past the end: (g, do) = (1, 0) change nothing
                gl = t < remu ? gl : 1.0f;
                a = t < remu ? a : 0.0f;
            }
            if constexpr (!AGG) {
                float hv = bits_val<T>(hr[t]);
                if (t == 0) hv = back || u > 0 ? hv : hinit;
                hr[t] = __float_as_uint(LOG ? hv * gl : hv);
                dr[t] = __float_as_uint(a);
                gr[t] = __float_as_uint(gl);
            }
            a = fmaf(last, glast, a);
            last = a;
            glast = gl;
            P *= gl;
        }
        const float l = last * glast;
        float lin, Pin, lb, Pb;
        compose_parts<LS, true>(l, P, u, ch, lin, Pin, lb, Pb);
        wait_turn(turn, n);
        const float cb = carry_l[ch];
        carry_l[ch] = fold(lb, Pb, cb);                                 // (the parts of a channel write the same value)
        if constexpr (AGG) carry_p[ch] *= Pb;
        __hip_atomic_store(&turn, n + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        if constexpr (!AGG) {
            const __amdgpu_buffer_rsrc_t rx = rsrc(dx + row0), ry = rsrc(dg + row0);
            float dh = fold(lin, Pin, cb), gate = 1.0f;                 // of the step behind
#pragma unroll
            for (int t = kBlk - 1; t >= 0; --t) {
                dh = fmaf(dh, gate, __uint_as_float(dr[t]));
                gate = __uint_as_float(gr[t]);
                if (FULL || t < remu) {
                    buf_put<T>(rx, voff, (uint32_t)t * rowb, dh);
                    buf_put<T>(ry, voff, (uint32_t)t * rowb, dh * __uint_as_float(hr[t]));
                }
            }
        }
    };
    for (int n = wave; n < nblk; n += nw) {
        const int64_t tb = t0 + (int64_t)(nblk - 1 - n) * kStep;        // blocks from the latest to the earliest
        const int rem = __builtin_amdgcn_readfirstlane((int)((t1 - tb) < (int64_t)kStep ? (t1 - tb) : (int64_t)kStep));
        if (rem == kStep) block(n, tb, rem, std::true_type{});
        else block(n, tb, rem, std::false_type{});
    }
    if constexpr (AGG) {
        if (wave == 0) {
            wait_turn(turn, nblk);
            if (active) {
                float* ag = agg + (bh * NS + seg) * 2 * D;
                ag[d] = carry_p[ch];
                ag[D + d] = carry_l[ch];
            }
        }
    }
}

// wgs = workgroups that columns of 64 channels give.  From 256 on nothing is split.  From 128 on a column is halved (LS = 2:
// 55 -> 48 us for 4 x 2048 x 2048 bf16) rather than cut in time, whose pair launch reads two of the five streams again (68 us).
// Below, short sequences are halved too (8.5 -> 6 us for 2 x 333 x 1024 fp32); from 2048 steps on whole 128-byte rows
// (LS = 1: 113 against 126 us for 1 x 16384 x 2048) in time segments for about two workgroups per CU.  A segment is at
// least four blocks long.
struct Plan {
    int64_t seg_len;
    int NS, LS;
};
Plan plan(int64_t BH, int64_t Tlen, int64_t D, int blk, bool split) {
    Plan p;
    const int64_t wgs = BH * mmf_ceil_div(D, 64);
    p.LS = wgs < 256 && (wgs >= 128 || Tlen < 2048) ? 2 : 1;
    const int64_t now = BH * mmf_ceil_div(D, 64 / p.LS), step = p.LS * blk;
    int64_t ns = 1;
    if (split && now < 128) {
        const int64_t want = mmf_ceil_div(512, now), most = Tlen / (4 * step);
        ns = want < most ? want : most;
        ns = ns < 1 ? 1 : ns > 64 ? 64 : ns;
    }
    p.seg_len = mmf_round_up(mmf_ceil_div(Tlen, ns), step);
    p.NS = (int)mmf_ceil_div(Tlen, p.seg_len);
    return p;
}
// The forward cuts time only where few columns meet eight of the blocks that `chunk` makes (whole chunks, at most 8 and at most 64
// steps): there, and nowhere else, mmf_hgrn_chunk_workspace_bytes asks for a workspace, also where plan() then leaves the sequence whole.
bool fwd_takes_workspace(int64_t BH, int64_t Tlen, int64_t D, int chunk) {
    const int64_t block = (64 / chunk > 8 ? 8 : 64 / chunk) * (int64_t)chunk;
    return BH * mmf_ceil_div(D, 64) < 256 && Tlen >= 8 * block;
}
Plan fwd_plan(int64_t BH, int64_t Tlen, int64_t D, int chunk) { return plan(BH, Tlen, D, kFwdBlk, fwd_takes_workspace(BH, Tlen, D, chunk)); }
int64_t pair_bytes(const Plan& p, int64_t BH, int64_t D) { return p.NS > 1 ? BH * p.NS * 2 * D * (int64_t)sizeof(float) : 0; }
// The kernels address a block of at most 64 rows with 32-bit offsets and count blocks in an int.
bool fits(int64_t Tlen, int64_t D, int dtype) {
    return Tlen / kBwdBlk < (1ll << 30) && 64 * D * (int64_t)(dtype == MMF_F32 ? 4 : 2) < (1ll << 31);
}

template <typename T, int LS>
int launch_fwd_ls(const Plan& p, const T* x, const T* g, const float* h0, T* o, float* ht, float* agg, int64_t BH, int64_t Tlen,
                  int64_t D, hipStream_t s) {
    const int64_t nblk = p.seg_len / (LS * kFwdBlk);
    const unsigned threads = 64u * (unsigned)(nblk < kMaxWaves ? nblk : kMaxWaves), gx = (unsigned)mmf_ceil_div(D, 64 / LS);
    if (p.NS > 1) {
        hgrn_scan_fwd_kernel<T, true, LS><<<dim3(gx, (unsigned)BH, (unsigned)(p.NS - 1)), threads, 0, s>>>(x, g, h0, o, ht, agg, Tlen, D,
                                                                                                  p.seg_len, p.NS);
        MMF_CHECK_LAUNCH();
    }
    hgrn_scan_fwd_kernel<T, false, LS><<<dim3(gx, (unsigned)BH, (unsigned)p.NS), threads, 0, s>>>(x, g, h0, o, ht, agg, Tlen, D,
                                                                                         p.seg_len, p.NS);
    MMF_CHECK_LAUNCH();
    return 0;
}
template <typename T>
int launch_fwd(const void* x, const void* g, const float* h0, void* o, float* ht, float* agg, int64_t BH, int64_t Tlen, int64_t D,
               int chunk, hipStream_t s) {
    const Plan p = fwd_plan(BH, Tlen, D, chunk);
    if (p.NS > 1 && !agg) return MMF_ERR_ARG;
    const T* xp = static_cast<const T*>(x);
    const T* gp = static_cast<const T*>(g);
    T* op = static_cast<T*>(o);
    return p.LS == 2 ? launch_fwd_ls<T, 2>(p, xp, gp, h0, op, ht, agg, BH, Tlen, D, s)
                     : launch_fwd_ls<T, 1>(p, xp, gp, h0, op, ht, agg, BH, Tlen, D, s);
}

template <typename T, bool LOG, int LS>
int launch_bwd_ls(const Plan& p, const T* g, const T* o, const T* dout, const float* h0, T* dx, T* dg, float* agg, int64_t BH,
                  int64_t Tlen, int64_t D, hipStream_t s) {
    const int64_t nblk = p.seg_len / (LS * kBwdBlk);
    const unsigned threads = 64u * (unsigned)(nblk < kMaxWaves ? nblk : kMaxWaves), gx = (unsigned)mmf_ceil_div(D, 64 / LS);
    if (p.NS > 1) {
        hgrn_scan_bwd_kernel<T, LOG, true, LS><<<dim3(gx, (unsigned)BH, (unsigned)(p.NS - 1)), threads, 0, s>>>(
            g, o, dout, h0, dx, dg, agg, Tlen, D, p.seg_len, p.NS);
        MMF_CHECK_LAUNCH();
    }
    hgrn_scan_bwd_kernel<T, LOG, false, LS><<<dim3(gx, (unsigned)BH, (unsigned)p.NS), threads, 0, s>>>(g, o, dout, h0, dx, dg, agg, Tlen,
                                                                                              D, p.seg_len, p.NS);
    MMF_CHECK_LAUNCH();
    return 0;
}
template <typename T, bool LOG>
int launch_bwd(const void* g, const void* o, const void* dout, const float* h0, void* dx, void* dg, float* agg, int64_t BH,
               int64_t Tlen, int64_t D, hipStream_t s) {
    const Plan p = plan(BH, Tlen, D, kBwdBlk, agg != nullptr);
    const T* gp = static_cast<const T*>(g);
    const T* op = static_cast<const T*>(o);
    const T* dp = static_cast<const T*>(dout);
    T* xp = static_cast<T*>(dx);
    T* yp = static_cast<T*>(dg);
    return p.LS == 2 ? launch_bwd_ls<T, LOG, 2>(p, gp, op, dp, h0, xp, yp, agg, BH, Tlen, D, s)
                     : launch_bwd_ls<T, LOG, 1>(p, gp, op, dp, h0, xp, yp, agg, BH, Tlen, D, s);
}

// ht = h0 (or zeros) for an empty sequence; a kernel, not a memset, so it can be graph captured.
__global__ __launch_bounds__(256) void state_init_kernel(const float* __restrict__ h0, float* __restrict__ ht, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) ht[i] = h0 ? h0[i] : 0.0f;
}

}  // namespace

extern "C" {

// chunk: the reference's chunk length.  The register blocks play its part: it decides from which length on a sequence may be cut
// and changes the result by rounding at most.
int64_t mmf_hgrn_chunk_workspace_bytes(int64_t BH, int64_t T, int64_t D, int chunk) {
    if (BH <= 0 || T <= 0 || D <= 0 || chunk < 1 || chunk > 64) return 0;
    if (!fwd_takes_workspace(BH, T, D, chunk)) return 0;
    return BH * fwd_plan(BH, T, D, chunk).NS * 2 * D * (int64_t)sizeof(float);
}

int mmf_hgrn_chunk(const void* x, const void* g, const float* h0, void* o, float* ht, int64_t BH, int64_t T, int64_t D,
                   int chunk, int dtype, void* workspace, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (BH < 0 || T < 0 || D <= 0 || BH > 65535 || chunk < 1 || chunk > 64) return MMF_ERR_ARG;
    if (BH == 0) return 0;
    if (T == 0) {
        if (ht) {
            state_init_kernel<<<(unsigned)mmf_ceil_div(BH * D, 256), 256, 0, stream>>>(h0, ht, BH * D);
            MMF_CHECK_LAUNCH();
        }
        return 0;
    }
    if (!x || !g || !o) return MMF_ERR_ARG;
    if (!fits(T, D, dtype)) return MMF_ERR_WIDE;
    float* agg = static_cast<float*>(workspace);
    switch (dtype) {
        case MMF_F32: return launch_fwd<float>(x, g, h0, o, ht, agg, BH, T, D, chunk, stream);
        case MMF_BF16: return launch_fwd<bf16_t>(x, g, h0, o, ht, agg, BH, T, D, chunk, stream);
        case MMF_F16: return launch_fwd<f16_t>(x, g, h0, o, ht, agg, BH, T, D, chunk, stream);
    }
    return MMF_ERR_ARG;
}

int64_t mmf_hgrn_recurrent_bwd_workspace_bytes(int64_t BH, int64_t T, int64_t D) {
    if (BH <= 0 || T <= 0 || D <= 0) return 0;
    return pair_bytes(plan(BH, T, D, kBwdBlk, true), BH, D);
}

int mmf_hgrn_recurrent_bwd_split(const void* g, const void* o, const void* grad_o, const float* h0, void* dx, void* dg, int64_t BH,
                                 int64_t T, int64_t D, int log_gates, int dtype, void* workspace, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (BH < 0 || T < 0 || D <= 0 || BH > 65535) return MMF_ERR_ARG;
    if (BH == 0 || T == 0) return 0;
    if (!g || !o || !grad_o || !dx || !dg) return MMF_ERR_ARG;
    if (!fits(T, D, dtype)) return MMF_ERR_WIDE;
    float* agg = static_cast<float*>(workspace);
#define MMF_RB(T_) return log_gates ? launch_bwd<T_, true>(g, o, grad_o, h0, dx, dg, agg, BH, T, D, stream) \
                                    : launch_bwd<T_, false>(g, o, grad_o, h0, dx, dg, agg, BH, T, D, stream)
    switch (dtype) {
        case MMF_F32: MMF_RB(float);
        case MMF_BF16: MMF_RB(bf16_t);
        case MMF_F16: MMF_RB(f16_t);
    }
#undef MMF_RB
    return MMF_ERR_ARG;
}

int mmf_hgrn_recurrent_bwd(const void* g, const void* o, const void* grad_o, const float* h0, void* dx, void* dg, int64_t BH,
                           int64_t T, int64_t D, int log_gates, int dtype, void* stream) {
    return mmf_hgrn_recurrent_bwd_split(g, o, grad_o, h0, dx, dg, BH, T, D, log_gates, dtype, nullptr, stream);
}

}  // extern "C"
