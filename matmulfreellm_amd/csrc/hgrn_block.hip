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
// Measured, bf16, backward: 8 x 1024 x 2048 145 -> 36 us in a training step (4.7 TB/s), 64 x 16384 x 128 with log gates 2290 -> 254 us
// (5.3 TB/s), against a kernel that loaded under a branch per step, so one load after the other, and read g and do twice.
// 16 to 28 steps a block and 8 or 16 waves a workgroup lie within 10 % of each other.  Forward, bf16:
// 64 x 16384 x 128 317 -> 160 us (5.0 TB/s), 4 x 2048 x 2048 61 -> 28 us (20 with the tensors in the last-level cache), against 64-step blocks that took a second exp per step
// for P_t and cut these shapes in time, two launches over x and g.
#include <type_traits>
#include "mmf_common.h"

namespace {

constexpr int kMaxWaves = 8, kFwdBlk = 28, kBwdBlk = 24;

// NT: streamed past the caches (each value is read or written once).
template <typename T, bool NT>
__device__ __forceinline__ uint32_t buf_bits(__amdgpu_buffer_rsrc_t r, uint32_t vo, uint32_t so) {   // a register per value: no packing of pairs
    if constexpr (sizeof(T) == 2) return (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, vo, so, NT ? 2 : 0);
    else return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, vo, so, NT ? 2 : 0);
}
template <typename T, bool NT>
__device__ __forceinline__ void buf_put(__amdgpu_buffer_rsrc_t r, uint32_t vo, uint32_t so, float v) {
    if constexpr (sizeof(T) == 2) __builtin_amdgcn_raw_buffer_store_b16(mmf_bits16(mmf_from_float<T>(v)), r, vo, so, NT ? 2 : 0);
    else __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, vo, so, NT ? 2 : 0);
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
// The carry of a channel that enters block n, as one LDS word with the block's number beside the value: a poll that finds the
// number has the value, and passing it on is one write.  (A turn counter with the carries behind it cost two more trips through
// LDS a turn: 350 ns, 205 of the 208 us of 64 x 16384 x 128, whose 585 blocks follow one another.)
__device__ __forceinline__ void pass_carry(uint64_t& word, float c, int n) {
    __hip_atomic_store(&word, (uint64_t)(uint32_t)n << 32 | __float_as_uint(c), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ float take_carry(uint64_t& word, int n) {
    uint64_t w = __hip_atomic_load(&word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    while ((int)(w >> 32) != n) {                               // all lanes see the same number
        if ((int)(w >> 32) < n - 1) __builtin_amdgcn_s_sleep(1);   // not the next one in line: leave LDS to the others
        w = __hip_atomic_load(&word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    return __uint_as_float((uint32_t)w);
}
// AGG: the product of the gates in front of block n travels in a word of its own, so that it is taken in the blocks' order (grouped by wave, a product
// that stays in range can meet an infinite partial one, and NaN where another is zero).  Both words are read in one trip.
__device__ __forceinline__ float take_pair(uint64_t& word, uint64_t& word_p, int n, float& p) {
    uint64_t c, q;
    do {
        c = __hip_atomic_load(&word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        q = __hip_atomic_load(&word_p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    } while ((int)(c >> 32) != n || (int)(q >> 32) != n);
    p = __uint_as_float((uint32_t)q);
    return __uint_as_float((uint32_t)c);
}
// The local pass ends here.  Left to itself the compiler moves it behind the wait, next to the first use of its results, and the
// turns that were to be a handful of instructions each take the loads' latency and all the arithmetic of a block: 570 ns a turn
// (64 x 16384 x 128 on 128 workgroups: 333 us forward, 218 with this line).
__device__ __forceinline__ void done_before_the_turn(float& l, float& P, float& lin, float& Pin, float& lb, float& Pb) {
    asm volatile("" : "+v"(l), "+v"(P), "+v"(lin), "+v"(Pin), "+v"(lb), "+v"(Pb)::"memory");
}
// JOINT: G workgroups share a column; each claims the column's next superblock (a block for each wave) from a counter.  What enters superblock
// n travels in a word of memory per channel, number beside value as in LDS.  A member composes its waves' blocks before the carry
// arrives, so between taking it and passing it on lies one multiply-add.
// Every wait ends, however few members run at once and whatever else the GPU runs: a member works on what it has claimed, claims are in order,
// and so everything that it waits for is in the hands of a running member, whose own wait is for something earlier still.  (With every
// G-th superblock assigned to a member, members that run could wait for one that found no room beside other kernels.)  The polls are bounded
// all the same; one that gave up would go on with NaN, which the results show.
// A claim is made when the carry is there, in the order in which the carry passes: the members keep taking turns, and the claim travels while the block
// is stored.  Made earlier, the claims came in no particular order and the chain waited for loads (64 x 16384 x 128 bf16 forward: every G-th
// 156 us, claimed so 156, in front of a superblock's loads 171 to 174, behind them 178).
struct Joint {
    uint64_t* words;      // per column: 64 carries, and behind all of them a counter each; zeroed in front of the launch
    int G;                // members of a column
    int64_t BH, columns;
};
constexpr int kJointPolls = 1 << 22;                                    // seconds
__device__ __forceinline__ void pass_joint(uint64_t* word, float c, int n) {
    __hip_atomic_store(word, (uint64_t)(uint32_t)n << 32 | __float_as_uint(c), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float take_joint(uint64_t* word, int n) {
    uint64_t w = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (int i = 0; __builtin_amdgcn_ballot_w64((int)(w >> 32) != n) != 0 && i < kJointPolls; ++i) {
        __builtin_amdgcn_s_sleep(2);
        w = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return (int)(w >> 32) == n ? __uint_as_float((uint32_t)w) : __builtin_nanf("");
}
// What the carry c makes of a run of steps with the product P and the own contribution l.  (A zero carry stays zero also where
// a product of gates beyond one has overflowed.)
__device__ __forceinline__ float fold(float l, float P, float c) { return c == 0.0f ? l : fmaf(P, c, l); }
// A workgroup's work on a column: the superblock it holds, the one it has claimed to follow (thread 0), how many it has taken.
struct Turns {
    uint64_t* word;       // this lane's carry
    uint64_t* counter;
    uint64_t next;
    int n, taken;
};
struct JointLds {
    float2 pair[2][kMaxWaves][64];
    uint64_t next[2];                                                   // how many were taken | the next one
};
__device__ __forceinline__ uint64_t claim(uint64_t* counter) {
    uint32_t at = 0;                                                    // an offset of the lane's own: for a uniform address the compiler waits on the spot
    asm volatile("" : "+v"(at));
    uint64_t n = 0;
    if (threadIdx.x == 0) n = __hip_atomic_fetch_add(counter + at, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return n;
}
// The carry that enters this wave's block (l, P) of superblock t.n, whose `nw` waves all come here.  last: no superblock follows.
// Composed only while every block's product is at most one (and NaN nowhere): beyond, the product of eight overflows where a step for each block
// stays in range, and an infinite one that meets a zero gives NaN.  There the blocks are folded in one by one, as without members.
__device__ __forceinline__ float joint_carry(float l, float P, Turns& t, bool last, int wave, int nw, JointLds& lds, uint64_t* carry, float first) {
    const int lane = (int)threadIdx.x & 63, n = t.n;
    float2 (*pair)[64] = lds.pair[t.taken & 1];
    pair[wave][lane] = make_float2(l, P);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");     // LDS only: loads and stores stay in flight
    float lin = 0.0f, Pin = 1.0f, most = fabsf(P), least = most;
    for (int w = 0; w < wave; ++w) {
        const float2 q = pair[w][lane];
        lin = fold(q.x, q.y, lin);
        Pin *= q.y;
        most = fmaxf(most, fabsf(q.y));
        least = fminf(least, fabsf(q.y));
    }
    float Pt = P * Pin;
    const bool composed = __builtin_amdgcn_ballot_w64(!(most <= 1.0f) || Pt != Pt) == 0;
    // only a zero gate makes a product zero: an infinite carry stays infinite as it does block by block
    if (least > 0.0f) {
        Pin = Pin == 0.0f ? copysignf(0x1p-149f, Pin) : Pin;
        Pt = Pt == 0.0f ? copysignf(0x1p-149f, Pt) : Pt;
    }
    auto enter = [&](float c) __attribute__((always_inline)) {           // what the carry c of the superblock is in front of this wave's block
        if (composed) return fold(lin, Pin, c);
        for (int w = 0; w < wave; ++w) c = fold(pair[w][lane].x, pair[w][lane].y, c);
        return c;
    };
    float c;
    if (wave == nw - 1) {
        const float lt = fold(l, P, lin);
        c = n == 0 ? first : take_joint(t.word, n);
        if (!last) pass_joint(t.word, composed ? fold(lt, Pt, c) : fold(l, P, enter(c)), n + 1);
        pass_carry(carry[lane], c, n);
    } else {
        c = take_carry(carry[lane], n);
    }
    t.next = claim(t.counter);
    return enter(c);
}
// Which column a workgroup of a joint launch works on: the G members of a column follow one another on one XCD.
__device__ __forceinline__ bool joint_place(const Joint& jt, int64_t D, int64_t& bh, unsigned& cb, Turns& t) {
    const unsigned G = (unsigned)jt.G, nd = (unsigned)((D + 63) / 64), col = blockIdx.x / (8u * G) * 8u + blockIdx.x % 8u;
    bh = col / nd;
    cb = col % nd;
    t = Turns{jt.words + (int64_t)col * 64 + (threadIdx.x & 63), jt.words + jt.columns * 64 + col, 0, 0, 0};   // (lanes past D: words of their own)
    return bh < jt.BH;                                                  // columns are padded to eights
}
// run(n): the block n of a wave, through joint_carry; idle(): its part in that where the superblock has no block left for it.
template <typename Run, typename Idle>
__device__ __forceinline__ void joint_turns(Turns& t, JointLds& lds, int nblk, int wave, int nw, Run&& run, Idle&& idle) {
    while (t.n * nw < nblk) {
        if (t.n * nw + wave < nblk) run(t.n * nw + wave);
        else idle();
        uint64_t* const slot = &lds.next[t.taken & 1];                  // (written again two superblocks on, a barrier behind everyone's read)
        if (threadIdx.x == 0) __hip_atomic_store(slot, (uint64_t)(uint32_t)(t.taken + 1) << 32 | (uint32_t)t.next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        ++t.taken;
        uint64_t w;
        do w = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        while ((int)(w >> 32) != t.taken);
        t.n = __builtin_amdgcn_readfirstlane((int)w);
    }
}
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

// ONE: halved columns that are not cut have at most one workgroup a CU and use the registers they need; held to 128 for two of them, their 16-bit backward
// took 7.4 for 6.8 us (8 x 333 x 1024, linear gates), 9.5 for 8.8 (8 x 500 x 1024 fp16), 6.2 for 5.6 (2 x 333 x 1024).  (Cut ones have two, and took 11.4
// for 10.2 us without the limit: 2 x 1000 x 1024.)
template <typename T, bool AGG, int LS, bool NT, bool JOINT, bool ONE = false>
__global__ __launch_bounds__(64 * kMaxWaves, ONE ? 2 : 4) void hgrn_scan_fwd_kernel(const T* __restrict__ x, const T* __restrict__ g,
                                                                       const float* __restrict__ h0, T* __restrict__ o,
                                                                       float* __restrict__ ht, float* __restrict__ agg,
                                                                       int64_t Tlen, int64_t D, int64_t seg_len, int NS, Joint jt) {
    constexpr int CH = 64 / LS, kBlk = kFwdBlk, kStep = LS * kBlk;      // channels of a workgroup, steps of a wave's block
    __shared__ uint64_t carry[CH];
    __shared__ uint64_t carry_p[AGG ? CH : 1];
    __shared__ typename std::conditional<JOINT, JointLds, int>::type joint_lds;
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), nw = (int)blockDim.x >> 6;
    const int ch = lane % CH, u = lane / CH;                            // channel, and which kBlk steps of the wave's block
    int64_t bh = blockIdx.y;
    const int seg = JOINT ? 0 : (int)blockIdx.z;                        // AGG: nobody folds the pair of the last segment
    unsigned cb = JOINT ? 0u : column_block<LS>();
    Turns turns{};
    if constexpr (JOINT) {
        if (!joint_place(jt, D, bh, cb, turns)) return;
    }
    const int64_t d = (int64_t)cb * CH + ch;
    const bool active = d < D;
    const int64_t dl = active ? d : D - 1;
    const uint32_t rowb = (uint32_t)D * (uint32_t)sizeof(T);
    const uint32_t cho = active ? (uint32_t)d * (uint32_t)sizeof(T) : 0x80000000u;    // lanes past D: out of range, nothing stored
    const uint32_t voff = cho + (uint32_t)(u * kBlk) * rowb;
    const int64_t t0 = (int64_t)seg * seg_len, t1 = t0 + seg_len < Tlen ? t0 + seg_len : Tlen;
    const int nblk = (int)((t1 - t0 + kStep - 1) / kStep);
    const float first = JOINT && h0 ? h0[bh * D + dl] : 0.0f;
    if constexpr (JOINT) {
        if (wave == 0) pass_carry(carry[ch], 0.0f, -1);
        const uint64_t n = claim(turns.counter);
        if (threadIdx.x == 0) {
            joint_lds.next[0] = 0;
            joint_lds.next[1] = (uint32_t)n;
        }
    }
    if (!JOINT && wave == 0) {
        float c = h0 && (!AGG || seg == 0) ? h0[bh * D + dl] : 0.0f;    // h0 enters the fold through segment 0's pair
        if constexpr (!AGG) {
            if (seg > 0) c = 0.0f;
            for (int j = 0; j < seg; ++j) {
                const float* ag = agg + (bh * NS + j) * 2 * D + dl;
                c = fold(ag[D], ag[0], c);
            }
        }
        pass_carry(carry[ch], c, 0);
        if constexpr (AGG) pass_carry(carry_p[ch], 1.0f, 0);
    }
    __syncthreads();
    if constexpr (JOINT) turns.n = __builtin_amdgcn_readfirstlane((int)joint_lds.next[1]);
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
                gr[t] = buf_bits<T, NT>(rg, voff, (uint32_t)t * rowb);
                xr[t] = buf_bits<T, NT>(rx, voff, (uint32_t)t * rowb);
            } else {                                                     // rows past the end re-read the last one
                const int row = u * kBlk + t < rem ? u * kBlk + t : rem - 1;
                gr[t] = buf_bits<T, NT>(rg, cho + (uint32_t)row * rowb, 0);
                xr[t] = buf_bits<T, NT>(rx, cho + (uint32_t)row * rowb, 0);
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
        done_before_the_turn(l, P, lin, Pin, lb, Pb);
        float cb;
        if constexpr (JOINT) {
            cb = joint_carry(lb, Pb, turns, (turns.n + 1) * nw >= nblk, wave, nw, joint_lds, carry, first);
        } else {
            float p = 1.0f;
            if constexpr (AGG) cb = take_pair(carry[ch], carry_p[ch], n, p);
            else cb = take_carry(carry[ch], n);
            pass_carry(carry[ch], fold(lb, Pb, cb), n + 1);             // (the parts of a channel write the same value)
            if constexpr (AGG) pass_carry(carry_p[ch], p * Pb, n + 1);
        }
        if constexpr (!AGG) {
            const __amdgpu_buffer_rsrc_t ro = rsrc(o + row0);
            float h = fold(lin, Pin, cb);
#pragma unroll
            for (int t = 0; t < kBlk; ++t) {
                h = fmaf(h, __uint_as_float(gr[t]), __uint_as_float(xr[t]));
                if (FULL || t < remu) buf_put<T, NT>(ro, voff, (uint32_t)t * rowb, h);
            }
            // (steps past the end have left h alone; the part that holds the last step knows the state)
            if (ht && seg == NS - 1 && n == nblk - 1 && active && u == (rem - 1) / kBlk) ht[bh * D + d] = h;
        }
    };
    auto run = [&](int n) __attribute__((always_inline)) {
        const int64_t tb = t0 + (int64_t)n * kStep;
        const int rem = __builtin_amdgcn_readfirstlane((int)((t1 - tb) < (int64_t)kStep ? (t1 - tb) : (int64_t)kStep));
        if (rem == kStep) block(n, tb, rem, std::true_type{});
        else block(n, tb, rem, std::false_type{});
    };
    if constexpr (JOINT) {
        joint_turns(turns, joint_lds, nblk, wave, nw, run, [&] { joint_carry(0.0f, 1.0f, turns, true, wave, nw, joint_lds, carry, first); });
    } else {
        for (int n = wave; n < nblk; n += nw) run(n);
    }
    if constexpr (AGG) {
        if (wave == 0) {
            float p;
            const float c = take_pair(carry[ch], carry_p[ch], nblk, p);
            if (active) {
                float* ag = agg + (bh * NS + seg) * 2 * D;
                ag[d] = p;
                ag[D + d] = c;
            }
        }
    }
}

// -------------------------------------------------------------------------- backward
template <typename T, bool LOG, bool AGG, int LS, bool NT, bool JOINT, bool ONE = false>
__global__ __launch_bounds__(64 * kMaxWaves, ONE ? 2 : 4) void hgrn_scan_bwd_kernel(const T* __restrict__ g, const T* __restrict__ o,
                                                                       const T* __restrict__ dout, const float* __restrict__ h0,
                                                                       T* __restrict__ dx, T* __restrict__ dg,
                                                                       float* __restrict__ agg, int64_t Tlen, int64_t D,
                                                                       int64_t seg_len, int NS, Joint jt) {
    constexpr int CH = 64 / LS, kBlk = kBwdBlk, kStep = LS * kBlk;                      // channels of a workgroup, steps of a wave's block
    __shared__ uint64_t carry[CH];
    __shared__ uint64_t carry_p[AGG ? CH : 1];
    __shared__ typename std::conditional<JOINT, JointLds, int>::type joint_lds;
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), nw = (int)blockDim.x >> 6;
    const int ch = lane % CH, u = lane / CH;                            // channel, and which kBlk steps of the wave's block
    int64_t bh = blockIdx.y;
    const int seg = JOINT ? 0 : AGG ? (int)blockIdx.z + 1 : (int)blockIdx.z;   // nobody folds the pair of segment 0
    unsigned cb = JOINT ? 0u : column_block<LS>();
    Turns turns{};
    if constexpr (JOINT) {
        if (!joint_place(jt, D, bh, cb, turns)) return;
    }
    const int64_t d = (int64_t)cb * CH + ch;
    const bool active = d < D;
    const int64_t dl = active ? d : D - 1;
    const uint32_t rowb = (uint32_t)D * (uint32_t)sizeof(T);
    const uint32_t cho = active ? (uint32_t)d * (uint32_t)sizeof(T) : 0x80000000u;    // lanes past D: out of range, nothing stored
    const uint32_t voff = cho + (uint32_t)(u * kBlk) * rowb;
    const int64_t t0 = (int64_t)seg * seg_len, t1 = t0 + seg_len < Tlen ? t0 + seg_len : Tlen;
    const int nblk = (int)((t1 - t0 + kStep - 1) / kStep);
    const float hinit = !AGG && h0 ? h0[bh * D + dl] : 0.0f;
    if constexpr (JOINT) {
        if (wave == 0) pass_carry(carry[ch], 0.0f, -1);
        const uint64_t n = claim(turns.counter);
        if (threadIdx.x == 0) {
            joint_lds.next[0] = 0;
            joint_lds.next[1] = (uint32_t)n;
        }
    }
    if (!JOINT && wave == 0) {
        float c = 0.0f;
        if constexpr (!AGG) {
            for (int j = NS - 1; j > seg; --j) {
                const float* ag = agg + (bh * NS + j) * 2 * D + dl;
                c = fold(ag[D], ag[0], c);
            }
        }
        pass_carry(carry[ch], c, 0);
        if constexpr (AGG) pass_carry(carry_p[ch], 1.0f, 0);
    }
    __syncthreads();
    if constexpr (JOINT) turns.n = __builtin_amdgcn_readfirstlane((int)joint_lds.next[1]);
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
                gr[t] = buf_bits<T, NT>(rg, voff, (uint32_t)t * rowb);
                dr[t] = buf_bits<T, NT>(rd, voff, (uint32_t)t * rowb);
                if constexpr (!AGG) {
                    if (t > 0) hr[t] = buf_bits<T, NT>(ro, voff, (uint32_t)(t - 1) * rowb + first);
                    else hr[t] = buf_bits<T, NT>(ro, back || u == 0 ? voff : voff - rowb, 0);
                }
            } else {                                                     // rows past the end re-read the last one
                const int row = u * kBlk + t < rem ? u * kBlk + t : rem - 1, prev = row - 1 + back;
                gr[t] = buf_bits<T, NT>(rg, cho + (uint32_t)row * rowb, 0);
                dr[t] = buf_bits<T, NT>(rd, cho + (uint32_t)row * rowb, 0);
                if constexpr (!AGG) hr[t] = buf_bits<T, NT>(ro, cho + (uint32_t)(prev > 0 ? prev : 0) * rowb, 0);
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
        float l = last * glast;
        float lin, Pin, lb, Pb;
        compose_parts<LS, true>(l, P, u, ch, lin, Pin, lb, Pb);
        done_before_the_turn(l, P, lin, Pin, lb, Pb);
        float cb;
        if constexpr (JOINT) {
            cb = joint_carry(lb, Pb, turns, (turns.n + 1) * nw >= nblk, wave, nw, joint_lds, carry, 0.0f);
        } else {
            float p = 1.0f;
            if constexpr (AGG) cb = take_pair(carry[ch], carry_p[ch], n, p);
            else cb = take_carry(carry[ch], n);
            pass_carry(carry[ch], fold(lb, Pb, cb), n + 1);             // (the parts of a channel write the same value)
            if constexpr (AGG) pass_carry(carry_p[ch], p * Pb, n + 1);
        }
        if constexpr (!AGG) {
            const __amdgpu_buffer_rsrc_t rx = rsrc(dx + row0), ry = rsrc(dg + row0);
            float dh = fold(lin, Pin, cb), gate = 1.0f;                 // of the step behind
#pragma unroll
            for (int t = kBlk - 1; t >= 0; --t) {
                dh = fmaf(dh, gate, __uint_as_float(dr[t]));
                gate = __uint_as_float(gr[t]);
                if (FULL || t < remu) {
                    buf_put<T, NT>(rx, voff, (uint32_t)t * rowb, dh);
                    buf_put<T, NT>(ry, voff, (uint32_t)t * rowb, dh * __uint_as_float(hr[t]));
                }
            }
        }
    };
    auto run = [&](int n) __attribute__((always_inline)) {
        const int64_t tb = t0 + (int64_t)(nblk - 1 - n) * kStep;        // blocks from the latest to the earliest
        const int rem = __builtin_amdgcn_readfirstlane((int)((t1 - tb) < (int64_t)kStep ? (t1 - tb) : (int64_t)kStep));
        if (rem == kStep) block(n, tb, rem, std::true_type{});
        else block(n, tb, rem, std::false_type{});
    };
    if constexpr (JOINT) {
        joint_turns(turns, joint_lds, nblk, wave, nw, run, [&] { joint_carry(0.0f, 1.0f, turns, true, wave, nw, joint_lds, carry, 0.0f); });
    } else {
        for (int n = wave; n < nblk; n += nw) run(n);
    }
    if constexpr (AGG) {
        if (wave == 0) {
            float p;
            const float c = take_pair(carry[ch], carry_p[ch], nblk, p);
            if (active) {
                float* ag = agg + (bh * NS + seg) * 2 * D;
                ag[d] = p;
                ag[D + d] = c;
            }
        }
    }
}

// wgs = workgroups that columns of 64 channels give.  A CU keeps about 60 KB of loads in flight, whole 128-byte lines, so fewer workgroups
// than CUs leave bandwidth unused: 128 of them reach 3.7 TB/s where 256 reach 5.2.  From 171 on nothing is split.
//   32 to 170, long sequences: G workgroups share a column's superblocks (JOINT), about 256 workgroups up to 64 columns and 512 (two a CU)
//      beyond.  bf16, forward + backward against the plans below: 64 x 16384 x 128 220 + 374 -> 160 + 262 us, 6 x 16384 x 1024 189 + 277 ->
//      136 + 220, 16 x 16384 x 128 64 + 84 -> 50 + 71, 9 x 5000 x 1024 74 + 124 -> 69 + 109.  Below 3072 steps the hand-overs between
//      workgroups show (64 x 2048 x 64 18 + 22 against 18 + 24, 7 x 1024 x 1024 11 + 16 against 17 + 22), below 32 columns the cut in time is as
//      good (24 x 16384 x 64 48 + 63 / 48 + 64, 8 x 16384 x 64 28 + 31 / 45 + 60).
//   up to 128, where they are not shared: a column is halved (LS = 2; 8.5 -> 6 us for 2 x 333 x 1024 fp32), at half a line a row and so half the
//      bytes in flight; with more columns than that whole ones win at every length (12 x 2048 x 1024 35 + 58 against 50 + 79; halved against whole,
//      forward + backward: 132 columns of 150 to 2500 steps 6.0 + 7.8 / 5.7 + 7.3 to 46 + 71 / 33 + 50, 192 of 300 9.2 + 13.1 / 8.0 + 11.2; 128 of 300
//      6.6 + 9.6 / 7.6 + 10.8).
//   64 columns and fewer, in fp32 40 (half a column's row is a whole line there), 2048 steps and more: whole 128-byte rows in time segments for about two workgroups per CU, a segment at least four
//      blocks long; a first launch reads x and g (g and do) of all but one segment once more.  Halved against cut, forward + backward, 2500 steps, bf16 and
//      fp32: 56 columns 49 / 48 and 53 / 73, 66 columns 52 / 52 and 59 / 87, 80 (of 1024-wide rows) 52 / 66 and 78 / 104, 96 54 / 76 and 99 / 123, 112 57 / 88
//      and 116 / 143; 127 (of 64-wide rows, whose halves no neighbour shares) 87 / 90 and 122 / 155.  fp32 alone: 32 columns 47 to 53 / 44, 40 47 to 54 / 55,
//      44 48 / 61, 64 58 to 63 / 80 to 84.
struct Plan {
    int64_t seg_len;
    int NS, LS, G;
};
Plan plan(int64_t BH, int64_t Tlen, int64_t D, int blk, bool split, bool joint, int elem) {
    Plan p;
    const int64_t wgs = BH * mmf_ceil_div(D, 64);
    p.G = joint && wgs >= 32 && wgs <= 170 && Tlen >= 3072 ? (int)((wgs <= 64 ? 256 : 512) / wgs) : 1;
    if (p.G > 1) {
        p.LS = p.NS = 1;
        p.seg_len = mmf_round_up(Tlen, blk);
        return p;
    }
    p.LS = wgs <= 128 && (wgs > (elem == 4 ? 40 : 64) || Tlen < 2048) ? 2 : 1;
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
Plan fwd_plan(int64_t BH, int64_t Tlen, int64_t D, int chunk, bool joint, int elem) {
    const bool split = fwd_takes_workspace(BH, Tlen, D, chunk);
    return plan(BH, Tlen, D, kFwdBlk, split, split && joint, elem);
}
int64_t joint_columns(int64_t BH, int64_t D) { return BH * mmf_ceil_div(D, 64); }
int64_t joint_bytes(int64_t BH, int64_t D) { return joint_columns(BH, D) * 65 * 8 + 8; }   // (8 over: the words begin at the workspace's first multiple of 8)
int64_t pair_bytes(const Plan& p, int64_t BH, int64_t D) {
    return p.G > 1 ? joint_bytes(BH, D) : p.NS > 1 ? BH * p.NS * 2 * D * (int64_t)sizeof(float) : 0;
}
// A forward of 65 to 128 columns up to 5120 steps whose three tensors fit the 256 MB last-level cache, or nearly, is faster halved than shared, as long as the halves'
// half lines come together: rows of 512 channels and more (column_block), or of fp32, where a half is a line.  Halved / shared, us: 8 x 3072 x 1024 bf16
// 29 / 35, 8 x 5000 x 1024 50 / 58, 5 x 5000 x 1024 37 / 37, 8 x 6500 x 1024 87 / 74; fp32 112 x 3072 x 64 49 / 55, 68 x 4000 x 64 39 / 45, 96 x 4000 x 64 (94 MB)
// 56 / 58, 128 x 3072 x 64 (96 MB) 59 / 62, 112 x 4000 x 64 (109 MB) 69 / 68; bf16 128 x 4000 x 64, whose halves are apart, 53 / 42.  The backward's five tensors fit it up to half that
// length: 8 x 3072 x 1024 44 / 49, 8 x 4000 x 1024 90 / 79, and with its forward just before 106 / 99.
bool fwd_halves(int64_t BH, int64_t Tlen, int64_t D, int64_t elem) {
    const int64_t columns = BH * mmf_ceil_div(D, 64);
    return columns > 64 && columns <= 128 && Tlen <= 5120 && BH * Tlen * D * elem <= (96ll << 20) && (D % 512 == 0 || (elem == 4 && D % 32 == 0));
}
// The kernels address a block of at most 64 rows with 32-bit offsets and count blocks in an int.
bool fits(int64_t Tlen, int64_t D, int dtype) {
    return Tlen / kBwdBlk < (1ll << 30) && 64 * D * (int64_t)(dtype == MMF_F32 ? 4 : 2) < (1ll << 31);
}

__global__ __launch_bounds__(256) void joint_words_kernel(uint64_t* __restrict__ words, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) words[i] = 0;
}
int64_t joint_grid(const Plan& p, int64_t BH, int64_t D) { return mmf_round_up(joint_columns(BH, D), 8) * p.G; }
Joint joint_begin(const Plan& p, float* workspace, int64_t BH, int64_t D, hipStream_t s) {
    uint64_t* words = reinterpret_cast<uint64_t*>((reinterpret_cast<uintptr_t>(workspace) + 7) & ~(uintptr_t)7);
    const int64_t n = joint_columns(BH, D) * 65;
    joint_words_kernel<<<(unsigned)mmf_ceil_div(n, 256), 256, 0, s>>>(words, n);
    return Joint{words, p.G, BH, joint_columns(BH, D)};
}
// Whether loads and stores are streamed past the caches.  Large tensors gain (40 x 2048 x 1024 bf16 118 + 198 -> 111 + 188 us, 128 x
// 8192 x 128 156 + 259 -> 138 + 241, 5.8 TB/s), smaller ones are found in the 256 MB last-level cache, by the scan or by what reads its results.  With
// x and g (do) written just before and the results read next, 16 x T x 1024 bf16, forward, streamed / not: 40 MB a tensor 65 / 62 us, 64 116 / 116, 85
// 157 / 151, 100 175 / 169, 130 222 / 223; backward 80 / 78, 123 / 126, 176 / 171, 198 / 198, 253 / 258; by itself on the same buffers the forward turns
// at 85 MB (64 MB 40 / 36, 100 MB 63 / 67), the backward at 60 (64 MB 67 / 71).  In the second launch over time segments from 24 MB on (6000 x 64 columns
// 46 + 69 -> 45 + 62).  Shared columns as whole ones (6 x 16384 x 1024 110 + 118 for 114 + 126; 4 x 5000 x 1024, 39 MB, forward and backward 86 / 77).
// Only whole lines: where a row is no multiple of 128 bytes neighbouring columns share lines, which streamed are fetched twice (9 x 3068 x 1808
// bf16, forward and backward, 312 us, streamed 418; columns shared by workgroups: 30 x 12073 x 144 288 and 406, 8 x 4049 x 720 148 and 169).
constexpr int64_t kFwdStream = 90ll << 20, kBwdStream = 64ll << 20;      // bytes of a tensor
bool whole_lines(int64_t row_bytes) { return row_bytes % 128 == 0; }
bool streams(const Plan& p, int64_t row_bytes, int64_t rows, int64_t from) {
    return whole_lines(row_bytes) && rows * row_bytes >= (p.NS > 1 ? 24ll << 20 : from);
}
template <typename T, int LS, bool NT>
int launch_fwd_ls(const Plan& p, const T* x, const T* g, const float* h0, T* o, float* ht, float* agg, int64_t BH, int64_t Tlen,
                  int64_t D, hipStream_t s) {
    const int64_t nblk = p.seg_len / (LS * kFwdBlk);
    const unsigned threads = 64u * (unsigned)(nblk < kMaxWaves ? nblk : kMaxWaves), gx = (unsigned)mmf_ceil_div(D, 64 / LS);
    if (p.NS > 1) {
        hgrn_scan_fwd_kernel<T, true, LS, false, false><<<dim3(gx, (unsigned)BH, (unsigned)(p.NS - 1)), threads, 0, s>>>(
            x, g, h0, o, ht, agg, Tlen, D, p.seg_len, p.NS, Joint{});
        MMF_CHECK_LAUNCH();
    }
    auto kern = LS == 2 && p.NS == 1 ? hgrn_scan_fwd_kernel<T, false, LS, NT, false, LS == 2> : hgrn_scan_fwd_kernel<T, false, LS, NT, false>;
    kern<<<dim3(gx, (unsigned)BH, (unsigned)p.NS), threads, 0, s>>>(
        x, g, h0, o, ht, agg, Tlen, D, p.seg_len, p.NS, Joint{});
    MMF_CHECK_LAUNCH();
    return 0;
}
template <typename T>
int launch_fwd(const void* x, const void* g, const float* h0, void* o, float* ht, float* agg, int64_t BH, int64_t Tlen, int64_t D,
               int chunk, hipStream_t s) {
    const Plan p = fwd_plan(BH, Tlen, D, chunk, agg && !fwd_halves(BH, Tlen, D, sizeof(T)), sizeof(T));
    if (!agg && (p.NS > 1 || (fwd_takes_workspace(BH, Tlen, D, chunk) && BH * mmf_ceil_div(D, 64) < 128 && Tlen >= 2048))) return MMF_ERR_ARG;
    const T* xp = static_cast<const T*>(x);
    const T* gp = static_cast<const T*>(g);
    T* op = static_cast<T*>(o);
    if (p.G > 1) {
        const Joint jt = joint_begin(p, agg, BH, D, s);
        MMF_CHECK_LAUNCH();
        auto kern = streams(p, D * (int64_t)sizeof(T), BH * Tlen, kFwdStream) ? hgrn_scan_fwd_kernel<T, false, 1, true, true> : hgrn_scan_fwd_kernel<T, false, 1, false, true>;
        kern<<<(unsigned)joint_grid(p, BH, D), 64 * kMaxWaves, 0, s>>>(
            xp, gp, h0, op, ht, nullptr, Tlen, D, p.seg_len, 1, jt);
        MMF_CHECK_LAUNCH();
        return 0;
    }
    return p.LS == 2 ? launch_fwd_ls<T, 2, false>(p, xp, gp, h0, op, ht, agg, BH, Tlen, D, s)
           : streams(p, D * (int64_t)sizeof(T), BH * Tlen, kFwdStream) ? launch_fwd_ls<T, 1, true>(p, xp, gp, h0, op, ht, agg, BH, Tlen, D, s)
                                                        : launch_fwd_ls<T, 1, false>(p, xp, gp, h0, op, ht, agg, BH, Tlen, D, s);
}

template <typename T, bool LOG, int LS, bool NT>
int launch_bwd_ls(const Plan& p, const T* g, const T* o, const T* dout, const float* h0, T* dx, T* dg, float* agg, int64_t BH,
                  int64_t Tlen, int64_t D, hipStream_t s) {
    const int64_t nblk = p.seg_len / (LS * kBwdBlk);
    const unsigned threads = 64u * (unsigned)(nblk < kMaxWaves ? nblk : kMaxWaves), gx = (unsigned)mmf_ceil_div(D, 64 / LS);
    if (p.NS > 1) {
        hgrn_scan_bwd_kernel<T, LOG, true, LS, false, false><<<dim3(gx, (unsigned)BH, (unsigned)(p.NS - 1)), threads, 0, s>>>(
            g, o, dout, h0, dx, dg, agg, Tlen, D, p.seg_len, p.NS, Joint{});
        MMF_CHECK_LAUNCH();
    }
    auto kern = LS == 2 && p.NS == 1 ? hgrn_scan_bwd_kernel<T, LOG, false, LS, NT, false, LS == 2> : hgrn_scan_bwd_kernel<T, LOG, false, LS, NT, false>;
    kern<<<dim3(gx, (unsigned)BH, (unsigned)p.NS), threads, 0, s>>>(
        g, o, dout, h0, dx, dg, agg, Tlen, D, p.seg_len, p.NS, Joint{});
    MMF_CHECK_LAUNCH();
    return 0;
}
template <typename T, bool LOG>
int launch_bwd(const void* g, const void* o, const void* dout, const float* h0, void* dx, void* dg, float* agg, int64_t BH,
               int64_t Tlen, int64_t D, hipStream_t s) {
    const Plan p = plan(BH, Tlen, D, kBwdBlk, agg != nullptr, agg != nullptr, sizeof(T));
    const T* gp = static_cast<const T*>(g);
    const T* op = static_cast<const T*>(o);
    const T* dp = static_cast<const T*>(dout);
    T* xp = static_cast<T*>(dx);
    T* yp = static_cast<T*>(dg);
    if (p.G > 1) {
        const Joint jt = joint_begin(p, agg, BH, D, s);
        MMF_CHECK_LAUNCH();
        auto kern = streams(p, D * (int64_t)sizeof(T), BH * Tlen, kBwdStream) ? hgrn_scan_bwd_kernel<T, LOG, false, 1, true, true> : hgrn_scan_bwd_kernel<T, LOG, false, 1, false, true>;
        kern<<<(unsigned)joint_grid(p, BH, D), 64 * kMaxWaves, 0, s>>>(
            gp, op, dp, h0, xp, yp, nullptr, Tlen, D, p.seg_len, 1, jt);
        MMF_CHECK_LAUNCH();
        return 0;
    }
    return p.LS == 2 ? launch_bwd_ls<T, LOG, 2, false>(p, gp, op, dp, h0, xp, yp, agg, BH, Tlen, D, s)
           : streams(p, D * (int64_t)sizeof(T), BH * Tlen, kBwdStream) ? launch_bwd_ls<T, LOG, 1, true>(p, gp, op, dp, h0, xp, yp, agg, BH, Tlen, D, s)
                                                        : launch_bwd_ls<T, LOG, 1, false>(p, gp, op, dp, h0, xp, yp, agg, BH, Tlen, D, s);
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
    const Plan p = fwd_plan(BH, T, D, chunk, true, 2);   // (fp32 is cut in no more places)
    return p.G > 1 ? joint_bytes(BH, D) : BH * p.NS * 2 * D * (int64_t)sizeof(float);
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
    return pair_bytes(plan(BH, T, D, kBwdBlk, true, true, 2), BH, D);
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
