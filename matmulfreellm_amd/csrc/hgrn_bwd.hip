// Backward of the HGRN recurrence (mmfreelm/ops/hgrn/recurrent_fuse.py:89-133; with log gates the gradient that
// mmfreelm/ops/hgrn/chunk.py:137-220 computes chunk-wise):
//   time runs backwards, dh += do_t; dx_t = dh; dg_t = dh * h_{t-1} (* exp(g_t) for log gates); dh *= g_t (exp(g_t)).
//
// Five streams of [BH, T, D] pass through once (g, o, do in; dx, dg out), so HBM is the bound.  A lane owns a channel, a
// workgroup 64 channels of one sequence (or of one time segment of it), a wave register blocks of 24 steps:
//   1. it loads its block's g, do and the outputs one step earlier (72 loads in flight per lane, none behind a branch);
//   2. local pass from a zero carry: l_t = gradient of the block's own steps, P_t = product of the gates behind step t;
//   3. its turn (blocks in order, latest first; the carry sits in LDS): ONE dependent step, carry = l_end + P_end * carry;
//   4. dh_t = l_t + P_t * carry for the whole block, stores.
// The waves run steps 1, 2 and 4 concurrently; what is serial across blocks is step 3, a handful of instructions.
// LS = 2: a workgroup owns 32 channels and the halves of a wave two consecutive runs of 24 steps, for twice the workgroups.
// When there are still too few, a first launch (AGG) runs steps 1-3 on g and do only and leaves per time segment
// the pair (P, l); the second enters segment s with the fold carry = l_j + P_j * carry over the segments behind it.
// Measured, bf16: 8 x 1024 x 2048 145 -> 40 us (4.1 TB/s), 64 x 16384 x 128 with log gates 2290 -> 369 us (3.6 TB/s), against
// a kernel that loaded under a branch per step, so one load after the other, and read g and do twice.  16 to 28 steps a block
// and 8 or 16 waves a workgroup lie within 10 % of each other.
#include <type_traits>
#include "mmf_common.h"

namespace {

constexpr int kBlk = 24, kMaxWaves = 8;

template <typename T, bool LOG, bool AGG, int LS>
__global__ __launch_bounds__(64 * kMaxWaves) void hgrn_scan_bwd_kernel(const T* __restrict__ g, const T* __restrict__ o,
                                                                       const T* __restrict__ dout, const float* __restrict__ h0,
                                                                       T* __restrict__ dx, T* __restrict__ dg,
                                                                       float* __restrict__ agg, int64_t Tlen, int64_t D,
                                                                       int64_t seg_len, int NS) {
    constexpr int CH = 64 / LS, kStep = LS * kBlk;                      // channels of a workgroup, steps of a wave's block
    __shared__ float carry_l[CH], carry_p[CH];
    __shared__ int turn;
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), nw = (int)blockDim.x >> 6;
    const int ch = lane % CH, u = lane / CH;                            // channel, and which kBlk steps of the wave's block
    const int64_t bh = blockIdx.y;
    const int seg = AGG ? (int)blockIdx.z + 1 : (int)blockIdx.z;       // nobody folds the pair of segment 0
    // The two halves of a 128-byte row go to workgroups 8 apart, which run on one XCD and share its L2.
    const unsigned bx = LS == 2 && gridDim.x % 16 == 0 ? (blockIdx.x & ~15u) + (blockIdx.x & 7u) * 2 + ((blockIdx.x >> 3) & 1u)
                                                       : blockIdx.x;
    const int64_t d = (int64_t)bx * CH + ch;
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
                c = ag[D] + ag[0] * c;
            }
        }
        carry_l[ch] = c;
        carry_p[ch] = 1.0f;
        if (lane == 0) turn = 0;
    }
    __syncthreads();
    auto wait_turn = [&](int n) __attribute__((always_inline)) {
        while (__hip_atomic_load(&turn, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) != n) __builtin_amdgcn_s_sleep(1);
    };
    auto bits = [](__amdgpu_buffer_rsrc_t r, uint32_t vo, uint32_t so) __attribute__((always_inline)) -> uint32_t {   // no packing of pairs
        if constexpr (sizeof(T) == 2) return (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, vo, so, 0);
        else return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, vo, so, 0);
    };
    auto store = [&](__amdgpu_buffer_rsrc_t r, uint32_t so, float v) __attribute__((always_inline)) {
        if constexpr (sizeof(T) == 2) __builtin_amdgcn_raw_buffer_store_b16(mmf_bits16(mmf_from_float<T>(v)), r, voff, so, 0);
        else __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, voff, so, 0);
    };
    auto rsrc = [](const T* p) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, 0x7fffffff, 0x00020000);
    };
    auto val = [](uint32_t v) __attribute__((always_inline)) -> float {
        if constexpr (sizeof(T) == 2) return mmf_to_float(mmf_from_bits16<T>((uint16_t)v));
        else return __uint_as_float(v);
    };

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
                gr[t] = bits(rg, voff, (uint32_t)t * rowb);
                dr[t] = bits(rd, voff, (uint32_t)t * rowb);
                if constexpr (!AGG) {
                    if (t > 0) hr[t] = bits(ro, voff, (uint32_t)(t - 1) * rowb + first);
                    else hr[t] = bits(ro, back || u == 0 ? voff : voff - rowb, 0);
                }
            } else {                                                     // rows past the end re-read the last one
                const int row = u * kBlk + t < rem ? u * kBlk + t : rem - 1, prev = row - 1 + back;
                gr[t] = bits(rg, cho + (uint32_t)row * rowb, 0);
                dr[t] = bits(rd, cho + (uint32_t)row * rowb, 0);
                if constexpr (!AGG) hr[t] = bits(ro, cho + (uint32_t)(prev > 0 ? prev : 0) * rowb, 0);
            }
        }
        float l = 0.0f, P = 1.0f;
#pragma unroll
        for (int t = kBlk - 1; t >= 0; --t) {
            float gl = val(gr[t]), a = val(dr[t]);
            if constexpr (LOG) gl = __expf(gl);
            if constexpr (!FULL) {                                       // steps past the end: (g, do) = (1, 0) change nothing
                gl = t < remu ? gl : 1.0f;
                a = t < remu ? a : 0.0f;
            }
            a += l;
            if constexpr (!AGG) {
                float hv = val(hr[t]);
                if (t == 0) hv = back || u > 0 ? hv : hinit;
                hr[t] = __float_as_uint(LOG ? hv * gl : hv);
                dr[t] = __float_as_uint(a);
                gr[t] = __float_as_uint(P);
            }
            l = a * gl;
            P *= gl;
        }
        // the parts behind this lane's, and the whole block, as one pair each
        float lb = l, Pb = P, lin = 0.0f, Pin = 1.0f;
        if constexpr (LS > 1) {
            lb = 0.0f;
            Pb = 1.0f;
#pragma unroll
            for (int k = LS - 1; k >= 0; --k) {
                if (u == k) {
                    lin = lb;
                    Pin = Pb;
                }
                const float lk = __shfl(l, k * CH + ch, 64), Pk = __shfl(P, k * CH + ch, 64);
                lb = lk + Pk * lb;
                Pb *= Pk;
            }
        }
        wait_turn(n);
        const float cb = carry_l[ch], c = LS > 1 ? lin + Pin * cb : cb;
        carry_l[ch] = lb + Pb * cb;                                     // (the parts of a channel write the same value)
        if constexpr (AGG) carry_p[ch] *= Pb;
        __hip_atomic_store(&turn, n + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        if constexpr (!AGG) {
            const __amdgpu_buffer_rsrc_t rx = rsrc(dx + row0), ry = rsrc(dg + row0);
#pragma unroll
            for (int t = kBlk - 1; t >= 0; --t) {
                if (FULL || t < remu) {
                    const float dh = __uint_as_float(dr[t]) + __uint_as_float(gr[t]) * c;
                    store(rx, (uint32_t)t * rowb, dh);
                    store(ry, (uint32_t)t * rowb, dh * __uint_as_float(hr[t]));
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
            wait_turn(nblk);
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
struct BwdPlan {
    int64_t seg_len;
    int NS, LS;
};
BwdPlan bwd_plan(int64_t BH, int64_t Tlen, int64_t D, bool split) {
    BwdPlan p;
    const int64_t wgs = BH * mmf_ceil_div(D, 64);
    p.LS = wgs < 256 && (wgs >= 128 || Tlen < 2048) ? 2 : 1;
    const int64_t now = BH * mmf_ceil_div(D, 64 / p.LS), step = p.LS * kBlk;
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

template <typename T, bool LOG, int LS>
int launch_bwd_ls(const BwdPlan& p, const T* g, const T* o, const T* dout, const float* h0, T* dx, T* dg, float* agg, int64_t BH,
                  int64_t Tlen, int64_t D, hipStream_t s) {
    const int64_t nblk = p.seg_len / (LS * kBlk);
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
    const BwdPlan p = bwd_plan(BH, Tlen, D, agg != nullptr);
    const T* gp = static_cast<const T*>(g);
    const T* op = static_cast<const T*>(o);
    const T* dp = static_cast<const T*>(dout);
    T* xp = static_cast<T*>(dx);
    T* yp = static_cast<T*>(dg);
    return p.LS == 2 ? launch_bwd_ls<T, LOG, 2>(p, gp, op, dp, h0, xp, yp, agg, BH, Tlen, D, s)
                     : launch_bwd_ls<T, LOG, 1>(p, gp, op, dp, h0, xp, yp, agg, BH, Tlen, D, s);
}

}  // namespace

extern "C" {

int64_t mmf_hgrn_recurrent_bwd_workspace_bytes(int64_t BH, int64_t T, int64_t D) {
    if (BH <= 0 || T <= 0 || D <= 0) return 0;
    const BwdPlan p = bwd_plan(BH, T, D, true);
    return p.NS > 1 ? BH * p.NS * 2 * D * (int64_t)sizeof(float) : 0;
}

int mmf_hgrn_recurrent_bwd_split(const void* g, const void* o, const void* grad_o, const float* h0, void* dx, void* dg, int64_t BH,
                                 int64_t T, int64_t D, int log_gates, int dtype, void* workspace, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (BH < 0 || T < 0 || D <= 0 || BH > 65535) return MMF_ERR_ARG;
    if (BH == 0 || T == 0) return 0;
    if (!g || !o || !grad_o || !dx || !dg) return MMF_ERR_ARG;
    if (T / kBlk >= (1ll << 30) || 64 * D * (int64_t)(dtype == MMF_F32 ? 4 : 2) >= (1ll << 31)) return MMF_ERR_WIDE;   // as the forward
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
