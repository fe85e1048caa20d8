// Top-p (nucleus) sampling of one token per row of logits, in one launch and without a sort.
//
// Replaces, for the loop that mmfreelm's generate.py:11 runs (model.generate(do_sample=True, top_p=0.4,
// temperature=0.6)), the per-token chain temperature scaling -> softmax -> descending sort -> cumulative sum ->
// nucleus mask -> renormalise -> multinomial draw that transformers' sampling path performs on the logits of
// HGRNBitForCausalLM.forward (mmfreelm/models/hgrn_bit/modeling_hgrn_bit.py:386).
//
// Every decision is made on integers, so the result does not depend on any summation order and a CPU restatement
// reproduces it exactly:
//   l_i   = logit_i / temperature                      (fp32 division; NaN counts as -inf)
//   p_i   = 1 if l_i == max l, else exp(l_i - max l)   (the deterministic fp32 exp of mmf_common.h)
//   top_k > 0:  l_i = -inf unless l_i >= the top_k-th largest l        (transformers' TopKLogitsWarper, which the
//               reference's call gets from the default generation parameters, top_k = 50; equal values stay together)
//   m_i   = trunc(p_i * 2^31)                          (uint32 probability mass; the row maximum has 2^31)
//   Z     = sum m_i,  P = max(1, trunc(double(top_p) * double(Z)))
//   keep i  iff  m_i > 0 and  sum{ m_j : m_j > m_i } < P     (the smallest set of most probable tokens whose mass
//                                                             reaches top_p; tokens of equal mass stay together)
//   S     = sum of kept m_i,  target = trunc(double(u) * double(S)),  u in [0, 1) supplied by the caller
//   token = the lowest index whose running sum of kept masses (in index order) exceeds target.
//
// One workgroup of 1024 threads per row; a thread owns NPT consecutive vocabulary entries and keeps their masses in
// registers.  The nucleus threshold (the smallest kept mass) is found by a radix descent over the 32-bit mass, 8 bits
// a pass: a 256-bin histogram of mass (LDS atomics on 64-bit integers, 16 interleaved copies of every bin so that
// neighbouring lanes hit different banks; a thread merges runs of equal bins before it touches LDS), a suffix scan of
// the bins by one wave, and the digit whose bin straddles P.  The top_k-th largest scaled logit comes from the same
// descent on token counts over an order-preserving integer image of the floats, BEFORE the exp: only the kept tokens
// (some 50 of 32000) then pay for it.  Limits of at most 64 take no descent at all where they can (samp_pick_few).
#include "mmf_common.h"

namespace {

typedef unsigned long long u64;
constexpr int kSampThreads = 1024, kSampWaves = 16, kSampBins = 256, kSampCopies = 16;
constexpr int64_t kSampMaxV = 65536;

struct SampleArgs {
    const void* logits;
    int64_t ld;
    int V;
    float temperature, top_p;
    int top_k;              // 0: no limit
    const float* params;    // null, or {temperature, top_p, bits of top_k} in device memory instead of the three above
    const int* pos;         // null, or per row which row of u [*, rows] holds its number
    const float* u;
    int64_t* out;
};

__device__ __forceinline__ u64 samp_shfl_down(u64 v, int o) {
    const unsigned lo = (unsigned)__shfl_down((int)(unsigned)v, o, 64), hi = (unsigned)__shfl_down((int)(unsigned)(v >> 32), o, 64);
    return ((u64)hi << 32) | lo;
}
__device__ __forceinline__ u64 samp_shfl_up(u64 v, int o) {
    const unsigned lo = (unsigned)__shfl_up((int)(unsigned)v, o, 64), hi = (unsigned)__shfl_up((int)(unsigned)(v >> 32), o, 64);
    return ((u64)hi << 32) | lo;
}

// Radix descent over the 32-bit masses, 8 bits a pass.  With W(S) the mass (COUNT false) or the number (COUNT true) of
// the non-zero entries in S, returns the lowest v with W({m > v}) < limit: the smallest kept mass of the nucleus, or the
// limit-th largest mass.  prefix = the high digits found so far, above = W of everything larger than any mass with that prefix.
template <bool COUNT, int NPT>
__device__ __forceinline__ unsigned samp_descent(const unsigned (&m)[NPT], u64 limit, u64* hist, u64* hsum, u64* sel) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const u64 P = limit;
    unsigned prefix = 0;
    u64 above = 0;
#pragma unroll
    for (int pass = 0; pass < 4; ++pass) {
        const int shift = 24 - 8 * pass;
        int cur = -1;
        u64 acc = 0;
#pragma unroll
        for (int j = 0; j < NPT; ++j) {
            const unsigned mj = m[j];
            const bool match = mj != 0 && (pass == 0 || (mj >> ((shift + 8) & 31)) == prefix);
            if (match) {
                const int b = (int)((mj >> shift) & 255u);
                if (b != cur) {
                    if (cur >= 0) atomicAdd(&hist[cur * kSampCopies + (lane & (kSampCopies - 1))], acc);
                    cur = b;
                    acc = 0;
                }
                acc += COUNT ? 1u : mj;
            }
        }
        if (cur >= 0) atomicAdd(&hist[cur * kSampCopies + (lane & (kSampCopies - 1))], acc);
        __syncthreads();
        if (t < kSampBins) {
            u64 h = 0;
#pragma unroll
            for (int c = 0; c < kSampCopies; ++c) {
                const int s = t * kSampCopies + ((c + t) & (kSampCopies - 1));   // rotated: lanes start on different banks
                h += hist[s];
                hist[s] = 0;                                                     // ready for the next pass
            }
            hsum[t] = h;
        }
        __syncthreads();
        if (wave == 0) {
            // lane owns bins 4*lane .. 4*lane+3; A(d) = above + mass of the bins over d; take the lowest d with A(d) < P
            u64 h[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) h[i] = hsum[lane * 4 + i];
            const u64 mine = h[0] + h[1] + h[2] + h[3];
            u64 suf = mine;                                       // inclusive suffix sum over the lanes
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const u64 y = samp_shfl_down(suf, o);
                if (lane + o < 64) suf += y;
            }
            u64 A = above + (suf - mine);                         // mass over this lane's bins
            int best = 256;
            u64 bestA = 0;
#pragma unroll
            for (int i = 3; i >= 0; --i) {
                if (A < P) { best = lane * 4 + i; bestA = A; }
                A += h[i];
            }
            int lowest = best;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) lowest = min(lowest, __shfl_xor(lowest, o, 64));
            if (best == lowest && best < 256) { sel[0] = bestA; sel[1] = (u64)best; }
        }
        __syncthreads();
        above = sel[0];
        prefix = (prefix << 8) | (unsigned)sel[1];
    }
    return prefix;
}

// One wave, n <= 64 kept tokens with their masses in any order: the nucleus and the draw by direct comparison (64 x 64), same rule as below.
__device__ __forceinline__ void samp_finish_few(const unsigned* few_m, const int* few_i, int n, float top_p, float u, int64_t* out) {
    const int lane = threadIdx.x & 63;
    const unsigned mi = lane < n ? few_m[lane] : 0u;
    const int ii = lane < n ? few_i[lane] : 0x7fffffff;
    u64 Zf = mi;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) Zf += samp_shfl_down(Zf, o);
    Zf = ((u64)(unsigned)__builtin_amdgcn_readfirstlane((int)(Zf >> 32)) << 32) | (unsigned)__builtin_amdgcn_readfirstlane((int)Zf);
    u64 Pf = (u64)((double)top_p * (double)Zf);
    if (Pf < 1) Pf = 1;
    u64 heavier = 0;
#pragma unroll
    for (int j = 0; j < 64; ++j) {
        const unsigned mj = (unsigned)__builtin_amdgcn_readlane((int)mi, j);
        heavier += mj > mi ? mj : 0u;
    }
    const unsigned kept = (mi != 0u && heavier < Pf) ? mi : 0u;
    u64 Sf = kept;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) Sf += samp_shfl_down(Sf, o);
    Sf = ((u64)(unsigned)__builtin_amdgcn_readfirstlane((int)(Sf >> 32)) << 32) | (unsigned)__builtin_amdgcn_readfirstlane((int)Sf);
    float uf = u;
    uf = uf >= 0.0f ? uf : 0.0f;
    u64 target = (u64)((double)uf * (double)Sf);
    if (target >= Sf) target = Sf - 1;
    u64 before = 0;                                   // kept mass at lower vocabulary indices
#pragma unroll
    for (int j = 0; j < 64; ++j) {
        const unsigned kj = (unsigned)__builtin_amdgcn_readlane((int)kept, j);
        const int ij = __builtin_amdgcn_readlane(ii, j);
        before += ij < ii ? kj : 0u;
    }
    if (kept != 0u && before <= target && target < before + kept) *out = ii;
}

// The lowest float above -inf that scales to no less than `low` does.
__device__ __forceinline__ float samp_lowest_reaching(float low, float temperature) {
    constexpr unsigned kBottom = 0x007fffffu;                     // -inf in the order of the floats
    auto order = [](float f) { const unsigned b = __float_as_uint(f); return b & 0x80000000u ? ~b : b | 0x80000000u; };
    auto value = [](unsigned k) { return __uint_as_float(k & 0x80000000u ? k & 0x7fffffffu : ~k); };
    const float reach = __fdiv_rn(low, temperature);
    unsigned no = kBottom, yes = order(low) > kBottom ? order(low) : kBottom + 1;
    while (yes - no > 1) {
        const unsigned mid = no + (yes - no) / 2;
        if (__fdiv_rn(value(mid), temperature) >= reach) yes = mid; else no = mid;
    }
    return value(yes);
}

// The tokens of a limit of at most 64, without a histogram: a bound no higher than the top_k-th largest logit first, then exact ranks among the few
// logits that reach it.  Scaling does not change the order, so only those are divided.  The bound: every wave's fourth largest (or third, ..: 16 waves have top_k
// between them) of its threads' maxima, the least of them; or, where the large logits lie close together, the least maximum of some wave's 64 threads.  A thread's
// logits come from all over the vocabulary, so that no wave has only rare tokens.  200 to 300 of 32000 normal logits reach it, 505 of sorted ones.  Two unequal
// logits can scale to equal ones: what lies less than 2^-21 below the bound is ranked too; where the bound or its scaled value is not in the
// middle range, where that covers such pairs, the lowest float that reaches it is searched for (all finite logits, where there are few).
// Returns the number of kept tokens (more than top_k on ties), their masses and places in ps.mass, ps.at; -1, for the whole workgroup, when the
// caller has to go the general way.
// Bound by latency: a row has one CU, whose waves wait for each other four times.  32000 logits, limit 50, 1 to 64 rows, us, descent and ranks: bf16 23.0 to
// 24.9 and 9.4 to 11.8, fp16 22.8 to 24.7 and 9.0 to 12.3, fp32 33 and 19 to 21 (128 KB through one CU); limit 64 with ties at it 39.5 to 41.6 and 10.8 to
// 12.7, limit 1 22 and 8; sorted logits bf16 25.6 and 13.7, fp32 35.4 and 22.4; all but 20 masked 19.9 and 7.6, 29.9 and 16.5; out of the middle range 23.6 and
// 13.4, 33.0 and 22.1.  What goes the general way after all has spent 5 us (fp32 15, its second read) and gets 10 back if a thousand ties at the bound are why:
// equal logits bf16 46.5 and 41.2, fp32 56.2 and 59.6.
constexpr int kPickMax = 1024;
// Four of each wave's 64 maxima bound 64 tokens (more maxima a wave cost what they save), where every thread has logits.
__host__ __device__ __forceinline__ bool samp_picks(int top_k, int V) { return top_k > 0 && top_k <= 64 && V >= 8 * kSampThreads; }
struct PickShared { float l[kPickMax], top[kSampWaves], low[kSampWaves], least[kSampWaves]; int idx[kPickMax], at[kPickMax]; unsigned mass[kPickMax], kept[kPickMax]; int n, few; };
template <typename T, int NPT>
__device__ __forceinline__ int samp_pick_few(const T* row, int V, bool vec_ok, int top_k, float temperature, float& reach, PickShared& ps) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    Raw8<T> raw[NPT / 8];
#pragma unroll
    for (int c = 0; c < NPT / 8; ++c) raw[c] = mmf_load8_raw<T>(row, ((int64_t)c * kSampThreads + t) * 8, V, vec_ok);
    if (t == 0) { ps.n = 0; ps.few = 0; }
    float x[NPT], most = -INFINITY;
#pragma unroll
    for (int c = 0; c < NPT / 8; ++c) {
        float v[8];
        mmf_unpack8<T>(raw[c], v);
        const int at = (c * kSampThreads + t) * 8;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            x[c * 8 + i] = at + i < V ? v[i] : -INFINITY;
            most = fmaxf(most, x[c * 8 + i]);                     // (NaN counts as -inf, here and in the comparisons below)
        }
    }
    const int q = (top_k + kSampWaves - 1) / kSampWaves;
    float rest = most, first = 0.0f, low = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i < q) {
            low = mmf_wave_max(rest);
            if (i == 0) first = low;
            const u64 at = __builtin_amdgcn_ballot_w64(rest == low);
            if (at != 0 && lane == (int)__builtin_ctzll(at)) rest = -INFINITY;
        }
    }
    const float least = -mmf_wave_max(-most);
    if (lane == 0) { ps.top[wave] = first; ps.low[wave] = low; ps.least[wave] = least; }
    __syncthreads();
    float mx = -INFINITY, close = -INFINITY;
    low = INFINITY;
#pragma unroll
    for (int w = 0; w < kSampWaves; ++w) {
        mx = fmaxf(mx, ps.top[w]);
        low = fminf(low, ps.low[w]);
        close = fmaxf(close, ps.least[w]);
    }
    low = fmaxf(low, close);
    reach = __fdiv_rn(low, temperature);
    if (mx == -INFINITY) return -1;
    float cut = __fsub_rn(low, __fmul_rn(fabsf(low), 0x1p-21f));
    if (!(fabsf(low) >= 0x1p-100f && fabsf(low) <= 0x1p100f && fabsf(reach) >= 0x1p-100f && fabsf(reach) <= 0x1p100f))
        cut = samp_lowest_reaching(low, temperature);
    if (most >= cut) {
#pragma unroll
        for (int j = 0; j < NPT; ++j) {
            if (x[j] >= cut) {
                const int pos = atomicAdd(&ps.n, 1);
                if (pos < kPickMax) { ps.l[pos] = __fdiv_rn(x[j], temperature); ps.idx[pos] = ((j >> 3) * kSampThreads + t) * 8 + (j & 7); }
            }
        }
    }
    __syncthreads();
    const int n = ps.n;
    if (n > kPickMax) return -1;
    mx = __fdiv_rn(mx, temperature);
    if (wave * 64 < n) {
        const float mine = t < n ? ps.l[t] : -INFINITY;
        int larger = 0;
        int j = 0;
        for (; j + 8 <= n; j += 8) {
            const float4 a = *reinterpret_cast<const float4*>(&ps.l[j]), b = *reinterpret_cast<const float4*>(&ps.l[j + 4]);
            larger += (a.x > mine) + (a.y > mine) + (a.z > mine) + (a.w > mine) + (b.x > mine) + (b.y > mine) + (b.z > mine) + (b.w > mine);
        }
        for (; j < n; ++j) larger += ps.l[j] > mine;
        if (t < n && larger < top_k) {                            // = no less than the top_k-th largest
            const float p = mine == mx ? 1.0f : mmf_exp(__fsub_rn(mine, mx));
            const int pos = atomicAdd(&ps.few, 1);
            ps.mass[pos] = (unsigned)__fmul_rn(p, 2147483648.0f);
            ps.at[pos] = ps.idx[t];
        }
    }
    __syncthreads();
    return ps.few;
}

// The nucleus and the draw among up to kPickMax kept tokens (more than 64: ties at the limit), a thread each over all of them.
__device__ __forceinline__ void samp_finish_listed(PickShared& ps, int n, float top_p, float u, int64_t* out) {
    const int t = threadIdx.x;
    const unsigned mine = t < n ? ps.mass[t] : 0u;
    const int at = t < n ? ps.at[t] : 0;
    if ((t & ~63) < n) {
        u64 Z = 0, heavier = 0;
        for (int j = 0; j < n; ++j) {
            const unsigned m = ps.mass[j];
            Z += m;
            heavier += m > mine ? m : 0u;
        }
        u64 P = (u64)((double)top_p * (double)Z);
        if (P < 1) P = 1;
        if (t < n) ps.kept[t] = mine != 0u && heavier < P ? mine : 0u;
    }
    __syncthreads();
    if ((t & ~63) < n) {
        u64 S = 0, before = 0;
        for (int j = 0; j < n; ++j) {
            const unsigned m = ps.kept[j];
            S += m;
            before += ps.at[j] < at ? m : 0u;
        }
        u = u >= 0.0f ? u : 0.0f;
        u64 target = (u64)((double)u * (double)S);
        if (target >= S) target = S - 1;
        const unsigned kept = t < n ? ps.kept[t] : 0u;
        if (kept != 0u && before <= target && target < before + kept) *out = at;
    }
}

// Beyond 32768 tokens an instance for each kind of limit that the host knows: the registers that a thread's 64 logits leave do not hold all ways.  50257 tokens, one row,
// all in one instance / one each, us: bf16 no limit 115 / 108, 1000 152 / 149, 65 137 / 132; fp32 113 / 112, 146 / 143, 134 / 131.  32 logits a thread take the
// same time either way (32000 tokens, no limit: 27.8 and 27.9).
enum Limit : int { kNoLimit, kLargeLimit, kAnyLimit };
template <typename T, int NPT, int LIMIT>
__global__ __launch_bounds__(kSampThreads) void sample_top_p_kernel(SampleArgs a) {
    __shared__ u64 hist[kSampBins * kSampCopies];                // 32 KiB
    __shared__ u64 hsum[kSampBins];
    __shared__ u64 wtot[kSampWaves], wtot2[kSampWaves];
    __shared__ u64 sel[2];
    __shared__ float wmax[kSampWaves];
    __shared__ int wcand[kSampWaves];
    __shared__ int few_n, few_i[64];
    __shared__ unsigned few_m[64];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int V = a.V;
    const float temperature = a.params ? a.params[0] : a.temperature, top_p = a.params ? a.params[1] : a.top_p;
    const int top_k = a.params ? __float_as_int(a.params[2]) : a.top_k;
    const T* row = static_cast<const T*>(a.logits) + (int64_t)blockIdx.x * a.ld;
    const int base = t * NPT;
    const int64_t u_at = blockIdx.x + (a.pos ? (int64_t)a.pos[blockIdx.x] * gridDim.x : 0);
    const bool vec_ok = (V % 8) == 0 && (a.ld % 8) == 0 && (reinterpret_cast<uintptr_t>(a.logits) & 15u) == 0;

    const bool pick = LIMIT == kAnyLimit && samp_picks(top_k, V) && temperature > 0.0f;
    float reach = 0.0f;                                           // no more than the top_k-th largest scaled logit
    __shared__ __align__(16) PickShared ps;
    if constexpr (LIMIT == kAnyLimit) {
        if (pick) {
            const int n = samp_pick_few<T, NPT>(row, V, vec_ok, top_k, temperature, reach, ps);
            if (n >= 0) {
                if (n > 64) samp_finish_listed(ps, n, top_p, a.u[u_at], a.out + blockIdx.x);
                else if (wave == 0) samp_finish_few(ps.mass, ps.at, n, top_p, a.u[u_at], a.out + blockIdx.x);
                return;
            }
        }   // a thousand ties, clusters in several places, no finite logit: the general way
    }
    Raw8<T> raw[NPT / 8];
#pragma unroll
    for (int c = 0; c < NPT / 8; ++c) raw[c] = mmf_load8_raw<T>(row, (int64_t)base + c * 8, V, vec_ok);
#pragma unroll
    for (int i = 0; i < kSampBins * kSampCopies / kSampThreads; ++i) hist[i * kSampThreads + t] = 0;

    float l[NPT];
    float mx = -INFINITY;
#pragma unroll
    for (int c = 0; c < NPT / 8; ++c) {
        float v[8];
        mmf_unpack8<T>(raw[c], v);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int idx = base + c * 8 + i;
            float x = v[i];
            x = (idx < V && x == x) ? __fdiv_rn(x, temperature) : -INFINITY;
            l[c * 8 + i] = x;
            mx = fmaxf(mx, x);
        }
    }
    mx = mmf_wave_max(mx);
    constexpr bool TIES = LIMIT == kAnyLimit && NPT <= 32;                      // (more logits a thread leave no registers for it)
    if (TIES && pick) {                                           // ties at the bound: it is the top_k-th largest
        int larger = 0;
#pragma unroll
        for (int j = 0; j < NPT; ++j) larger += l[j] > reach;
        larger = mmf_wave_sum(larger);
        if (lane == 0) atomicAdd(&ps.few, larger);
    }
    if (lane == 0) wmax[wave] = mx;
    __syncthreads();                                              // also publishes the zeroed histogram
#pragma unroll
    for (int w = 0; w < kSampWaves; ++w) mx = fmaxf(mx, wmax[w]);

    unsigned m[NPT];
    if (LIMIT != kNoLimit && top_k > 0 && top_k < V && mx != -INFINITY) {          // a row without a finite logit has no top_k-th largest: it is drawn
                                                                   // uniformly like without the limit (every mass is 2^31)
        // order-preserving image of the scaled logits: non-negative floats above the negative ones, -inf and the slots
        // past V at 0 (which the descent ignores)
#pragma unroll
        for (int j = 0; j < NPT; ++j) {
            const unsigned b = __float_as_uint(__fadd_rn(l[j], 0.0f));       // -0 counts as +0, as the comparison of floats does
            m[j] = l[j] == -INFINITY ? 0u : (b & 0x80000000u) ? ~b : (b | 0x80000000u);
        }
        unsigned kth;
        if (TIES && pick && ps.few < top_k) {
            const unsigned b = __float_as_uint(__fadd_rn(reach, 0.0f));
            kth = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
        } else kth = samp_descent<true, NPT>(m, (u64)top_k, hist, hsum, sel);
        // the kept tokens (top_k of them, more on ties) with their masses, in any order, for one wave to finish
        if (t == 0) few_n = 0;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < NPT; ++j) {
            const bool keep = m[j] != 0u && m[j] >= kth;
            float p = 0.0f;
            if (__builtin_amdgcn_ballot_w64(keep) != 0) {         // wave-uniform: most waves skip the exp for most slots
                p = l[j] == mx ? 1.0f : mmf_exp(__fsub_rn(l[j], mx));
                p = keep ? p : 0.0f;
            }
            m[j] = (unsigned)__fmul_rn(p, 2147483648.0f);
            if (keep) {
                const int pos = atomicAdd(&few_n, 1);
                if (pos < 64) { few_m[pos] = m[j]; few_i[pos] = base + j; }
            }
        }
        __syncthreads();
        const int n = few_n;
        if (n <= 64) {
            // few enough for one lane each
            if (wave == 0) samp_finish_few(few_m, few_i, n, top_p, a.u[u_at], a.out + blockIdx.x);
            return;
        }
    } else {
#pragma unroll
        for (int j = 0; j < NPT; ++j) {
            const float p = l[j] == mx ? 1.0f : mmf_exp(__fsub_rn(l[j], mx));
            m[j] = base + j < V ? (unsigned)__fmul_rn(p, 2147483648.0f) : 0u;
        }
    }
    u64 zs = 0;
#pragma unroll
    for (int j = 0; j < NPT; ++j) zs += m[j];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) zs += samp_shfl_down(zs, o);
    if (lane == 0) wtot[wave] = zs;
    __syncthreads();
    u64 Z = 0;
#pragma unroll
    for (int w = 0; w < kSampWaves; ++w) Z += wtot[w];
    u64 P = (u64)((double)top_p * (double)Z);
    if (P < 1) P = 1;

    // ---- the nucleus: the smallest kept mass
    const unsigned thr = samp_descent<false, NPT>(m, P, hist, hsum, sel);

    // ---- the draw: inverse CDF over the kept masses in index order
    u64 s = 0;
#pragma unroll
    for (int j = 0; j < NPT; ++j) s += m[j] >= thr ? m[j] : 0u;
    u64 inc = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const u64 y = samp_shfl_up(inc, o);
        if (lane >= o) inc += y;
    }
    if (lane == 63) wtot2[wave] = inc;
    __syncthreads();
    u64 S = 0, before = 0;
#pragma unroll
    for (int w = 0; w < kSampWaves; ++w) {
        const u64 x = wtot2[w];
        S += x;
        if (w < wave) before += x;
    }
    float u = a.u[u_at];
    u = u >= 0.0f ? u : 0.0f;                                     // NaN and negatives draw the first kept token
    u64 target = (u64)((double)u * (double)S);
    if (target >= S) target = S - 1;                              // u >= 1
    u64 run = before + inc - s;
    int cand = 0x7fffffff;
#pragma unroll
    for (int j = 0; j < NPT; ++j) {
        if (m[j] >= thr) {
            run += m[j];
            if (run > target && cand == 0x7fffffff) cand = base + j;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cand = min(cand, __shfl_xor(cand, o, 64));
    if (lane == 0) wcand[wave] = cand;
    __syncthreads();
    if (t == 0) {
#pragma unroll
        for (int w = 0; w < kSampWaves; ++w) cand = min(cand, wcand[w]);
        a.out[blockIdx.x] = cand < V ? cand : 0;
    }
}

template <typename T>
int launch_sample(const SampleArgs& a, int64_t rows, hipStream_t s) {
    auto launch = [&](auto* kernel) { kernel<<<(unsigned)rows, kSampThreads, 0, s>>>(a); };
    if (a.V <= 32 * kSampThreads) launch(sample_top_p_kernel<T, 32, kAnyLimit>);
    else if (a.params || samp_picks(a.top_k, a.V)) launch(sample_top_p_kernel<T, 64, kAnyLimit>);
    else if (a.top_k > 0) launch(sample_top_p_kernel<T, 64, kLargeLimit>);
    else launch(sample_top_p_kernel<T, 64, kNoLimit>);
    MMF_CHECK_LAUNCH();
    return 0;
}

}  // namespace

extern "C" {

int64_t mmf_sample_top_p_max_vocab(void) { return kSampMaxV; }

int mmf_sample_top_p(const void* logits, int64_t ld, int64_t rows, int64_t V, float temperature, float top_p,
                     int64_t top_k, const float* u, int64_t* out, int dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (rows < 0 || V <= 0 || ld < V || rows > 0x7fffffff || top_k < 0) return MMF_ERR_ARG;
    if (!(temperature > 0.0f) || !(top_p == top_p)) return MMF_ERR_ARG;
    if (rows == 0) return 0;
    if (!logits || !u || !out) return MMF_ERR_ARG;
    if (V > kSampMaxV) return MMF_ERR_WIDE;
    SampleArgs a{};
    a.logits = logits; a.ld = ld; a.V = (int)V; a.temperature = temperature;
    a.top_p = top_p < 0.0f ? 0.0f : top_p > 1.0f ? 1.0f : top_p;
    a.top_k = top_k >= V ? 0 : (int)top_k;
    a.u = u; a.out = out;
    switch (dtype) {
        case MMF_F32: return launch_sample<float>(a, rows, stream);
        case MMF_BF16: return launch_sample<bf16_t>(a, rows, stream);
        case MMF_F16: return launch_sample<f16_t>(a, rows, stream);
    }
    return MMF_ERR_ARG;
}

int mmf_sample_top_p_recorded(const void* logits, int64_t ld, int64_t rows, int64_t V, const float* params, const float* u,
                              const int* pos, int64_t* out, int dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (rows < 0 || V <= 0 || ld < V || rows > 0x7fffffff) return MMF_ERR_ARG;
    if (rows == 0) return 0;
    if (!logits || !params || !u || !pos || !out) return MMF_ERR_ARG;
    if (V > kSampMaxV) return MMF_ERR_WIDE;
    SampleArgs a{};
    a.logits = logits; a.ld = ld; a.V = (int)V; a.params = params; a.u = u; a.pos = pos; a.out = out;
    switch (dtype) {
        case MMF_F32: return launch_sample<float>(a, rows, stream);
        case MMF_BF16: return launch_sample<bf16_t>(a, rows, stream);
        case MMF_F16: return launch_sample<f16_t>(a, rows, stream);
    }
    return MMF_ERR_ARG;
}

}  // extern "C"
