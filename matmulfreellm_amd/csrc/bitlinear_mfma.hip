// Ternary-weight contraction on the int8 matrix cores (v_mfma_i32_16x16x64_i8 and v_mfma_i32_32x32x32_i8, gfx950).
//
//   out[m, n] = T( fp32( sum_k q[m,k] * t[n,k] ) * deq[m] * wdeq[seg(n)] (+ bias[n]) )
//
// Replaces the dense F.linear on de-quantised weights at mmfreelm/ops/fusedbitnet.py:458
// (and the weight_quant at :456, done once at pack time instead).
//
// Operands
//   A  int8 activation codes in the fragment-tiled layout the quantiser writes:
//      [ceil32(M)/32][Kp/16][32 rows][16 bytes]; the 1 KiB at (mb, 2*ks .. 2*ks+1) is one
//      32x32 A fragment in lane order (lane l: row l%32, k = 16*(l/32) .. +15).
//   B  2-bit packed ternary codes (t+1), block layout [Np/32][Kp/128][64 lanes][4 dwords];
//      dword ks of lane l expands with 3 shifts + 4 masks into the 16 bytes lane l feeds
//      the MFMA for k-step ks.  B never touches LDS: every wave streams its own n-blocks
//      straight from global memory (they are 16x smaller than the int8 tile they become).
//   The stored code is t+1 in {0,1,2}; the epilogue subtracts sum_k q[m,k] (qsum).
//
// Three kernels, chosen by a measured cost model (dispatch_mfma):
//   large problems : a workgroup of WGM x WGN waves computes a (WGM*WM*32) x (WGN*WN*32) tile; each
//                    wave owns WM x WN accumulators of 32x32 (16 VGPRs each, four 16x16x64 blocks); A is staged through
//                    LDS by DMA in k-blocks of 128, three buffers, one barrier per k-block
//                    (bitlinear_mfma_dma3_kernel);
//   small problems : one 32x32 output block per workgroup, 8 waves split K, operands straight
//                    into registers (bitlinear_mfma_skinny_kernel);
//   small M with K > 8192 : A staged through registers, double buffered (bitlinear_mfma_kernel).
#include "mmf_common.h"
#include "../../include/mmf.h"

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

struct MfmaArgs {
    const int8_t* a;      // tiled codes
    const uint4* b;       // packed weights
    const float* deq;     // [M]
    const int* qsum;      // [M]
    const float* wdeq;    // per segment
    const void* bias;     // [N] or null
    const void* addend;   // [M, N] (leading dimension ldo) or null: out = T(T(o) + addend)
    void* out;            // [M, N]
    int64_t M, N, Kp, seg_rows, ldo;
    int64_t a_seg, m_seg; // 0, or the bytes from one weight segment's codes to the next's, and the entries between their deq and qsum: stacked
                          // projections whose inner norms differ contract each its own codes of the same rows
    int tiles_m, tiles_n;
    int rows_per_xcd;     // tile rows an XCD keeps in its L2 while it walks the columns (0: row-major tile order)
    int vec_store;        // outputs can be written as aligned 16-byte vectors
    long long* clocks;    // null, or [clock_cap][2]: shader-clock and 100 MHz ticks a workgroup spent in the kernel
    int64_t clock_cap;
};

// Where the tiled kernel notes its clocks (mmf_bitlinear_mfma_clock_sink); null: nothing is noted.
long long* g_clock_sink = nullptr;
int64_t g_clock_cap = 0;

// The operands of the weight segment that n-block nb0 lies in (wave-uniform; a workgroup's tile lies in one segment).
__device__ __forceinline__ void mfma_select_segment(MfmaArgs& p, int64_t nb0) {
    if (p.a_seg == 0) return;
    const int64_t seg = (int64_t)((uint32_t)(nb0 * 32) / (uint32_t)p.seg_rows);
    p.a += seg * p.a_seg;
    p.deq += seg * p.m_seg;
    p.qsum += seg * p.m_seg;
}

// Pack rounded outputs: two floats -> one dword of bf16/f16 (round to nearest even).
template <typename T>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    const T ta = mmf_from_float<T>(a), tb = mmf_from_float<T>(b);
    return (uint32_t)mmf_bits16(ta) | ((uint32_t)mmf_bits16(tb) << 16);
}

// Where the four groups of four accumulators that a lane holds of a 32 x 32 block lie.  The MFMAs are issued with the weights as
// the first operand, so a group is four consecutive output COLUMNS of one row, and packs into one 8-byte piece with no
// cross-lane traffic.
//   Lay32  one v_mfma_i32_32x32x32_i8 block: group g is column 8 g + 4 (l / 32), row l % 32
//   Lay16  four v_mfma_i32_16x16x64_i8 blocks, g = 2 * (row half) + (column half): column 16 (g % 2) + 4 (l / 16), row 16 (g / 2) + l % 16
struct Lay32 {
    static constexpr int RH = 1;                                 // rows of a lane
    static __device__ __forceinline__ int row(int lane, int) { return lane & 31; }
    static __device__ __forceinline__ int col(int lane, int g) { return 8 * g + 4 * (lane >> 5); }
    static __device__ __forceinline__ constexpr int half(int) { return 0; }
};
struct Lay16 {
    static constexpr int RH = 2;
    static __device__ __forceinline__ int row(int lane, int g) { return 16 * (g >> 1) + (lane & 15); }
    static __device__ __forceinline__ int col(int lane, int g) { return 16 * (g & 1) + 4 * (lane >> 4); }
    static __device__ __forceinline__ constexpr int half(int g) { return g >> 1; }
};
struct Acc16 { v4i g[4]; };                                      // a 32 x 32 block in Lay16
__device__ __forceinline__ int acc_at(const v16i& a, int g, int t) { return a[4 * g + t]; }
__device__ __forceinline__ int acc_at(const Acc16& a, int g, int t) { return a.g[g][t]; }
__device__ __forceinline__ void acc_set(v16i& a, int g, int t, int v) { a[4 * g + t] = v; }
__device__ __forceinline__ void acc_set(Acc16& a, int g, int t, int v) { a.g[g][t] = v; }

// Epilogue of the tiled kernels.  The wave stages its 32 x (WN*32) outputs in a
// private LDS region and writes them out as aligned 16-byte vectors (128-byte row segments).
// Per-lane row scales and per-block weight scales of the epilogue, fetched at kernel start so
// their latency hides behind the whole K loop.
template <class L, int WM, int WN>
struct EpiScales { float dq[WM][L::RH]; int qs[WM][L::RH]; float wdq[WN]; };

template <class L, int WM, int WN>
__device__ __forceinline__ void mfma_prefetch_scales(const MfmaArgs& p, EpiScales<L, WM, WN>& sc, int lane, int wm,
                                                     int64_t mb0, int64_t nb0) {
    const int64_t NB = (p.N + 31) >> 5;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int h = 0; h < L::RH; ++h) {
            const int64_t m = (mb0 + wm * WM + i) * 32 + L::row(lane, 2 * h);
            sc.dq[i][h] = m < p.M ? p.deq[m] : 0.0f;
            sc.qs[i][h] = m < p.M ? p.qsum[m] : 0;
        }
#pragma unroll
    for (int j = 0; j < WN; ++j)   // seg_rows is a multiple of 32: one weight scale per n-block
        sc.wdq[j] = (nb0 + j < NB) ? p.wdeq[(uint32_t)((nb0 + j) * 32) / (uint32_t)p.seg_rows] : 0.0f;
}

template <typename T, class L, class A, int WM, int WN>
__device__ __forceinline__ void mfma_epilogue(const MfmaArgs& p, A (&acc)[WM][WN], const EpiScales<L, WM, WN>& sc,
                                              unsigned char* smem, int lane, int wave, int wm, int64_t mb0, int64_t nb0) {
    const T* bias = static_cast<const T*>(p.bias);
    const T* addend = static_cast<const T*>(p.addend);
    T* out = static_cast<T*>(p.out);
    const float (&wdq)[WN] = sc.wdq;
    constexpr int E = sizeof(T);
    constexpr int RS = WN * 32 * E + 16;          // LDS row stride of a wave's 32 x (WN*32) staging tile
    constexpr int CPR = WN * 32 * E / 16;         // 16-byte chunks per row
    unsigned char* stage = smem + wave * (32 * RS);
#pragma unroll
    for (int i = 0; i < WM; ++i) {
        const int64_t mblk = (mb0 + wm * WM + i) * 32;
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float dq = sc.dq[i][L::half(g)];
                const int qs = sc.qs[i][L::half(g)], mloc = L::row(lane, g);
                const int64_t m = mblk + mloc;
                const int ncol = j * 32 + L::col(lane, g);           // first of 4 consecutive columns, tile-relative
                float o[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    o[t] = __fmul_rn(__fmul_rn((float)(acc_at(acc[i][j], g, t) - qs), dq), wdq[j]);
                    if (bias) {
                        const int64_t n = nb0 * 32 + ncol + t;
                        o[t] = __fadd_rn(o[t], n < p.N ? mmf_to_float(bias[n]) : 0.0f);
                    }
                }
                if (p.vec_store) {
                    if constexpr (E == 2)
                        *reinterpret_cast<uint2*>(stage + mloc * RS + ncol * 2) = make_uint2(pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3]));
                    else
                        *reinterpret_cast<float4*>(stage + mloc * RS + ncol * 4) = make_float4(o[0], o[1], o[2], o[3]);
                } else if (m < p.M) {
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        const int64_t n = nb0 * 32 + ncol + t;
                        if (n < p.N) {
                            float v = o[t];
                            if (addend) v = __fadd_rn(mmf_round_to<T>(v), mmf_to_float(addend[m * p.ldo + n]));
                            out[m * p.ldo + n] = mmf_from_float<T>(v);
                        }
                    }
                }
            }
        if (p.vec_store) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
            for (int c0 = 0; c0 < 32 * CPR; c0 += 64) {
                const int c = c0 + lane;
                const int row = c / CPR, cc = c % CPR;
                const int64_t mr = mblk + row, n = nb0 * 32 + cc * (16 / E);
                if (mr < p.M && n < p.N) {
                    uint4 v = *reinterpret_cast<const uint4*>(stage + row * RS + cc * 16);
                    if (addend) {
                        const uint4 av = *reinterpret_cast<const uint4*>(addend + mr * p.ldo + n);
                        T pe[16 / E], ae[16 / E], oe[16 / E];
                        __builtin_memcpy(pe, &v, 16);
                        __builtin_memcpy(ae, &av, 16);
#pragma unroll
                        for (int e = 0; e < 16 / E; ++e) oe[e] = mmf_from_float<T>(__fadd_rn(mmf_to_float(pe[e]), mmf_to_float(ae[e])));
                        __builtin_memcpy(&v, oe, 16);
                    }
                    *reinterpret_cast<uint4*>(out + mr * p.ldo + n) = v;
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
}

// Lean epilogue of the common case (16-byte stores possible, no bias): the accumulators were
// started at -qsum[m], so a value costs one convert and two multiplies; lane-constant parts of the
// store addresses are computed once; interior tiles skip the bounds tests.
template <bool STREAM, typename T, class L, class A, int WM, int WN>
__device__ __forceinline__ void mfma_epilogue_fast(const MfmaArgs& p, A (&acc)[WM][WN], const EpiScales<L, WM, WN>& sc,
                                                   unsigned char* smem, int lane, int wave, int wm, int64_t mb0, int64_t nb0) {
    const T* addend = static_cast<const T*>(p.addend);
    T* out = static_cast<T*>(p.out);
    constexpr int E = sizeof(T);
    constexpr int RS = WN * 32 * E + 16;          // LDS row stride of a wave's 32 x (WN*32) staging tile
    constexpr int CPR = WN * 32 * E / 16;         // 16-byte chunks per row (divides 64)
    constexpr int RPI = 64 / CPR;                 // rows covered by one 64-lane store
    unsigned char* stage = smem + wave * (32 * RS);
    const int cc = lane % CPR, rsub = lane / CPR;
    const int64_t m_first = (mb0 + wm * WM) * 32, n_first = nb0 * 32;
    const bool interior = m_first + WM * 32 <= p.M && n_first + WN * 32 <= p.N;
    const int64_t n = n_first + cc * (16 / E);
    const int64_t lane_off = (m_first + rsub) * p.ldo + n;         // element offset of this lane's first chunk
    unsigned char* wr = stage + L::row(lane, 0) * RS + L::col(lane, 0) * E;
    const unsigned char* rd = stage + rsub * RS + cc * 16;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float dq = sc.dq[i][L::half(g)];
                float o[4];
#pragma unroll
                for (int t = 0; t < 4; ++t) o[t] = __fmul_rn(__fmul_rn((float)acc_at(acc[i][j], g, t), dq), sc.wdq[j]);
                unsigned char* w = wr + L::row(0, g) * RS + (j * 32 + L::col(0, g)) * E;
                if constexpr (E == 2) *reinterpret_cast<uint2*>(w) = make_uint2(pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3]));
                else *reinterpret_cast<float4*>(w) = make_float4(o[0], o[1], o[2], o[3]);
            }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int r0 = 0; r0 < 32; r0 += RPI) {
            const int64_t off = lane_off + (int64_t)(i * 32 + r0) * p.ldo;
            if (interior || (m_first + i * 32 + r0 + rsub < p.M && n < p.N)) {
                uint4 v = *reinterpret_cast<const uint4*>(rd + r0 * RS);
                if (addend) {
                    const uint4 av = *reinterpret_cast<const uint4*>(addend + off);
                    T pe[16 / E], ae[16 / E], oe[16 / E];
                    __builtin_memcpy(pe, &v, 16);
                    __builtin_memcpy(ae, &av, 16);
#pragma unroll
                    for (int e = 0; e < 16 / E; ++e) oe[e] = mmf_from_float<T>(__fadd_rn(mmf_to_float(pe[e]), mmf_to_float(ae[e])));
                    __builtin_memcpy(&v, oe, 16);
                }
                if constexpr (STREAM) __builtin_nontemporal_store(*reinterpret_cast<const v4i*>(&v), reinterpret_cast<v4i*>(out + off));
                else *reinterpret_cast<uint4*>(out + off) = v;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// Epilogue of the gate/up contraction with the MLP activation folded in (mmfreelm/models/hgrn_bit/modeling_hgrn_bit.py:55-59):
// the wave's two n-blocks are the gate and the up projection of the same 32 channels, so a lane holds both operands of
// out = T((g * u) / (1 + exp(-g))), g = T(gate), u = T(up), and the wave writes 32 columns of the [M, N/2] result.
// Same conditions as the lean epilogue (accumulators started at -qsum, 16-byte stores).  The activation was most of what this
// launch took beyond the plain one: 16384 x 2048 -> 11264 in bf16 356 us with the exact exp and divide, 322 with mmf_swiglu_n (the plain
// contraction of as many columns about 300); 2002 rows 57 and 54; fp16, whose elements fall back eight times as often, 1377 rows 36.8 and 36.3.
template <typename T, class L, class A, int WM>
__device__ __forceinline__ void mfma_epilogue_swiglu(const MfmaArgs& p, A (&acc)[WM][2], const EpiScales<L, WM, 2>& sc,
                                                     unsigned char* smem, int lane, int wave, int wm, int64_t mb0, int64_t nbg) {
    T* out = static_cast<T*>(p.out);
    constexpr int E = sizeof(T);
    constexpr int RS = 32 * E + 16;               // LDS row stride of a wave's 32 x 32 staging tile
    constexpr int CPR = 32 * E / 16;              // 16-byte chunks per row
    constexpr int RPI = 64 / CPR;                 // rows covered by one 64-lane store
    unsigned char* stage = smem + wave * (32 * RS);
    const int cc = lane % CPR, rsub = lane / CPR;
    const int64_t nseg = p.N >> 1;
    const int64_t m_first = (mb0 + wm * WM) * 32, n_first = nbg * 32;
    const bool interior = m_first + WM * 32 <= p.M && n_first + 32 <= nseg;
    const int64_t n = n_first + cc * (16 / E);
    const int64_t lane_off = (m_first + rsub) * p.ldo + n;
    unsigned char* wr = stage + L::row(lane, 0) * RS + L::col(lane, 0) * E;
    const unsigned char* rd = stage + rsub * RS + cc * 16;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const float dq = sc.dq[i][L::half(g)];
            float gv[4], uv[4], o[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                gv[t] = mmf_round_to<T>(__fmul_rn(__fmul_rn((float)acc_at(acc[i][0], g, t), dq), sc.wdq[0]));
                uv[t] = mmf_round_to<T>(__fmul_rn(__fmul_rn((float)acc_at(acc[i][1], g, t), dq), sc.wdq[1]));
            }
            mmf_swiglu_n<T, 4>(gv, uv, o);
            unsigned char* w = wr + L::row(0, g) * RS + L::col(0, g) * E;
            if constexpr (E == 2) *reinterpret_cast<uint2*>(w) = make_uint2(pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3]));
            else *reinterpret_cast<float4*>(w) = make_float4(o[0], o[1], o[2], o[3]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int r0 = 0; r0 < 32; r0 += RPI) {
            const int64_t off = lane_off + (int64_t)(i * 32 + r0) * p.ldo;
            if (interior || (m_first + i * 32 + r0 + rsub < p.M && n < nseg))
                *reinterpret_cast<uint4*>(out + off) = *reinterpret_cast<const uint4*>(rd + r0 * RS);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

template <typename T, int WGM, int WGN, int WM, int WN, int KSL>
__global__ __launch_bounds__(64 * WGM * WGN) void bitlinear_mfma_kernel(MfmaArgs p) {
    constexpr int NT = 64 * WGM * WGN;
    constexpr int BMB = WGM * WM;                 // m-blocks (of 32 rows) per workgroup tile
    constexpr int BNB = WGN * WN;                 // n-blocks per workgroup tile
    constexpr int CH = KSL * 4096;                // bytes of one m-block's slab (KSL k-blocks of 128)
    constexpr int PIECES = BMB * (CH / 16);       // 16-byte pieces of one A slab
    constexpr int NPA = (PIECES + NT - 1) / NT;   // pieces per thread
    extern __shared__ __align__(16) unsigned char smem[];   // 2 x BMB x CH bytes

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // wave-uniform: keep it in a scalar register
    const int wm = wave / WGN, wn = wave % WGN;

    // XCD-aware tile order: hardware deals consecutive workgroup ids round-robin to the 8
    // XCDs; remap so each XCD walks a contiguous run of tiles (shared A panel stays in its L2).
    int64_t wg = blockIdx.x;
    const int64_t total = (int64_t)p.tiles_m * p.tiles_n;
    if (total % 8 == 0) wg = (wg % 8) * (total / 8) + wg / 8;
    const int64_t tile_m = wg / p.tiles_n, tile_n = wg % p.tiles_n;

    const int64_t MB = (p.M + 31) >> 5, NB = (p.N + 31) >> 5;
    const int64_t KB = p.Kp >> 7, KG = p.Kp >> 4;
    const int64_t mb0 = tile_m * BMB, nb0 = tile_n * BNB + wn * WN;
    EpiScales<Lay32, WM, WN> sc;
    mfma_prefetch_scales<Lay32, WM, WN>(p, sc, lane, wm, mb0, nb0);

    v16i acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

    uint4 areg[NPA];
    uint4 breg[KSL][WN], bnext[KSL][WN];

    auto load_a = [&](int64_t kb) {
#pragma unroll
        for (int i = 0; i < NPA; ++i) {
            const int pc = threadIdx.x + i * NT;
            const int chunk = pc / (CH / 16), within = pc % (CH / 16);
            areg[i] = make_uint4(0, 0, 0, 0);
            if (pc < PIECES && mb0 + chunk < MB && kb * 8 + (within >> 5) < KG)
                areg[i] = *reinterpret_cast<const uint4*>(p.a + ((mb0 + chunk) * KG + kb * 8) * 512 + within * 16);
        }
    };
    auto store_a = [&](int buf) {
#pragma unroll
        for (int i = 0; i < NPA; ++i) {
            const int pc = threadIdx.x + i * NT;
            if (pc < PIECES) *reinterpret_cast<uint4*>(smem + buf * (BMB * CH) + pc * 16) = areg[i];
        }
    };
    auto load_b = [&](int64_t kb, uint4 (&dst)[KSL][WN]) {
#pragma unroll
        for (int q = 0; q < KSL; ++q)
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                dst[q][j] = make_uint4(0x55555555u, 0x55555555u, 0x55555555u, 0x55555555u);   // all codes 1 = ternary 0
                if (nb0 + j < NB && kb + q < KB) dst[q][j] = p.b[((nb0 + j) * KB + kb + q) * 64 + lane];
            }
    };

    load_a(0);
    load_b(0, breg);
    store_a(0);
    __syncthreads();

    for (int64_t kb = 0; kb < KB; kb += KSL) {
        const int buf = (int)((kb / KSL) & 1);
        const bool more = kb + KSL < KB;
        if (more) {
            load_a(kb + KSL);
            load_b(kb + KSL, bnext);
        }
        const unsigned char* abase = smem + buf * (BMB * CH) + (wm * WM) * CH + lane * 16;
        // Software pipeline over the 32-wide k-steps of the slab: the LDS reads of step ks+1
        // are issued before the MFMAs of step ks.
        v4i af[2][WM];
#pragma unroll
        for (int i = 0; i < WM; ++i) af[0][i] = *reinterpret_cast<const v4i*>(abase + i * CH);
#pragma unroll
        for (int ks = 0; ks < 4 * KSL; ++ks) {
            if (ks + 1 < 4 * KSL) {
#pragma unroll
                for (int i = 0; i < WM; ++i)
                    af[(ks + 1) & 1][i] = *reinterpret_cast<const v4i*>(abase + i * CH + (ks + 1) * 1024);
            }
            v4i bf[WN];
#pragma unroll
            for (int j = 0; j < WN; ++j) {
                const uint4 bq = breg[ks >> 2][j];
                const uint32_t w = (ks & 3) == 0 ? bq.x : (ks & 3) == 1 ? bq.y : (ks & 3) == 2 ? bq.z : bq.w;
                bf[j][0] = (int)(w & 0x03030303u);
                bf[j][1] = (int)((w >> 2) & 0x03030303u);
                bf[j][2] = (int)((w >> 4) & 0x03030303u);
                bf[j][3] = (int)((w >> 6) & 0x03030303u);
            }
#pragma unroll
            for (int i = 0; i < WM; ++i)
#pragma unroll
                for (int j = 0; j < WN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bf[j], af[ks & 1][i], acc[i][j], 0, 0, 0);
        }
        if (more) {
            store_a(buf ^ 1);
#pragma unroll
            for (int q = 0; q < KSL; ++q)
#pragma unroll
                for (int j = 0; j < WN; ++j) breg[q][j] = bnext[q][j];
        }
        __syncthreads();
    }

    mfma_epilogue<T, Lay32>(p, acc, sc, smem, lane, wave, wm, mb0, nb0);
}

// One 1 KiB wave-load global -> LDS (16 bytes per lane; lane l lands at lds + 16 l) from `base` (wave-uniform) + 16 l.
// Written in assembly so that the compiler does not know of an LDS write in flight: it answers the builtin with waits
// for all vector-memory traffic in front of later LDS reads and barriers, at places of its own choosing (the top of the
// k-loop, half a k-block after the request).  The kernel waits for its transfers itself, once per k-block, where the
// data is needed.
__device__ __forceinline__ void mfma_dma_1k(const void* base, uint32_t lane16, const unsigned char* lds) {
    const uint32_t l = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)lds;
    const uint64_t b = (uint64_t)base;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(l), "v"(lane16), "s"(b) : "memory");
}
// acc += b x a on a 16 x 16 block over 64 inputs, in place.  (From the builtin the compiler gives every product a destination of its own
// and the 16 four-register accumulators wander through the registers until some are spilled.)  What the compiler would see to for
// the builtin: the two wait states behind the vector operations that wrote b (FRESH: its first use); before anything else reads the
// accumulators, mfma_done().  That no copy of an accumulator and no other write falls between is this compiler's choice of registers:
// tests/test_product_hazards.py reads the assembly for it.
template <bool FRESH>
__device__ __forceinline__ void mfma_16x16x64(v4i& acc, const v4i& b, const v4i& a) {
    if constexpr (FRESH) asm volatile("s_nop 1\n\tv_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+v"(acc) : "v"(b), "v"(a));
    else asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+v"(acc) : "v"(b), "v"(a));
}
template <int WM, int WN>
__device__ __forceinline__ void mfma_done(Acc16 (&acc)[WM][WN]) {
    asm volatile("s_nop 15\n\ts_nop 15");
#pragma unroll
    for (int t = 0; t < WM * WN * 4; ++t) asm volatile("" : "+v"(acc[t / (WN * 4)][t / 4 % WN].g[t & 3]));   // no reader moves in front of the wait
}
// Workgroup barrier behind an explicit wait: at most `VM` vector-memory operations may stay in flight, LDS traffic done.
// Only VM = 0 says anything about a transfer into LDS: such transfers and ordinary loads complete in no fixed order.
template <int VM>
__device__ __forceinline__ void mfma_barrier_vm() {
    static_assert(VM >= 0 && VM < 64, "vmcnt is a 6-bit count");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(VM) : "memory");
}

// LDS of the large-M kernel: three activation buffers, the exchange of partial sums or the epilogue's staging area, whichever is largest; behind
// them the rows' scales and code sums (registers held through the k-loop otherwise).
template <typename T, int WGM, int WGN, int WM, int WN, int KS, bool SWI>
constexpr int dma3_work_bytes() {
    constexpr int waves = WGM * WGN * KS, a = 3 * WGM * WM * 4096 * KS, e = waves * 32 * ((SWI ? 1 : WN) * 32 * (int)sizeof(T) + 16),
                  x = KS > 1 ? waves * (KS - 1) * WN * 4096 : 0;
    return a > e ? (a > x ? a : x) : (e > x ? e : x);
}

// ------------------------------------------------------------------------------------------
// The large-M kernel.  Same tiling, but A goes global -> LDS by DMA (global_load_lds_dwordx4:
// lane l's 16 bytes land at the wave-uniform LDS base + 16*l, which is exactly the
// fragment-tiled layout), so no VGPRs stage it and no ds_write sits in the instruction stream.
// Three A buffers of one 128-wide k-block each and ONE barrier per k-block,
// placed between its two k-steps of 64.  At that barrier every wave has left the previous
// k-block, so its buffer is free for the DMA of k-block s+2, and k-block s+1 (issued one k-block
// earlier, waited for by each wave just before the barrier, together with the packed weights
// requested with it) is complete for everybody.  K-block
// boundaries therefore carry no synchronisation: the A fragments of the next k-block's first
// step are read while the current one's last MFMAs run, and the matrix pipe never drains.
// FAST (chosen by the launcher): 16-byte stores possible and no bias -> lean epilogue, accumulators start at -qsum.  2: stores past the caches.
// SWI: the weight is the stacked [gate; up] projection (N = 2 * I): a wave's two n-blocks are the gate and the up rows
// of the same 32 channels, a workgroup tile covers WGN such channel blocks, and the epilogue writes swiglu(gate, up).
// KS > 1: the workgroup's waves form KS groups that take every KS-th k-block of the same (KS times narrower) tile: a mid-sized
// problem then has KS times as many tiles at the same work per wave, and each wave's chain is KS times shorter.  The groups
// exchange partial sums through LDS at the end (integers: exact), each finishing its share of the wave tile.
// What bounds it: on many tiles the power that the matrix cores draw on real codes.  On register operands v_mfma_i32_32x32x32_i8 reaches
// 3.6 P op/s before the clock gives way, v_mfma_i32_16x16x64_i8 4.8, which is why the products are of the second form although there are twice as
// many of them.  Measured with 32x32x32, then with
// 16x16x64, us: 16384 x 2048 -> 6144 204 and 172-180 (2.4 P op/s), x 5632 -> 2048 147 and 126-130 (3.0), x 2048 -> 11264 with swiglu 363-369 and
// 316-325; 4096 x 2048 -> 11264 83 and 73, 2002 rows 44 and 40.
// W32: the first form, for at most one split tile per CU: what counts there is each wave's chain of instructions, which has half as many products and no
// exchange of half-waves, and in front of it no rows' scales to pass through LDS.  us, 32x32x32 and 16x16x64: 5632 -> 2048, 1377 rows 21.6 and 23.1, 700 rows
// 19.8 and 21.3, 2002 rows (a tile for every CU) 24.3 and 24.1, 2500 (on some two) 35.4 and 33.3; 2048 -> 6144, 460 rows 11.8 and 12.4; 1024 -> 1024, 128
// to 4096 rows 7.4 to 9.2 and 8.0 to 9.7.  Whole tiles, one per CU, differ by 2 % either way.
template <typename T, int WGM, int WGN, int WM, int WN, int KS, int FAST, bool SWI = false, bool W32 = false>
__global__ __launch_bounds__(64 * WGM * WGN * KS, (WM * WN <= 4 ? 4 : 1))   // small wave tiles: 4 waves per SIMD = two workgroups per CU
void bitlinear_mfma_dma3_kernel(MfmaArgs p) {
    using L = typename std::conditional<W32, Lay32, Lay16>::type;
    using Acc = typename std::conditional<W32, v16i, Acc16>::type;
    constexpr int NT = WGM * WGN;                  // waves that cover the tile once
    constexpr int NW = NT * KS;
    constexpr int BMB = WGM * WM;
    constexpr int BNB = WGN * WN;
    constexpr int CH = 4096;                       // bytes of one m-block's k-block
    constexpr int BUF = BMB * CH * KS;             // one step: a k-block for each group
    constexpr int WPIECES = BUF / 1024;            // 1 KiB wave-loads per step
    constexpr int NDMA = (WPIECES + NW - 1) / NW;  // per wave
    static_assert(WPIECES % NW == 0, "every wave issues the same number of DMA pieces");
    extern __shared__ __align__(16) unsigned char smem[];

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wk = wave / NT, wm = wave % NT / WGN, wn = wave % WGN;
    long long clk0 = 0, wall0 = 0;
    if (p.clocks) { clk0 = __builtin_amdgcn_s_memtime(); wall0 = __builtin_amdgcn_s_memrealtime(); }
    // Workgroup ids are dealt round-robin to the 8 XCDs.  The tile rows are cut into bands of 8 * RB rows; inside a band
    // XCD x owns rows [x * RB, (x + 1) * RB) and walks the columns with the rows running fastest: the RB workgroups that
    // share a weight tile run together, and the RB activation panels (sized by the host to stay in that XCD's L2) are
    // re-read from L2 for every column.  Bands follow one another.
    uint32_t wg = blockIdx.x;                                     // 32 bits: a 64-bit division is 200 scalar instructions in front of the first load
    const uint32_t total = gridDim.x, tiles_n = (uint32_t)p.tiles_n;
    int64_t tile_m, tile_n;
    if (p.rows_per_xcd > 0) {
        const uint32_t RB = (uint32_t)p.rows_per_xcd, x = wg & 7;
        const uint32_t l = wg >> 3, per_band = RB * tiles_n;
        const uint32_t band = l / per_band, l2 = l % per_band;
        tile_m = band * 8 * RB + x * RB + l2 % RB;
        tile_n = l2 / RB;
    } else {
        if (total % 8 == 0) wg = (wg % 8) * (total / 8) + wg / 8;
        tile_m = wg / tiles_n;
        tile_n = wg % tiles_n;
    }
    const int64_t MB = (p.M + 31) >> 5, NB = (p.N + 31) >> 5;
    const int KB = (int)(p.Kp >> 7), KBs = KB / KS;               // k-blocks of the row, steps (the launcher: KB % KS == 0)
    const int64_t KG = p.Kp >> 4;
    static_assert(!SWI || (WN == 2 && FAST), "the swiglu epilogue pairs a gate and an up n-block per wave");
    const int64_t NBs = NB >> 1;                                  // SWI: n-blocks per stacked segment
    const int64_t mb0 = tile_m * BMB, nb0 = SWI ? tile_n * WGN + wn : tile_n * BNB + wn * WN;
    // the n-block behind accumulator column j (columns past the end re-read a valid block and are never stored)
    auto nblock = [&](int j) -> int64_t {
        if constexpr (SWI) return (nb0 < NBs ? nb0 : NBs - 1) + j * NBs;
        else return nb0 + j < NB ? nb0 + j : NB - 1;
    };
    if constexpr (!SWI) mfma_select_segment(p, tile_n * BNB);
    float* const row_dq = reinterpret_cast<float*>(smem + dma3_work_bytes<T, WGM, WGN, WM, WN, KS, SWI>());
    int* const row_qs = reinterpret_cast<int*>(row_dq + BMB * 32);
    static_assert(BMB * 32 <= 64 * NW, "a row's scale and code sum per thread");
    float my_dq = 0.0f;                            // on their way while the first transfers are requested; into LDS behind the first wait
    int my_qs = 0;
    EpiScales<L, WM, WN> sc;
    if constexpr (W32) mfma_prefetch_scales<L, WM, WN>(p, sc, lane, wm, mb0, nb0);   // one row a lane: into registers
    else if (const int64_t m = mb0 * 32 + threadIdx.x; threadIdx.x < BMB * 32 && m < p.M) {
        my_dq = p.deq[m];
        my_qs = p.qsum[m];
    }
#pragma unroll
    for (int j = 0; j < WN; ++j)   // seg_rows is a multiple of 32: one weight scale per n-block
        sc.wdq[j] = p.wdeq[(uint32_t)(nblock(j) * 32) / (uint32_t)p.seg_rows];

    auto dma_block = [&](int kb, int boff) {                      // k-block kb -> buffer at byte offset boff
#pragma unroll
        for (int i = 0; i < NDMA; ++i) {
            const int w = i * NW + wave;
            const int sub = w / (BMB * 4), chunk = (w >> 2) % BMB, within = w & 3;   // 4 pieces per m-block
            int64_t mb = mb0 + chunk;
            if (mb >= MB) mb = MB - 1;                            // rows past M are never stored: any valid data will do
            const int kbc = (kb < KBs ? kb : KBs - 1) * KS + sub; // past the end: harmless re-read, never consumed
            const unsigned char* g = reinterpret_cast<const unsigned char*>(p.a) + (mb * KG + kbc * 8 + within * 2) * 512;
            mfma_dma_1k(g, (uint32_t)lane * 16u, smem + boff + w * 1024);
        }
    };
    const uint32_t boff = W32 ? (uint32_t)lane * 16u : (uint32_t)(((lane >> 4) & 1) * 32 + (lane >> 5) * 16 + (lane & 15)) * 16u;
    auto load_b = [&](int kb, uint4 (&dst)[WN]) {                 // unconditional: the barrier's vmcnt counts on WN loads
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            const int64_t nb = nblock(j);
            const int kbc = (kb < KBs ? kb : KBs - 1) * KS + wk;  // past the end: never consumed
            // wave-uniform block address + a 32-bit lane offset: the load then takes its base from scalar registers and
            // no 64-bit per-lane address is kept alive
            const unsigned char* blk = reinterpret_cast<const unsigned char*>(p.b + (nb * KB + kbc) * 64);
            dst[j] = *reinterpret_cast<const uint4*>(blk + boff);
        }
    };
    // A loaded set as operands.  Lane l loaded the dwords of weight row 16 (l / 32) + l % 16, k-half (l / 16) % 2; exchanging the upper half of the
    // lanes of the first dword with the lower half of the second leaves rows 0-15 in x and rows 16-31 in y, the lanes' fourths on
    // inputs 0-15, 16-31, 32-47, 48-63 of the k-block; z and w the same of its second half.
    auto arrange_b = [&](uint4 (&s)[WN]) {
#pragma unroll
        for (int j = 0; j < WN; ++j) {
            const auto lo = __builtin_amdgcn_permlane32_swap(s[j].x, s[j].y, false, false);
            const auto hi = __builtin_amdgcn_permlane32_swap(s[j].z, s[j].w, false, false);
            s[j] = make_uint4(lo[0], lo[1], hi[0], hi[1]);
        }
    };
    auto expand = [](uint32_t w) {
        v4i b;
        b[0] = (int)(w & 0x03030303u);
        b[1] = (int)((w >> 2) & 0x03030303u);
        b[2] = (int)((w >> 4) & 0x03030303u);
        b[3] = (int)((w >> 6) & 0x03030303u);
        return b;
    };

    // B is requested a k-block and a half before its first use, into a ring of three register sets.  The ring is walked
    // by unrolling the k-loop three times, so a set keeps its registers from its load to its last use (rotating the sets
    // with copies at the loop's back edge makes the compiler wait there for everything in flight: the copy reads the set
    // loaded last).
    uint4 bset0[WN], bset1[WN], bset2[WN];
    dma_block(0, 0);
    dma_block(1, BUF);
    load_b(0, bset0);
    load_b(1, bset1);
    __builtin_amdgcn_s_waitcnt(0x0F70);            // vmcnt(0): this wave's pieces of k-blocks 0 and 1 have landed
    if (!W32 && threadIdx.x < BMB * 32) {
        row_dq[threadIdx.x] = my_dq;
        row_qs[threadIdx.x] = my_qs;
    }
    __syncthreads();

    if constexpr (!W32) arrange_b(bset0);

    // FAST: a lane's accumulators start at -qsum of their row (read for every group and masked: as a choice the compiler branches around
    // a read of its own for each of the accumulators, 2 us of a launch)
    Acc acc[WM][WN];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int qs = W32 ? sc.qs[i][0] : FAST ? row_qs[(wm * WM + i) * 32 + L::row(lane, g)] : 0;
            const int init = FAST ? -qs & (KS == 1 || wk == 0 ? -1 : 0) : 0;
#pragma unroll
            for (int j = 0; j < WN; ++j)
#pragma unroll
                for (int t = 0; t < 4; ++t) acc_set(acc[i][j], g, t, init);
        }
    int cur = 0, nxt = BUF, fre = 2 * BUF;         // byte offsets of the buffers of k-blocks s, s+1, s+2
    auto k_loop = [&](auto&& kblock) __attribute__((always_inline)) {
        int kb = 0;
        for (;;) {                                 // left in the middle: no copy of a k-block for the remainder, whose code a launch would fetch cold
            kblock(kb, bset0, bset1, bset2);
            if (++kb >= KBs) break;
            kblock(kb, bset1, bset2, bset0);
            if (++kb >= KBs) break;
            kblock(kb, bset2, bset0, bset1);
            if (++kb >= KBs) break;
        }
    };
    if constexpr (W32) {
        // One k-block in four steps of 32; the requests go out right behind the barrier, and a step's weights are expanded under the MFMAs of the
        // step before, columns outermost: once the MFMAs of a column are issued, its registers take the next step's.
        const int aoff = (wk * BMB + wm * WM) * CH + lane * 16;
        v4i af[2][WM], bf[WN];
#pragma unroll
        for (int i = 0; i < WM; ++i) af[0][i] = *reinterpret_cast<const v4i*>(smem + cur + aoff + i * CH);
#pragma unroll
        for (int j = 0; j < WN; ++j) bf[j] = expand(bset0[j].x);
        k_loop([&](int kb, const uint4 (&bcur)[WN], const uint4 (&bnxt)[WN], uint4 (&bfar)[WN]) __attribute__((always_inline)) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) {
                if (ks == 2) {                                     // (the wait of the other form below)
                    mfma_barrier_vm<0>();
                    dma_block(kb + 2, fre);
                    load_b(kb + 2, bfar);
                }
                const unsigned char* nsrc = ks < 3 ? smem + cur + aoff + (ks + 1) * 1024 : smem + nxt + aoff;
#pragma unroll
                for (int i = 0; i < WM; ++i) af[(ks + 1) & 1][i] = *reinterpret_cast<const v4i*>(nsrc + i * CH);
                v4i bn[WN];
#pragma unroll
                for (int j = 0; j < WN; ++j) {
#pragma unroll
                    for (int i = 0; i < WM; ++i) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bf[j], af[ks & 1][i], acc[i][j], 0, 0, 0);
                    bn[j] = expand(ks == 0 ? bcur[j].y : ks == 1 ? bcur[j].z : ks == 2 ? bcur[j].w : bnxt[j].x);
                }
                __builtin_amdgcn_sched_group_barrier(0x100, WM, 0);
#pragma unroll
                for (int j = 0; j < WN; ++j) {
                    __builtin_amdgcn_sched_group_barrier(0x008, WM, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, 7, 0);
                }
#pragma unroll
                for (int j = 0; j < WN; ++j) bf[j] = bn[j];
                __builtin_amdgcn_sched_barrier(0);
            }
            const int t = cur; cur = nxt; nxt = fre; fre = t;
        });
    } else {
        // A 16 x 64 fragment: lane l reads input group l / 16 of row l % 16
        const int aoff = (wk * BMB + wm * WM) * CH + (lane >> 4) * 512 + (lane & 15) * 16;
        constexpr int MF = 2 * WM, NF = 2 * WN;        // 16-row and 16-column fragments of the wave tile
        auto read_a = [&](int off, int f) { return *reinterpret_cast<const v4i*>(smem + off + aoff + (f >> 1) * CH + (f & 1) * 256); };
        // word of the arranged set for step q of its k-block, column fragment c
        auto word = [](const uint4 (&s)[WN], int q, int c) {
            const uint4 w = s[c >> 1];
            return q == 0 ? ((c & 1) == 0 ? w.x : w.y) : (c & 1) == 0 ? w.z : w.w;
        };
        v4i af[2], bf[NF];
        af[0] = read_a(cur, 0);
#pragma unroll
        for (int c = 0; c < NF; ++c) bf[c] = expand(word(bset0, 0, c));

        // One k-block in two steps of 64: contracts with the set `bcur`, requests k-block kb + 2 into `bfar`.  Activation rows outermost, the next
        // row's fragment on its way from LDS under this row's MFMAs; under the last row every weight fragment is replaced by the next step's
        // as soon as its MFMA has been issued.  (A step's weights and two row fragments: 24 registers, which is what 64 accumulators, three
        // sets in flight and addresses leave of 128.  Columns outermost, two more weight fragments expanded a row earlier, or four and eight row fragments
        // ahead, where one workgroup per CU leaves the registers, all measured the same or slower.)
        auto kblock = [&](int kb, const uint4 (&bcur)[WN], uint4 (&bnxt)[WN], uint4 (&bfar)[WN]) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                if (q == 1) {
                    // Everything requested one k-block ago -- this wave's pieces of A k-block kb+1 and the weights of kb+1 --
                    // has to be here now.  The wait is for ALL vector-memory traffic: a transfer into LDS and an ordinary load
                    // do not complete in the order they were issued (a count that leaves the younger weight loads in flight let
                    // warm weight loads overtake a cold A transfer and gave wrong sums), so the next requests go out after
                    // the barrier, between the rows' MFMAs (ahead of them all waves' address arithmetic left the matrix pipe idle: 0.64 us a k-block
                    // with one workgroup per CU, 0.61 so), and have the rest of the k-block and half the next to land.  The weights that have
                    // come in are arranged ahead of them: the compiler waits for them by a count that does not know of the transfer, which behind it
                    // would be a wait for the transfer.
                    mfma_barrier_vm<0>();
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int f = 0; f < MF; ++f) {
                    const int t = q * MF + f + 1;                      // of the 2 MF fragments of this k-block, then the next one's first
                    af[t & 1] = t < 2 * MF ? read_a(cur + t / MF * 2048, t % MF) : read_a(nxt, 0);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int c = 0; c < NF; ++c) {
                        v4i& d = acc[f >> 1][c >> 1].g[2 * (f & 1) + (c & 1)];
                        if (f == 0 && c == 0) mfma_16x16x64<true>(d, bf[c], af[f & 1]);
                        else mfma_16x16x64<false>(d, bf[c], af[f & 1]);
                        if (f == MF - 1) bf[c] = expand(q == 0 ? word(bcur, 1, c) : word(bnxt, 0, c));
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if (q == 1) {
                        if (f == 0) arrange_b(bnxt);
                        if (f == 1 || MF == 1) dma_block(kb + 2, fre);
                        if (f == (MF > 2 ? 2 : MF - 1)) load_b(kb + 2, bfar);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
            const int t = cur; cur = nxt; nxt = fre; fre = t;
        };
        k_loop(kblock);
        mfma_done(acc);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);            // the trailing DMA must not land in the epilogue's staging area
    __syncthreads();
    if constexpr (!W32) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                sc.dq[i][h] = row_dq[(wm * WM + i) * 32 + L::row(lane, 2 * h)];
                sc.qs[i][h] = FAST ? 0 : row_qs[(wm * WM + i) * 32 + L::row(lane, 2 * h)];
            }
    }
    if constexpr (KS == 1) {
        if constexpr (SWI) mfma_epilogue_swiglu<T, L>(p, acc, sc, smem, lane, wave, wm, mb0, nb0);
        else if constexpr (FAST) mfma_epilogue_fast<FAST == 2, T, L>(p, acc, sc, smem, lane, wave, wm, mb0, nb0);
        else mfma_epilogue<T, L>(p, acc, sc, smem, lane, wave, wm, mb0, nb0);
    } else {
        // group g finishes row block g of the wave tile: it takes the other groups' partial sums of that block
        static_assert(KS == WM, "a row block of the wave tile per group");
        int* const ex = reinterpret_cast<int*>(smem);            // [source wave][KS - 1 blocks][WN][16][64]
        constexpr int BLK = WN * 16 * 64;
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            if (i != wk) {
                int* dst = ex + (wave * (KS - 1) + (i > wk ? i - 1 : i)) * BLK + lane;
#pragma unroll
                for (int j = 0; j < WN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) dst[(j * 16 + r) * 64] = acc_at(acc[i][j], r >> 2, r & 3);
            }
        }
        __syncthreads();
        Acc mine[1][WN];
        EpiScales<L, 1, WN> sc1;
#pragma unroll
        for (int i = 0; i < WM; ++i) {
            if (i == wk) {
#pragma unroll
                for (int h = 0; h < L::RH; ++h) {
                    sc1.dq[0][h] = sc.dq[i][h];
                    sc1.qs[0][h] = sc.qs[i][h];
                }
#pragma unroll
                for (int j = 0; j < WN; ++j) mine[0][j] = acc[i][j];
            }
        }
#pragma unroll
        for (int j = 0; j < WN; ++j) sc1.wdq[j] = sc.wdq[j];
#pragma unroll
        for (int o = 0; o < KS; ++o) {
            if (o != wk) {
                const int* src = ex + ((o * NT + wave % NT) * (KS - 1) + (wk > o ? wk - 1 : wk)) * BLK + lane;
#pragma unroll
                for (int j = 0; j < WN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc_set(mine[0][j], r >> 2, r & 3, acc_at(mine[0][j], r >> 2, r & 3) + src[(j * 16 + r) * 64]);
            }
        }
        __syncthreads();                                         // the exchange area becomes the epilogue's staging area
        const int wm1 = wm * WM + wk;
        if constexpr (SWI) mfma_epilogue_swiglu<T, L>(p, mine, sc1, smem, lane, wave, wm1, mb0, nb0);
        else if constexpr (FAST) mfma_epilogue_fast<FAST == 2, T, L>(p, mine, sc1, smem, lane, wave, wm1, mb0, nb0);
        else mfma_epilogue<T, L>(p, mine, sc1, smem, lane, wave, wm1, mb0, nb0);
    }
    if (p.clocks && threadIdx.x == 0 && (int64_t)blockIdx.x < p.clock_cap) {
        p.clocks[2 * blockIdx.x] = __builtin_amdgcn_s_memtime() - clk0;
        p.clocks[2 * blockIdx.x + 1] = __builtin_amdgcn_s_memrealtime() - wall0;
    }
}

// Tile rows per XCD and band (see the kernel): the largest divisor of tiles_m / 8 whose activation panels
// (tile_rows * Kp bytes each) stay within 1.5 MiB of an XCD's 4 MiB L2 (measured at 16384 x 2048 x 11264: 0.389 ms
// against 0.410 ms with all 32 panels of an XCD in one band; smaller budgets are no better); 0 when tiles_m is not a
// multiple of 8.
inline int mfma_rows_per_xcd(int tiles_m, int tile_rows, int64_t Kp) {
    if (tiles_m % 8 != 0) return 0;
    const int R = tiles_m / 8;
    const int64_t budget = 1536 << 10;
    int64_t cap = budget / ((int64_t)tile_rows * Kp);
    if (cap < 1) cap = 1;
    int best = 1;
    for (int d = 1; d <= R && d <= cap; ++d)
        if (R % d == 0) best = d;
    return best;
}

template <typename T, int WGM, int WGN, int WM, int WN, int KS, bool SWI>
int launch_mfma_dma3(MfmaArgs a, hipStream_t s) {
    constexpr int BM = WGM * WM * 32, BN = WGN * WN * 32;        // SWI: BN rows of the stacked weight, BN / 2 channels
    a.clocks = g_clock_sink; a.clock_cap = g_clock_cap;
    a.tiles_m = (int)mmf_ceil_div(a.M, BM);
    a.tiles_n = SWI ? (int)mmf_ceil_div(a.N / 2, BN / 2) : (int)mmf_ceil_div(a.N, BN);
    a.rows_per_xcd = mfma_rows_per_xcd(a.tiles_m, BM, a.Kp);
    constexpr int waves = WGM * WGN * KS;
    constexpr size_t lds = dma3_work_bytes<T, WGM, WGN, WM, WN, KS, SWI>() + BM * 8;
    const int per_vec = 16 / (int)sizeof(T);
    a.vec_store = SWI || ((a.N % per_vec == 0) && (a.ldo % per_vec == 0) && ((reinterpret_cast<uintptr_t>(a.out) & 15u) == 0) &&
                          ((reinterpret_cast<uintptr_t>(a.addend) & 15u) == 0));
    // 16-bit outputs of 20 MB and more leave the caches to the activations and weights.  bf16, the launch and what reads its output next, us: 16384 x 2048 ->
    // 6144 (201 MB) 148 and 70 (gate and scan), streamed 147 and 62; -> 2048 and 5632 -> 2048 (67 MB) 98.5 on average and 46.9 (residual norm), 94.6
    // and 44.6; 2002 x 2048 -> 6144 (25 MB) 31.7 and 16.4, 29.5 and 17.0.  1377 rows (17 MB): 26.3 and 12.5, 25.1 and 13.2, no gain.  Whole forwards: 16384
    // tokens 21.01 ms, streamed 20.77, 2002 tokens with logits and loss 4.45 and 4.41.  By itself the launch is 2 to 4 % shorter over outputs of 1024 to 11264
    // columns and 20 to 160 MB, with a copy behind it as long.  Only whole lines: rows that share theirs are written twice, alone and with a copy behind
    // it 40 MB of 1000 columns 25.9 and 40.6, streamed 27.6 and 43.7, of 1960 39.0 and 52.9, 40.4 and 53.8, of 4104 37.3 and 52.1, 39.9 and 54.8.  Not the swiglu
    // form, whose output is half as large for its time: 293 and 54 (quantiser), 297 and 65; nor fp32: 666 x 1024 -> 32000 (85 MB) 36.6 and 18.9 (loss), 34.7 and 30.0.
    auto kern = bitlinear_mfma_dma3_kernel<T, WGM, WGN, WM, WN, KS, 1, SWI>;
    if constexpr (!SWI) {
        if (!a.vec_store || a.bias) kern = bitlinear_mfma_dma3_kernel<T, WGM, WGN, WM, WN, KS, 0, false>;
        else if constexpr (sizeof(T) == 2) {
            if (a.M * a.N * 2 >= (20 << 20) && a.ldo % 64 == 0 && (reinterpret_cast<uintptr_t>(a.out) & 127u) == 0) kern = bitlinear_mfma_dma3_kernel<T, WGM, WGN, WM, WN, KS, 2, false>;
        }
    }
    if constexpr (KS > 1) {
        if ((int64_t)a.tiles_m * a.tiles_n <= 256) {             // (too small an output to be streamed)
            kern = bitlinear_mfma_dma3_kernel<T, WGM, WGN, WM, WN, KS, 1, SWI, true>;
            if constexpr (!SWI) {
                if (!a.vec_store || a.bias) kern = bitlinear_mfma_dma3_kernel<T, WGM, WGN, WM, WN, KS, 0, false, true>;
            }
        }
    }
    if (lds > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)lds);
        if (e != hipSuccess) return (int)e;
    }
    kern<<<dim3((unsigned)((int64_t)a.tiles_m * a.tiles_n)), dim3(64 * waves), lds, s>>>(a);
    MMF_CHECK_LAUNCH();
    return 0;
}

// ------------------------------------------------------------------------------------------
// Small problems (decode batches, short prompts): the contraction is a weight stream, not a
// GEMM, and the enemy is latency, so nothing is staged and nothing waits on a barrier until the
// very end.  One workgroup of NWV waves owns a 32x32 output block (grid.y walks M); wave w takes the k-blocks
// w, w + NWV, ...: at most ITER of them, with the loads of PF in flight.
// A fragments (1 KiB each, L2 resident: the whole A is M x K bytes) and the packed B block
// are loaded straight into registers; the partial accumulators meet in LDS and all threads run the epilogue.
// NWV = 16 where that still leaves a CU per workgroup: half the k-blocks in a wave's chain.  NWV = 8 otherwise, in few enough
// registers for three workgroups a CU when the row is short (a gate/up projection of 704 blocks took two rounds at two a
// CU).  Measured at 64 rows, 1.3B shape: gate/up 7.9 -> 6.6 us, down_proj 7.2 -> 6.1 us against 8 waves and three k-blocks in
// flight for every shape.
// SWI: the weight is stacked [gate; up] (N = 2 I) and a workgroup contracts the gate and the up rows of the same 32 channels with
// shared A fragments, half of their traffic; the epilogue writes swiglu(gate, up), so the exp and divide of the MLP activation
// run spread over all workgroups instead of in the next quantiser's one workgroup per row: 6.6 + 5.9 -> 6.4 + 4.2 us for the two.
// (Two plain n-blocks per workgroup measured no faster than one.)
template <typename T, int NWV, int ITER, bool SWI>
__global__ __launch_bounds__(64 * NWV, NWV == 8 && ITER <= 2 && !SWI ? 6 : 4) void bitlinear_mfma_skinny_kernel(MfmaArgs p) {
    constexpr int NB = SWI ? 2 : 1, PF = ITER < 3 ? ITER : 3, NT = 64 * NWV, EL = 1024 / NT;   // outputs per thread
    __shared__ int red[NWV][NB][16][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // wave-uniform: keep it in a scalar register
    const int64_t nb = blockIdx.x, nb1 = nb + (p.N >> 6), mb = blockIdx.y;           // SWI: nb1 holds the up rows
    mfma_select_segment(p, nb);
    const int KB = (int)(p.Kp >> 7);
    const int8_t* abase = p.a + mb * (p.Kp >> 4) * 512;
    const uint4* const bbase[2] = {p.b + nb * KB * 64, p.b + nb1 * KB * 64};

    v16i acc[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0;
    uint4 breg[PF][NB];
    v4i areg[PF][4];
    auto load_stage = [&](int st, int kb) __attribute__((always_inline)) {
        if (kb < KB) {
#pragma unroll
            for (int i = 0; i < NB; ++i) breg[st][i] = bbase[i][kb * 64 + lane];
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) areg[st][ks] = *reinterpret_cast<const v4i*>(abase + (kb * 8 + ks * 2) * 512 + lane * 16);
        }
    };
#pragma unroll
    for (int st = 0; st < PF; ++st) load_stage(st, wave + st * NWV);

    // the epilogue's operands, requested now so that the end of the kernel waits for nothing
    const T* bias = static_cast<const T*>(p.bias);
    const T* addend = static_cast<const T*>(p.addend);
    T* out = static_cast<T*>(p.out);
    const int64_t n_ep = nb * 32 + (lane & 31);
    const bool n_ok = SWI || n_ep < p.N;
    float ep_wdeq[NB];                                   // an n-block never straddles a segment
#pragma unroll
    for (int i = 0; i < NB; ++i) ep_wdeq[i] = p.wdeq[(uint32_t)((i ? nb1 : nb) * 32) / (uint32_t)p.seg_rows];
    const float ep_bias = (bias && n_ok) ? mmf_to_float(bias[n_ep]) : 0.0f;
    int ep_qsum[EL];
    float ep_deq[EL], ep_add[EL];
#pragma unroll
    for (int j = 0; j < EL; ++j) {
        const int r = wave + j * NWV;                    // accumulator register of this thread's j-th output
        const int64_t m = mb * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        const int64_t mc = m < p.M ? m : 0;
        ep_qsum[j] = p.qsum[mc];
        ep_deq[j] = p.deq[mc];
        ep_add[j] = (addend && n_ok) ? mmf_to_float(addend[mc * p.ldo + n_ep]) : 0.0f;
    }

#pragma unroll
    for (int it = 0; it < ITER; ++it) {
        const int st = it % PF, kb = wave + it * NWV;
        if (kb < KB) {
#pragma unroll
            for (int ks = 0; ks < 4; ++ks)
#pragma unroll
                for (int i = 0; i < NB; ++i) {
                    const uint4 bq = breg[st][i];
                    const uint32_t w = ks == 0 ? bq.x : ks == 1 ? bq.y : ks == 2 ? bq.z : bq.w;
                    v4i bf;
                    bf[0] = (int)(w & 0x03030303u);
                    bf[1] = (int)((w >> 2) & 0x03030303u);
                    bf[2] = (int)((w >> 4) & 0x03030303u);
                    bf[3] = (int)((w >> 6) & 0x03030303u);
                    acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(areg[st][ks], bf, acc[i], 0, 0, 0);
                }
        }
        if (it + PF < ITER) load_stage(st, wave + (it + PF) * NWV);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) red[wave][i][r][lane] = acc[i][r];
    __syncthreads();

#pragma unroll
    for (int j = 0; j < EL; ++j) {
        const int r = wave + j * NWV;
        const int64_t m = mb * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        float o[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            int tot = 0;
#pragma unroll
            for (int w = 0; w < NWV; ++w) tot += red[w][i][r][lane];
            o[i] = __fmul_rn(__fmul_rn((float)(tot - ep_qsum[j]), ep_deq[j]), ep_wdeq[i]);
        }
        if constexpr (SWI) {
            const float g[1] = {mmf_round_to<T>(o[0])}, u[1] = {mmf_round_to<T>(o[1])};
            float z[1];
            mmf_swiglu_n<T, 1>(g, u, z);
            if (m < p.M) out[m * p.ldo + n_ep] = mmf_from_float<T>(z[0]);
        } else if (m < p.M && n_ok) {
            if (bias) o[0] = __fadd_rn(o[0], ep_bias);
            if (addend) o[0] = __fadd_rn(mmf_round_to<T>(o[0]), ep_add[j]);
            out[m * p.ldo + n_ep] = mmf_from_float<T>(o[0]);
        }
    }
}

template <typename T, int NWV, bool SWI>
void launch_skinny_waves(const MfmaArgs& a, dim3 grid, hipStream_t s) {
    const int64_t it = mmf_ceil_div(a.Kp >> 7, (int64_t)NWV);
    if (it <= 1) bitlinear_mfma_skinny_kernel<T, NWV, 1, SWI><<<grid, dim3(64 * NWV), 0, s>>>(a);
    else if (it <= 2) bitlinear_mfma_skinny_kernel<T, NWV, 2, SWI><<<grid, dim3(64 * NWV), 0, s>>>(a);
    else if (it <= 3) bitlinear_mfma_skinny_kernel<T, NWV, 3, SWI><<<grid, dim3(64 * NWV), 0, s>>>(a);
    else if (it <= 4) bitlinear_mfma_skinny_kernel<T, NWV, 4, SWI><<<grid, dim3(64 * NWV), 0, s>>>(a);
    else if constexpr (NWV == 8) {
        if (it <= 6) bitlinear_mfma_skinny_kernel<T, NWV, 6, SWI><<<grid, dim3(64 * NWV), 0, s>>>(a);
        else bitlinear_mfma_skinny_kernel<T, NWV, 8, SWI><<<grid, dim3(64 * NWV), 0, s>>>(a);
    }
}
// Kp <= 8192: at most 64 k-blocks, four per wave of 16 or eight per wave of 8
template <typename T>
int launch_skinny(const MfmaArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)mmf_ceil_div(a.N, 32), (unsigned)mmf_ceil_div(a.M, 32));
    if ((int64_t)grid.x * grid.y <= 256) launch_skinny_waves<T, 16, false>(a, grid, s);
    else launch_skinny_waves<T, 8, false>(a, grid, s);
    MMF_CHECK_LAUNCH();
    return 0;
}
template <typename T>
int launch_skinny_swiglu(const MfmaArgs& a, hipStream_t s) {
    launch_skinny_waves<T, 8, true>(a, dim3((unsigned)(a.N / 64), (unsigned)mmf_ceil_div(a.M, 32)), s);
    MMF_CHECK_LAUNCH();
    return 0;
}

template <typename T, int WGM, int WGN, int WM, int WN, int KSL = 1>
int launch_mfma(MfmaArgs a, hipStream_t s) {
    constexpr int BM = WGM * WM * 32, BN = WGN * WN * 32;
    a.tiles_m = (int)mmf_ceil_div(a.M, BM);
    a.tiles_n = (int)mmf_ceil_div(a.N, BN);
    size_t lds = 2u * (WGM * WM) * 4096u * KSL;
    const size_t lds_epi = (size_t)(WGM * WGN) * 32u * (WN * 32u * sizeof(T) + 16u);   // per-wave output staging
    if (lds_epi > lds) lds = lds_epi;
    const int per_vec = 16 / (int)sizeof(T);
    a.vec_store = (a.N % per_vec == 0) && (a.ldo % per_vec == 0) && ((reinterpret_cast<uintptr_t>(a.out) & 15u) == 0) &&
                  ((reinterpret_cast<uintptr_t>(a.addend) & 15u) == 0);
    auto kern = bitlinear_mfma_kernel<T, WGM, WGN, WM, WN, KSL>;
    if (lds > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)lds);
        if (e != hipSuccess) return (int)e;
    }
    kern<<<dim3((unsigned)((int64_t)a.tiles_m * a.tiles_n)), dim3(64 * WGM * WGN), lds, s>>>(a);
    MMF_CHECK_LAUNCH();
    return 0;
}

// Which kernel is the fastest, from its measured time on MI355X (us; N from 1024 to 11264, K from 1024 to 9216, M from 77 to 9600):
//   weight stream  3 + 0.7 ns per output block + 0.18 ns per output block and k-block, as long as the row fits its LDS;
//   split tiles    (64 x 256, two groups of waves on every second k-block) at most one tile per CU: a chain of 0.29 us per k-block, and
//                  what a fuller chip adds.  At most two per CU run side by side and share it: one time, whatever their number.  Beyond
//                  that, 3.9 + 0.295 us per k-block for every 256;
//   tiles          (64 x 512) at most one per CU: 4.4 + 0.58 us per k-block and what a fuller chip adds; beyond, 4.4 + 0.62 per 256.
// A whole tile is worth two split ones, so against an even number of split rounds whole tiles win or tie, but for two rounds of long rows,
// and where the last round of whole tiles would be less than half full, an odd number of split rounds does instead.  Split against whole:
// 5632 -> 2048 (44 k-blocks), 2002 rows (256 split tiles) 23.4 / 33.8, 3600 (456) 34.6 / 38.8, 9600 82.1 / 87.2; 6912 -> 2560 (54), 2300 rows
// 39.7 / 43.3, 6500 86.5 / 77.4; 2048 -> 2048 (16), 2002 rows 12.2 / 15.1, 3600 18.0 / 18.5; 2048 -> 6144, 2002 rows (768) 27.1 / 26.4.  Stream against split:
// 1024 -> 5632, 300 rows 6.0 / 8.4, 700 9.9 / 9.4; 2048 -> 2048, 1203 rows 10.9 / 11.4, 1395 12.1 / 11.3.
// Over 389 shapes, 66 to 8000 rows, the choice costs 0.01 % against the best of the three on average, 15 % at most (377 x 1536 -> 4608: 1.2 us).
//   narrow tiles   (64 x 128, split like the others) where they give every CU at most one, or three in all; with rows of 2560 to 6144 also instead of a
//                  split one on nearly every CU (481 to 512 of them: over 72 shapes 1.4 % less on average, from 10 % less to 4 % more, most where their last row of
//                  tiles is nearly empty; rows of 6912 0.6 % more).  us, best of the others / narrow: 5632 -> 2048, 700 rows 15.6 / 12.8, 1001 (256 narrow tiles) 19.0 / 13.9, 1377 (352)
//                  20.1 / 20.5, 2002 (512) 24.5 / 23.2, 2400 (608) 32.9 / 29.2; 2048 -> 2048, 830 rows 8.3 / 7.4, 1001 9.2 / 7.8, 1200 (304) 10.4 / 10.8, 2002
//                  11.7 / 11.8; 2816 -> 1024, 1600 rows 11.9 / 8.4, 4022 (504) 16.4 / 14.5, 4100 (520) 19.7 / 17.4; 2560 -> 2560, 711 rows 11.3 / 8.4, 1491 (480) 13.0 / 13.2,
//                  1966 (620) 20.3 / 18.4; 2048 -> 6144, 320 rows 9.3 / 7.6.  Weights that an XCD's L2 does not hold cost it more (6912 -> 2560, 580 rows 18.9 / 19.2,
//                  700 21.3 / 19.6).  Against the stream, whose time is overestimated where it is short, with a margin (670 rows of 1536 -> 1536 stream 5.4, narrow 6.3).
//                  Over 110 shapes, 163 to 6000 rows, the choice with it takes 5.5 % less, at best 35.  Two groups of two waves, 64 columns each: 3 to 12 % slower
//                  than of four with 32.
// With the swiglu epilogue (M from 66 to 6300, K from 512 to 4096, N from 2048 to 22016) the stream's workgroups each own two blocks, of gate and of up, and
// take 1.3 + 0.1 ns per k-block a block; a tile's epilogue, which nothing hides where a CU has one, is 3 to 5 us.  Over 461 shapes beside the 357 fitted the choice costs 0.25 %
// on average, 8 % at most; with the plain products' times it cost 4 %, and 58 % at most (106 x 2560 -> 13824, stream / split 9.7 / 15.3 us; 410 x 1024 -> 5632
// 9.1 / 12.1 in a model).
enum class MfmaPick { kStream, kSplit, kNarrow, kTiles };
struct MfmaChoice { MfmaPick pick; double us; };
inline MfmaChoice mfma_choice(int64_t M, int64_t N, int64_t Kp, bool swiglu) {
    const int64_t KB = Kp >> 7;
    const double kb = (double)KB, blocks = (double)mmf_ceil_div(M, 32) * (double)mmf_ceil_div(N, 32);
    const int64_t half = mmf_ceil_div(M, 64) * mmf_ceil_div(N, 256), full = mmf_ceil_div(M, 64) * mmf_ceil_div(N, 512);
    const double halves = (double)half / 256.0, wholes = (double)full / 256.0, half_rounds = (double)mmf_ceil_div(half, 256), rounds = (double)mmf_ceil_div(full, 256);
    double t_stream, t_tiles, t_split, t_narrow = 1e30;
    if (swiglu) {
        t_stream = 3.5 + blocks * (0.0013 + 0.0001 * kb);
        t_tiles = full <= 256 ? 9.2 + 0.585 * kb + wholes * (0.19 * kb - 1.0) : 6.5 + rounds * (3.5 + 0.54 * kb);
        t_split = half <= 256 ? 8.0 + 0.285 * kb + halves * 0.1 * kb : half <= 512 ? 10.5 + 0.595 * kb : 5.8 + half_rounds * (2.4 + 0.297 * kb);
    } else {
        t_stream = 3.0 + blocks * (0.0007 + 0.00018 * (double)((KB + 7) / 8 * 8));
        t_tiles = full <= 256 ? 4.4 + 0.58 * kb + wholes * (1.0 + 0.18 * kb) : rounds * (4.4 + 0.62 * kb);
        t_split = half <= 256 ? 4.4 + 0.29 * kb + halves * (1.0 + 0.1 * kb) : half <= 512 ? 8.5 + 0.59 * kb : half_rounds * (3.9 + 0.295 * kb);
    }
    if (!swiglu) {
        const int64_t narrow = mmf_ceil_div(M, 64) * mmf_ceil_div(N, 128);
        if (narrow <= 256) t_narrow = 3.9 + 0.17 * kb + (double)narrow / 256.0 * (0.3 + 0.045 * kb) + (N * Kp > 16 << 20 ? 0.1 * kb : 0.0);
        else if (narrow > 480 && half <= 256 && KB >= 20 && KB <= 48) t_narrow = t_split - 0.1;   // (instead of a split one, whatever that is estimated at)
        else if (narrow > 512 && narrow <= 768) t_narrow = 7.0 + 0.54 * kb;
    }
    if (KB % 2 != 0) t_split = t_narrow = 1e30;
    if (Kp <= 8192 && M <= 65535 * 32 && (M <= 64 || (t_stream <= t_split && t_stream <= t_tiles && t_stream * (KB < 20 ? 0.85 : 0.95) <= t_narrow))) return {MfmaPick::kStream, t_stream};
    if (t_narrow < t_split && t_narrow < t_tiles) return {MfmaPick::kNarrow, t_narrow};
    if (t_split < t_tiles) return {MfmaPick::kSplit, t_split};
    return {MfmaPick::kTiles, t_tiles};
}

// The kernel of a choice (dispatch_mfma's numbers), and the columns of its tiles: 0 where they are never several segments' in one launch.
inline int mfma_config(MfmaPick pick, int64_t M, int64_t N) {
    if (pick == MfmaPick::kStream) return 5;
    if (M <= 64) return M <= 32 ? 0 : 1;
    return pick == MfmaPick::kSplit ? 18 : pick == MfmaPick::kNarrow ? 19 : N >= 512 ? 17 : 16;
}
inline int64_t mfma_tile_cols(int config) { return config == 5 ? 32 : config == 19 ? 128 : config == 16 || config == 18 ? 256 : config == 17 ? 512 : 0; }
// tiles that suit segments with codes of their own (of seg columns; 0: one set of codes)
inline bool mfma_suits(int config, int64_t N, int64_t seg) { return seg == 0 || N <= seg || (mfma_tile_cols(config) && seg % mfma_tile_cols(config) == 0); }

// The rows of the first of two launches, or all of them: where the tiles' last round holds a few of them, its rows go in a launch of their own, most
// often the stream's.  us, one launch / two (rows of the second): 2048 -> 6144, 1377 rows (528 split tiles; 33) 27.2 / 23.3, 2693 (5) 36.6 / 29.0, 5549 (109)
// 59.6 / 54.5; gate and up to 5632 with swiglu, 3066 (122) 80.6 / 73.7, 715 (11) 26.3 / 25.2; 5632 -> 2048, 2096 (48) 32.6 / 27.7; 1536 -> 4608, 3586 (2)
// 30.9 / 23.7; 6912 -> 2560, 3357 (93) 61.2 / 49.2.  Over 87 shapes with at most 320 rows in the second, 65 to 16384 in all, that were estimated to gain 3 %: 5 % less
// on average, 15 % more at most.  Where the estimate has to promise 7 % (10 % from 129 rows on; 3 % with swiglu, whose rounds take longer than
// estimated) none took longer.  With 340 to 600 rows in the second two launches took between 12 % less and 12 % more (2048 -> 6144, 4843 (747)
// 47.7 / 53.5; 6912 -> 2560, 5431 (567) 70.6 / 79.2).  The sums are integers and a row's do not depend on the others: the same bits.
// Segments with codes of their own (seg columns) that do not suit a launch's tiles take a launch each, which no estimate covers: rows are cut only where all three
// launches suit them (three of 2304, cut all the same / in one go: 1157 rows 53.1 / 27.9 us, 2445 61.8 / 47.8; of 1152, 2473 36.1 / 32.4).
constexpr int64_t kCutRows = 320;
inline int64_t mfma_first_rows(int64_t M, int64_t N, int64_t Kp, int64_t seg, bool swiglu) {
    auto suits = [&](const MfmaChoice& c, int64_t m) { return mfma_suits(mfma_config(c.pick, m, N), N, seg); };
    const MfmaChoice all = mfma_choice(M, N, Kp, swiglu);
    const double whole = all.us;
    if (!suits(all, M)) return M;
    double least = whole;
    int64_t first = M;
    for (const int64_t cols : {256, 512}) {
        const int64_t across = mmf_ceil_div(N, cols), rounds = mmf_ceil_div(mmf_ceil_div(M, 64) * across, 256);
        for (int64_t r = rounds - 1; r >= 1 && r >= rounds - 2; --r) {
            const int64_t m = 256 * r / across * 64;
            if (m < 64 || m >= M || M - m > kCutRows) continue;
            const MfmaChoice head = mfma_choice(m, N, Kp, swiglu), tail = mfma_choice(M - m, N, Kp, swiglu);
            const double us = head.us + tail.us;
            if (suits(head, m) && suits(tail, M - m) && us < least && us < (swiglu ? 0.97 : M - m <= 128 ? 0.93 : 0.90) * whole) {
                least = us;
                first = m;
            }
        }
    }
    return first;
}
// rows m0 to m0 + m of a contraction (m0 a multiple of 32)
template <typename T>
MfmaArgs mfma_rows(MfmaArgs a, int64_t m0, int64_t m) {
    a.a += m0 * a.Kp;
    a.deq += m0;
    a.qsum += m0;
    if (a.addend) a.addend = static_cast<const T*>(a.addend) + m0 * a.ldo;
    a.out = static_cast<T*>(a.out) + m0 * a.ldo;
    a.M = m;
    return a;
}

template <typename T>
int dispatch_mfma(const MfmaArgs& a, int config, hipStream_t s, bool cut = true) {
    // config < 0: pick by shape, the rows in two launches where that is estimated to be faster (cut).
    //   5        weight-stream kernel: one 32x32 output block per workgroup, 8 waves split K (needs Kp <= 8192)
    //   0 / 1    32x256 / 64x256 tiles, A staged through registers (small M with Kp > 8192)
    //   18 / 19  64x256 / 64x128 tiles, two groups of waves on every second k-block (need an even number of k-blocks)
    //   15 / 16 / 17  256x256 / 128x256 / 64x512 tiles, A staged by DMA (17: every wave reads the whole activation
    //            tile from LDS and owns its own weight columns, so no weight block is fetched twice)
    if (config < 0) {
        const int64_t first = cut ? mfma_first_rows(a.M, a.N, a.Kp, a.a_seg ? a.seg_rows : 0, false) : a.M;
        if (first < a.M) {
            if (const int rc = dispatch_mfma<T>(mfma_rows<T>(a, 0, first), -1, s, false)) return rc;
            return dispatch_mfma<T>(mfma_rows<T>(a, first, a.M - first), -1, s, false);
        }
        config = mfma_config(mfma_choice(a.M, a.N, a.Kp, false).pick, a.M, a.N);
    }
    if ((config == 18 || config == 19) && (a.Kp >> 7) % 2 != 0) return MMF_ERR_ARG;
    if (config == 5 && (a.Kp > 8192 || a.M > 65535 * 32)) return MMF_ERR_ARG;
    if (a.a_seg != 0 && !mfma_suits(config, a.N, a.seg_rows)) {
        // tiles that would straddle two segments (or tiles of the kernels that take one set of codes): a launch per segment
        for (int64_t n0 = 0; n0 < a.N; n0 += a.seg_rows) {
            const int64_t seg = n0 / a.seg_rows;
            MfmaArgs b = a;
            b.a += seg * a.a_seg;
            b.deq += seg * a.m_seg;
            b.qsum += seg * a.m_seg;
            b.a_seg = 0;
            b.b += (n0 >> 5) * (a.Kp >> 7) * 64;
            b.wdeq += seg;
            b.N = a.N - n0 < a.seg_rows ? a.N - n0 : a.seg_rows;
            b.out = static_cast<T*>(a.out) + n0;
            if (const int rc = dispatch_mfma<T>(b, config, s)) return rc;
        }
        return 0;
    }
    switch (config) {
        case 5: return launch_skinny<T>(a, s);
        case 0: return launch_mfma<T, 1, 8, 1, 1>(a, s);
        case 1: return launch_mfma<T, 1, 8, 2, 1>(a, s);
        case 15: return launch_mfma_dma3<T, 2, 4, 4, 2, 1, false>(a, s);
        case 16: return launch_mfma_dma3<T, 2, 4, 2, 2, 1, false>(a, s);
        case 17: return launch_mfma_dma3<T, 1, 8, 2, 2, 1, false>(a, s);
        case 18: return launch_mfma_dma3<T, 1, 4, 2, 2, 2, false>(a, s);
        case 19: return launch_mfma_dma3<T, 1, 4, 2, 1, 2, false>(a, s);
    }
    return MMF_ERR_ARG;
}

template <typename T>
int dispatch_mfma_swiglu(const MfmaArgs& a, hipStream_t s, bool cut = true) {
    const int64_t first = cut ? mfma_first_rows(a.M, a.N, a.Kp, 0, true) : a.M;
    if (first < a.M) {
        if (const int rc = dispatch_mfma_swiglu<T>(mfma_rows<T>(a, 0, first), s, false)) return rc;
        return dispatch_mfma_swiglu<T>(mfma_rows<T>(a, first, a.M - first), s, false);
    }
    switch (mfma_choice(a.M, a.N, a.Kp, true).pick) {
        case MfmaPick::kStream: return launch_skinny_swiglu<T>(a, s);
        case MfmaPick::kSplit: return launch_mfma_dma3<T, 1, 4, 2, 2, 2, true>(a, s);
        case MfmaPick::kNarrow:
        case MfmaPick::kTiles: return launch_mfma_dma3<T, 1, 8, 2, 2, 1, true>(a, s);
    }
    return MMF_ERR_ARG;
}

// The matrix pipe with nothing else to do: every wave issues four independent 32x32x32 int8 MFMAs per
// step on operands that never leave its registers (8 waves per workgroup, 4 waves per SIMD with two workgroups per CU).
// random_operands: int8 codes and ternary weights drawn per lane (the switching activity of real operands) instead of the
// constant 1s, on which the pipe draws far less power.
__global__ __launch_bounds__(512, 4) void mfma_pipe_probe_kernel(int64_t steps, int random_operands, long long* clocks, int* sink) {
    const long long clk0 = __builtin_amdgcn_s_memtime(), wall0 = __builtin_amdgcn_s_memrealtime();
    auto mix = [](uint32_t x) { x ^= x >> 16; x *= 0x7feb352du; x ^= x >> 15; x *= 0x846ca68bu; x ^= x >> 16; return x; };
    v4i a[2], b[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            a[h][i] = random_operands ? (int)mix(threadIdx.x * 16 + h * 4 + i) : 0x01010101 * (int)(threadIdx.x & 1);
            b[h][i] = random_operands ? (int)(mix(threadIdx.x * 16 + 8 + h * 4 + i) & 0x03030303u) : 0x01010101;
        }
    v16i acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0;
    for (int64_t s = 0; s < steps; ++s) {
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(b[t & 1], a[t >> 1], acc[t], 0, 0, 0);
    }
    int x = 0;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) x ^= acc[t][r];
    if (x == 0x7fffffff) *sink = x;                              // keeps the accumulators live; never true
    if (threadIdx.x == 0) {
        clocks[2 * blockIdx.x] = __builtin_amdgcn_s_memtime() - clk0;
        clocks[2 * blockIdx.x + 1] = __builtin_amdgcn_s_memrealtime() - wall0;
    }
}

}  // namespace

extern "C" {

int mmf_bitlinear_mfma_clock_sink(int64_t* sink, int64_t workgroups) {
    if (workgroups < 0 || (sink && workgroups == 0)) return MMF_ERR_ARG;
    g_clock_sink = reinterpret_cast<long long*>(sink);
    g_clock_cap = sink ? workgroups : 0;
    return 0;
}

int mmf_mfma_pipe_probe(int64_t steps, int64_t workgroups, int random_operands, int64_t* clocks, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (steps < 0 || workgroups <= 0 || workgroups > 65535 || !clocks) return MMF_ERR_ARG;
    // the word after the clocks is the sink of the never-taken store
    mfma_pipe_probe_kernel<<<(unsigned)workgroups, 512, 0, stream>>>(steps, random_operands, reinterpret_cast<long long*>(clocks),
                                                                    reinterpret_cast<int*>(clocks + 2 * workgroups));
    MMF_CHECK_LAUNCH();
    return 0;
}

int mmf_bitlinear_mfma_plan(int64_t M, int64_t K, int64_t N, int64_t seg, int swiglu, int64_t* first_rows, int* configs) {
    if (M < 1 || K < 1 || N < 1 || N > 0x7fffffff || seg < 0 || !first_rows || !configs) return MMF_ERR_ARG;
    const int64_t Kp = mmf_round_up(K, 128), first = mfma_first_rows(M, N, Kp, seg, swiglu != 0);
    auto config = [&](int64_t m) {
        const MfmaPick pick = mfma_choice(m, N, Kp, swiglu != 0).pick;
        return !swiglu ? mfma_config(pick, m, N) : pick == MfmaPick::kStream ? 5 : pick == MfmaPick::kSplit ? 18 : 17;
    };
    *first_rows = first;
    configs[0] = config(first);
    configs[1] = first < M ? config(M - first) : -1;
    return 0;
}

int mmf_bitlinear_mfma(const int8_t* codes_tiled, const float* deq, const int* qsum, const void* packed,
                       const float* wdeq, int64_t seg_rows, const void* bias, const void* addend, void* out, int64_t ldo,
                       int64_t M,
                       int64_t K, int64_t N, int out_dtype, int config, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (M < 0 || K <= 0 || N <= 0 || seg_rows <= 0 || seg_rows % 32 != 0 || ldo < N || N > 0x7fffffff) return MMF_ERR_ARG;
    if (M == 0) return 0;
    if (!codes_tiled || !deq || !qsum || !packed || !wdeq || !out) return MMF_ERR_ARG;
    if ((reinterpret_cast<uintptr_t>(codes_tiled) & 15u) || (reinterpret_cast<uintptr_t>(packed) & 15u)) return MMF_ERR_ALIGN;
    MfmaArgs a{};
    a.a = codes_tiled; a.b = static_cast<const uint4*>(packed); a.deq = deq; a.qsum = qsum; a.wdeq = wdeq; a.bias = bias; a.addend = addend;
    a.out = out; a.M = M; a.N = N; a.Kp = mmf_round_up(K, 128); a.seg_rows = seg_rows; a.ldo = ldo;
    switch (out_dtype) {
        case MMF_F32: return dispatch_mfma<float>(a, config, stream);
        case MMF_BF16: return dispatch_mfma<bf16_t>(a, config, stream);
        case MMF_F16: return dispatch_mfma<f16_t>(a, config, stream);
    }
    return MMF_ERR_ARG;
}

int mmf_bitlinear_mfma_multi(const int8_t* codes_tiled, int64_t codes_stride, const float* deq, const int* qsum, const void* packed,
                             const float* wdeq, int64_t seg_rows, void* out, int64_t ldo, int64_t M, int64_t K, int64_t N,
                             int out_dtype, int config, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (M < 0 || K <= 0 || N <= 0 || seg_rows <= 0 || seg_rows % 32 != 0 || ldo < N || N > 0x7fffffff) return MMF_ERR_ARG;
    if (M == 0) return 0;
    if (!codes_tiled || !deq || !qsum || !packed || !wdeq || !out || codes_stride < 0) return MMF_ERR_ARG;
    if ((reinterpret_cast<uintptr_t>(codes_tiled) & 15u) || (codes_stride & 15) || (reinterpret_cast<uintptr_t>(packed) & 15u))
        return MMF_ERR_ALIGN;
    MfmaArgs a{};
    a.a = codes_tiled; a.a_seg = codes_stride; a.m_seg = M; a.b = static_cast<const uint4*>(packed); a.deq = deq; a.qsum = qsum; a.wdeq = wdeq;
    a.out = out; a.M = M; a.N = N; a.Kp = mmf_round_up(K, 128); a.seg_rows = seg_rows; a.ldo = ldo;
    switch (out_dtype) {
        case MMF_F32: return dispatch_mfma<float>(a, config, stream);
        case MMF_BF16: return dispatch_mfma<bf16_t>(a, config, stream);
        case MMF_F16: return dispatch_mfma<f16_t>(a, config, stream);
    }
    return MMF_ERR_ARG;
}

int mmf_bitlinear_mfma_swiglu(const int8_t* codes_tiled, const float* deq, const int* qsum, const void* packed,
                              const float* wdeq, int64_t seg_rows, void* out, int64_t ldo, int64_t M, int64_t K, int64_t N,
                              int out_dtype, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (M < 0 || K <= 0 || N <= 0 || N % 64 != 0 || seg_rows <= 0 || seg_rows % 32 != 0 || ldo < N / 2 || N > 0x7fffffff)
        return MMF_ERR_ARG;
    if (M == 0) return 0;
    if (!codes_tiled || !deq || !qsum || !packed || !wdeq || !out) return MMF_ERR_ARG;
    const int64_t per_vec = out_dtype == MMF_F32 ? 4 : 8;
    if ((reinterpret_cast<uintptr_t>(codes_tiled) & 15u) || (reinterpret_cast<uintptr_t>(packed) & 15u) ||
        (reinterpret_cast<uintptr_t>(out) & 15u) || ldo % per_vec != 0)
        return MMF_ERR_ALIGN;
    MfmaArgs a{};
    a.a = codes_tiled; a.b = static_cast<const uint4*>(packed); a.deq = deq; a.qsum = qsum; a.wdeq = wdeq;
    a.out = out; a.M = M; a.N = N; a.Kp = mmf_round_up(K, 128); a.seg_rows = seg_rows; a.ldo = ldo;
    switch (out_dtype) {
        case MMF_F32: return dispatch_mfma_swiglu<float>(a, stream);
        case MMF_BF16: return dispatch_mfma_swiglu<bf16_t>(a, stream);
        case MMF_F16: return dispatch_mfma_swiglu<f16_t>(a, stream);
    }
    return MMF_ERR_ARG;
}

}  // extern "C"
