// The weight gradients of a training step's BitLinears: dw[N, K] = dout[M, N]^T @ y[M, K], several products over the same
// M rows in one launch (the six of an HGRNBitBlock), fp32 sums, one rounding (mmfreelm/ops/fusedbitnet.py:498).
#include "mmf_common.h"

#include <type_traits>

namespace {

// Both operands have the contraction as their slow axis.  A workgroup owns 256 x 256 outputs, its four waves 128 x 128 each (256
// accumulators a lane, one wave per SIMD): a row of either operand is read from LDS twice, where eight waves of 128 x 64 would keep
// the LDS as busy as the matrix cores.  Rows travel from memory straight into LDS, 32 at a time into one of four buffers, up to
// three buffers ahead of the products; ds_read_b64_tr_b16 turns four rows of 16 columns round on the way into the registers.  A
// row's 64-byte pieces change places by its index's low two bits on the way in, which puts the four rows that a turning read
// touches into different banks.  Reads and transfers are issued one between two products each.
//
// The bound is the matrix cores, at the clock that they run at under this load: four products of 2048 x 2048 over 8192 rows take
// 215 us, the bare products without reads and transfers 159.  Two buffers of 64 rows took 236 us, four reads in front of four
// products and their transfers in pairs behind them 231; a fifth buffer changes nothing.
// The six gradients of a 2048-wide block over 8192 rows: 686 us (1.23 PFLOP/s), as a library product each 892; 2048 rows 207 and
// 270, 1024 rows 118 and 190: by themselves 64 or 352 tiles leave much of the chip idle, 784 together do not.
constexpr int kSide = 256, kSide32 = 128, kRows = 32, kOperand = kRows * kSide * 2, kBuffer = 2 * kOperand, kBuffers = 4, kCUs = 256, kMaxProducts = 8;
constexpr int kRows32 = 16, kOperand32 = kRows32 * kSide32 * 4, kBuffer32 = 2 * kOperand32, kFlight32 = kBuffer32 / 1024 / 4;
constexpr int kFlight = kBuffer / 1024 / 4;                         // transfers of 1 KiB that a wave issues per buffer
constexpr int kMaxSplit = 16, kMaxSlices = 768, kMaxSlices32 = 3072;  // 192 MiB

struct Product {
    const void* p;          // dout, row stride ldp
    const void* q;          // y, row stride ldq
    void* out;              // [N, K]
    int64_t ldp, ldq;
    int N, K, tiles_k, tile0;
};
struct GradArgs {
    Product pr[kMaxProducts];
    int n, full, rest, split;       // `full` tiles over all rows, then `rest` tiles in `split` slices of the rows each
    int64_t M;
    float* part;                    // [split][rest][side * side] in the order of waves, accumulators and lanes
};

typedef short v4s __attribute__((ext_vector_type(4)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
union Frag { v4s h[2]; v8b b; v8h f; };

// 64 lanes x 16 bytes from `base` + off to LDS, lane order.  In assembly so that the compiler, which would answer the builtin with a wait
// for every transfer in front of the next LDS read, does not see an LDS write in flight: the kernel waits itself, by a count of those that may
// still be on their way.  Among themselves transfers complete in the order issued (what keeps no order is a transfer and an ordinary load); the 16-bit kernels
// spill a register in front of the first of them (six or seven more behind the loop, none in it), and one more operation on its way can only make a
// counted wait longer.  The same bits as with waits for all of them, operands cold, warm and beside other traffic.
__device__ __forceinline__ void grad_dma(const void* base, uint32_t off, uint32_t lds) {
    const uint64_t b = (uint64_t)base;
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(b) : "memory");
}
template <int VM>
__device__ __forceinline__ void grad_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(VM) : "memory");
}
__device__ __forceinline__ v4s grad_turn(uint32_t lds) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)(uintptr_t)lds);
}
template <typename T>
__device__ __forceinline__ v16f grad_mul(const Frag& a, const Frag& b, const v16f& c) {
    if constexpr (std::is_same_v<T, bf16_t>) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.b, b.b, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_32x32x16_f16(a.f, b.f, c, 0, 0, 0);
}
template <typename T>
__device__ __forceinline__ uint2 grad_round(float a, float b, float c, float d) {
    union { T t[4]; uint2 u; } r;
    r.t[0] = mmf_from_float<T>(a);
    r.t[1] = mmf_from_float<T>(b);
    r.t[2] = mmf_from_float<T>(c);
    r.t[3] = mmf_from_float<T>(d);
    return r.u;
}

// The product that a tile belongs to and its first output: panels of four tiles along K, so that the 32 tiles that an XCD holds at a time
// share eight strips of dout and four of y.
struct GradTile { int w, n0, k0; };
template <int SIDE>
__device__ __forceinline__ GradTile grad_tile(const GradArgs& a, int tile) {
    GradTile t{0, 0, 0};
    while (t.w + 1 < a.n && tile >= a.pr[t.w + 1].tile0) ++t.w;
    const Product& pr = a.pr[t.w];
    const int i = tile - pr.tile0, tn = (pr.N + SIDE - 1) / SIDE, panel = i / (4 * tn), r = i - panel * 4 * tn;
    const int left = pr.tiles_k - panel * 4, width = left < 4 ? left : 4;
    t.n0 = r / width * SIDE;
    t.k0 = (panel * 4 + r % width) * SIDE;
    return t;
}
// Workgroup b of `total` runs on XCD b % 8: each XCD walks a stretch of its own.
__device__ __forceinline__ int grad_stretch(int b, int total) {
    const int x = b & 7, base = total >> 3, more = total & 7;
    return x * base + (x < more ? x : more) + (b >> 3);
}

template <typename T>
__global__ __launch_bounds__(256, 1) void weight_grad_kernel(GradArgs a) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), wp = wave & 1, wq = wave >> 1;
    int tile, slice = 0, piece = -1;
    if ((int)blockIdx.x < a.full) tile = grad_stretch((int)blockIdx.x, a.full);
    else {                                                           // (`full` is a multiple of 8 where there is a rest)
        piece = grad_stretch((int)blockIdx.x - a.full, a.rest * a.split);
        slice = piece / a.rest;
        tile = a.full + piece % a.rest;
    }
    const GradTile t = grad_tile<kSide>(a, tile);
    const Product& pr = a.pr[t.w];
    const int N = pr.N, K = pr.K, n0 = t.n0, k0 = t.k0;
    const int64_t stages = (a.M + kRows - 1) / kRows;
    const int64_t s0 = stages * slice / a.split, s1 = piece < 0 ? stages : stages * (slice + 1) / a.split;
    const int count = (int)(s1 - s0);
    // rows of the last stage, where it is not a whole one: the others are read again from the last row and zeroed in LDS
    const int valid = s1 == stages && a.M % kRows ? (int)(a.M % kRows) : kRows;

    // A wave's q-th transfer of an operand moves rows 8 * wave + 2 * q and the next one; columns past the edge read the tile's first ones.
    uint32_t offp[4], offq[4];
    auto offsets = [&](int rows) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int r = wave * 8 + 2 * q + (lane >> 5), src = r < rows ? r : rows - 1, piece16 = lane & 31;
            const int col = (((piece16 >> 2) ^ (r & 3)) << 5) + (piece16 & 3) * 8;
            offp[q] = (uint32_t)(src * (int)pr.ldp + (n0 + col < N ? col : 0)) * 2;
            offq[q] = (uint32_t)(src * (int)pr.ldq + (k0 + col < K ? col : 0)) * 2;
        }
    };
    offsets(count == 1 ? valid : kRows);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    const uint16_t* gp = static_cast<const uint16_t*>(pr.p) + n0 + s0 * kRows * pr.ldp;
    const uint16_t* gq = static_cast<const uint16_t*>(pr.q) + k0 + s0 * kRows * pr.ldq;
    const int64_t stepp = kRows * pr.ldp, stepq = kRows * pr.ldq;
    auto dma = [&](int q, int side, uint32_t into) __attribute__((always_inline)) {
        if (side == 0) grad_dma(gp, offp[q], lds0 + into + (wave * 4 + q) * 1024);
        else grad_dma(gq, offq[q], lds0 + into + kOperand + (wave * 4 + q) * 1024);
    };
    auto clear = [&](uint32_t into) __attribute__((always_inline)) {
        for (int i = (int)threadIdx.x; i < 2 * (kRows - valid) * 32; i += 256) {
            const int side = i >= (kRows - valid) * 32, j = i - side * (kRows - valid) * 32;
            *reinterpret_cast<uint4*>(smem + into + side * kOperand + valid * 512 + j * 16) = uint4{0, 0, 0, 0};
        }
        grad_barrier<0>();
    };

    // A turning read: lane i of 16 names four columns of row i / 4 and receives column i of the four rows.  A fragment is 32 columns
    // and 16 rows, eight of them a lane in two reads.
    uint32_t rp[4], rq[4];
    {
        const int i = lane & 15, g = lane >> 4, at = ((g >> 1) * 8 + (i >> 2)) * 512 + (g & 1) * 32 + (i & 3) * 8;
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            rp[f] = lds0 + at + (wp * 4 + (f ^ (i >> 2))) * 64;
            rq[f] = lds0 + at + (wq * 4 + (f ^ (i >> 2))) * 64 + kOperand;
        }
    }
    v16f acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    Frag fp[2][4], fq[2][4];
    uint32_t buf = 0;
    // the x-th read of the g-th four: first the fragments of dout, which the first four products all need
    auto turn = [&](int set, int g, int x, uint32_t b, int half) __attribute__((always_inline)) {
        const int f = (g & 1) * 2 + (x >> 1);
        Frag& d = g < 2 ? fp[set][f] : fq[set][f];
        d.h[x & 1] = grad_turn((g < 2 ? rp[f] : rq[f]) + b + half * (16 * 512) + (x & 1) * (4 * 512));
    };
    // sixteen products of one set of fragments; the other set arrives from rows 16 * half, .. of buffer b, the next transfers leave
    auto products = [&](int set, uint32_t b, int half, bool more) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                acc[g][j] = grad_mul<T>(fq[set][g], fp[set][j], acc[g][j]);
                turn(set ^ 1, g, j, b, half);
                if (more && (j & 1)) dma(g, j >> 1, buf);
                __builtin_amdgcn_sched_barrier(0);
            }
    };

#pragma unroll
    for (int b = 0; b < kBuffers; ++b)
        if (b < count) {
            if (b > 0 && b == count - 1) offsets(valid);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                dma(q, 0, b * kBuffer);
                dma(q, 1, b * kBuffer);
            }
            gp += stepp;
            gq += stepq;
        }
    if (count >= kBuffers) grad_barrier<(kBuffers - 1) * kFlight>();
    else grad_barrier<0>();
    if (count == 1 && valid < kRows) clear(0);
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int x = 0; x < 4; ++x) turn(0, g, x, 0, 0);
    for (int s = 0; s < count; ++s) {
        const uint32_t next = buf == (kBuffers - 1) * kBuffer ? 0 : buf + kBuffer;
        products(0, buf, 1, false);
        // Every wave has read this stage's buffer out; of the three stages in flight the next has to be there.
        if (s + kBuffers - 1 < count) grad_barrier<(kBuffers - 2) * kFlight>();
        else grad_barrier<0>();
        if (s + 2 == count && valid < kRows) clear(next);
        if (s + kBuffers + 1 == count && valid < kRows) offsets(valid);
        products(1, next, 0, s + kBuffers < count);                  // (behind the last stage the reads bring what nothing uses)
        gp += stepp;
        gq += stepq;
        buf = next;
    }
    __syncthreads();

    if (piece >= 0) {
        float* o = a.part + (int64_t)piece * kSide * kSide + wave * 16384 + lane * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const v16f& c = acc[i][j];
                    *reinterpret_cast<v4f*>(o + ((i * 4 + j) * 4 + e) * 256) = v4f{c[4 * e], c[4 * e + 1], c[4 * e + 2], c[4 * e + 3]};
                }
        return;
    }
    // A lane holds one row n and four neighbouring k at a time; 32 rows of the wave go through LDS into 16-byte stores.
    constexpr int kPitch = 272;
    unsigned char* st = smem + wave * 32 * kPitch;
    const int nw = n0 + wp * 128, kw = k0 + wq * 128;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const v16f& c = acc[i][j];
                *reinterpret_cast<uint2*>(st + (lane & 31) * kPitch + i * 64 + e * 16 + (lane >> 5) * 8) =
                    grad_round<T>(c[4 * e], c[4 * e + 1], c[4 * e + 2], c[4 * e + 3]);
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int h = 0; h < 8; ++h) {
            const int row = h * 4 + (lane >> 4), col = (lane & 15) * 8, n = nw + j * 32 + row;
            const uint4 v = *reinterpret_cast<const uint4*>(st + row * kPitch + col * 2);
            if (n < N && kw + col < K) *reinterpret_cast<uint4*>(static_cast<uint16_t*>(pr.out) + (int64_t)n * K + kw + col) = v;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    }
}

// In single precision the matrix cores are the bound by far (157 TFLOP/s dense): 16 rows of 128 x 128 outputs take 2048 cycles and 16 KiB.  A
// row of 128 floats is as long as one of 256 16-bit elements and travels as above; a fragment of two rows is read as it lies.  Two
// workgroups on a CU cover each other's barriers, starts and ends: the six gradients of a 1024-wide block over 666 rows 143 us, one
// workgroup with buffers of 32 rows 163, and 172 where its transfers left together and no read crossed a stage's end; one library
// product each 220.  Tiles of 128 leave a smaller rest than tiles of 256.
__global__ __launch_bounds__(256, 2) void weight_grad32_kernel(GradArgs a) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), wp = wave & 1, wq = wave >> 1;
    int tile, slice = 0, piece = -1;
    if ((int)blockIdx.x < a.full) tile = grad_stretch((int)blockIdx.x, a.full);
    else {
        piece = grad_stretch((int)blockIdx.x - a.full, a.rest * a.split);
        slice = piece / a.rest;
        tile = a.full + piece % a.rest;
    }
    const GradTile t = grad_tile<kSide32>(a, tile);
    const Product& pr = a.pr[t.w];
    const int N = pr.N, K = pr.K, n0 = t.n0, k0 = t.k0;
    const int64_t stages = (a.M + kRows32 - 1) / kRows32;
    const int64_t s0 = stages * slice / a.split, s1 = piece < 0 ? stages : stages * (slice + 1) / a.split;
    const int count = (int)(s1 - s0);
    const int valid = s1 == stages && a.M % kRows32 ? (int)(a.M % kRows32) : kRows32;

    uint32_t offp[2], offq[2];
    auto offsets = [&](int rows) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int r = wave * 4 + 2 * q + (lane >> 5), src = r < rows ? r : rows - 1, col = (lane & 31) * 4;
            offp[q] = (uint32_t)(src * (int)pr.ldp + (n0 + col < N ? col : 0)) * 4;
            offq[q] = (uint32_t)(src * (int)pr.ldq + (k0 + col < K ? col : 0)) * 4;
        }
    };
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    const float* gp = static_cast<const float*>(pr.p) + n0 + s0 * kRows32 * pr.ldp;
    const float* gq = static_cast<const float*>(pr.q) + k0 + s0 * kRows32 * pr.ldq;
    auto dma = [&](int q, int side, uint32_t into) __attribute__((always_inline)) {
        if (side == 0) grad_dma(gp, offp[q], lds0 + into + (wave * 2 + q) * 1024);
        else grad_dma(gq, offq[q], lds0 + into + kOperand32 + (wave * 2 + q) * 1024);
    };
    v16f acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    auto clear = [&](uint32_t into) __attribute__((always_inline)) {
        for (int i = (int)threadIdx.x; i < 2 * (kRows32 - valid) * 32; i += 256) {
            const int side = i >= (kRows32 - valid) * 32, j = i - side * (kRows32 - valid) * 32;
            *reinterpret_cast<uint4*>(smem + into + side * kOperand32 + valid * 512 + j * 16) = uint4{0, 0, 0, 0};
        }
        grad_barrier<0>();
    };
    offsets(count == 1 ? valid : kRows32);
#pragma unroll
    for (int b = 0; b < kBuffers - 1; ++b)
        if (b < count) {
            if (b > 0 && b == count - 1) offsets(valid);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                dma(q, 0, b * kBuffer32);
                dma(q, 1, b * kBuffer32);
            }
            gp += kRows32 * pr.ldp;
            gq += kRows32 * pr.ldq;
        }
    if (count >= kBuffers - 1) grad_barrier<(kBuffers - 2) * kFlight32>();
    else grad_barrier<0>();
    if (count == 1 && valid < kRows32) clear(0);
    const unsigned char* atp = smem + (lane >> 5) * 512 + wp * 256 + (lane & 31) * 4;
    const unsigned char* atq = smem + kOperand32 + (lane >> 5) * 512 + wq * 256 + (lane & 31) * 4;
    float pf[2][2], qf[2][2];
    auto read = [&](int set, uint32_t b, int k) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            pf[set][i] = *reinterpret_cast<const float*>(atp + b + k * 1024 + i * 128);
            qf[set][i] = *reinterpret_cast<const float*>(atq + b + k * 1024 + i * 128);
        }
    };
    read(0, 0, 0);
    uint32_t buf = 0;
    for (int s = 0; s < count; ++s) {
        const uint32_t next = (buf + kBuffer32) & (kBuffers * kBuffer32 - 1), last = (buf - kBuffer32) & (kBuffers * kBuffer32 - 1);
        const bool more = s + kBuffers - 1 < count;
        if (s + kBuffers == count && valid < kRows32) offsets(valid);
#pragma unroll
        for (int k = 0; k < kRows32 / 2; ++k) {                        // the next two rows arrive under four products
            if (k + 1 < kRows32 / 2) read((k + 1) & 1, buf, k + 1);
            else {
                // Every wave has read this stage's buffer out; of the three stages in flight the next has to be there.
                if (more) grad_barrier<(kBuffers - 2) * kFlight32>();
                else grad_barrier<0>();
                if (s + 2 == count && valid < kRows32) clear(next);
                read(0, next, 0);                                    // (behind the last stage: what nothing uses)
            }
            __builtin_amdgcn_sched_barrier(0);                       // the reads leave first: four products cover them, one would not
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(qf[k & 1][i], pf[k & 1][j], acc[i][j], 0, 0, 0);
            if (more && k < 4) dma(k >> 1, k & 1, last);
            __builtin_amdgcn_sched_barrier(0);
        }
        gp += kRows32 * pr.ldp;
        gq += kRows32 * pr.ldq;
        buf = next;
    }
    float* o = piece < 0 ? nullptr : a.part + (int64_t)piece * kSide32 * kSide32 + wave * 4096 + lane * 4;
    float* out = static_cast<float*>(pr.out);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const v4f v = v4f{acc[i][j][4 * e], acc[i][j][4 * e + 1], acc[i][j][4 * e + 2], acc[i][j][4 * e + 3]};
                const int n = n0 + wp * 64 + j * 32 + (lane & 31), k = k0 + wq * 64 + i * 32 + e * 8 + (lane >> 5) * 4;
                if (o) *reinterpret_cast<v4f*>(o + ((i * 2 + j) * 4 + e) * 256) = v;
                else if (n < N && k < K) *reinterpret_cast<v4f*>(out + (int64_t)n * K + k) = v;
            }
}

// The slices of the split tiles added up in their order, 1024 outputs a workgroup.
template <typename T, int SIDE>
__global__ __launch_bounds__(256) void weight_grad_sum_kernel(GradArgs a) {
    constexpr int kSubs = SIDE * SIDE / 1024, F = SIDE / 64;          // a wave's tile: F x F fragments, one a workgroup
    const int r = (int)blockIdx.x / kSubs, sub = (int)blockIdx.x % kSubs;
    const GradTile t = grad_tile<SIDE>(a, a.full + r);
    const Product& pr = a.pr[t.w];
    const float* o = a.part + (int64_t)r * SIDE * SIDE + sub * 1024 + (int)threadIdx.x * 4;
    v4f v = *reinterpret_cast<const v4f*>(o);
    for (int s = 1; s < a.split; ++s) {
        const v4f w = *reinterpret_cast<const v4f*>(o + (int64_t)s * a.rest * SIDE * SIDE);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = __fadd_rn(v[i], w[i]);
    }
    const int wave = sub / (F * F), i = sub / F % F, j = sub % F, e = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
    const int n = t.n0 + (wave & 1) * (SIDE / 2) + j * 32 + (lane & 31), k = t.k0 + (wave >> 1) * (SIDE / 2) + i * 32 + e * 8 + (lane >> 5) * 4;
    if (n >= pr.N || k >= pr.K) return;
    T* out = static_cast<T*>(pr.out) + (int64_t)n * pr.K + k;
    if constexpr (std::is_same_v<T, float>) *reinterpret_cast<v4f*>(out) = v;
    else *reinterpret_cast<uint2*>(out) = grad_round<T>(v[0], v[1], v[2], v[3]);
}

// The tiles behind the last whole round of the chip, cut into slices of the rows where that is estimated to end sooner: microseconds from a stage's
// 0.85, a workgroup's start and end 5, the second launch 4 and 0.1 per slice written and read.  8192 rows, as they are / cut: one product of
// 2048 x 2048 (64 tiles, 4 slices) 167 / 80 us, 11264 x 2048 (96 of 352 tiles, 2 slices) 360 / 313, 2048 x 5632 (176 tiles) 179 whole, 228 in 4.
// Single precision: 0.95 a stage, 0.025 a slice.  The slices of a launch are held to 192 MiB of workspace: for blocks of widths 256 to 4096 the estimate is that
// without a bound up to 16384 rows, and 0 to 7 % above it at 32768, 0 to 15 % at 65536 (1024 wide).
struct GradPlan { int full, rest, split; };
GradPlan grad_plan(int64_t tiles, int64_t M, bool f32) {
    const int64_t stages = mmf_ceil_div(M, f32 ? kRows32 : kRows), rest = tiles % kCUs;
    const double stage = f32 ? 0.95 : 0.85, slice = f32 ? 0.025 : 0.1;
    int best = 1;
    double least = 0.0;
    for (int s = 1; s <= kMaxSplit && (s == 1 || rest * s <= (f32 ? kMaxSlices32 : kMaxSlices)) && stages / s >= (f32 ? 2 : 4); ++s) {
        const double us = (double)mmf_ceil_div(rest * s, kCUs) * ((double)mmf_ceil_div(stages, s) * stage + 5.0) + (s > 1 ? 4.0 + slice * (double)(rest * s) : 0.0);
        if (s == 1 || us < least) {
            best = s;
            least = us;
        }
    }
    if (rest == 0 || best == 1) return GradPlan{(int)tiles, 0, 1};
    return GradPlan{(int)(tiles - rest), (int)rest, best};
}
int64_t grad_tiles(int n, const int64_t* N, const int64_t* K, int side) {
    int64_t t = 0;
    for (int i = 0; i < n; ++i) t += mmf_ceil_div(N[i], side) * mmf_ceil_div(K[i], side);
    return t;
}

template <typename T>
int launch_grad(const GradArgs& a, hipStream_t s) {
    constexpr bool f32 = std::is_same_v<T, float>;
    constexpr int side = f32 ? kSide32 : kSide;
    void (*kern)(GradArgs);
    if constexpr (f32) kern = weight_grad32_kernel;
    else kern = weight_grad_kernel<T>;
    constexpr int lds = kBuffers * (f32 ? kBuffer32 : kBuffer);
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return (int)e;
    kern<<<(unsigned)(a.full + a.rest * a.split), 256, lds, s>>>(a);
    MMF_CHECK_LAUNCH();
    if (a.rest) {
        weight_grad_sum_kernel<T, side><<<(unsigned)(a.rest * (side * side / 1024)), 256, 0, s>>>(a);
        MMF_CHECK_LAUNCH();
    }
    return 0;
}

}  // namespace

extern "C" {

int64_t mmf_weight_grad_workspace_bytes(int products, const int64_t* N, const int64_t* K, int64_t M, int dtype) {
    if (products < 1 || products > kMaxProducts || !N || !K || M < 1) return 0;
    for (int i = 0; i < products; ++i)
        if (N[i] < 1 || K[i] < 1 || N[i] > 0x7fffff00 || K[i] > 0x7fffff00) return 0;
    const bool f32 = dtype == MMF_F32;
    const int side = f32 ? kSide32 : kSide;
    const GradPlan plan = grad_plan(grad_tiles(products, N, K, side), M, f32);
    return (int64_t)plan.rest * (plan.split > 1 ? plan.split : 0) * side * side * 4;
}

int mmf_weight_grad(int products, const void* const* dout, const int64_t* lddout, const void* const* y, const int64_t* ldy, void* const* dw,
                    const int64_t* N, const int64_t* K, int64_t M, int dtype, void* workspace, void* stream_) {
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    if (products < 1 || products > kMaxProducts || !dout || !lddout || !y || !ldy || !dw || !N || !K || M < 1) return MMF_ERR_ARG;
    if (dtype != MMF_BF16 && dtype != MMF_F16 && dtype != MMF_F32) return MMF_ERR_ARG;
    if (M > 0x7fffffff) return MMF_ERR_WIDE;
    const bool f32 = dtype == MMF_F32;
    const int side = f32 ? kSide32 : kSide, whole = f32 ? 4 : 8;                               // elements of 16 bytes
    GradArgs a{};
    int64_t tiles = 0;
    auto off = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) != 0; };
    for (int i = 0; i < products; ++i) {
        if (N[i] < 1 || K[i] < 1 || lddout[i] < N[i] || ldy[i] < K[i] || !dout[i] || !y[i] || !dw[i]) return MMF_ERR_ARG;
        if (N[i] % whole || K[i] % whole || lddout[i] % whole || ldy[i] % whole || off(dout[i]) || off(y[i]) || off(dw[i])) return MMF_ERR_ALIGN;
        if (lddout[i] > 1 << 24 || ldy[i] > 1 << 24) return MMF_ERR_WIDE;                      // 32 rows in 32-bit byte offsets
        const int64_t tk = mmf_ceil_div(K[i], side);
        a.pr[i] = Product{dout[i], y[i], dw[i], lddout[i], ldy[i], (int)N[i], (int)K[i], (int)tk, (int)tiles};
        tiles += tk * mmf_ceil_div(N[i], side);
        if (tiles > 0x3fffffff) return MMF_ERR_WIDE;
    }
    const GradPlan plan = grad_plan(tiles, M, f32);
    if (plan.rest && !workspace) return MMF_ERR_ARG;
    if (plan.rest && off(workspace)) return MMF_ERR_ALIGN;
    a.n = products; a.full = plan.full; a.rest = plan.rest; a.split = plan.split; a.M = M; a.part = static_cast<float*>(workspace);
    switch (dtype) {
        case MMF_F32: return launch_grad<float>(a, stream);
        case MMF_BF16: return launch_grad<bf16_t>(a, stream);
        case MMF_F16: return launch_grad<f16_t>(a, stream);
    }
    return MMF_ERR_ARG;
}

}  // extern "C"
