// bf16 / f16 / s8 / f32 GEMM on gfx950 MFMA for grids too small for the large tiles: one BM x BN output tile per workgroup,
// its K dealt to the workgroup's waves. (The kernel; gemm_wavek.hip and gemm_wavek8.hip hold its instances.)
//
// Computes Y = epilogue(A[M][K] x B[N][K]^T) as the 4-wave kernel does (gemm_mfma.hip), for products whose M is a few
// tens to a few hundred rows: their time is the weight's way from HBM, and a chain of k-tiles with a barrier each
// (copies issued, waited for, read, multiplied, one after the other by all waves of a tile) holds it up: bf16 64 x 4096
// x 4096, weights from HBM, 43.3 us a call on 128 x 128 tiles and 30.8 with K in four slices over workgroups, whose
// sums meet in a second launch, against 14.5 here; 64 x 11008 x 4096 45.2 against 28.2. Nothing in the K loop is shared:
//  - Wave w of W takes k-tiles w, w + W, w + 2 W, ... (128 bytes of each weight row) and accumulates the whole tile over
//    them. It owns a stage of LDS for one k-tile of A and B; it waits for its own copies (vmcnt), reads all fragments
//    into registers, issues the copies of its next k-tile into the same stage, and runs the MFMAs while they fly. No
//    barrier orders the waves, so they drift apart and hide one another's waits; a CU holds 64 to 160 KB of stages.
//  - At the end the waves' sums meet in LDS, in wave order (the same bits every run), and every thread applies the
//    epilogue to runs of 8 columns.
//  - K needs no padding to whole k-tiles: a copy of the last k-tile reads zeros for the 16-byte chunks past K. Rows that
//    are no multiple of 16 bytes apart, or end inside a chunk, go through registers instead of the LDS DMA (REG): loads
//    at any element alignment, written to the stage once the previous k-tile's fragments are out of it.
// What bounds it, by counters: the bytes of weight in flight over the whole chip against HBM's latency where calls are
// small (64 x 4096 x 4096: waves wait 0.72 of their cycles), and from 64 x 11008 x 4096 up as much the copies through a
// CU's address unit, (BM + BN) x 128 bytes per k-tile at 21 to 27 of its cycles per KB (busy 0.4 to 0.7 of the time; the
// MFMAs are busy 0.3 at most). So a tile is small where the grid is small, and the narrow ones (BN = 16, on 16 x 16
// MFMAs) give N = 4096 a workgroup per CU.
// A 16-bit weight stored [K][N] is read in place by the tiles of BN >= 64 (KM): a k-tile of B is then 64 k-rows of whole
// 128-byte lines, and gfx950's transposing LDS read hands each lane 4 consecutive k of one n.
// An 8-bit weight of an f16 product stays 8-bit up to the registers: a k-tile is then 128 k (two 128-byte pieces of an A
// row), a lane reads 16 weights as one LDS read and turns them into f16 exactly (1024 + b as f16 bits, minus the
// offset) for two MFMA steps, whose A chunks are those k. Packing the weight to f16 first moved 2.5 times its bytes
// twice: 4 x 4096 x 4096 21.5 us a call.
// An integer product runs on v_mfma_i32_*_i8; a u8 A is shifted by -128 in registers (one XOR), and the term the shift
// removes, 128 times the weight's row sums, comes from one more MFMA per weight fragment against ones, whose
// accumulators lie as the product's do.
#ifndef KUDNN_GEMM_WAVEK_H
#define KUDNN_GEMM_WAVEK_H

#include <algorithm>
#include <cstdint>
#include <type_traits>
#include <utility>

#include "device_common.h"
#include "kernels.h"

namespace {

using namespace kudnn_dev;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kChunks = 8;  // 16-byte chunks per 128-byte k-tile row

// What a copy reads for the chunks of the last k-tile that lie past K.
__device__ __align__(16) const uint32_t kZeroChunk[4] = {0u, 0u, 0u, 0u};

// 8 8-bit integers as f16, exactly: b (u8; s8 + 128) under the exponent of 1024 is the f16 number 1024 + b.
template <int BT>
__device__ __forceinline__ uint4 cvt8_f16(uint32_t w0, uint32_t w1)
{
    constexpr bool S8 = BT == KUDNN_DT_S8;
    w0 = S8 ? w0 ^ 0x80808080u : w0;
    w1 = S8 ? w1 ^ 0x80808080u : w1;
    const f16x2_t off = {static_cast<_Float16>(S8 ? -1152.0f : -1024.0f), static_cast<_Float16>(S8 ? -1152.0f : -1024.0f)};
    auto pair = [&](uint32_t w, uint32_t sel) __attribute__((always_inline)) {
        const f16x2_t h = __builtin_bit_cast(f16x2_t, __builtin_amdgcn_perm(w, 0x64646464u, sel)) + off;
        return __builtin_bit_cast(uint32_t, h);
    };
    return make_uint4(pair(w0, 0x00050004u), pair(w0, 0x00070006u), pair(w1, 0x00050004u), pair(w1, 0x00070006u));
}

__device__ __forceinline__ uint32_t lds_byte(const uint4 *p)
{
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void *)p));
}

// One LDS DMA copy: lane l's 16 bytes at src land in LDS at lds + 16 l. Inline asm, so that the compiler neither tracks
// nor waits for it; the s_nop is the wait state between the write of M0 and the copy that reads it. `lds` is scalar
// arithmetic on the wave index.
__device__ __forceinline__ void dma16(const void *src, uint32_t lds)
{
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds) : "memory", "m0");
}

// 16 bytes at an address that is a multiple of the element size only.
template <typename E>
__device__ __forceinline__ uint4 load16(const E *p)
{
    struct __attribute__((packed, aligned(alignof(E)))) Any16 {
        uint32_t w[4];
    };
    const Any16 v = *reinterpret_cast<const Any16 *>(p);
    return make_uint4(v.w[0], v.w[1], v.w[2], v.w[3]);
}

// The chunk at p of which only the first `valid` elements belong to the row (any count, also none): the rest are zeros.
// It reads the row's last 16 bytes and shifts them down, so no byte past the row's end is touched.
template <typename E>
__device__ __forceinline__ uint4 load16_tail(const E *p, int valid)
{
    constexpr int N = 16 / static_cast<int>(sizeof(E));
    if (valid >= N) {
        return load16(p);
    }
    const uint4 v = load16(p + valid - N);
    uint64_t lo = v.x | static_cast<uint64_t>(v.y) << 32, hi = v.z | static_cast<uint64_t>(v.w) << 32;
    const int sh = (N - (valid > 0 ? valid : 0)) * static_cast<int>(sizeof(E)) * 8;  // 8 .. 128 bits
    if (sh >= 64) {
        lo = sh < 128 ? hi >> (sh & 63) : 0u;
        hi = 0u;
    } else {
        lo = lo >> sh | hi << (64 - sh);
        hi >>= sh;
    }
    return make_uint4(static_cast<uint32_t>(lo), static_cast<uint32_t>(lo >> 32), static_cast<uint32_t>(hi),
                      static_cast<uint32_t>(hi >> 32));
}

template <int... I, typename F>
__device__ __forceinline__ void sfor_impl(std::integer_sequence<int, I...>, F &&f)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void sfor(F &&f)
{
    sfor_impl(std::make_integer_sequence<int, N>{}, f);
}

// CT: compute type, KUDNN_DT_BF16 / F16 / S8 / F32. BT: type of the stored weight: CT's, S8 or U8 under F16, and U8 under S8
// stands for a u8 A beside an s8 weight (the shift's term is added). KM: B is stored [K][N] (16-bit; row pitch ldb along
// k, whole 16-byte chunks of columns). REG: rows of any alignment, K of at least one chunk.
template <int CT, int BT, int BM, int BN, int W, bool KM, bool REG>
__global__ __launch_bounds__(W * 64, 1) void gemm_wavek_kernel(GemmOperands op, EpiParams ep, int tilesM)
{
    constexpr bool INT = CT == KUDNN_DT_S8;
    constexpr bool B8 = CT == KUDNN_DT_F16 && BT != CT;  // an 8-bit weight of an f16 product
    constexpr bool UA = INT && BT == KUDNN_DT_U8;
    constexpr bool F32 = CT == KUDNN_DT_F32;
    using TA = std::conditional_t<F32, uint32_t, std::conditional_t<INT, uint8_t, uint16_t>>;
    using TB = std::conditional_t<F32, uint32_t, std::conditional_t<INT || B8, uint8_t, uint16_t>>;
    constexpr int EA = 16 / static_cast<int>(sizeof(TA)), EB = 16 / static_cast<int>(sizeof(TB));  // elements per chunk
    constexpr int AH = B8 ? 2 : 1;                // 128-byte pieces of an A row in a k-tile
    constexpr int kBK = kChunks * EB;             // k of a k-tile
    constexpr int TS = BM == 16 || BN == 16 ? 16 : 32;  // side of the MFMA's output block
    constexpr int G = 64 / TS;                    // lane groups, each with a chunk (16 bytes of k) of a step
    constexpr int FM = BM / TS, FN = BN / TS;     // blocks of the tile
    constexpr int KS = kChunks * AH / G;          // MFMA steps of a k-tile
    constexpr int NR = TS == 32 ? 16 : 4;         // accumulators a lane holds of a block
    constexpr int GA = BM / 8, GB = BN / 8;       // 1 KB copies of a k-tile (A: per piece)
    constexpr int kStage = (BM * AH + BN) * kChunks;  // uint4 per wave
    static_assert(!KM || (BN >= 64 && !INT && !B8 && !F32 && !REG), "K-major B: 16-bit elements, whole lines of columns");
    // K-major B: a copy covers kRpc k-rows of a segment of kSegN columns (128 bytes of a k-row). kSeg: segments of the tile;
    // narrower tiles have no K-major form, and only a divisor's value
    constexpr int kSegN = 64, kSeg = BN < 64 ? 1 : BN / kSegN, kRpc = 8, kRowC = 8;
    // blocks of columns whose sums are exchanged at a time: the most that fit a wave's stage
    constexpr int JP = BM * BN * 4 <= kStage * 16 ? FN : (BM * BN * 2 <= kStage * 16 ? FN / 2 : 1);
    constexpr int PC = JP * TS;                   // ... in columns
    static_assert(BM * PC * 4 <= kStage * 16 && FN % JP == 0, "a wave's sums fit its stage");
    using Acc = std::conditional_t<INT, std::conditional_t<TS == 32, i32x16_t, i32x4_t>,
                                   std::conditional_t<TS == 32, f32x16_t, f32x4_t>>;
    __shared__ uint4 lds[W * kStage];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the tiles of one column panel follow one another on one XCD, whose L2 then reads the panel's weight once
    const int lid = xcd_remap(blockIdx.x, gridDim.x);
    const int tm = lid % tilesM, tn = lid / tilesM;
    const int64_t m0 = static_cast<int64_t>(tm) * BM, n0 = static_cast<int64_t>(tn) * BN;
    const int64_t M = op.M, N = op.N, K = op.K;
    const int64_t batch = blockIdx.y;
    const int64_t i2 = batch % ep.bdim[2];
    const int64_t i1 = (batch / ep.bdim[2]) % ep.bdim[1];
    const int64_t i0 = batch / (ep.bdim[2] * ep.bdim[1]);
    const TA *A = static_cast<const TA *>(op.a) + i0 * op.a_bs[0] + i1 * op.a_bs[1] + i2 * op.a_bs[2];
    const TB *B = static_cast<const TB *>(op.b) + i0 * op.b_bs[0] + i1 * op.b_bs[1] + i2 * op.b_bs[2];

    uint4 *stage = lds + wave * kStage;
    const uint4 *sA = stage, *sB = stage + BM * AH * kChunks;
    const uint32_t ldsA = __builtin_amdgcn_readfirstlane(lds_byte(stage));
    const uint32_t ldsB = ldsA + BM * AH * kChunks * 16;
    // copy addressing: 8 rows x 128 bytes per copy; lane l fills slot l % 8 of row l / 8 with the chunk that the XOR
    // swizzle (chunk ^ (row % 8)) keeps there, so that the fragment reads of 8 rows at one chunk hit every bank once
    const int lrow8 = lane >> 3, lchunk = (lane & 7) ^ lrow8;
    const TA *pa[GA];
    const TB *pb[GB];
#pragma unroll
    for (int j = 0; j < GA; ++j) {
        int64_t r = m0 + j * 8 + lrow8;
        r = r < M ? r : M - 1;  // rows past M are read and never stored
        pa[j] = A + r * op.lda + lchunk * EA;
    }
#pragma unroll
    for (int j = 0; j < GB; ++j) {
        if constexpr (KM) {
            // copy j: k-rows kRpc (j / kSeg) .. of segment j % kSeg. Row k keeps chunk c in slot c ^ 4 ((k / 2) % 2): the
            // four k-rows that a transposing read takes at a time then lie in four different quarters of the banks.
            // Chunks past N are clamped to the last one (read, never stored). (Half lines of 32 columns were no faster:
            // 32 x 5120 x 12928 77 us either way.)
            const int r = lane / kRowC, c = (lane % kRowC) ^ (4 * ((r >> 1) & 1));
            int64_t n = n0 + j % kSeg * kSegN + c * 8;
            n = n + 8 <= N ? n : N - 8;
            pb[j] = B + (j / kSeg * kRpc + r) * op.ldb + n;
        } else {
            int64_t r = n0 + j * 8 + lrow8;
            r = r < N ? r : N - 1;
            pb[j] = B + r * op.ldb + lchunk * EB;
        }
    }
    const int KT = static_cast<int>((K + kBK - 1) / kBK);
    const int kLast = static_cast<int>(K - static_cast<int64_t>(KT - 1) * kBK);  // k of the last k-tile
    auto issue = [&](int kt) __attribute__((always_inline)) {
        const int64_t k0 = static_cast<int64_t>(kt) * kBK;
        const int64_t kb = KM ? k0 * op.ldb : k0;
        if (kt == KT - 1 && kLast < kBK) {
            // a chunk of a row that starts past K, or a k-row past K, is zeros (a packed row holds zeros up to the chunk;
            // a shifted u8 row's zeros become -128 and meet the weight's zeros)
            const TA *padA = reinterpret_cast<const TA *>(kZeroChunk);
            const TB *padB = reinterpret_cast<const TB *>(kZeroChunk);
#pragma unroll
            for (int h = 0; h < AH; ++h) {
                const bool in = (h * kChunks + lchunk) * EA < kLast;
#pragma unroll
                for (int j = 0; j < GA; ++j) dma16(in ? pa[j] + k0 + h * 64 : padA, ldsA + (h * GA + j) * 1024);
            }
#pragma unroll
            for (int j = 0; j < GB; ++j) {
                const bool in = KM ? j / kSeg * kRpc + lane / kRowC < kLast : lchunk * EB < kLast;
                dma16(in ? pb[j] + kb : padB, ldsB + j * 1024);
            }
        } else {
#pragma unroll
            for (int h = 0; h < AH; ++h) {
#pragma unroll
                for (int j = 0; j < GA; ++j) dma16(pa[j] + k0 + h * 64, ldsA + (h * GA + j) * 1024);
            }
#pragma unroll
            for (int j = 0; j < GB; ++j) dma16(pb[j] + kb, ldsB + j * 1024);
        }
    };

    // REG: the next k-tile's chunks, in registers from their loads until the stage is free
    uint4 ra[REG ? AH * GA : 1], rb[REG ? GB : 1];
    auto fetch = [&](int kt) __attribute__((always_inline)) {
        const int64_t k0 = static_cast<int64_t>(kt) * kBK;
        if (kt == KT - 1) {
#pragma unroll
            for (int h = 0; h < AH; ++h) {
                const int valid = kLast - (h * kChunks + lchunk) * EA;
#pragma unroll
                for (int j = 0; j < GA; ++j) ra[h * GA + j] = load16_tail(pa[j] + k0 + h * 64, valid);
            }
#pragma unroll
            for (int j = 0; j < GB; ++j) rb[j] = load16_tail(pb[j] + k0, kLast - lchunk * EB);
        } else {
#pragma unroll
            for (int h = 0; h < AH; ++h) {
#pragma unroll
                for (int j = 0; j < GA; ++j) ra[h * GA + j] = load16(pa[j] + k0 + h * 64);
            }
#pragma unroll
            for (int j = 0; j < GB; ++j) rb[j] = load16(pb[j] + k0);
        }
    };
    auto next = [&](int kt) __attribute__((always_inline)) {
        if constexpr (REG) {
            fetch(kt);
        } else {
            issue(kt);
        }
    };

    Acc acc[FN][FM], rsum[UA ? FN : 1];
#pragma unroll
    for (int j = 0; j < FN; ++j) {
#pragma unroll
        for (int i = 0; i < FM; ++i) acc[j][i] = Acc{};
        if constexpr (UA) {
            rsum[j] = Acc{};
        }
    }
    const int lrow = lane & (TS - 1), lgrp = lane / TS;  // a lane's row of a block, and which chunk of a step it holds
    const uint32_t xorA = UA && op.a_u8 ? 0x80808080u : 0u;
    if (wave < KT) {
        next(wave);
    }
    for (int kt = wave; kt < KT; kt += W) {
        if constexpr (REG) {
#pragma unroll
            for (int j = 0; j < AH * GA; ++j) stage[j * 64 + lane] = ra[j];
#pragma unroll
            for (int j = 0; j < GB; ++j) stage[(AH * GA + j) * 64 + lane] = rb[j];
            // a wave's LDS accesses run in order; the fence keeps the compiler from moving the reads up
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's copies have landed
        }
        uint4 va[KS][FM], vb[KS / AH][FN];
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            // the chunk of A a lane multiplies at step s; with an 8-bit weight, half s % 2 of the 16 k of its B chunk
            const int ca = AH == 2 ? 2 * (G * (s / 2) + lgrp) + s % 2 : G * s + lgrp;
            const int h = ca / kChunks, c = (ca % kChunks) ^ (lrow & 7);
#pragma unroll
            for (int i = 0; i < FM; ++i) va[s][i] = sA[(h * BM + i * TS + lrow) * kChunks + c];
        }
#pragma unroll
        for (int s = 0; s < KS / AH; ++s) {
            const int c = (G * s + lgrp) ^ (lrow & 7);
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                if constexpr (KM) {
                    // address lane 4 q + c of a 16-lane group: 4 columns n .. n + 3 of k-row k + q; lane i of the group
                    // receives column i at k .. k + 3. Two reads give the 8 k of step s and lane half lgrp.
                    typedef short v4i16_t __attribute__((ext_vector_type(4)));
                    typedef __attribute__((address_space(3))) v4i16_t lds_v4i16;
                    typedef __attribute__((address_space(3))) const char lds_char;
                    const int q = (lane & 15) >> 2;
                    const int col = (j * 32) % kSegN + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);  // within the segment
                    const int chunk = (col / 8) ^ (4 * ((q >> 1) & 1));
                    lds_char *p = (lds_char *)(reinterpret_cast<const char *>(sB)) + j * 32 / kSegN * 1024 + chunk * 16 +
                                  (lane & 1) * 8;
                    uint2 hf[2];
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const int k = 16 * s + 8 * lgrp + 4 * t + q;  // its copy's group of rows, then the row within
                        const int off = k / kRpc * kSeg * 1024 + k % kRpc * (kSegN * 2);
                        hf[t] = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16 *)(p + off)));
                    }
                    vb[s][j] = make_uint4(hf[0].x, hf[0].y, hf[1].x, hf[1].y);
                } else {
                    vb[s][j] = sB[(j * TS + lrow) * kChunks + c];
                }
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the fragments are in registers: the stage is free
        __builtin_amdgcn_sched_barrier(0);
        if (kt + W < KT) {
            next(kt + W);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            if constexpr (UA) {
#pragma unroll
                for (int i = 0; i < FM; ++i) {
                    va[s][i] = make_uint4(va[s][i].x ^ xorA, va[s][i].y ^ xorA, va[s][i].z ^ xorA, va[s][i].w ^ xorA);
                }
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                uint4 b;
                if constexpr (B8) {
                    const uint4 w = vb[s / 2][j];
                    b = s % 2 == 0 ? cvt8_f16<BT>(w.x, w.y) : cvt8_f16<BT>(w.z, w.w);
                } else {
                    b = vb[s][j];
                }
                // the weight is the first operand: a lane then holds one output row and runs of 4 columns
                if constexpr (F32) {
                    // MFMA q multiplies element q of the lane groups' chunks
                    const f32x4_t b4 = __builtin_bit_cast(f32x4_t, b);
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
#pragma unroll
                        for (int i = 0; i < FM; ++i) {
                            const f32x4_t a4 = __builtin_bit_cast(f32x4_t, va[s][i]);
                            if constexpr (TS == 32) {
                                acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x2f32(b4[q], a4[q], acc[j][i], 0, 0, 0);
                            } else {
                                acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(b4[q], a4[q], acc[j][i], 0, 0, 0);
                            }
                        }
                    }
                } else if constexpr (INT) {
                    const i32x4_t bi = __builtin_bit_cast(i32x4_t, b);
                    const int one = 0x01010101;
                    const i32x4_t ones = {one, one, one, one};
                    auto mfma = [&](i32x4_t a, Acc c) __attribute__((always_inline)) {
                        if constexpr (TS == 32) {
                            return __builtin_amdgcn_mfma_i32_32x32x32_i8(bi, a, c, 0, 0, 0);
                        } else {
                            return __builtin_amdgcn_mfma_i32_16x16x64_i8(bi, a, c, 0, 0, 0);
                        }
                    };
#pragma unroll
                    for (int i = 0; i < FM; ++i) acc[j][i] = mfma(__builtin_bit_cast(i32x4_t, va[s][i]), acc[j][i]);
                    if constexpr (UA) {
                        rsum[j] = mfma(ones, rsum[j]);
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < FM; ++i) {
                        if constexpr (CT == KUDNN_DT_BF16) {
                            const bf16x8_t bb = __builtin_bit_cast(bf16x8_t, b), a = __builtin_bit_cast(bf16x8_t, va[s][i]);
                            if constexpr (TS == 32) {
                                acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bb, a, acc[j][i], 0, 0, 0);
                            } else {
                                acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bb, a, acc[j][i], 0, 0, 0);
                            }
                        } else {
                            const f16x8_t bb = __builtin_bit_cast(f16x8_t, b), a = __builtin_bit_cast(f16x8_t, va[s][i]);
                            if constexpr (TS == 32) {
                                acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bb, a, acc[j][i], 0, 0, 0);
                            } else {
                                acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bb, a, acc[j][i], 0, 0, 0);
                            }
                        }
                    }
                }
            }
        }
    }

    // the waves' sums meet in LDS, PC columns at a time: row m's 16-byte piece p lies at piece p ^ (m % PR)
    constexpr int PR = PC / 4;
    uint4 *mine = stage;
    const EpiBatch ob = epi_batch_offsets(ep, batch);
    sfor<FN / JP>([&](auto pc) __attribute__((always_inline)) {
        constexpr int J0 = decltype(pc)::value * JP;
        if constexpr (J0 > 0) {
            __syncthreads();  // every thread has read the previous columns
        }
#pragma unroll
        for (int j = 0; j < JP; ++j) {
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                Acc a = acc[J0 + j][i];
                if constexpr (UA) {
#pragma unroll
                    for (int r = 0; r < NR; ++r) a[r] = static_cast<int>(static_cast<uint32_t>(a[r]) + 128u * static_cast<uint32_t>(rsum[J0 + j][r]));
                }
#pragma unroll
                for (int g = 0; g < NR / 4; ++g) {
                    const int m = i * TS + lrow, p = j * (TS / 4) + g * 2 + lgrp;
                    // elements are copied out first: __builtin_bit_cast of an element of an ext_vector_type reads element 0
                    const auto e0 = a[4 * g], e1 = a[4 * g + 1], e2 = a[4 * g + 2], e3 = a[4 * g + 3];
                    mine[m * PR + (p ^ (m & (PR - 1)))] =
                        make_uint4(__builtin_bit_cast(uint32_t, e0), __builtin_bit_cast(uint32_t, e1),
                                   __builtin_bit_cast(uint32_t, e2), __builtin_bit_cast(uint32_t, e3));
                }
            }
        }
        __syncthreads();
        for (int r = tid; r < BM * PC / 8; r += W * 64) {
            const int row = r / (PC / 8), p0 = (r % (PC / 8)) * 2;
            const int64_t m = m0 + row, n = n0 + J0 * TS + p0 * 4;
            if (m >= M || n >= N) {
                continue;
            }
            float v[8];
            uint32_t u[8];
#pragma unroll
            for (int w = 0; w < W; ++w) {
                const uint4 *s = lds + w * kStage + row * PR;
                const uint4 lo = s[p0 ^ (row & (PR - 1))], hi = s[(p0 + 1) ^ (row & (PR - 1))];
                const uint32_t x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    if constexpr (INT) {
                        u[e] = w == 0 ? x[e] : u[e] + x[e];
                    } else {
                        v[e] = w == 0 ? u2f(x[e]) : v[e] + u2f(x[e]);
                    }
                }
            }
            if constexpr (INT) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = u2f(u[e]);
                if (ep.fast8 && n + 7 < N) {
                    epi_i32_8(ep, ob, m, n, v);
                } else {
#pragma unroll
                    for (int q = 0; q < 8; ++q) {
                        if (n + q < N) {
                            epi_i32_1(ep, ob, m, n + q, v[q]);
                        }
                    }
                }
            } else if (ep.vec8 && n + 7 < N) {
                epi_apply8(ep, ob, m, n, v);
            } else {
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    if (n + q < N) {
                        epi_apply(ep, ob, m, n + q, v[q]);
                    }
                }
            }
        }
    });
}

template <int CT, int BT, int BM, int BN, int W>
int launch_tile(const GemmOperands &op, const EpiParams &ep, int64_t batches, bool reg, hipStream_t stream)
{
    const int64_t tilesM = (op.M + BM - 1) / BM, tiles = tilesM * ((op.N + BN - 1) / BN);
    if (tiles > INT32_MAX) {
        return -1;
    }
    constexpr bool k16 = CT == BT && (CT == KUDNN_DT_BF16 || CT == KUDNN_DT_F16);
    decltype(&gemm_wavek_kernel<CT, BT, BM, BN, W, false, false>) kernel = nullptr;
    if (op.b_kmajor) {
        if constexpr (k16 && BN >= 64) {
            kernel = gemm_wavek_kernel<CT, BT, BM, BN, W, true, false>;
        }
    } else if (reg) {
        if constexpr (kudnn_wavek_reg_tile(BM, BN, W)) {
            kernel = gemm_wavek_kernel<CT, BT, BM, BN, W, false, true>;
        }
    } else if constexpr (!(k16 && BM == 16)) {  // (aligned 16-bit decode has kernels of its own, skinny_bf16.hip)
        kernel = gemm_wavek_kernel<CT, BT, BM, BN, W, false, false>;
    }
    if (kernel == nullptr) {
        return -1;
    }
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(tiles), static_cast<unsigned>(batches)), dim3(W * 64), 0, stream,
                       op, ep, static_cast<int>(tilesM));
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <int CT, int BT>
int launch_type(const GemmOperands &op, const EpiParams &ep, int64_t batches, int cfg, bool reg, hipStream_t stream)
{
    constexpr bool f16w8 = CT == KUDNN_DT_F16 && BT != CT;  // two pieces of A a k-tile: fewer waves
    if (reg) {
        cfg = cfg == KUDNN_CFG_WAVEK_32x16 ? KUDNN_CFG_WAVEK_32x32
                                           : (cfg == KUDNN_CFG_WAVEK_64x64 || cfg == KUDNN_CFG_WAVEK_64x128
                                                  ? KUDNN_CFG_WAVEK_64x64_W4 : cfg);
    } else if (CT == BT && CT != KUDNN_DT_S8 && CT != KUDNN_DT_F32) {
        cfg = cfg == KUDNN_CFG_WAVEK_16x16 ? KUDNN_CFG_WAVEK_32x16 : (cfg == KUDNN_CFG_WAVEK_16x32 ? KUDNN_CFG_WAVEK_32x32 : cfg);
    }
    switch (cfg) {
        case KUDNN_CFG_WAVEK_16x16: return launch_tile<CT, BT, 16, 16, 8>(op, ep, batches, reg, stream);
        case KUDNN_CFG_WAVEK_16x32: return launch_tile<CT, BT, 16, 32, 8>(op, ep, batches, reg, stream);
        case KUDNN_CFG_WAVEK_32x16: return launch_tile<CT, BT, 32, 16, 8>(op, ep, batches, reg, stream);
        case KUDNN_CFG_WAVEK_32x32: return launch_tile<CT, BT, 32, 32, 8>(op, ep, batches, reg, stream);
        case KUDNN_CFG_WAVEK_32x64: return launch_tile<CT, BT, 32, 64, 6>(op, ep, batches, reg, stream);
        // 6 waves of f16 with 8-bit weights spill a register or two in one form each: 64 x 32 with rows of any alignment
        // 12 bytes a lane, 64 x 64 in whole chunks 8; outside those forms no instance spills
        case KUDNN_CFG_WAVEK_64x32: return launch_tile<CT, BT, 64, 32, 6>(op, ep, batches, reg, stream);
        case KUDNN_CFG_WAVEK_64x64: return launch_tile<CT, BT, 64, 64, f16w8 ? 6 : 8>(op, ep, batches, reg, stream);
        case KUDNN_CFG_WAVEK_64x64_W4: return launch_tile<CT, BT, 64, 64, f16w8 ? 3 : 4>(op, ep, batches, reg, stream);
        case KUDNN_CFG_WAVEK_64x128: return launch_tile<CT, BT, 64, 128, 4>(op, ep, batches, reg, stream);
        case KUDNN_CFG_WAVEK_64x64_W1:
            if constexpr (CT == BT && (CT == KUDNN_DT_BF16 || CT == KUDNN_DT_F16)) {
                return reg ? -1 : launch_tile<CT, BT, 64, 64, 1>(op, ep, batches, false, stream);
            }
            return -1;
        default: return -1;
    }
}

}  // namespace

#endif  // KUDNN_GEMM_WAVEK_H
