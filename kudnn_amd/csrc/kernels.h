// Host-side launchers of the HIP kernels (one translation unit per kernel family).
#ifndef KUDNN_KERNELS_H
#define KUDNN_KERNELS_H

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "plan_types.h"

// Tile configurations of the dispatcher (values are stable: they appear in plan descriptions).
enum {
    KUDNN_CFG_BF16_256x256 = 1,
    KUDNN_CFG_BF16_256x128 = 2,
    KUDNN_CFG_BF16_128x128 = 3,
    KUDNN_CFG_BF16_PINGPONG_256x256 = 4,
    KUDNN_CFG_F32_128x128 = 10,
    KUDNN_CFG_F32_64x64 = 11,
    KUDNN_CFG_F32_KSLICE_16x32 = 12,  // small f32 grids: 16 x 32 tiles, K split over the waves of the workgroup
    KUDNN_CFG_SKINNY_BF16 = 20,
    KUDNN_CFG_GEMV_BF16 = 21,  // M == 1: one wave per weight row, X staged in LDS (skinny engine)
    KUDNN_CFG_GEMV_MULTI_BF16 = 22,  // 2 <= M <= 5 (M <= 8 forced): one wave per weight row, X staged in LDS
    KUDNN_CFG_GEMV_KSPLIT_BF16 = 23,  // 2 <= M <= 16, K <= 4096, one batch: K split over 8 waves, X in registers
    // a small tile per workgroup, its K dealt to the waves (gemm_wavek.hip, kudnn_wavek_rule)
    KUDNN_CFG_WAVEK_16x16 = 28,    // 8 waves; 8-bit weights
    KUDNN_CFG_WAVEK_16x32 = 29,    // 8; 8-bit weights
    KUDNN_CFG_WAVEK_32x16 = 30,    // 8
    KUDNN_CFG_WAVEK_32x32 = 31,    // 8
    KUDNN_CFG_WAVEK_32x64 = 32,    // 6
    KUDNN_CFG_WAVEK_64x32 = 33,    // 6
    KUDNN_CFG_WAVEK_64x64 = 34,    // 8 (8-bit weights of f16: 6)
    KUDNN_CFG_WAVEK_64x64_W4 = 35, // 4 (8-bit weights of f16: 3)
    KUDNN_CFG_WAVEK_64x128 = 36,   // 4
    KUDNN_CFG_WAVEK_64x64_W1 = 37, // 1: batches of 16-bit products with a short K
};
inline bool kudnn_is_wavek(int cfg) { return cfg >= KUDNN_CFG_WAVEK_16x16 && cfg <= KUDNN_CFG_WAVEK_64x64_W1; }

// Returns 0 on success, -1 if the launch failed or cfg is unknown. `ct` is the operand (compute) type of the 16- and
// 8-bit kernels: KUDNN_DT_BF16, KUDNN_DT_F16 (f32 accumulation) or KUDNN_DT_S8 (int32 accumulation, integer
// epilogue only). Their tile configurations keep the bf16 names; an s8 k-tile is 128 elements instead of 64.
// 4-wave MFMA kernels (gemm_mfma.hip). A grid too small for the chip is split along K, in the same launch, when `ws`
// (device memory of at least kudnn_gemm_workspace_bytes bytes, 256-byte aligned) and `counters` (at least
// KUDNN_SPLIT_MAX_TILES uint32, zero; a split launch leaves them zero) are given; with nullptr it runs unsplit. s8
// launches are never split.
constexpr int KUDNN_SPLIT_MAX_TILES = 128;
size_t kudnn_gemm_workspace_bytes(const GemmOperands &op, int64_t batches, int cfg, int ct);
int kudnn_launch_gemm_mfma(const GemmOperands &op, const EpiParams &ep, int64_t batches, int cfg, int ct, void *ws,
                           uint32_t *counters, hipStream_t stream);
// 8-wave ping-pong schedule, 256x256 tile (gemm_pingpong.hip). Needs K a whole number of 128-byte k-tiles, 16-byte
// aligned rows and 32-bit operand offsets; kudnn_pingpong_eligible says whether `op` qualifies.
bool kudnn_pingpong_eligible(const GemmOperands &op, int ct);
// Bytes of workspace the launch wants for its K slices (slicesOk) or its tail split (0: one data-parallel launch);
// `ws` of at least that many bytes, or nullptr to run without either. The launch takes the same slicesOk.
size_t kudnn_pingpong_workspace_bytes(const GemmOperands &op, int64_t batches, int ct, bool slicesOk);
// The split the launch would make: tiles of the data-parallel launch, tail tiles, k-iterations per tail workgroup
// (all 0 when it makes none).
void kudnn_pingpong_split(const GemmOperands &op, int64_t batches, int ct, int *dpTiles, int *tailTiles, int *iters);
// The K slices the launch would make when allowed (0: none).
int kudnn_pingpong_slices(const GemmOperands &op, int64_t batches, int ct);
// Tiles in slices when only the last partial round is sliced (0: none, or every tile).
int kudnn_pingpong_slice_tail(const GemmOperands &op, int64_t batches, int ct);
// Device scratch of the allocation-free entry point: the split-K counters (KUDNN_SPLIT_MAX_TILES uint32), then the
// workspace.
constexpr int64_t KUDNN_FIXED_BYTES = int64_t(64) << 20, KUDNN_FIXED_COUNTERS = 512;
constexpr int64_t KUDNN_FIXED_WORKSPACE = KUDNN_FIXED_BYTES - KUDNN_FIXED_COUNTERS;
// Whether S slices leave every call of the allocation-free entry point accepted that is accepted unsliced: with no
// operand packed, either or both (16-bit), what fits the scratch without the sums fits with them. `base`: the columns a row
// of sums takes in the calls that have to stay accepted (0: no sums), `ld`: the ones it is to take.
inline bool kudnn_slices_fit(int64_t M, int64_t N, int64_t K, int64_t S, int64_t base, int64_t ld)
{
    const auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
    const int64_t a = up(M * K * 2), b = up(N * K * 2), from = up(S * M * base * 4), to = up(S * M * ld * 4);
    for (const int64_t packs : {int64_t(0), a, b, a + b}) {
        if (packs + from <= KUDNN_FIXED_WORKSPACE && packs + to > KUDNN_FIXED_WORKSPACE) {
            return false;
        }
    }
    return true;
}
// Columns that a row of the slices' sums takes: whole 128-byte lines (816 x 7048 x 4096 in two slices 103 -> 80 us) where
// every call that fits the scratch with whole 32-byte chunks still fits it, else those (512 x 3073 x 6784 with a packed
// weight needs 66.93 MB of 67.11 that way, 67.12 with lines).
inline int64_t kudnn_slice_pitch(int64_t M, int64_t N, int64_t K, int64_t S)
{
    const int64_t lines = (N + 31) / 32 * 32, chunks = (N + 7) / 8 * 8;
    return kudnn_slices_fit(M, N, K, S, chunks, lines) ? lines : chunks;
}
// The planner's K-slice count for the ping-pong kernel (0: none) of an M x N grid with KT k-tiles of 128 bytes.
// Measured on MI355X over 26 shapes (M 256..4096, N 1152..14336, K 2048..14336, against the unsliced ping-pong, its
// tail split and the 4-wave kernel): up to 64 tiles of 256 x 256, as many slices as keep tiles x slices <= 128 (at
// most 8), each of at least 16 k-tiles, were 1.07-2.4x faster than the best of those, except at 64 tiles with fewer
// than 64 k-tiles, where the 4-wave kernel's 128 x 128 tiles fill the CUs (2048 x 2048 x 2048: 49 against 38 us);
// 80-96 tiles with M >= 1024 and at least 48 k-tiles: two slices, 7-23 % faster (M = 512 lost 3 %, 112-128 tiles up
// to 47 %).
// 65-120 tiles otherwise: two slices where 9 us + 0.6 us a k-tile (10 % more from 97 tiles on) + the sums' way at 3.6
// TB/s is 5 % less than 5 us + 1.05 us a k-tile of the whole tiles (1.2 where M is off the tile: edge rows are copied
// one block at a time). Measured (bf16, unsliced against two slices): 738 x 5896 x 10112 178 -> 110 us, 512 x 11008 x
// 14336 281 -> 180, 376 x 11840 x 3584 72 -> 62, 768 x 8192 x 8192 140 -> 116; below the line 1100 x 4096 x 2560 50
// against 54, 700 x 8192 x 2048 48 against 57; 128 tiles fill the chip twice over (2048 x 4096 x 8192 143 against 155).
// Three slices gained 3 % on two at 72 tiles and lost 35-60 % at 86.
inline int kudnn_kslice_rule(int64_t M, int64_t N, int64_t KT, int64_t batches, int ct)
{
    if (batches != 1 || ct == KUDNN_DT_S8 || M <= 0 || N <= 0) {
        return 0;
    }
    const int64_t tiles = (M + 255) / 256 * ((N + 255) / 256);
    int64_t S = 0;
    if (tiles <= 64) {
        S = 128 / tiles;
        S = S < 8 ? S : 8;
        S = S < KT / 16 ? S : KT / 16;
        if (tiles * 4 >= 256 && KT < 64) {
            S = 0;
        }
    } else if (tiles <= 96 && M >= 1024 && KT >= 48) {
        S = 2;
    } else if (tiles <= 120) {
        const double kt = static_cast<double>(KT), mn = static_cast<double>(M) * static_cast<double>(N);
        const double whole = 5.0 + (M % 256 != 0 ? 1.2 : 1.05) * kt;
        const double half = 9.0 + 0.6 * kt * (tiles > 96 ? 1.1 : 1.0) + mn * 16.0 / 3.6e6;
        S = half * 1.05 < whole && kudnn_slices_fit(M, N, KT * 64, 2, 0, (N + 31) / 32 * 32) ? 2 : 0;
    }
    return S >= 2 ? static_cast<int>(S) : 0;
}

// Slices of the last partial round of a 16-bit grid of more tiles than CUs, whose full rounds run whole tiles (0:
// none). With R tiles in that round (R = tiles mod CUs): R at most an eighth of the CUs, S = min(CUs / 2 / R, 8,
// KT / 16) when that is at least 2. Measured on MI355X against the unsliced grid (bf16, bias): 3072 x 11008 x 4096
// (R = 4) 265 -> 231 us, 4352 x 4096 x 4096 (R = 16) 168 -> 136 us, 4096 x 4608 x 4096 and 2304 x 8192 x 4096
// (R = 32) 168 -> 148-149 us; R = 64 with 48 k-tiles even, with 24 k-tiles 15 % slower; R = 88, 128 and 176 (C3)
// slower at every S; 18 k-tiles slower at every S.
inline int kudnn_tail_slice_rule(int64_t M, int64_t N, int64_t KT, int64_t batches, int ct, int cus)
{
    if (batches != 1 || ct == KUDNN_DT_S8 || M <= 0 || N <= 0 || cus <= 0) {
        return 0;
    }
    const int64_t tiles = (M + 255) / 256 * ((N + 255) / 256);
    const int64_t rem = tiles % cus;
    if (tiles <= cus || rem == 0 || rem * 8 > cus) {
        return 0;
    }
    int64_t S = cus / 2 / rem;
    S = S < 8 ? S : 8;
    S = S < KT / 16 ? S : KT / 16;
    return S >= 2 ? static_cast<int>(S) : 0;
}

// The wave-K tiles that can take rows of any alignment through registers (the wider ones have none to spare).
constexpr bool kudnn_wavek_reg_tile(int bm, int bn, int waves)
{
    return bn >= bm / 2 && bm * bn <= 64 * 64 && (bm * bn < 64 * 64 || waves <= 4) && (bm != 32 || bn != 16);
}

// Tiles whose K is dealt to the workgroup's waves (gemm_wavek.hip). op.K is the true K; k_padded says that packed rows
// hold zeros up to a whole 16-byte chunk. Operands that are not whole chunks (rows, K, bases) take the register form.
// b_kmajor (16-bit): whole chunks of columns, tiles of 64 columns or more. `bt` is the weight's stored type: ct, s8 or u8
// under f16, and u8 under s8 for a u8 A beside an s8 weight (the term of the -128 shift is added here; op.a_u8 says whether
// A still has to be shifted). No workspace.
int kudnn_launch_gemm_wavek(const GemmOperands &op, const EpiParams &ep, int64_t batches, int ct, int bt, int cfg,
                            hipStream_t stream);
// Its 8-bit and f32 instances (a translation unit of their own); `reg`: the register form.
int kudnn_launch_gemm_wavek8(const GemmOperands &op, const EpiParams &ep, int64_t batches, int ct, int bt, int cfg, bool reg,
                             hipStream_t stream);

// The wave-K tile for a product (0: the kernel the other rules chose). The tile is the one with the least estimate, which
// is what the measurements of 7 tiles over M = 17..1030 and N, K = 2048..14336 (weights rotated past the Infinity Cache)
// fit: 4.2 us a call, plus the largest of the weight's stream from HBM at 6.6 TB/s, the busiest CU's copies, nsPerKB per KB
// of A and B (`over` times that when more tiles come to a CU than fit beside one another), and the products at 0.8 PFLOP/s
// (8-bit 1.4; f32 by the tile's rate on the busiest CU), plus a part of the stream. Over 26 drawn bf16 shapes the choice was
// within 7 % of the best tile but for 3 (19 %).
// That tile is taken where its cost is below otherUs, the cost of the other rules' kernel (BuildCore). The estimate orders
// the tiles but is 15-50 % low where K is short, the output large, the rows unaligned or the batches many, so the cost is a
// fit of its own, over 5600 products (M = 1..8192, N = 1..16384, K = 64..16384, up to 64 batches; half of them drawn as the
// layers of a model are) timed on the chosen tile and on the other kernel, with a mean error of 10 %: the copies or half the
// stream, whichever is longer, plus most of the stream (waves that share nothing overlap them badly), 0.3 ns per output of
// the busiest CU, 2.2 us per million outputs, and the tiles' own packs (packUs); rows of any alignment take twice the
// copies' time, and batches with a weight each (`weights`) stream all of A and B. f32: the estimate, which was within 8 %,
// or nine tenths of it and 0.45 ns per output of the busiest CU. Of 20000 drawn layers 793 change sides against the
// comparison of the bare estimates: 176 of them had been slower than the other kernel by 3 % and more (up to 1.5 times), 5
// are now (up to 10 %); the 793 take 0.89 of the time.
// Measured, against the other kernel: bf16 64 x 4096 x 4096 10 us (31), 64 x 11008 x 4096 22 (48), 192 x 4096 x 11008 45
// (48), 400 x 4096 x 4096 27 (45), 16 batches of 32 x 1024 x 4096 33 (91); f16 x s8 4 x 4096 x 4096 6.1 (21.5), 128 x 4096 x
// 4096 12 (55); u8 x s8 64 x 4096 x 4096 7.5 (47), 1024 x 4096 x 4096 40 (51). The others stay where a weight is wide for
// its depth (bf16 255 x 14336 x 4096 55 against 47, 742 x 7968 x 256 34 against 22; f32 10925 x 2304 x 376 304 against 223)
// and where the small tiles re-read A and B too often (M large; 64 batches of 128 x 512 x 2048 72 against 51).
// 16-bit products of up to 16 rows have the decode kernels. Whole 256-row tiles of 16-bit products with whole k-tiles keep
// the plans that tests of the dispatch name, although up to 32 tiles of 256 x 256 the wave-K tiles are the faster ones (256
// x 4096 x 4096 23 against 38 us, 512 x 4096 x 4096 35 against 49; from 43 tiles on slower: 256 x 11008 x 4096 57 against
// 50, 1024 x 4096 x 4096 65 against 51). Less than 4 whole k-tiles leave most waves without one. minParts (f32): the fewest
// chains of 2-k steps that K is dealt to, for no longer chain of rounded sums than otherUs' kernel has: a wave's MFMAs are
// of 2 k, with 16 rows or columns of 4. binary: the epilogue reads a second operand. bareUs: the other kernel's estimate for
// the comparison of the bare estimates, 0 where it does not count.
inline int kudnn_wavek_rule(int64_t M, int64_t N, int64_t K, int64_t batches, int64_t weights, int ct, bool weight8,
                            bool kmajor, bool byRow, bool binary, double packUs, double otherUs, double bareUs,
                            int minParts = 1)
{
    struct Tile {
        int cfg, bm, bn, waves;
        double nsPerKB, over, f32Rate;  // f32Rate: f32 TFLOP/s of a CU
    };
    static const Tile kTiles[] = {{KUDNN_CFG_WAVEK_16x16, 16, 16, 8, 11.5, 1.1, 0.25}, {KUDNN_CFG_WAVEK_16x32, 16, 32, 8, 11.6, 1.1, 0.28},
                                  {KUDNN_CFG_WAVEK_32x16, 32, 16, 8, 11.5, 1.1, 0.28}, {KUDNN_CFG_WAVEK_32x32, 32, 32, 8, 11.7, 1.1, 0.32},
                                  {KUDNN_CFG_WAVEK_64x32, 64, 32, 6, 11.3, 1.1, 0.32}, {KUDNN_CFG_WAVEK_32x64, 32, 64, 6, 11.8, 1.1, 0.32},
                                  {KUDNN_CFG_WAVEK_64x64, 64, 64, 8, 12.6, 1.25, 0.34}, {KUDNN_CFG_WAVEK_64x64_W4, 64, 64, 4, 12.9, 1.1, 0.40},
                                  {KUDNN_CFG_WAVEK_64x128, 64, 128, 4, 15.5, 1.1, 0.45}};
    const bool f16w8 = weight8 && ct != KUDNN_DT_S8;          // two 128-byte pieces of an A row a k-tile
    const bool f32 = ct == KUDNN_DT_F32;
    const int64_t bk = f32 ? 32 : (weight8 || ct == KUDNN_DT_S8 ? 128 : 64);
    const int64_t KT = (K + bk - 1) / bk;
    if ((bk == 64 && M >= 256 && M % 256 == 0 && K % 64 == 0) || K < 4 * bk) {
        return 0;
    }
    const double mac = static_cast<double>(M) * static_cast<double>(N) * static_cast<double>(K * batches);
    const double mn = static_cast<double>(M * N * batches) * 1e-6;
    const double lineUs = static_cast<double>(K) * 128.0 / static_cast<double>(bk) / 6.6e6;  // a row of k at 6.6 TB/s
    const double stream = static_cast<double>(N) * lineUs;
    const double streamAll = static_cast<double>(N * weights + (weights > 1 ? M * batches : 0)) * lineUs;
    int best = 0;
    double bestUs = 0.0, cost = 0.0;
    for (const Tile &t : kTiles) {
        if ((kmajor && t.bn < 64) || (t.bm == 16 && (M > 16 || (bk == 64 && !byRow))) ||
            (byRow && !kudnn_wavek_reg_tile(t.bm, t.bn, t.waves)) || t.waves * (t.bm == 16 || t.bn == 16 ? 2 : 1) < minParts) {
            continue;
        }
        const int64_t waves = f16w8 && t.bm == 64 && t.bn == 64 ? t.waves * 3 / 4 : t.waves;
        const double kb = (t.bm * (f16w8 ? 2 : 1) + t.bn) / 8.0;  // KB of a k-tile: a wave's stage
        const int64_t tiles = (M + t.bm - 1) / t.bm * ((N + t.bn - 1) / t.bn) * batches;
        const int64_t perCu = (tiles + 255) / 256, ktiles = (KT + waves - 1) / waves * waves;
        const double copies = static_cast<double>(perCu * ktiles) * kb * t.nsPerKB * 1e-3 *
                              (static_cast<double>(perCu * waves) * kb > 160.0 ? t.over : 1.0);
        const double mfma = f32 ? static_cast<double>(perCu * t.bm * t.bn) * 2e-6 * static_cast<double>(ktiles * bk) / t.f32Rate
                                : mac * 2.0 / (ct == KUDNN_DT_S8 ? 1.4e9 : 0.8e9);
        // a part of the CUs streams a part of HBM's rate: in proportion for k-rows, less so for rows
        double part = tiles < 256 ? 256.0 / static_cast<double>(tiles) : 1.0;
        part = kmajor ? part : std::sqrt(part);
        const double copyUs = copies * (byRow ? 1.15 : (kmajor ? 1.08 : 1.0)), busy = std::max(copyUs, mfma), hbm = stream * part;
        const double us = 4.2 + (busy > hbm ? busy + 0.15 * stream : hbm + 0.15 * copyUs);
        if (best == 0 || us < bestUs) {
            best = t.cfg;
            bestUs = us;
            const double out = static_cast<double>(perCu * t.bm * t.bn) * 1e-3;
            if (f32) {
                cost = std::max(us, 0.9 * us + 0.45 * out);
            } else {
                cost = 4.0 + std::max(0.9 * std::max(copies * (byRow ? 1.95 : 1.0), mfma), 0.58 * streamAll * part) +
                       0.79 * streamAll + 0.31 * (t.cfg == KUDNN_CFG_WAVEK_64x64_W4 ? 0.63 : 1.0) * out +
                       (binary ? 2.57 : 2.2) * mn + packUs;
            }
        }
    }
    return cost < otherUs || bestUs < bareUs ? best : 0;
}

// The same for batches of 16-bit products of at most 256 k (scores of attention heads, say), which spend their time on
// tiles that start and end. One wave per 64 x 64 tile took 7 us + 2.5 ns a tile + 1 ns a k-tile of it; the ping-pong
// kernel 3 us + 7.5 us a round of 256 tiles of 256 x 256, which ragged M and N leave partly empty, + 1.9 us a k-tile of
// it; the 4-wave kernel 4 us + 4.2 us a round of 256 tiles of 128 x 128 + 0.9 us a k-tile. packUs: what these two pack on
// each call. Up to 768 tiles, three a CU, four waves share one: 5.3 us + 2.5 ns a tile, or, with several tiles a CU and
// short products, 4.5 us + 0.22 us a tile of the busiest CU + 0.4 us a k-tile of it + 1.4 us per million outputs. A binary
// operand, which only the other kernels read ahead, adds to both. Measured (bf16, against the other kernel): 63 x
// (192 x 376 x 80) 31 -> 12 us, 32 x (256 x 256 x 96) 21 -> 7, 64 x (2048 x 128 x 128) 32 -> 26, 20 x (300 x 1000 x 128)
// 15.4 -> 12.6; these stay: 32 x (1024 x 1024 x 128) 44 against 27, 13 x (640 x 256 x 64) 10.2 against 7.9, 39 x (256 x 576
// x 64) with an addend 19.5 against 14.8. Over 579 batches the side taken costs 1.1 % more than the better one. bare: the
// comparison without the several tiles' and the operand's terms.
inline int kudnn_wavek_batch_rule(int64_t M, int64_t N, int64_t K, int64_t batches, bool pingpong, bool binary, double packUs,
                                  bool bare)
{
    const int64_t KT = (K + 63) / 64;
    if (batches < 2 || KT > 4) {
        return 0;
    }
    const int64_t bm = pingpong ? 256 : 128;
    const int64_t tiles = (M + 63) / 64 * ((N + 63) / 64) * batches;
    const double rounds = static_cast<double>(((M + bm - 1) / bm * ((N + bm - 1) / bm) * batches + 255) / 256);
    const double kt = static_cast<double>(KT), t = static_cast<double>(tiles), perCu = static_cast<double>((tiles + 255) / 256);
    const double mn = static_cast<double>(M * N * batches) * 1e-6;
    const double other = packUs + (pingpong ? 3.0 + rounds * (7.5 + 1.9 * kt) : 4.0 + rounds * (4.2 + 0.9 * kt));
    const bool four = tiles <= 768;
    double us = four ? 5.3 + 2.5e-3 * t : 7.0 + t * (2.5e-3 + 1e-3 * kt);
    if (!bare) {
        us = four ? std::max(us, 4.5 + perCu * (0.22 + 0.4 * kt) + 1.4 * mn) : us;
        us += binary ? (four ? 0.5 : 1.0) + 0.3 * mn : 0.0;
    }
    return us < other ? (four ? KUDNN_CFG_WAVEK_64x64_W4 : KUDNN_CFG_WAVEK_64x64_W1) : 0;
}
int kudnn_launch_gemm_pingpong(const GemmOperands &op, const EpiParams &ep, int64_t batches, int ct, void *ws,
                               bool slicesOk, hipStream_t stream);
int kudnn_launch_gemm_f32(const GemmOperands &op, const EpiParams &ep, int64_t batches, int cfg, void *ws,
                          uint32_t *counters, hipStream_t stream);
// f32, one 16 x 32 tile per workgroup with K split over its waves (gemm_kslice.hip): no workspace. Needs K a multiple
// of 16, 16-byte aligned operands and row strides; kudnn_kslice_eligible says whether `op` qualifies.
bool kudnn_kslice_eligible(const GemmOperands &op);
int kudnn_launch_gemm_f32_kslice(const GemmOperands &op, const EpiParams &ep, int64_t batches, hipStream_t stream);
// M <= 16, bf16 or f16 operands (`ct`), B contiguous along K (M == 1, and M <= 8 under cfg KUDNN_CFG_GEMV_MULTI_BF16:
// row-per-wave GEMV with X staged in LDS; otherwise 16-row MFMA tiles; 64-bit addressed forms for operands of 2 GiB or
// more).
int kudnn_launch_skinny(const GemmOperands &op, const EpiParams &ep, int64_t batches, int ct, int cfg, hipStream_t stream);

// Pack: dst[b][r][k] (row pitch kp, zero for k >= cols) = convert(src element (b, r, k)) where the source
// element sits at src + b-offset + r*s_r + k*s_k. dst dtype is the compute type: F32, BF16, F16 or S8 (conversions are
// exact: widening, 8-bit integers to f16 or f32, or a copy).
struct PackArgs {
    const void *src;
    int src_dt;
    int64_t rows, cols;      // logical rows (M or N) and K
    int64_t s_r, s_k;        // source strides (elements)
    int64_t bdim[3];
    int64_t bs[3];           // source batch strides
    void *dst;
    int dst_dt;
    int64_t kp;              // destination row pitch (elements), >= cols
    int64_t dst_bstride;     // destination batch stride (elements)
    int shift;               // subtracted from every element (128: u8 -> s8 for the integer MFMA); padding stays 0
};
int kudnn_launch_pack(const PackArgs &p, int64_t batches, hipStream_t stream);
// out[c * rows + r] = scale * (sum over the kp int8 of row r of copy c of a packed operand), in wrapping 32-bit
// arithmetic: the correction terms of an integer GEMM whose other operand was a shifted u8.
int kudnn_launch_rowsum_s8(const int8_t *p, int64_t rows, int64_t kp, int64_t copies, int64_t bstride, uint32_t scale,
                           int32_t *out, hipStream_t stream);

#endif  // KUDNN_KERNELS_H
