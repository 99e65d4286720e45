// CPU check of the row pitch of the K slices' sums (kudnn_slice_pitch, kudnn_amd/csrc/kernels.h) over the grids that the
// planner slices: a call of the allocation-free entry point that fits its scratch with rows of whole 32-byte chunks still
// fits it, whichever operands it packs, and rows are whole 128-byte lines everywhere else. Exit status 0 when all hold.
#include <cstdint>
#include <cstdio>

#include "kernels.h"

int main()
{
    const auto up = [](int64_t v) { return (v + 255) / 256 * 256; };
    long grids = 0, chunks = 0, refused = 0, wrong = 0;
    for (int64_t M = 256; M <= 8192; M += 128) {
        for (int64_t N = 8; N <= 16384; N += N % 64 == 1 ? 7 : (N % 64 == 0 ? 1 : 8)) {
            for (int64_t K = 512; K <= 14336; K += 448) {
                const int S = kudnn_kslice_rule(M, N, K / 64, 1, KUDNN_DT_BF16);
                if (S < 2) {
                    continue;
                }
                ++grids;
                const int64_t n8 = (N + 7) / 8 * 8, n32 = (N + 31) / 32 * 32, ld = kudnn_slice_pitch(M, N, K, S);
                if (ld != n8 && ld != n32) {
                    ++wrong;
                }
                chunks += ld != n32;
                bool lines = true;
                for (int p = 0; p < 4; ++p) {
                    const int64_t packs = (p & 1 ? up(M * K * 2) : 0) + (p & 2 ? up(N * K * 2) : 0);
                    const bool before = packs + up(S * M * n8 * 4) <= KUDNN_FIXED_WORKSPACE;
                    refused += before && packs + up(S * M * ld * 4) > KUDNN_FIXED_WORKSPACE;
                    lines = lines && !(before && packs + up(S * M * n32 * 4) > KUDNN_FIXED_WORKSPACE);
                }
                wrong += lines != (ld == n32);
            }
        }
    }
    std::printf("%ld sliced grids, %ld with rows of chunks, %ld refused, %ld wrong\n", grids, chunks, refused, wrong);
    return grids > 10000 && chunks > 0 && refused == 0 && wrong == 0 ? 0 : 1;
}
