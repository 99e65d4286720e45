// The wave-K kernel's launch and its bf16 and f16 instances (gemm_wavek.h).
#include "gemm_wavek.h"

int kudnn_launch_gemm_wavek(const GemmOperands &op, const EpiParams &ep, int64_t batches, int ct, int bt, int cfg,
                            hipStream_t stream)
{
    // whole 16-byte chunks (rows, batches and bases) go through the LDS DMA, others through registers
    auto size = [](int dt) { return dt == KUDNN_DT_F32 ? 4 : (dt == KUDNN_DT_S8 || dt == KUDNN_DT_U8 ? 1 : 2); };
    const int ea = 16 / size(ct), eb = 16 / size(bt);
    auto whole = [&](const void *p, int64_t ld, const int64_t bs[3], int e) {
        return reinterpret_cast<uintptr_t>(p) % 16 == 0 && ld % e == 0 && bs[0] % e == 0 && bs[1] % e == 0 && bs[2] % e == 0;
    };
    const bool kWhole = op.k_padded || (op.K % ea == 0 && (op.b_kmajor || op.K % eb == 0));
    const bool reg = !kWhole || !whole(op.a, op.lda, op.a_bs, ea) || !whole(op.b, op.ldb, op.b_bs, eb);
    if (op.K <= 0 || (reg && (op.b_kmajor || op.K < std::max(ea, eb))) || (op.b_kmajor && (op.N % 8 != 0 || op.ldb < op.N))) {
        return -1;
    }
    switch (ct * 16 + bt) {
        case KUDNN_DT_BF16 * 16 + KUDNN_DT_BF16: return launch_type<KUDNN_DT_BF16, KUDNN_DT_BF16>(op, ep, batches, cfg, reg, stream);
        case KUDNN_DT_F16 * 16 + KUDNN_DT_F16: return launch_type<KUDNN_DT_F16, KUDNN_DT_F16>(op, ep, batches, cfg, reg, stream);
        default: return kudnn_launch_gemm_wavek8(op, ep, batches, ct, bt, cfg, reg, stream);
    }
}
