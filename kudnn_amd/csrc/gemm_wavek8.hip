// The wave-K kernel's instances with 8-bit weights and in f32 (gemm_wavek.h).
#include "gemm_wavek.h"

int kudnn_launch_gemm_wavek8(const GemmOperands &op, const EpiParams &ep, int64_t batches, int ct, int bt, int cfg, bool reg,
                             hipStream_t stream)
{
    switch (ct * 16 + bt) {
        case KUDNN_DT_F16 * 16 + KUDNN_DT_S8: return launch_type<KUDNN_DT_F16, KUDNN_DT_S8>(op, ep, batches, cfg, reg, stream);
        case KUDNN_DT_F16 * 16 + KUDNN_DT_U8: return launch_type<KUDNN_DT_F16, KUDNN_DT_U8>(op, ep, batches, cfg, reg, stream);
        case KUDNN_DT_S8 * 16 + KUDNN_DT_S8: return launch_type<KUDNN_DT_S8, KUDNN_DT_S8>(op, ep, batches, cfg, reg, stream);
        case KUDNN_DT_S8 * 16 + KUDNN_DT_U8: return launch_type<KUDNN_DT_S8, KUDNN_DT_U8>(op, ep, batches, cfg, reg, stream);
        case KUDNN_DT_F32 * 16 + KUDNN_DT_F32: return launch_type<KUDNN_DT_F32, KUDNN_DT_F32>(op, ep, batches, cfg, reg, stream);
        default: return -1;
    }
}
