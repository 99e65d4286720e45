// Operand packing: any strided layout / floating dtype -> K-contiguous rows in the compute dtype.
//
// The reference reorders non-standard layouts into f32 temporaries before calling BLAS
// (BatchedExtendedGemm, src/dnn/src/kudnn_gemm.cpp:725-765) and widens mismatched dtypes through
// MatrixConverter (:655-670). Here one launch does both for the operands that the MFMA kernels
// cannot read directly: it converts the element type exactly (bf16/f16 -> f32, or bf16 copy; u8 -> s8
// shifted by -128 for the integer MFMA), and zero-fills the row tail up to the padded pitch so the GEMM needs no
// K-tail handling.
//
// Three kernels, by where the source is contiguous; each is bound by HBM (source read once, packed copy written once):
//  - pack_rows_kernel: along K (rows whose pitch, K or type the GEMM cannot take). A lane converts 16 bytes of the
//    packed row per step from one vector load.
//  - pack_cols_kernel: along the rows (a weight stored [K][N]). A 64 x 64 tile goes through LDS in the source's own
//    type, so that both sides move 16-byte pieces.
//  - pack_kernel: any other strides, one element at a time.
// Source rows may start at any multiple of the element size (K is odd in the calls that need a pack most), so the
// vector loads are declared with the element's alignment; gfx950 serves such loads at nearly the aligned rate.
#include <type_traits>

#include "device_common.h"
#include "kernels.h"

using namespace kudnn_dev;

namespace {

constexpr int kTile = 64;

// One element at a time: a 64 x 64 tile through LDS as f32.
__global__ __launch_bounds__(256) void pack_kernel(PackArgs p)
{
    __shared__ float tile[kTile][kTile + 1];
    const int tid = threadIdx.x;
    // rows on x (up to 2^31 - 1 workgroups: a folded batch makes M large), K on y
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * kTile;
    const int64_t k0 = static_cast<int64_t>(blockIdx.y) * kTile;
    const int64_t b = blockIdx.z;
    const int64_t i2 = b % p.bdim[2];
    const int64_t i1 = (b / p.bdim[2]) % p.bdim[1];
    const int64_t i0 = b / (p.bdim[2] * p.bdim[1]);
    const int64_t srcOff = i0 * p.bs[0] + i1 * p.bs[1] + i2 * p.bs[2];

    // Read so that consecutive threads touch consecutive source addresses.
    const bool rFast = (p.s_r == 1 && p.s_k != 1);
    for (int i = 0; i < kTile * kTile / 256; ++i) {
        int e = tid + i * 256;
        int rr = rFast ? (e % kTile) : (e / kTile);
        int kk = rFast ? (e / kTile) : (e % kTile);
        int64_t r = r0 + rr, k = k0 + kk;
        float v = 0.0f;
        if (r < p.rows && k < p.cols) {
            v = load_elem(p.src, p.src_dt, srcOff + r * p.s_r + k * p.s_k) - static_cast<float>(p.shift);
        }
        tile[rr][kk] = v;
    }
    __syncthreads();
    for (int i = 0; i < kTile * kTile / 256; ++i) {
        int e = tid + i * 256;
        int rr = e / kTile, kk = e % kTile;
        int64_t r = r0 + rr, k = k0 + kk;
        if (r < p.rows && k < p.kp) {
            store_elem(p.dst, p.dst_dt, b * p.dst_bstride + r * p.kp + k, tile[rr][kk]);
        }
    }
}

// Storage type of an element type.
template <int DT>
using Elem = std::conditional_t<DT == KUDNN_DT_F32, uint32_t,
                                std::conditional_t<DT == KUDNN_DT_S8 || DT == KUDNN_DT_U8, uint8_t, uint16_t>>;

// Exact conversion of one element's bits, as load_elem / store_elem do it: a copy within one type, u8 -> s8 shifted by
// -128, 8-bit integers -> f16, anything -> f32.
template <int SRC, int DST>
__device__ __forceinline__ Elem<DST> convert(Elem<SRC> v)
{
    if constexpr (SRC == DST) {
        return v;
    } else if constexpr (DST == KUDNN_DT_S8) {
        static_assert(SRC == KUDNN_DT_U8, "an s8 operand comes from s8 or u8");
        return static_cast<uint8_t>(v ^ 0x80u);
    } else {
        float f;
        if constexpr (SRC == KUDNN_DT_S8) {
            f = static_cast<float>(static_cast<int8_t>(v));
        } else if constexpr (SRC == KUDNN_DT_U8) {
            f = static_cast<float>(v);
        } else if constexpr (SRC == KUDNN_DT_BF16) {
            f = bf16_to_f32(v);
        } else {
            f = f16_to_f32(v);
        }
        if constexpr (DST == KUDNN_DT_F32) {
            return f2u(f);
        } else {
            static_assert(DST == KUDNN_DT_F16 && (SRC == KUDNN_DT_S8 || SRC == KUDNN_DT_U8), "f16 from 8-bit integers");
            return f32_to_f16_rne(f);
        }
    }
}

// N source elements at any element-aligned address, one (or a few) vector loads.
template <typename E, int N>
struct __attribute__((packed, aligned(alignof(E)))) Vec {
    E v[N];
};

// Batch base offset of the source (elements).
__device__ __forceinline__ int64_t batch_off(const PackArgs &p, int64_t b)
{
    return b / (p.bdim[2] * p.bdim[1]) * p.bs[0] + (b / p.bdim[2]) % p.bdim[1] * p.bs[1] + b % p.bdim[2] * p.bs[2];
}

// Source contiguous along K. A workgroup of 4 waves takes 16 rows x 64 chunks of 16 packed bytes: wave w's lane l
// converts chunk l of rows w, w + 4, w + 8, w + 12, all four loads issued before the first store. A call of M = 4 on an
// s8 weight of 4096 x 4096 (f16 x s8: 16.8 MB read, 33.6 MB written) takes 21.5 us, 36.1 one element at a time. Packed
// rows of at most 32 chunks share a wave, 2^laneBits lanes to a row (a row of one k-tile is 8 chunks: with a wave each,
// 56 lanes of 64 did nothing: 165504 x 256 x 40 bf16, which packs its source, 59 us a call, 48 this way).
constexpr int kRowsPerGroup = 16;  // with a wave to a row

template <int SRC, int DST>
__global__ __launch_bounds__(256) void pack_rows_kernel(PackArgs p, int laneBits)
{
    using S = Elem<SRC>;
    using D = Elem<DST>;
    constexpr int EPC = 16 / static_cast<int>(sizeof(D));
    const int chunk = threadIdx.x & ((1 << laneBits) - 1);
    const int step = 256 >> laneBits;  // rows a workgroup takes at a time
    const int64_t b = blockIdx.z;
    const int64_t k = ((static_cast<int64_t>(blockIdx.y) << laneBits) + chunk) * EPC;
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * (kRowsPerGroup / 4 * step) + (threadIdx.x >> laneBits);
    if (k >= p.kp) {
        return;  // no barrier below
    }
    const S *src = static_cast<const S *>(p.src) + batch_off(p, b) + k;
    D *dst = static_cast<D *>(p.dst) + b * p.dst_bstride + k;
    union Chunk {
        D e[EPC];
        uint4 q;
    };
    if (k + EPC <= p.cols) {
        Vec<S, EPC> in[kRowsPerGroup / 4];
#pragma unroll
        for (int i = 0; i < kRowsPerGroup / 4; ++i) {
            const int64_t r = r0 + step * i;
            in[i] = *reinterpret_cast<const Vec<S, EPC> *>(src + (r < p.rows ? r : p.rows - 1) * p.s_r);
        }
#pragma unroll
        for (int i = 0; i < kRowsPerGroup / 4; ++i) {
            const int64_t r = r0 + step * i;
            if (r < p.rows) {
                Chunk c;
#pragma unroll
                for (int e = 0; e < EPC; ++e) c.e[e] = convert<SRC, DST>(in[i].v[e]);
                *reinterpret_cast<uint4 *>(dst + r * p.kp) = c.q;
            }
        }
        return;
    }
    // the chunk that column K ends in, and the padding after it
    for (int64_t r = r0; r < p.rows && r < r0 + kRowsPerGroup / 4 * step; r += step) {
        Chunk c;
#pragma unroll
        for (int e = 0; e < EPC; ++e) c.e[e] = k + e < p.cols ? convert<SRC, DST>(src[r * p.s_r + e]) : D(0);
        *reinterpret_cast<uint4 *>(dst + r * p.kp) = c.q;
    }
}

// Source contiguous along the rows (a weight stored [K][N]): a tile of 64 rows x 64 k through LDS in the source's type.
// Loads are 16 bytes of one k (or single elements at the edge), stores 16 bytes of one packed row, 8 lanes to a
// 128-byte line. 4096 x 1152 x 3256 in bf16 (both operands packed, the weight [K][N]): 89 us a call, 110 one element
// at a time. The LDS pitch of one extra dword per k keeps the column reads free of bank conflicts: a lane's k step
// moves it by an odd number of dwords.
template <int SRC, int DST>
__global__ __launch_bounds__(256) void pack_cols_kernel(PackArgs p)
{
    using S = Elem<SRC>;
    using D = Elem<DST>;
    constexpr int EPC = 16 / static_cast<int>(sizeof(D));   // packed elements per store
    constexpr int EPL = 16 / static_cast<int>(sizeof(S));   // source elements per load
    constexpr int PD = kTile * static_cast<int>(sizeof(S)) / 4 + 1;  // LDS pitch of one k, dwords
    constexpr int P = PD * 4 / static_cast<int>(sizeof(S));          // ... in elements
    __shared__ uint32_t lds[kTile * PD];
    const S *tile = reinterpret_cast<const S *>(lds);
    const int tid = threadIdx.x;
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * kTile;
    const int64_t k0 = static_cast<int64_t>(blockIdx.y) * kTile;
    const int64_t b = blockIdx.z;
    const S *src = static_cast<const S *>(p.src) + batch_off(p, b);
    constexpr int kLoads = kTile * kTile / EPL;  // 16-byte pieces of the tile
    constexpr int kIn = (kLoads + 255) / 256;
    Vec<S, EPL> in[kIn];
#pragma unroll
    for (int i = 0; i < kIn; ++i) {
        const int c = tid + i * 256;
        const int64_t k = k0 + c / (kTile / EPL), r = r0 + (c % (kTile / EPL)) * EPL;
        if (k < p.cols && r + EPL <= p.rows) {
            in[i] = *reinterpret_cast<const Vec<S, EPL> *>(src + k * p.s_k + r);
        } else {
#pragma unroll
            for (int e = 0; e < EPL; ++e) in[i].v[e] = k < p.cols && r + e < p.rows ? src[k * p.s_k + r + e] : S(0);
        }
    }
#pragma unroll
    for (int i = 0; i < kIn; ++i) {
        const int c = tid + i * 256;
        uint32_t w[4];
        __builtin_memcpy(w, in[i].v, 16);
        uint32_t *row = lds + c / (kTile / EPL) * PD + (c % (kTile / EPL)) * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) row[e] = w[e];
    }
    __syncthreads();
    constexpr int kChunks = kTile / EPC;  // stores per packed row of the tile
#pragma unroll
    for (int c = tid; c < kTile * kChunks; c += 256) {
        const int rr = c / kChunks, kk = (c % kChunks) * EPC;
        const int64_t r = r0 + rr, k = k0 + kk;
        if (r < p.rows && k < p.kp) {
            union {
                D e[EPC];
                uint4 q;
            } o;
#pragma unroll
            for (int e = 0; e < EPC; ++e) o.e[e] = k + e < p.cols ? convert<SRC, DST>(tile[(kk + e) * P + rr]) : D(0);
            *reinterpret_cast<uint4 *>(static_cast<D *>(p.dst) + b * p.dst_bstride + r * p.kp + k) = o.q;
        }
    }
}

// One wave per row of a packed int8 operand: sums its kp elements (16 per lane and step), then scales.
__global__ __launch_bounds__(256) void rowsum_s8_kernel(const int8_t *p, int64_t rows, int64_t kp, int64_t copies,
                                                        int64_t bstride, uint32_t scale, int32_t *out)
{
    const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (row >= rows * copies) {
        return;  // no barrier below
    }
    const int64_t c = row / rows, r = row - c * rows;
    const int8_t *src = p + c * bstride + r * kp;
    int32_t sum = 0;
    // kp is a multiple of the 128-element k-tile, so whole 16-byte chunks are in bounds
    for (int64_t k = static_cast<int64_t>(lane) * 16; k < kp; k += 64 * 16) {
        const int4 v = *reinterpret_cast<const int4 *>(src + k);
        const int w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
            for (int b = 0; b < 4; ++b) sum += static_cast<int8_t>(static_cast<uint32_t>(w[j]) >> (8 * b));
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        sum += __shfl_xor(sum, o);
    }
    if (lane == 0) {
        out[c * rows + r] = static_cast<int32_t>(static_cast<uint32_t>(sum) * scale);
    }
}

template <int SRC, int DST>
void launch_vector(const PackArgs &p, int64_t batches, hipStream_t stream)
{
    constexpr int EPC = 16 / static_cast<int>(sizeof(Elem<DST>));
    if (p.s_k == 1) {
        int laneBits = 3;  // the fewest lanes that hold a packed row, up to a wave
        while (laneBits < 6 && (int64_t(EPC) << laneBits) < p.kp) {
            ++laneBits;
        }
        const int64_t rows = kRowsPerGroup / 4 * (256 >> laneBits), k = int64_t(EPC) << laneBits;
        const dim3 grid(static_cast<unsigned>((p.rows + rows - 1) / rows), static_cast<unsigned>((p.kp + k - 1) / k),
                        static_cast<unsigned>(batches));
        hipLaunchKernelGGL((pack_rows_kernel<SRC, DST>), grid, dim3(256), 0, stream, p, laneBits);
    } else {
        const dim3 grid(static_cast<unsigned>((p.rows + kTile - 1) / kTile),
                        static_cast<unsigned>((p.kp + kTile - 1) / kTile), static_cast<unsigned>(batches));
        hipLaunchKernelGGL((pack_cols_kernel<SRC, DST>), grid, dim3(256), 0, stream, p);
    }
}

}  // namespace

int kudnn_launch_rowsum_s8(const int8_t *p, int64_t rows, int64_t kp, int64_t copies, int64_t bstride, uint32_t scale,
                           int32_t *out, hipStream_t stream)
{
    if (kp % 16 != 0) {
        return -1;
    }
    const int64_t total = rows * copies;
    hipLaunchKernelGGL(rowsum_s8_kernel, dim3(static_cast<unsigned>((total + 3) / 4)), dim3(256), 0, stream, p, rows,
                       kp, copies, bstride, scale, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int kudnn_launch_pack(const PackArgs &p, int64_t batches, hipStream_t stream)
{
    // The vector kernels take the type pairs the planner makes, a source contiguous along K or along the rows, and a
    // packed pitch of whole 16-byte chunks (every k-tile is 128 bytes); a size-one dimension has stride 0, which
    // neither kernel ever steps over, so it may count as contiguous.
    const bool contiguous = p.s_k == 1 || p.s_r == 1;
    const int es = p.dst_dt == KUDNN_DT_F32 ? 4 : (p.dst_dt == KUDNN_DT_S8 ? 1 : 2);
    const int shift = p.src_dt == KUDNN_DT_U8 && p.dst_dt == KUDNN_DT_S8 ? 128 : 0;
    if (contiguous && p.kp * es % 16 == 0 && p.dst_bstride * es % 16 == 0 && p.shift == shift) {
        void (*launch)(const PackArgs &, int64_t, hipStream_t) = nullptr;
        switch (p.dst_dt * 16 + p.src_dt) {
            case KUDNN_DT_BF16 * 16 + KUDNN_DT_BF16:
            case KUDNN_DT_F16 * 16 + KUDNN_DT_F16: launch = launch_vector<KUDNN_DT_BF16, KUDNN_DT_BF16>; break;  // a copy
            case KUDNN_DT_F16 * 16 + KUDNN_DT_S8: launch = launch_vector<KUDNN_DT_S8, KUDNN_DT_F16>; break;
            case KUDNN_DT_F16 * 16 + KUDNN_DT_U8: launch = launch_vector<KUDNN_DT_U8, KUDNN_DT_F16>; break;
            case KUDNN_DT_S8 * 16 + KUDNN_DT_S8: launch = launch_vector<KUDNN_DT_S8, KUDNN_DT_S8>; break;
            case KUDNN_DT_S8 * 16 + KUDNN_DT_U8: launch = launch_vector<KUDNN_DT_U8, KUDNN_DT_S8>; break;
            case KUDNN_DT_F32 * 16 + KUDNN_DT_F32: launch = launch_vector<KUDNN_DT_F32, KUDNN_DT_F32>; break;
            case KUDNN_DT_F32 * 16 + KUDNN_DT_BF16: launch = launch_vector<KUDNN_DT_BF16, KUDNN_DT_F32>; break;
            case KUDNN_DT_F32 * 16 + KUDNN_DT_F16: launch = launch_vector<KUDNN_DT_F16, KUDNN_DT_F32>; break;
            case KUDNN_DT_F32 * 16 + KUDNN_DT_S8: launch = launch_vector<KUDNN_DT_S8, KUDNN_DT_F32>; break;
            case KUDNN_DT_F32 * 16 + KUDNN_DT_U8: launch = launch_vector<KUDNN_DT_U8, KUDNN_DT_F32>; break;
            default: break;
        }
        if (launch != nullptr) {
            launch(p, batches, stream);
            return hipGetLastError() == hipSuccess ? 0 : -1;
        }
    }
    dim3 grid(static_cast<unsigned>((p.rows + kTile - 1) / kTile), static_cast<unsigned>((p.kp + kTile - 1) / kTile),
              static_cast<unsigned>(batches));
    hipLaunchKernelGGL(pack_kernel, grid, dim3(256), 0, stream, p);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
