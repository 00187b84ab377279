// k_copy.hip -- bf16 copies of GEMM operands in workspace (gfx950): fp32
// operands of the fp32-input bf16 GEMM rounded once, ahead of the bf16-storage
// tiles, instead of by every tile that reads them (the reference rounds while
// packing, src/gemm/gemm_driver_generic.cpp with bfloat16_t packing).
#include "device_common.h"
#include "kernels.h"

using namespace dnnopt_dev;

namespace dnnopt_hip {

namespace {

constexpr int kRows = 4;   // rows of a wave's piece: 8 loads of 16 bytes in flight per lane
constexpr int kCols = 512;  // columns of a wave's piece, 8 per lane

struct CopyOperand {
    const float* src;
    uint16_t* dst;
    long long lds, ldd;
    int rows, cols;    // of the source
    int drows;         // rows of the copy (>= rows; the further ones are zero)
    int segs;          // pieces per row group
    int waves;         // pieces in all
};

// HBM-bound: 4 bytes read and 2 written per element (MI355X, 4096 x 11008:
// 41 us, 6.5 TB/s, as the best of a sweep of loads in flight and grid sizes;
// 46-50 us with a quarter of the workgroups).  One launch copies both
// operands: waves [0, a.waves) take A, the others B.
__global__ __launch_bounds__(256) void dnnopt_bf16_copy(CopyOperand a, CopyOperand b) {
    int w = (int)blockIdx.x * 4 + wave_id();
    const bool second = w >= a.waves;
    const CopyOperand& o = second ? b : a;
    if (second) w -= a.waves;
    if (w >= o.waves) return;
    const int r0 = w / o.segs * kRows, c0 = w % o.segs * kCols + 8 * lane_id();
    const int live = o.rows - r0 < kRows ? (o.rows - r0 > 0 ? o.rows - r0 : 0) : kRows;
    // Descriptor over the group's rows up to the last one's end.
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(
        o.src + (size_t)r0 * o.lds, live ? range31(((size_t)(live - 1) * o.lds + o.cols) * 4) : 0u);
    u32x4 lo[kRows], hi[kRows];
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        const uint32_t off = ((uint32_t)i * (uint32_t)o.lds + (uint32_t)c0) * 4u;
        lo[i] = buf_load_x4_stream(rs, i < live && c0 < o.cols ? off : kOobOffset);
        hi[i] = buf_load_x4_stream(rs, i < live && c0 < o.cols ? off + 16u : kOobOffset);
    }
    if (c0 >= o.ldd) return;
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
        if (r0 + i >= o.drows) break;
        u32x4 v;
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const uint32_t e0 = d < 2 ? lo[i][2 * d] : hi[i][2 * d - 4], e1 = d < 2 ? lo[i][2 * d + 1] : hi[i][2 * d - 3];
            // the padding columns of the copy are zero
            const uint32_t h0 = c0 + 2 * d < o.cols ? f32_to_bf16_bits(as_f32(e0)) : 0u;
            const uint32_t h1 = c0 + 2 * d + 1 < o.cols ? f32_to_bf16_bits(as_f32(e1)) : 0u;
            v[d] = h0 | (h1 << 16);
        }
        *reinterpret_cast<u32x4*>(o.dst + (size_t)(r0 + i) * o.ldd + c0) = v;
    }
}

CopyOperand operand(const float* src, long long lds, int rows, int cols, uint16_t* dst, long long ldd, int drows) {
    const int segs = (int)((ldd + kCols - 1) / kCols);
    return CopyOperand{src, dst, lds, ldd, rows, cols, drows, segs, (drows + kRows - 1) / kRows * segs};
}

}  // namespace

hipError_t launch_bf16_copy(const float* A, int lda, const float* B, int ldb, int M, int N, int K, uint16_t* dA,
                            int ldda, uint16_t* dB, int lddb, int dK, hipStream_t s) {
    if (ldda % 8 || ldda < K || (long long)lda * 16 >= 0x7FFFFFFFll) return hipErrorInvalidValue;
    if (dB && (lddb % 8 || lddb < N || dK < K || (long long)ldb * 16 >= 0x7FFFFFFFll)) return hipErrorInvalidValue;
    const CopyOperand a = operand(A, lda, M, K, dA, ldda, M);
    const CopyOperand b = dB ? operand(B, ldb, K, N, dB, lddb, dK) : CopyOperand{};
    const long long waves = (long long)a.waves + b.waves;
    if (waves > 0x7FFFFFF0ll) return hipErrorInvalidValue;
    hipLaunchKernelGGL(dnnopt_bf16_copy, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, a, b);
    return hipGetLastError();
}

}  // namespace dnnopt_hip
