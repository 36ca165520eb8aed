// SiLU * up over the fused gate||up projection: out[m, i] = fp16(silu(g) *
// u) with g = gate_up[m, i], u = gate_up[m, I + i], computed in fp32 --
// the reference's kernels/silu_mul.py:17-39 (x * sigmoid(x) * y in fp32,
// one rounding), reading the fused output in place instead of its two
// .contiguous() copies (model/qwen2.py:187-194): one pass, 6 bytes read and
// 2 written per output.  Each thread handles 8 consecutive outputs with
// 16-byte loads and stores (I % 8 == 0).
#include "awq_kernels.h"

namespace awq {
namespace {

// Bound by memory: at 1021 x 18944 116 MB, 18.7 us at 6.2 TB/s (inputs and
// outputs of repeated calls lie partly in the last-level cache), as long as the
// vector unit takes no longer.  With a 64-bit division per piece and the
// compiler's correctly rounded one per output it did: 23.3 us there; 19.6 with
// that division alone, 19.0 as it is, 18.6 with the bare reciprocal (silu_mul).
__global__ __launch_bounds__(256) void awq_silu_mul_kernel(const half_t* __restrict__ gu, half_t* __restrict__ out,
                                                           uint32_t items, uint32_t per_row, uint32_t inv) {
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t >= items) return;
    uint32_t piece;
    const uint32_t m = div_by(t, per_row, inv, piece);
    const half8_t* row = reinterpret_cast<const half8_t*>(gu) + (size_t)m * 2 * per_row;
    const half8_t g = row[piece];
    const half8_t u = row[per_row + piece];
    half8_t o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (half_t)silu_mul((float)g[e], (float)u[e]);
    reinterpret_cast<half8_t*>(out)[t] = o;
}

}  // namespace

hipError_t launch_silu_mul(const half_t* gate_up, half_t* out, int M, int I, hipStream_t stream) {
    if (M == 0) return hipSuccess;
    const uint32_t items = (uint32_t)((int64_t)M * (I / 8));  // below 2^27: the entry point bounds the operand
    hipLaunchKernelGGL(awq_silu_mul_kernel, dim3((items + 255) / 256), dim3(256), 0, stream, gate_up, out, items,
                       (uint32_t)(I / 8), div_inverse((uint32_t)(I / 8)));
    return hipGetLastError();
}

}  // namespace awq
