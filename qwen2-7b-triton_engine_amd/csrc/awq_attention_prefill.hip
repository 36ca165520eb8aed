// Causal attention of a prompt's positions 0 .. S - 1 for the Qwen2 engine,
// from the fused QKV projection to the attention output: rotate-half RoPE,
// the KV cache's rows, GQA softmax attention (model/qwen2.py:104-163).
//
// What bounds it: the matrix cores.  The torch form it replaces computed the
// full S x T scores in fp32 products and passed over the [heads, S, T] scores
// in memory about eight times (matmul, scale, mask, softmax, matmul).  Here
// the scores never leave registers.  Measured on Qwen2-7B's heads (28 of 128
// over 4 KV heads), both launches: 30 us at S = 700, 68 us at 1777 (about 1.2
// ms before, in some 25 launches), 250 us at 4096 -- there 0.95 PFLOP/s through
// the MFMA, the two parts of each operand counted; a 4-layer prefill of 1777
// tokens 9.03 -> 4.36 ms.
//
// Precision.  K and V are fp16 in the cache; q after RoPE and the
// probabilities are fp32 and stay so: each is split into two fp16 parts, hi =
// fp16(x) and lo = fp16(x - hi), and both go through the fp16 MFMA with its
// fp32 sums.  hi + lo carries 23 bits while lo is above fp16's smallest
// steps (2^-24), so both operands are scaled first: a query row by the power
// of two that brings its largest value to 2^14 .. 2^15 (RoPE makes up to 65504
// sqrt(2) of fp16 values, more than fp16 holds), the probabilities, at most
// 1, by 2^14.  Such scales cancel exactly.  log2(e) / sqrt(HD) is no power of
// two and multiplies the difference of a score and the maximum, in fp32: the
// scores reach 3e10, where the product's own rounding would be thousands.
// Outputs that land on another fp16 value than the 64-bit result's, per
// thousand, here / in plain fp32 attention (28 heads of 128, S = 1777): 1.1 /
// 1.9, 1.9 / 3.3, 4.3 / 7.0 for queries and keys of standard deviation 0.3, 1, 2.
#include "awq_kernels.h"

namespace awq {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = 4;
constexpr int kKeys = 64;           // keys per tile
constexpr int kPExp = 14;           // the probabilities' scale before they are split: 2^14

// Position of a key within its 64-key tile of the transposed V: the S^T
// product leaves lane group t (lanes 16 t ..) with keys 4 t .. 4 t + 3 of each
// 16-key block, and the P V product wants 8 consecutive k per lane, so 8
// consecutive places hold keys 4 t .. 4 t + 3 of two neighbouring blocks.
// key_of_place is a bijection of 0 .. 63.
__device__ __forceinline__ int key_of_place(int place) {
    const int half = place >> 5, t = (place >> 3) & 3, j = place & 7;
    return 32 * half + 16 * (j >> 2) + 4 * t + (j & 3);
}

// Swizzle of the 16-byte chunks of a tile row in LDS: rows a power of two
// bytes apart start on the same bank, and 16 rows' same chunk is what one
// MFMA operand read fetches.
template <int CHUNKS>
__device__ __forceinline__ int swizzled(int row, int chunk) {
    return chunk ^ (row & (CHUNKS < 16 ? CHUNKS - 1 : 15));
}

// Keys and values of 64 positions of one KV head: RoPE and the cache rows,
// and V transposed into the tile image that the attention kernel copies to
// LDS (vt: [kvh][tiles][HD][64], places permuted and chunks swizzled as
// above, zeros past the prompt).
template <int HD>
__global__ __launch_bounds__(kThreads) void awq_prefill_kv_kernel(const half_t* __restrict__ qkv,
                                                                  half_t* __restrict__ kc, half_t* __restrict__ vc,
                                                                  const float* __restrict__ cosp,
                                                                  const float* __restrict__ sinp,
                                                                  half_t* __restrict__ vt, int S, int nh, int kvh,
                                                                  int max_seq) {
    constexpr int kChunks = HD / 8;
    constexpr int kStride = HD + 8;   // halfs per LDS row
    __shared__ __align__(16) half_t lv[kKeys * kStride];
    const int tile = blockIdx.x, g = blockIdx.y;
    const size_t ld = (size_t)(nh + 2 * kvh) * HD;
    for (int i = threadIdx.x; i < kKeys * kChunks; i += kThreads) {
        const int row = i / kChunks, d0 = 8 * (i % kChunks);
        const int pos = tile * kKeys + row;
        half8_t v = {};
        if (pos < S) {
            const half_t* src = qkv + (size_t)pos * ld + (size_t)(nh + g) * HD;
            const bool low = d0 < HD / 2;
            const half8_t a = *reinterpret_cast<const half8_t*>(src + d0);
            const half8_t b = *reinterpret_cast<const half8_t*>(src + (low ? d0 + HD / 2 : d0 - HD / 2));
            const floatx4* c = reinterpret_cast<const floatx4*>(cosp + (size_t)pos * HD + d0);
            const floatx4* s = reinterpret_cast<const floatx4*>(sinp + (size_t)pos * HD + d0);
            half8_t k;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float p = (float)b[e];
                k[e] = (half_t)((float)a[e] * c[e / 4][e % 4] + (low ? -p : p) * s[e / 4][e % 4]);
            }
            v = *reinterpret_cast<const half8_t*>(src + (size_t)kvh * HD + d0);
            const size_t dst = ((size_t)g * max_seq + pos) * HD + d0;
            *reinterpret_cast<half8_t*>(kc + dst) = k;
            *reinterpret_cast<half8_t*>(vc + dst) = v;
        }
        *reinterpret_cast<half8_t*>(lv + row * kStride + d0) = v;
    }
    __syncthreads();
    half_t* dst = vt + ((size_t)g * gridDim.x + tile) * kKeys * HD;
    for (int i = threadIdx.x; i < HD * 8; i += kThreads) {
        const int d = i >> 3, chunk = swizzled<8>(d, i & 7);
        half8_t v;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = lv[key_of_place(8 * chunk + j) * kStride + d];
        *reinterpret_cast<half8_t*>(dst + 8 * i) = v;
    }
}

// One workgroup: 64 NQ queries of one head, 16 NQ per wave, over the 64-key
// tiles up to its last query.  S^T = K Q^T puts a query in each MFMA column,
// so a query's running maximum and sum are one value per lane column, and the
// exponentials are already laid out as the B operand of O^T = V^T P^T: no
// transposition and no LDS pass between the two products.  K and V tiles are
// double-buffered in LDS by direct loads, the next tile's issued before this
// one is computed.
template <int HD, int NQ>
__global__ __launch_bounds__(kThreads, 2) void awq_prefill_attn_kernel(
    const half_t* __restrict__ qkv, const half_t* __restrict__ kc, const half_t* __restrict__ vt,
    const float* __restrict__ cosp, const float* __restrict__ sinp, half_t* __restrict__ out, int S, int nh, int kvh,
    int max_seq) {
    constexpr int kSteps = HD / 32;       // MFMA k-steps of a q.k product
    constexpr int kDb = HD / 16;          // 16-column blocks of the output
    constexpr int kChunks = HD / 8;
    constexpr int kTile = kKeys * HD;     // halfs of a K or V tile
    constexpr int kLoads = kTile * 2 / 1024 / kWaves;
    __shared__ __align__(1024) half_t lds[4 * kTile];   // K0 V0 K1 V1

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, t = lane >> 4;
    const int tiles_q = (S + 64 * NQ - 1) / (64 * NQ);
    const int head = blockIdx.x % nh;
    const int qt = tiles_q - 1 - (int)blockIdx.x / nh;   // the longest key ranges start first
    const int g = head / (nh / kvh);
    const int q0 = qt * 64 * NQ + wave * 16 * NQ;        // this wave's first query
    const int last = qt * 64 * NQ + 64 * NQ - 1 < S - 1 ? qt * 64 * NQ + 64 * NQ - 1 : S - 1;
    const int tiles = last / kKeys + 1;
    const int tiles_all = (S + kKeys - 1) / kKeys;

    const u32x4 rk = raw_rsrc(kc + (size_t)g * max_seq * HD, (uint32_t)S * HD * 2u);
    const u32x4 rv = raw_rsrc(vt + (size_t)g * tiles_all * kTile, (uint32_t)tiles_all * kTile * 2u);
    uint32_t kofs[kLoads];   // byte offset within a K tile of this lane's 16 bytes
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int slot = (wave * kLoads + i) * 64 + lane;
        const int row = slot / kChunks;
        kofs[i] = (uint32_t)(row * HD * 2 + 16 * swizzled<kChunks>(row, slot % kChunks));
    }
    auto issue = [&](int tile, int buf) {
        const uint32_t base = lds_addr(lds + 2 * buf * kTile);
        const uint32_t gofs = (uint32_t)tile * (uint32_t)(kTile * 2);
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const uint32_t dst = (uint32_t)(wave * kLoads + i) * 1024u;
            buffer_load_lds_x4(rk, gofs + kofs[i], 0, base + dst);
            buffer_load_lds_x4(rv, gofs + dst + 16u * lane, 0, base + kTile * 2 + dst);
        }
    };
    issue(0, 0);

    half8_t qhi[NQ][kSteps], qlo[NQ][kSteps];
    float unit[NQ];            // exp(x / sqrt(HD)) = exp2(score * unit)
    {
        const size_t ld = (size_t)(nh + 2 * kvh) * HD;
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
            const int q = q0 + 16 * n + col < S ? q0 + 16 * n + col : S - 1;
            const half_t* src = qkv + (size_t)q * ld + (size_t)head * HD + 8 * t;
            half8_t raw[kSteps];
#pragma unroll
            for (int st = 0; st < kSteps; ++st) raw[st] = *reinterpret_cast<const half8_t*>(src + 32 * st);
            float x[kSteps][8], mx = 0.0f;
#pragma unroll
            for (int st = 0; st < kSteps; ++st) {
                const bool low = st < kSteps / 2;
                const half8_t b = raw[low ? st + kSteps / 2 : st - kSteps / 2];
                const floatx4* c = reinterpret_cast<const floatx4*>(cosp + (size_t)q * HD + 32 * st + 8 * t);
                const floatx4* s = reinterpret_cast<const floatx4*>(sinp + (size_t)q * HD + 32 * st + 8 * t);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float p = (float)b[e];
                    x[st][e] = (float)raw[st][e] * c[e / 4][e % 4] + (low ? -p : p) * s[e / 4][e % 4];
                    mx = fmaxf(mx, fabsf(x[st][e]));
                }
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const int exp = split16_exp(mx);
            unit[n] = __builtin_ldexpf(1.4426950408889634f / sqrtf((float)HD), -exp);
#pragma unroll
            for (int st = 0; st < kSteps; ++st) split16(x[st], exp, qhi[n][st], qlo[n][st]);
        }
    }

    float m[NQ], l[NQ];        // running maximum (of the scaled scores) and this lane's share of the sum
    floatx4 acc[NQ][kDb];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        m[n] = -INFINITY;
        l[n] = 0.0f;
#pragma unroll
        for (int d = 0; d < kDb; ++d) acc[n][d] = floatx4{0.f, 0.f, 0.f, 0.f};
    }

    for (int tile = 0; tile < tiles; ++tile) {
        // This wave's loads of the tile have landed; after the barrier every
        // wave's have, and no wave still reads the other buffer.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tile + 1 < tiles) issue(tile + 1, (tile + 1) & 1);
        const int key0 = tile * kKeys;
        if (key0 > q0 + 16 * NQ - 1) continue;   // past every query of this wave (its last tiles only)
        const half_t* lk = lds + 2 * (tile & 1) * kTile;
        const half_t* lv = lk + kTile;

        floatx4 s[NQ][4];
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
            const int row = 16 * kb + col;
#pragma unroll
            for (int n = 0; n < NQ; ++n) s[n][kb] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < kSteps; ++st) {
                const half8_t a =
                    *reinterpret_cast<const half8_t*>(lk + row * HD + 8 * swizzled<kChunks>(row, 4 * st + t));
#pragma unroll
                for (int n = 0; n < NQ; ++n) {
                    s[n][kb] = mfma16x16x32(a, qhi[n][st], s[n][kb]);
                    s[n][kb] = mfma16x16x32(a, qlo[n][st], s[n][kb]);
                }
            }
        }
        if (key0 + kKeys - 1 > q0) {   // the diagonal
#pragma unroll
            for (int n = 0; n < NQ; ++n)
#pragma unroll
                for (int kb = 0; kb < 4; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (key0 + 16 * kb + 4 * t + r > q0 + 16 * n + col) s[n][kb][r] = -INFINITY;
        }
        half8_t phi[NQ][2], plo[NQ][2];
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
            float mx = s[n][0][0];
#pragma unroll
            for (int kb = 0; kb < 4; ++kb)
#pragma unroll
                for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[n][kb][r]);
            mx = fmaxf(mx, __shfl_xor(mx, 16));
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const float mn = fmaxf(m[n], mx);
            const float ref = mn == -INFINITY ? 0.0f : mn;   // nothing yet: every exponential is 0
            if (__any(mn > m[n])) {
                const float alpha = __builtin_amdgcn_exp2f((m[n] - ref) * unit[n]);
                l[n] *= alpha;
#pragma unroll
                for (int d = 0; d < kDb; ++d) acc[n][d] *= alpha;
            }
            m[n] = mn;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float p[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    p[j] = __builtin_amdgcn_exp2f((s[n][2 * h + (j >> 2)][j & 3] - ref) * unit[n]);
                    l[n] += p[j];
                }
                split16(p, kPExp, phi[n][h], plo[n][h]);
            }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int d = 0; d < kDb; ++d) {
                const int row = 16 * d + col;
                const half8_t a =
                    *reinterpret_cast<const half8_t*>(lv + row * kKeys + 8 * swizzled<8>(row, 4 * h + t));
#pragma unroll
                for (int n = 0; n < NQ; ++n) {
                    acc[n][d] = mfma16x16x32(a, phi[n][h], acc[n][d]);
                    acc[n][d] = mfma16x16x32(a, plo[n][h], acc[n][d]);
                }
            }
    }

#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        float sum = l[n];
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        sum = __builtin_ldexpf(sum, kPExp);
        const int q = q0 + 16 * n + col;
        if (q >= S) continue;
        half_t* dst = out + ((size_t)q * nh + head) * HD + 4 * t;
#pragma unroll
        for (int d = 0; d < kDb; ++d) {
            half4_t o;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = (half_t)(acc[n][d][r] / sum);
            *reinterpret_cast<half4_t*>(dst + 16 * d) = o;
        }
    }
}

template <int HD>
hipError_t launch(const PrefillAttnArgs& a, int cus, hipStream_t stream) {
    const int tiles = (a.S + kKeys - 1) / kKeys;
    hipLaunchKernelGGL((awq_prefill_kv_kernel<HD>), dim3(tiles, a.kvh), dim3(kThreads), 0, stream, a.qkv, a.k_cache,
                       a.v_cache, a.cos, a.sin, a.vt, a.S, a.nh, a.kvh, a.max_seq);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // Two 16-query blocks per wave read K and V from LDS half as often, one
    // makes twice the workgroups.  A causal grid is uneven (the last query
    // tile has all the keys) and two workgroups share a CU, so the wide tile
    // needs at least three workgroups per CU to win.  28 heads of 128 over 4
    // KV heads, both launches, us narrow / wide: S = 700 30 / 38, 1200 43 / 58, 1777
    // 68 / 81, 4096 256 / 250.
    const int64_t wide = (int64_t)((a.S + 127) / 128) * a.nh, narrow = (int64_t)tiles * a.nh;
    if (wide >= 3 * cus)
        hipLaunchKernelGGL((awq_prefill_attn_kernel<HD, 2>), dim3((unsigned)wide), dim3(kThreads), 0, stream, a.qkv,
                           a.k_cache, a.vt, a.cos, a.sin, a.out, a.S, a.nh, a.kvh, a.max_seq);
    else
        hipLaunchKernelGGL((awq_prefill_attn_kernel<HD, 1>), dim3((unsigned)narrow), dim3(kThreads), 0, stream, a.qkv,
                           a.k_cache, a.vt, a.cos, a.sin, a.out, a.S, a.nh, a.kvh, a.max_seq);
    return hipGetLastError();
}

}  // namespace

size_t prefill_attn_workspace(int S, int kvh, int hd) {
    return (size_t)((S + kKeys - 1) / kKeys) * kKeys * kvh * hd * sizeof(half_t);
}

hipError_t launch_prefill_attn(const PrefillAttnArgs& a, int hd, int cus, hipStream_t stream) {
    if (a.S == 0) return hipSuccess;
    return hd == 64 ? launch<64>(a, cus, stream) : launch<128>(a, cus, stream);
}

}  // namespace awq
