// Decode attention of the Qwen2 engine: one new position against a static KV
// cache, from the fused QKV projection to the attention output
// (model/qwen2.py:104-163: rotate-half RoPE, cache update, GQA softmax
// attention).  fp16 operands, every product and sum in fp32; q stays fp32
// after RoPE, the probabilities stay fp32.
//
// What bounds it: latency.  A thousand positions of 4 KV heads are 2 MB, a
// third of a microsecond of HBM time; the torch form of the same step read
// the whole static cache several times through about 25 launches of 2 - 5 us.
// Here it is two launches: the cache is split along its positions over
// enough workgroups to load it at once, each keeps a running softmax of its
// range for all query heads of one KV head (so K and V are read once), and a
// second launch weights the ranges' partial sums.  Measured on Qwen2-7B: a
// 1024-token prompt and 48 greedy tokens, 28 layers, cache of 1152 positions,
// 301 -> 190 ms (2.3 ms less per token); eight eager steps of a 4-layer stack
// at position 900 of 2048, 13.9 -> 6.9 ms.
#include "awq_kernels.h"

namespace awq {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kKeys = 64;   // positions of one inner pass of a workgroup: 16 per wave

// Sum over aligned groups of 16 (8) lanes, left in every lane: rotations
// within a 16-lane DPP row (within its halves: mirror, quad permutations).
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
template <int LANES>
__device__ __forceinline__ float group_sum(float v) {
    v += dpp<0xB1>(v);    // quad_perm [1,0,3,2]
    v += dpp<0x4E>(v);    // quad_perm [2,3,0,1]
    v += dpp<0x141>(v);   // row_half_mirror: lane i <-> 7 - i
    if (LANES == 16) v += dpp<0x140>(v);   // row_mirror: lane i <-> 15 - i
    return v;
}

__device__ __forceinline__ float rope(float x, float partner, float c, float s, bool low) {
    return x * c + (low ? -partner : partner) * s;
}

// One workgroup: positions [split * chunk, ...) of one KV head for up to G
// query heads.  Within an inner pass of 64 positions each wave owns 16: its
// 16-lane (head size 64: 8-lane) groups each read one K row per load, 16 bytes
// a lane, and reduce the dot products within the group; the wave's own 16
// positions then go through its running softmax and its P V product, where
// a lane owns HD / 64 columns of V.  The four waves' results meet once, at
// the end.
template <int HD, int G>
__global__ __launch_bounds__(kThreads) void awq_decode_attn_kernel(
    const half_t* __restrict__ qkv, half_t* __restrict__ kc, half_t* __restrict__ vc, const float* __restrict__ cosp,
    const float* __restrict__ sinp, const int64_t* __restrict__ posp, float* __restrict__ part, int nh, int kvh,
    int groups, int max_seq, int chunk) {
    constexpr int kLpk = HD / 8;            // lanes per K row
    constexpr int kRows = 64 / kLpk;        // K rows per load of a wave
    constexpr int kPass = 16 / kRows;       // loads per 16 positions
    constexpr int kVc = HD / 64;            // V columns per lane
    typedef half_t vcols_t __attribute__((ext_vector_type(kVc)));
    __shared__ __align__(16) float p_lds[kWaves][16][G];
    __shared__ float m_lds[kWaves][G], l_lds[kWaves][G];
    __shared__ float o_lds[kWaves][G][HD];

    const int64_t pos64 = *posp;
    const int split = blockIdx.x, g = blockIdx.y;
    const int h0 = blockIdx.z * G;                       // first query head of this block within the group
    const int heads = groups - h0 < G ? groups - h0 : G;
    if (pos64 < 0 || pos64 >= max_seq || (int64_t)split * chunk > pos64) return;
    const int pos = (int)pos64;
    const int start = split * chunk;
    const int end = start + chunk < pos + 1 ? start + chunk : pos + 1;

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int sub = lane % kLpk, kr = lane / kLpk;
    const int d0 = 8 * sub, dp = d0 < HD / 2 ? d0 + HD / 2 : d0 - HD / 2;
    const bool low = d0 < HD / 2;
    half_t* kbase = kc + (size_t)g * max_seq * HD;
    half_t* vbase = vc + (size_t)g * max_seq * HD;
    const half_t* knew = qkv + (size_t)nh * HD + (size_t)g * HD;
    const half_t* vnew = knew + (size_t)kvh * HD;

    half8_t kraw[kPass];
    float vraw[16][kVc];
    auto load = [&](int first) {   // rows past the last position are not read
#pragma unroll
        for (int i = 0; i < kPass; ++i) {
            const int key = first + 16 * wave + i * kRows + kr;
            kraw[i] = half8_t{};
            if (key < end && key != pos) kraw[i] = *reinterpret_cast<const half8_t*>(kbase + (size_t)key * HD + d0);
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int key = first + 16 * wave + j;
            const half_t* row = (key == pos ? vnew : vbase + (size_t)key * HD) + kVc * lane;
            vcols_t v = {};
            if (key < end) v = *reinterpret_cast<const vcols_t*>(row);
#pragma unroll
            for (int c = 0; c < kVc; ++c) vraw[j][c] = (float)v[c];
        }
    };
    load(start);

    // RoPE of this lane's 8 columns of the query heads and of the new key.
    float cs[8], sn[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        cs[e] = cosp[(size_t)pos * HD + d0 + e];
        sn[e] = sinp[(size_t)pos * HD + d0 + e];
    }
    float q[G][8];
#pragma unroll
    for (int h = 0; h < G; ++h) {
        const half_t* qh = qkv + (size_t)(g * groups + h0 + (h < heads ? h : 0)) * HD;
        const half8_t a = *reinterpret_cast<const half8_t*>(qh + d0);
        const half8_t b = *reinterpret_cast<const half8_t*>(qh + dp);
#pragma unroll
        for (int e = 0; e < 8; ++e) q[h][e] = rope((float)a[e], (float)b[e], cs[e], sn[e], low);
    }
    half8_t kn;
    {
        const half8_t a = *reinterpret_cast<const half8_t*>(knew + d0);
        const half8_t b = *reinterpret_cast<const half8_t*>(knew + dp);
#pragma unroll
        for (int e = 0; e < 8; ++e) kn[e] = (half_t)rope((float)a[e], (float)b[e], cs[e], sn[e], low);
    }
    if (end == pos + 1 && blockIdx.z == 0 && threadIdx.x < kLpk) {   // the cache's new row
        *reinterpret_cast<half8_t*>(kbase + (size_t)pos * HD + d0) = kn;
        *reinterpret_cast<half8_t*>(vbase + (size_t)pos * HD + d0) = *reinterpret_cast<const half8_t*>(vnew + d0);
    }

    // exp(x / sqrt(HD) - max) = exp2(x c - max c)
    const float c2 = 1.4426950408889634f / sqrtf((float)HD);
    float m[G], l[G], o[G][kVc];
#pragma unroll
    for (int h = 0; h < G; ++h) {
        m[h] = -INFINITY;
        l[h] = 0.0f;
#pragma unroll
        for (int c = 0; c < kVc; ++c) o[h][c] = 0.0f;
    }

    for (int first = start; first < end; first += kKeys) {
        if (first != start) load(first);
        float s[kPass][G];
#pragma unroll
        for (int i = 0; i < kPass; ++i) {
            const int key = first + 16 * wave + i * kRows + kr;
            const half8_t kv = key == pos ? kn : kraw[i];
#pragma unroll
            for (int h = 0; h < G; ++h) {
                float a = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) a = fmaf((float)kv[e], q[h][e], a);
                a = group_sum<kLpk>(a) * c2;
                s[i][h] = key < end ? a : -INFINITY;
            }
        }
#pragma unroll
        for (int h = 0; h < G; ++h) {
            float mx = s[0][h];
#pragma unroll
            for (int i = 1; i < kPass; ++i) mx = fmaxf(mx, s[i][h]);
#pragma unroll
            for (int w = kLpk; w < 64; w *= 2) mx = fmaxf(mx, __shfl_xor(mx, w));
            const float mn = fmaxf(m[h], mx);
            const float ref = mn == -INFINITY ? 0.0f : mn;   // nothing yet: every exponential is 0
            const float alpha = __builtin_amdgcn_exp2f(m[h] - ref);
            float sum = 0.0f;
#pragma unroll
            for (int i = 0; i < kPass; ++i) {
                const float p = __builtin_amdgcn_exp2f(s[i][h] - ref);
                if (sub == 0) p_lds[wave][i * kRows + kr][h] = p;
                sum += p;
            }
#pragma unroll
            for (int w = kLpk; w < 64; w *= 2) sum += __shfl_xor(sum, w);
            m[h] = mn;
            l[h] = l[h] * alpha + sum;
#pragma unroll
            for (int c = 0; c < kVc; ++c) o[h][c] *= alpha;
        }
        __builtin_amdgcn_wave_barrier();   // p_lds[wave] is written and read by this wave only, in order
#pragma unroll
        for (int j = 0; j < 16; ++j)
#pragma unroll
            for (int h = 0; h < G; ++h) {
                const float p = p_lds[wave][j][h];
#pragma unroll
                for (int c = 0; c < kVc; ++c) o[h][c] = fmaf(p, vraw[j][c], o[h][c]);
            }
        __builtin_amdgcn_wave_barrier();
    }

#pragma unroll
    for (int h = 0; h < G; ++h) {
        if (lane == 0) {
            m_lds[wave][h] = m[h];
            l_lds[wave][h] = l[h];
        }
#pragma unroll
        for (int c = 0; c < kVc; ++c) o_lds[wave][h][kVc * lane + c] = o[h][c];
    }
    __syncthreads();
    // part: [split][head][HD + 2]: HD sums, the maximum, the sum of exponentials
    for (int i = threadIdx.x; i < heads * HD; i += kThreads) {
        const int h = i / HD, d = i - h * HD;
        float mx = m_lds[0][h];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) mx = fmaxf(mx, m_lds[w][h]);
        const float ref = mx == -INFINITY ? 0.0f : mx;
        float sum = 0.0f, ls = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float a = __builtin_amdgcn_exp2f(m_lds[w][h] - ref);
            sum = fmaf(a, o_lds[w][h][d], sum);
            ls = fmaf(a, l_lds[w][h], ls);
        }
        float* dst = part + ((size_t)split * nh + g * groups + h0 + h) * (HD + 2);
        dst[d] = sum;
        if (d == 0) {
            dst[HD] = mx;
            dst[HD + 1] = ls;
        }
    }
}

// out[head] = sum of the live ranges' partial sums, each weighted by
// exp2(its maximum - the overall maximum).  One workgroup per head; lane i of
// each wave holds range i's weight (at most kMaxRanges = 64 ranges); four
// threads share an output column's ranges, eight loads in flight each.
template <int HD>
__global__ __launch_bounds__(4 * HD) void awq_decode_combine_kernel(const float* __restrict__ part,
                                                                    const int64_t* __restrict__ posp,
                                                                    half_t* __restrict__ out, int nh, int max_seq,
                                                                    int chunk) {
    __shared__ float o_lds[4][HD];
    const int64_t pos = *posp;
    if (pos < 0 || pos >= max_seq) return;
    const int n = (int)(pos / chunk) + 1;
    const int head = blockIdx.x, d = threadIdx.x % HD, quarter = threadIdx.x / HD, lane = threadIdx.x & 63;
    const size_t step = (size_t)nh * (HD + 2);
    const float* base = part + (size_t)head * (HD + 2);
    const float mine = lane < n ? base[lane * step + HD] : -INFINITY;
    float l = lane < n ? base[lane * step + HD + 1] : 0.0f;
    float mx = mine;
#pragma unroll
    for (int w = 1; w < 64; w *= 2) mx = fmaxf(mx, __shfl_xor(mx, w));
    const float a = __builtin_amdgcn_exp2f(mine - (mx == -INFINITY ? 0.0f : mx));
    l *= a;
#pragma unroll
    for (int w = 1; w < 64; w *= 2) l += __shfl_xor(l, w);
    float sum = 0.0f;
    for (int i0 = quarter; i0 < n; i0 += 32) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = i0 + 4 * j < n ? base[(i0 + 4 * j) * step + d] : 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j)   // lanes past n hold weight 0
            sum = fmaf(__shfl(a, (i0 + 4 * j) & 63), v[j], sum);
    }
    o_lds[quarter][d] = sum;
    __syncthreads();
    if (quarter == 0)
        out[(size_t)head * HD + d] = (half_t)((o_lds[0][d] + o_lds[1][d] + o_lds[2][d] + o_lds[3][d]) / l);
}

// Ranges of a cache of max_seq positions: 64 positions each, at most 64
// ranges (longer caches take a multiple of 64 positions per range).
constexpr int kMaxRanges = 64;
int chunk_for(int64_t max_seq) { return (int)(kKeys * ((max_seq + kMaxRanges * kKeys - 1) / (kMaxRanges * kKeys))); }

template <int HD, int G>
hipError_t launch(const DecodeAttnArgs& a, hipStream_t stream) {
    const int groups = a.nh / a.kvh, chunk = chunk_for(a.max_seq);
    const int splits = (a.max_seq + chunk - 1) / chunk;
    hipLaunchKernelGGL((awq_decode_attn_kernel<HD, G>), dim3(splits, a.kvh, (groups + G - 1) / G), dim3(kThreads), 0,
                       stream, a.qkv, a.k_cache, a.v_cache, a.cos, a.sin, a.pos, a.part, a.nh, a.kvh, groups,
                       a.max_seq, chunk);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((awq_decode_combine_kernel<HD>), dim3(a.nh), dim3(4 * HD), 0, stream, a.part, a.pos, a.out,
                       a.nh, a.max_seq, chunk);
    return hipGetLastError();
}

// Query heads per workgroup: all of a KV head's up to 8 (K and V are then
// read once), the smallest instance that holds them.
template <int HD>
hipError_t launch_hd(const DecodeAttnArgs& a, hipStream_t stream) {
    const int groups = a.nh / a.kvh;
    if (groups == 1) return launch<HD, 1>(a, stream);
    if (groups == 2) return launch<HD, 2>(a, stream);
    if (groups <= 4) return launch<HD, 4>(a, stream);
    return launch<HD, 8>(a, stream);
}

}  // namespace

size_t decode_attn_workspace(int max_seq, int nh, int hd) {
    const int chunk = chunk_for(max_seq);
    return (size_t)((max_seq + chunk - 1) / chunk) * nh * (hd + 2) * sizeof(float);
}

hipError_t launch_decode_attn(const DecodeAttnArgs& a, int hd, hipStream_t stream) {
    return hd == 64 ? launch_hd<64>(a, stream) : launch_hd<128>(a, stream);
}

}  // namespace awq
