// Decode attention of the Qwen2 engine: one new position against a static KV
// cache, from the fused QKV projection to the attention output
// (model/qwen2.py:104-163: rotate-half RoPE, cache update, GQA softmax
// attention).  q after RoPE and the probabilities are fp32 values, split in
// two fp16 parts for the matrix cores, summed in fp32.  Outputs that land on
// another fp16 value than the 64-bit result's, per thousand, here / in plain
// fp32 attention (28 heads of 128, 1777 positions): 0.6 / 2.0, 1.3 / 2.6, 3.6 /
// 3.9 for queries and keys of standard deviation 0.3, 1, 2.
//
// What bounds it: latency.  A thousand positions of 4 KV heads are 2 MB, a
// third of a microsecond of HBM time; the torch form of the same step read
// the whole static cache several times through about 25 launches of 2 - 5 us.
// Here it is two launches: the cache is split along its positions over
// enough workgroups to load it at once, each keeps a running softmax of its
// range for all query heads of one KV head (so K and V are read once), and a
// second launch weights the ranges' partial sums.  Measured on Qwen2-7B's
// heads (28 of 128 over 4 KV heads, cache of 1152), graph replays: 8.7 us for
// the two at position 1100, where two small launches take 4; 10.2 with eight
// waves a workgroup (two per SIMD: the kernel is then bound by its own
// instructions) and its loads behind the position's; 17 with the scores, the
// softmax and P V on the vector unit, 16 lanes a key.
#include "awq_kernels.h"

namespace awq {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kHeads = 16;             // query heads of one workgroup: the columns of an MFMA
constexpr int kKeys = 16 * kWaves;     // positions of one inner pass of a workgroup: 16 per wave
constexpr int kPExp = 14;              // the probabilities' scale before they are split: 2^14

// exp(x / sqrt(HD)) = exp2(x exp2_factor)
template <int HD>
__device__ __forceinline__ float exp2_factor() {
    return 1.4426950408889634f / sqrtf((float)HD);
}

// One workgroup: positions [split * chunk, ...) of one KV head for up to 16
// query heads, 16 positions per wave and pass.  S^T = K Q^T on the MFMA: its
// columns are the heads, so one exponential covers four positions of every
// head, and the result is already the B operand of O^T = V^T P^T (16x16x16).
// V's row order in that product is free, so lane i takes columns i VC ..
// i VC + VC - 1 of a V row with one load and supplies one of them to each of
// VC products.  q and the probabilities are fp32 values split in two fp16
// parts, q scaled by its head's largest value and the probabilities by 2^14.
// Every exponent is a difference of two scores first: scores reach 3e10, and
// what they are rounded to on the way must be the same wherever two meet.
// K, V and q are loaded before the position is known (rows of the cache past
// it are masked), so the chain is two memory latencies long: the position,
// then the RoPE row it selects.  The waves' results meet once, at the end.
//
// LONG: ranges of several passes.  Their workgroups past the position return
// at once; a short range's go on (every position masked, nothing stored)
// instead of keeping all loads behind the position's.
template <int HD, bool LONG>
__global__ __launch_bounds__(kThreads) void awq_decode_attn_kernel(
    const half_t* __restrict__ qkv, half_t* kc, half_t* vc, const float* __restrict__ cosp,
    const float* __restrict__ sinp, const int64_t* __restrict__ posp, float* __restrict__ part, int nh, int kvh,
    int groups, int max_seq, int chunk) {
    constexpr int kSteps = HD / 32;
    constexpr int VC = HD / 16;            // V columns per lane
    constexpr int kStride = HD + 4;        // floats per head of the reduction buffer
    typedef half_t vcols_t __attribute__((ext_vector_type(VC)));
    __shared__ float m_lds[kWaves][kHeads], l_lds[kWaves][kHeads];
    __shared__ __align__(16) float o_lds[kWaves][kHeads][kStride];

    const int split = blockIdx.x, g = blockIdx.y;
    const int h0 = blockIdx.z * kHeads;    // first query head of this block within the group
    const int heads = groups - h0 < kHeads ? groups - h0 : kHeads;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, t = lane >> 4;
    const int start = split * chunk;
    const int64_t pos64 = *posp;

    half_t* kbase = kc + (size_t)g * max_seq * HD;
    half_t* vbase = vc + (size_t)g * max_seq * HD;
    const half_t* qh = qkv + (size_t)(g * groups + h0 + (col < heads ? col : 0)) * HD;
    const half_t* knew = qkv + (size_t)(nh + g) * HD;
    const half_t* vnew = knew + (size_t)kvh * HD;
    half8_t kf[kSteps];
    vcols_t vf[4];
    auto load = [&](int first) {
        const int krow = first + 16 * wave + col;
        const half_t* ks = kbase + (size_t)(krow < max_seq ? krow : max_seq - 1) * HD + 8 * t;
#pragma unroll
        for (int st = 0; st < kSteps; ++st) kf[st] = *reinterpret_cast<const half8_t*>(ks + 32 * st);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int vrow = first + 16 * wave + 4 * t + j;
            vf[j] = *reinterpret_cast<const vcols_t*>(vbase + (size_t)(vrow < max_seq ? vrow : max_seq - 1) * HD +
                                                      VC * col);
        }
    };
    if (LONG && start > pos64) return;
    load(start);
    half8_t qraw[kSteps], kraw[kSteps];
#pragma unroll
    for (int st = 0; st < kSteps; ++st) qraw[st] = *reinterpret_cast<const half8_t*>(qh + 32 * st + 8 * t);
#pragma unroll
    for (int st = 0; st < kSteps; ++st) kraw[st] = *reinterpret_cast<const half8_t*>(knew + 32 * st + 8 * t);
    const vcols_t vrow_new = *reinterpret_cast<const vcols_t*>(vnew + VC * col);

    const bool valid = pos64 >= 0 && pos64 < max_seq;
    const int pos = valid ? (int)pos64 : 0;
    const int end = start + chunk < pos + 1 ? start + chunk : pos + 1;
    floatx4 cs[kSteps][2], sn[kSteps][2];
#pragma unroll
    for (int st = 0; st < kSteps; ++st)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            cs[st][e] = reinterpret_cast<const floatx4*>(cosp + (size_t)pos * HD + 32 * st + 8 * t)[e];
            sn[st][e] = reinterpret_cast<const floatx4*>(sinp + (size_t)pos * HD + 32 * st + 8 * t)[e];
        }
    __builtin_amdgcn_sched_barrier(0);   // every load above is issued before the first is waited for

    // RoPE of this lane's columns 32 st + 8 t .. + 7 of its head, and of the
    // new key.
    const bool has_new = start <= pos && end == pos + 1;
    half8_t qhi[kSteps], qlo[kSteps], kn[kSteps] = {};
    float x[kSteps][8], qmax = 0.0f;
#pragma unroll
    for (int st = 0; st < kSteps; ++st) {
        const bool low = st < kSteps / 2;
        const int other = low ? st + kSteps / 2 : st - kSteps / 2;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float cc = cs[st][e / 4][e % 4], ss = low ? -sn[st][e / 4][e % 4] : sn[st][e / 4][e % 4];
            x[st][e] = (float)qraw[st][e] * cc + (float)qraw[other][e] * ss;
            qmax = fmaxf(qmax, fabsf(x[st][e]));
            if (has_new) kn[st][e] = (half_t)((float)kraw[st][e] * cc + (float)kraw[other][e] * ss);
        }
    }
    qmax = fmaxf(qmax, __shfl_xor(qmax, 16));
    qmax = fmaxf(qmax, __shfl_xor(qmax, 32));
    const int exp = split16_exp(qmax);
    const float c = exp2_factor<HD>(), unit = __builtin_ldexpf(c, -exp);   // the scores are scaled like q
#pragma unroll
    for (int st = 0; st < kSteps; ++st) split16(x[st], exp, qhi[st], qlo[st]);
    if (valid && has_new && blockIdx.z == 0 && wave == 0) {   // the caches' new row
        if (col == 0) {
#pragma unroll
            for (int st = 0; st < kSteps; ++st)
                *reinterpret_cast<half8_t*>(kbase + (size_t)pos * HD + 32 * st + 8 * t) = kn[st];
        }
        if (t == 0) *reinterpret_cast<vcols_t*>(vbase + (size_t)pos * HD + VC * col) = vrow_new;
    }

    float m = -INFINITY, l = 0.0f;   // of head `col`; l: this lane's positions only
    floatx4 acc[VC];
#pragma unroll
    for (int v = 0; v < VC; ++v) acc[v] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int first = start; first == start || (LONG && first < end); first += kKeys) {
        if (first != start) load(first);
        const int k0 = first + 16 * wave;
        // The new position's row comes from the projection (the cache's may
        // not be written yet), rows past it count as zeros.
        if (k0 + col == pos) {
#pragma unroll
            for (int st = 0; st < kSteps; ++st) kf[st] = kn[st];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int key = k0 + 4 * t + j;
            if (key >= pos) vf[j] = key == pos ? vrow_new : vcols_t{};
        }
        // The low parts first: their sum is small, and so are its roundings.
        floatx4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < kSteps; ++st) s = mfma16x16x32(kf[st], qlo[st], s);
#pragma unroll
        for (int st = 0; st < kSteps; ++st) s = mfma16x16x32(kf[st], qhi[st], s);
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (k0 + 4 * t + r >= end) s[r] = -INFINITY;
            mx = fmaxf(mx, s[r]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float mn = fmaxf(m, mx);
        const float ref = mn == -INFINITY ? 0.0f : mn;   // nothing yet: every exponential is 0
        const float alpha = __builtin_amdgcn_exp2f((m - ref) * unit);
        m = mn;
        float p[4];
        l *= alpha;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            p[r] = __builtin_amdgcn_exp2f((s[r] - ref) * unit);
            l += p[r];
        }
        half4_t phi, plo;
        split16(p, kPExp, phi, plo);
#pragma unroll
        for (int v = 0; v < VC; ++v) {
            const half4_t a = {vf[0][v], vf[1][v], vf[2][v], vf[3][v]};
            acc[v] *= alpha;
            acc[v] = __builtin_amdgcn_mfma_f32_16x16x16f16(a, phi, acc[v], 0, 0, 0);
            acc[v] = __builtin_amdgcn_mfma_f32_16x16x16f16(a, plo, acc[v], 0, 0, 0);
        }
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);

    // This lane: rows 4 t + r of each product, i.e. columns VC (4 t + r) + v of head `col`.
    if (col < heads) {
        if (t == 0) {
            m_lds[wave][col] = __builtin_ldexpf(m, -exp);   // of the scores themselves
            l_lds[wave][col] = l;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int v = 0; v < VC; v += 4)
                *reinterpret_cast<floatx4*>(&o_lds[wave][col][VC * (4 * t + r) + v]) =
                    floatx4{acc[v][r], acc[v + 1][r], acc[v + 2][r], acc[v + 3][r]};
    }
    if (!valid || start > pos) return;   // the whole workgroup
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
            const float a = __builtin_amdgcn_exp2f((m_lds[w][h] - ref) * c);
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
                                                                    int chunk, int ranges) {
    __shared__ float o_lds[4][HD];
    const int64_t pos = *posp;
    const int head = blockIdx.x, d = threadIdx.x % HD, lane = threadIdx.x & 63;
    const int quarter = __builtin_amdgcn_readfirstlane(threadIdx.x / HD);   // the same for a wave
    const size_t step = (size_t)nh * (HD + 2);
    const float* base = part + (size_t)head * (HD + 2);
    // Loaded before the position is known; what no range wrote this time is
    // masked below.
    const int lr = lane < ranges ? lane : 0;
    float mine = base[lr * step + HD], l = base[lr * step + HD + 1];
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = base[(quarter + 4 * j < ranges ? quarter + 4 * j : 0) * step + d];
    __builtin_amdgcn_sched_barrier(0);
    if (pos < 0 || pos >= max_seq) {   // the host has not seen the position: no output that could pass for one
        if (quarter == 0) out[(size_t)head * HD + d] = (half_t)NAN;
        return;
    }
    const int n = (int)pos / chunk + 1;
    if (lane >= n) {
        mine = -INFINITY;
        l = 0.0f;
    }
    const float mx = wave_max(mine);
    const float a = __builtin_amdgcn_exp2f((mine - (mx == -INFINITY ? 0.0f : mx)) * exp2_factor<HD>());
    l = wave_sum(l * a);
    float sum = 0.0f;
    for (int i0 = quarter; i0 < n; i0 += 32) {
        if (i0 != quarter) {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = i0 + 4 * j < n ? base[(i0 + 4 * j) * step + d] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float w = __builtin_bit_cast(
                float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, a), (i0 + 4 * j) & 63));
            sum = fmaf(w, i0 + 4 * j < n ? v[j] : 0.0f, sum);
        }
    }
    o_lds[quarter][d] = sum;
    __syncthreads();
    if (quarter == 0)
        out[(size_t)head * HD + d] = (half_t)((o_lds[0][d] + o_lds[1][d] + o_lds[2][d] + o_lds[3][d]) / __builtin_ldexpf(l, kPExp));
}

// Ranges of a cache of max_seq positions: one inner pass each, at most 64
// ranges (longer caches take a multiple of that per range).
constexpr int kMaxRanges = 64;
int chunk_for(int64_t max_seq) { return (int)(kKeys * ((max_seq + kMaxRanges * kKeys - 1) / (kMaxRanges * kKeys))); }

template <int HD>
hipError_t launch(const DecodeAttnArgs& a, hipStream_t stream) {
    const int groups = a.nh / a.kvh, chunk = chunk_for(a.max_seq);
    const int splits = (a.max_seq + chunk - 1) / chunk;
    auto kernel = chunk > kKeys ? awq_decode_attn_kernel<HD, true> : awq_decode_attn_kernel<HD, false>;
    hipLaunchKernelGGL(kernel, dim3(splits, a.kvh, (groups + kHeads - 1) / kHeads),
                       dim3(kThreads), 0, stream, a.qkv, a.k_cache, a.v_cache, a.cos, a.sin, a.pos, a.part, a.nh,
                       a.kvh, groups, a.max_seq, chunk);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((awq_decode_combine_kernel<HD>), dim3(a.nh), dim3(4 * HD), 0, stream, a.part, a.pos, a.out,
                       a.nh, a.max_seq, chunk, splits);
    return hipGetLastError();
}

}  // namespace

size_t decode_attn_workspace(int max_seq, int nh, int hd) {
    const int chunk = chunk_for(max_seq);
    return (size_t)((max_seq + chunk - 1) / chunk) * nh * (hd + 2) * sizeof(float);
}

hipError_t launch_decode_attn(const DecodeAttnArgs& a, int hd, hipStream_t stream) {
    return hd == 64 ? launch<64>(a, stream) : launch<128>(a, stream);
}

}  // namespace awq
