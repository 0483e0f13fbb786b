// The decision read-out on the device: DecisionModel.ReadOut
// (src/StructuredDecisions.Laya/Models/DecisionModel.cs:170-226) for every item of the last forward.
//
// From an item's option logits (the scorer's output): the untempered softmax
// as SimdOps.Softmax computes it (max, e = exp(v − max), Σe, then e·(1/Σe)), the entropy −Σ p·log(max(p,
// 1e-9)) over log(max(2, K)), the top probability and its margin over the second (strict comparisons in
// option order). With the item's first head-output row (pooled = h[start]) they form the act head's input
// [h, top1, top1 − top2, entropy, k/255]; its MLP (Linear → exact GELU → Linear) and a softmax give the
// action probabilities. Each output of a Linear is one wave's dot product.
#include "common.hpp"

namespace laya {
namespace {

// What bounds the read-out is fetching the act head's first weight ([256, d + 4], 0.8 MB at d = 768) for one
// item. One CU took 32 us for it, so its rows are dealt to RO_SPLIT workgroups per item of four waves, each wave
// with four rows' float4 loads in flight; every workgroup forms the item's features itself (K exponentials), and
// the small second product and the softmax follow in a launch of their own. One decision: 374 us with one
// workgroup of four waves taking a row of scalar loads at a time and one thread fetching the scores in turn, 32 us
// with one workgroup of sixteen waves, 11 + 4 us in these two launches.
constexpr int RO_THREADS = 256, RO_WAVES = RO_THREADS / 64, RO_ROWS = 4;
constexpr int RO_SPLIT = 16;     // workgroups the hidden units of one item are dealt to
constexpr int RO_OPTIONS = 256;  // options whose exponentials are formed in parallel and kept in LDS

typedef float f32x4 __attribute__((ext_vector_type(4)));

// The dot products of x (LDS) with rows o, o + step, … of w (RO_ROWS of them, clamped to the last row), each summed
// over the wave. V: floats per load (4 when n is a multiple of 4 and w is 16-byte aligned).
template <int V>
__device__ __forceinline__ void wave_dots(const float* x, const float* __restrict__ w, int n, int rows, int o, int step,
                                          int lane, float (&s)[RO_ROWS]) {
    typedef float vec __attribute__((ext_vector_type(V)));
    const float* row[RO_ROWS];
#pragma unroll
    for (int u = 0; u < RO_ROWS; ++u) {
        row[u] = w + (long)min(o + u * step, rows - 1) * n;
        s[u] = 0.0f;
    }
#pragma unroll 4
    for (int i = V * lane; i < n; i += V * 64) {
        const vec xi = *reinterpret_cast<const vec*>(x + i);
#pragma unroll
        for (int u = 0; u < RO_ROWS; ++u) {
            const vec wi = *reinterpret_cast<const vec*>(row[u] + i);
#pragma unroll
            for (int e = 0; e < V; ++e) s[u] = fmaf(xi[e], wi[e], s[u]);
        }
    }
#pragma unroll
    for (int u = 0; u < RO_ROWS; ++u) s[u] = wave_sum(s[u]);
}

__device__ __forceinline__ void wave_dots_any(const float* x, const float* __restrict__ w, int n, int rows, int o,
                                              int step, int lane, float (&s)[RO_ROWS]) {
    if (n % 4 == 0 && (reinterpret_cast<uintptr_t>(w) & 15u) == 0)
        wave_dots<4>(x, w, n, rows, o, step, lane, s);
    else
        wave_dots<1>(x, w, n, rows, o, step, lane, s);
}

__global__ __launch_bounds__(RO_THREADS) void readout_hidden_kernel(const float* __restrict__ scores,
                                                                    const int* __restrict__ opt_off,
                                                                    const int* __restrict__ seg_start,
                                                                    const float* __restrict__ states, int d,
                                                                    const float* __restrict__ w1,
                                                                    const float* __restrict__ b1, int a1,
                                                                    float* __restrict__ hidden,
                                                                    float* __restrict__ features) {
    extern __shared__ __attribute__((aligned(16))) float x[];  // the act head's input [d + 4]
    __shared__ float ex[RO_OPTIONS], top[RO_WAVES];
    const int item = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int o0 = opt_off[item], K = opt_off[item + 1] - o0;
    const float* h = states + (long)seg_start[item] * d;
    for (int i = tid; i < d; i += RO_THREADS) x[i] = h[i];
    float mx = -__builtin_huge_valf();
    for (int o = tid; o < K; o += RO_THREADS) mx = fmaxf(mx, scores[o0 + o]);
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) mx = fmaxf(mx, __shfl_xor(mx, s, 64));
    if (lane == 0) top[wave] = mx;
    __syncthreads();
    mx = top[0];
    for (int w = 1; w < RO_WAVES; ++w) mx = fmaxf(mx, top[w]);
    if (tid < min(K, RO_OPTIONS)) ex[tid] = expf(scores[o0 + tid] - mx);
    __syncthreads();
    if (tid == 0) {
        auto e = [&](int o) { return o < RO_OPTIONS ? ex[o] : expf(scores[o0 + o] - mx); };
        float top1 = 0.0f, top2 = 0.0f, entropy = 0.0f;
        if (K > 0 && mx != -__builtin_huge_valf()) {
            float total = 0.0f;
            for (int o = 0; o < K; ++o) total += e(o);
            const float scale = total > 0.0f ? 1.0f / total : 0.0f;
            for (int o = 0; o < K; ++o) {
                const float p = e(o) * scale;
                entropy -= p * logf(fmaxf(p, 1e-9f));
                if (p > top1) {
                    top2 = top1;
                    top1 = p;
                } else if (p > top2) {
                    top2 = p;
                }
            }
        }
        const float k = (float)max(2, K);
        entropy /= logf(k);
        x[d] = top1;
        x[d + 1] = top1 - top2;
        x[d + 2] = entropy;
        x[d + 3] = k / 255.0f;
        if (features && blockIdx.x == 0) {
            features[item * 4 + 0] = top1;
            features[item * 4 + 1] = top1 - top2;
            features[item * 4 + 2] = entropy;
            features[item * 4 + 3] = k / 255.0f;
        }
    }
    __syncthreads();
    const int step = RO_WAVES * gridDim.x;
    for (int o = blockIdx.x * RO_WAVES + wave; o < a1; o += step * RO_ROWS) {
        float s[RO_ROWS];
        wave_dots_any(x, w1, d + 4, a1, o, step, lane, s);
#pragma unroll
        for (int u = 0; u < RO_ROWS; ++u) {
            const int r = o + u * step;
            if (lane == 0 && r < a1) hidden[(long)item * a1 + r] = gelu_f(s[u] + b1[r]);
        }
    }
}

__global__ __launch_bounds__(RO_THREADS) void readout_action_kernel(const float* __restrict__ hidden, int a1,
                                                                    const float* __restrict__ w2,
                                                                    const float* __restrict__ b2, int na,
                                                                    float* __restrict__ probs) {
    extern __shared__ __attribute__((aligned(16))) float hid[];  // hidden [a1 rounded up to 4], act logits [na]
    float* out = hid + (a1 + 3) / 4 * 4;
    const int item = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int i = tid; i < a1; i += RO_THREADS) hid[i] = hidden[(long)item * a1 + i];
    __syncthreads();
    for (int o = wave; o < na; o += RO_WAVES * RO_ROWS) {
        float s[RO_ROWS];
        wave_dots_any(hid, w2, a1, na, o, RO_WAVES, lane, s);
#pragma unroll
        for (int u = 0; u < RO_ROWS; ++u) {
            const int r = o + u * RO_WAVES;
            if (lane == 0 && r < na) out[r] = s[u] + b2[r];
        }
    }
    __syncthreads();
    if (tid == 0) {
        float mx = -__builtin_huge_valf();
        for (int o = 0; o < na; ++o) mx = fmaxf(mx, out[o]);
        float total = 0.0f;
        for (int o = 0; o < na; ++o) total += expf(out[o] - mx);
        const float scale = total > 0.0f ? 1.0f / total : 0.0f;
        for (int o = 0; o < na; ++o) probs[item * na + o] = expf(out[o] - mx) * scale;
    }
}

}  // namespace

void decision_readout(laya_ctx* ctx, const float* scores, const int* opt_off, const int* seg_start, int n_items,
                      const float* states, int d, const float* w1, const float* b1, int a1, const float* w2,
                      const float* b2, int na, float* hidden, float* probs, float* features) {
    if (n_items <= 0) return;
    LAYA_REQUIRE(d > 0 && a1 > 0 && na > 0, "readout: bad act-head shape");
    const size_t lds = sizeof(float) * (size_t)(d + 4 + a1 + na);
    LAYA_REQUIRE(lds <= 64 * 1024, "readout: act-head input too wide for one workgroup");
    ProfileScope scope(ctx, "decision_readout", 0.0, 4.0 * n_items * ((double)d + (double)a1 * (d + 4)));
    for (int i0 = 0; i0 < n_items; i0 += 65535) {  // the grid's y limit
        const int n = std::min(65535, n_items - i0);
        LAYA_LAUNCH(readout_hidden_kernel, dim3(RO_SPLIT, n), dim3(RO_THREADS), sizeof(float) * (size_t)(d + 4),
                    ctx->stream, scores, opt_off + i0, seg_start + i0, states, d, w1, b1, a1,
                    hidden + (size_t)i0 * a1, features ? features + (size_t)i0 * 4 : nullptr);
        check_launch("readout_hidden_kernel");
    }
    LAYA_LAUNCH(readout_action_kernel, dim3(n_items), dim3(RO_THREADS), sizeof(float) * (size_t)((a1 + 3) / 4 * 4 + na),
                ctx->stream, hidden, a1, w2, b2, na, probs);
    check_launch("readout_action_kernel");
}

}  // namespace laya
