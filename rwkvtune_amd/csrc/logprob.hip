// Per-token log-probabilities of chosen tokens: out[r] = log_softmax(logits[r])[index[r]]
// without materialising the log-softmax (the selective_log_softmax of
// rwkvtune/training/grpo/utils.py:13-103, used by the GRPO log-prob recompute,
// grpo/lightning_module.py:1810-1964).
//
// One 256-thread block per row reads the row once with 16-byte loads, keeping an
// online (max, sum of exp(x - max)) per thread; the chosen logit is read once.
// Four loads per thread are in flight while the four before them are summed, and an
// exponential is one subtraction, one multiplication and v_exp_f32: with one load at a
// time and expf's range reduction the kernel was bound by VALU issue (4,096 rows of
// 65,536 bf16: 128 us, 4.2 TB/s; now 92 us, 5.8 TB/s, what a read-only stream reaches).
// Numerics follow the reference per dtype:
//   float32 logits:  out = x[i] - logsumexp(x)                       (fp32)
//   bf16 / fp16:     lse = logsumexp(float(x)) rounded to the dtype,
//                    out = round(float(x[i]) - float(lse))            (the dtype)
// (the reference computes torch.logsumexp(logits.float()).to(dtype) and
// subtracts in the dtype).  An index outside [0, V) gives NaN (the reference's
// gather raises instead; checking would cost a host synchronisation).
#include "common.hpp"

namespace {

constexpr int kT = 256;

__device__ __forceinline__ float block_reduce_max(float v, float* red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = red[0];
#pragma unroll
    for (int i = 1; i < kT / 64; ++i) s = fmaxf(s, red[i]);
    return s;
}

__device__ __forceinline__ float block_reduce_sum(float v, float* red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < kT / 64; ++i) s += red[i];
    return s;
}

constexpr int kU = 4;  // groups of 8 logits a thread has in flight
constexpr float kLog2e = 1.4426950408889634f;

// 8 consecutive logits of a row as loaded (16 or 32 bytes)
template <typename LT> struct Group8 {
    uint4 u[sizeof(LT) / 2];
    __device__ __forceinline__ void load(const LT* p) {
#pragma unroll
        for (int q = 0; q < (int)(sizeof(LT) / 2); ++q) u[q] = reinterpret_cast<const uint4*>(p)[q];
    }
    __device__ __forceinline__ void get(float* x) const {
        const LT* e = reinterpret_cast<const LT*>(u);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = io_traits<LT>::to_f32(e[j]);
    }
};

// (m, s) += the logits x[0 .. N)
template <int N>
__device__ __forceinline__ void take(const float (&x)[N], float& m, float& s) {
    float mc = x[0];
#pragma unroll
    for (int e = 1; e < N; ++e) mc = fmaxf(mc, x[e]);
    if (mc > m) {
        s = (m == -INFINITY) ? 0.f : s * expf(m - mc);
        m = mc;
    }
    if (m != -INFINITY && m != INFINITY) {
        float p[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < N; ++e) p[e & 3] += __builtin_amdgcn_exp2f((x[e] - m) * kLog2e);
        s += (p[0] + p[1]) + (p[2] + p[3]);
    }
}

// One pass over the row: each thread keeps a running (max, sum of exp(x - max))
// over its groups of 8 logits (rescaling the sum when the max grows), then the
// block combines the pairs.  vec: rows are 16-byte aligned and V % 8 == 0, else
// elements are read one by one.
template <typename LT>
__global__ __launch_bounds__(kT) void selective_logsoftmax_kernel(int V, const LT* __restrict__ logits, int64_t ld,
                                                                  const int64_t* __restrict__ index,
                                                                  LT* __restrict__ out, int vec)
{
    __shared__ float red[kT / 64];
    const int r = blockIdx.x, t = threadIdx.x;
    const LT* row = logits + (int64_t)r * ld;
    float m = -INFINITY, s = 0.f;
    int i0 = 8 * t;
    if (vec) {
        constexpr int step = 8 * kT;
        Group8<LT> cur[kU];
        if (i0 + (kU - 1) * step < V) {
#pragma unroll
            for (int u = 0; u < kU; ++u) cur[u].load(row + i0 + u * step);
        }
        for (; i0 + (kU - 1) * step < V; i0 += kU * step) {
            Group8<LT> nxt[kU];
            // (past the last full set: the same groups again, unused)
            const int j0 = i0 + (2 * kU - 1) * step < V ? i0 + kU * step : i0;
#pragma unroll
            for (int u = 0; u < kU; ++u) nxt[u].load(row + j0 + u * step);
            float x[8 * kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) cur[u].get(x + 8 * u);
            take(x, m, s);
#pragma unroll
            for (int u = 0; u < kU; ++u) cur[u] = nxt[u];
        }
    }
    for (; i0 < V; i0 += 8 * kT) {
        float x[8];
        if (vec) {
            Group8<LT> g;
            g.load(row + i0);
            g.get(x);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = (i0 + e < V) ? io_traits<LT>::to_f32(row[i0 + e]) : -INFINITY;
        }
        take(x, m, s);
    }
    const float M = block_reduce_max(m, red);
    const float part = (m == -INFINITY || M == INFINITY) ? 0.f : s * expf(m - M);
    const float S = block_reduce_sum(part, red);
    if (t == 0) {
        // logsumexp as torch defines it: max + log(sum exp(x - max)); an all -inf
        // row gives -inf, a +inf max gives +inf
        const float lse = (M == -INFINITY || M == INFINITY) ? M : M + logf(S);
        const int64_t id = index[r];
        const float xs = (id >= 0 && id < V) ? io_traits<LT>::to_f32(row[id]) : NAN;
        float o;
        if (sizeof(LT) == 4) o = xs - lse;
        else o = xs - io_traits<LT>::to_f32(io_traits<LT>::from_f32(lse));
        out[r] = io_traits<LT>::from_f32(o);
    }
}

}  // namespace

template <typename LT>
hipError_t launch_selective_logsoftmax(int R, int V, const void* logits, int64_t ld, const int64_t* index, void* out,
                                       hipStream_t st)
{
    const int vec = (((uintptr_t)logits) & 15) == 0 && (V % 8) == 0 && ((ld * (int64_t)sizeof(LT)) % 16) == 0;
    hipLaunchKernelGGL((selective_logsoftmax_kernel<LT>), dim3(R), dim3(kT), 0, st, V, (const LT*)logits, ld, index,
                       (LT*)out, vec);
    return hipGetLastError();
}

template hipError_t launch_selective_logsoftmax<float>(int, int, const void*, int64_t, const int64_t*, void*,
                                                       hipStream_t);
template hipError_t launch_selective_logsoftmax<bf16_t>(int, int, const void*, int64_t, const int64_t*, void*,
                                                        hipStream_t);
template hipError_t launch_selective_logsoftmax<f16_t>(int, int, const void*, int64_t, const int64_t*, void*,
                                                       hipStream_t);
