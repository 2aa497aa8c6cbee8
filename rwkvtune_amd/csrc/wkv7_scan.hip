// The scan between the two passes of a segmented WKV7 walk (wkv7_seg.hpp): X_i = X_{i-1} Q_i + H_i over the
// segments of one (sequence, head), written over H, X_0 being the first segment's H.
//
// Rows of X are independent, so a block takes 16 of a unit's 64 (wave w: columns 16 w ..) and four blocks
// share a unit; everything runs on v_mfma_f32_16x16x4_f32.  A step is a few hundred cycles of a serial chain
// against a memory latency of one to two microseconds, so Q and H are loaded kAhead segments ahead
// (16 segments of 12 units: 20 us when each step loaded its own, 10 us so).
#include "wkv7_mm.hpp"
#include "wkv7_seg.hpp"

namespace {

constexpr int NH = 64;
constexpr int kAhead = 4;

// steps 1 .. n of the chain whose step i is at float offset base + i * stride
__device__ __forceinline__ void scan(int n, size_t base, int64_t stride, int i0, const float* __restrict__ q_all,
                                     float* __restrict__ h_all)
{
    __shared__ __attribute__((aligned(16))) float x_sh[2][16][wkvmm::SP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 15, h = lane >> 4;
    const int er = tid >> 4, ec = 4 * (tid & 15);
    float q[kAhead][16], hh[kAhead][4];
    auto load = [&](int i, float (&qq)[16], float (&h4)[4]) {
        const float* Q = q_all + base + i * stride + 4 * h * NH + 16 * wave + c;
        const float* Hs = h_all + base + i * stride + (i0 + 4 * h) * NH + 16 * wave + c;
#pragma unroll
        for (int m = 0; m < 16; ++m) qq[m] = Q[(16 * (m >> 2) + (m & 3)) * NH];
#pragma unroll
        for (int e = 0; e < 4; ++e) h4[e] = Hs[e * NH];
    };
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
        if (u < n) load(1 + u, q[u], hh[u]);
    *reinterpret_cast<f32x4*>(&x_sh[0][er][ec]) =
        *reinterpret_cast<const f32x4*>(h_all + base + (i0 + er) * NH + ec);
    wkvmm::lds_barrier();
    for (int i1 = 1; i1 <= n; i1 += kAhead) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int i = i1 + u;
            if (i > n) break;  // uniform
            f32x4 acc0 = {hh[u][0], hh[u][1], hh[u][2], hh[u][3]}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int m4 = 0; m4 < 4; ++m4) {
                const f32x4 x = *reinterpret_cast<const f32x4*>(&x_sh[u & 1][c][16 * m4 + 4 * h]);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (m4 & 1) acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], q[u][4 * m4 + e], acc1, 0, 0, 0);
                    else acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], q[u][4 * m4 + e], acc0, 0, 0, 0);
                }
            }
            if (i + kAhead <= n) load(i + kAhead, q[u], hh[u]);
            float* Hs = h_all + base + i * stride + (i0 + 4 * h) * NH + 16 * wave + c;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x = acc0[e] + acc1[e];
                x_sh[(u & 1) ^ 1][4 * h + e][16 * wave + c] = x;
                Hs[e * NH] = x;
            }
            wkvmm::lds_barrier();
        }
    }
}

// blockIdx.x = 4 unit + row group
__global__ __launch_bounds__(256) void wkv7_scan_forward_kernel(WkvSegs m, int H, const float* __restrict__ q,
                                                                float* __restrict__ h)
{
    const int unit = blockIdx.x >> 2, s = unit / H, head = unit - s * H;
    int g0, n;
    wkvseg::range(m, s, g0, n);
    if (n < 3) return;
    scan(n - 2, ((size_t)g0 * H + head) * (NH * NH), (int64_t)H * (NH * NH), 16 * (blockIdx.x & 3), q, h);
}

__global__ __launch_bounds__(256) void wkv7_scan_backward_kernel(int nseg, const float* __restrict__ q,
                                                                 float* __restrict__ h)
{
    const size_t last = (size_t)(blockIdx.x >> 2) * nseg + nseg - 1;
    scan(nseg - 2, last * (NH * NH), -(int64_t)(NH * NH), 16 * (blockIdx.x & 3), q, h);
}

}  // namespace

hipError_t launch_wkv7_scan_forward(const WkvSegs& m, int H, const float* q, float* h, hipStream_t st)
{
    hipLaunchKernelGGL(wkv7_scan_forward_kernel, dim3(4u * (unsigned)m.nseq * (unsigned)H), dim3(256), 0, st, m, H, q,
                       h);
    return hipGetLastError();
}

hipError_t launch_wkv7_scan_backward(int64_t units, int nseg, const float* q, float* h, hipStream_t st)
{
    hipLaunchKernelGGL(wkv7_scan_backward_kernel, dim3((unsigned)(4 * units)), dim3(256), 0, st, nseg, q, h);
    return hipGetLastError();
}
