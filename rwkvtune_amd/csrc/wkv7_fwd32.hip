// Chunked WKV7 forward for float32 inputs on gfx950: prefill, and the training forward with its checkpoints.
//
// The chunk algebra of wkv7_chunk.hip (32 tokens as dense contractions, S the state at the chunk start),
//   X = S a~^T + V^T A_ak,  SA = X T,  T = (I - A_ab)^-1
//   Y = S r~^T + V^T B_rk + SA B_rb,  S' = (S + V^T k^ + SA b^) diag(D_L)
// with every product on v_mfma_f32_32x32x2_f32 and float32 operands in LDS.  A 1024-thread block walks the
// chunks of one (sequence, head) or of one segment of it (wkv7_seg.hpp); a wave owns one 32 x 32 tile per
// phase, and four waves keep S in their accumulators.  A chunk whose per-token log-decay lies below the matrix
// form's floor runs the exact token-serial update.
//
// The kernel before this one split each operand into three bf16 parts as it was read (six MFMAs per product
// step, the solve on one wave): 50 us per chunk against 8.5 us here.  Bound: the float32 MFMA rate (32 products
// of 32 x 32 x 32 per chunk take 8,200 cycles of the CU's matrix cores) and the phases' latencies.
// 4 sequences x 128 tokens x 12 heads 198 -> 36 us, 1 x 2,000 x 12 (segments) 3,370 -> 93 us, 8 x 1,500 x 64
// 5,800 -> 805 us.  Against float64: state 1.6e-7 -> 1.1e-7, y 1.6e-7 -> 1.5e-7 (relative, 2-norm).
#include "wkv7_mm.hpp"
#include "wkv7_seg.hpp"

namespace {

using namespace wkvmm;

constexpr int NH = 64;
constexpr int L = 32;
constexpr int TH = 1024;
constexpr int NW = TH / 64;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLog2DecayFloor = -1.25f * kLog2e;  // as in wkv7_chunk.hip

struct __attribute__((aligned(16))) FwdLds {
    float Rt[L][SP], At[L][SP], Kh[L][SP], Bh[L][SP];        // scaled operands [t][j]
    float V[L][SP], X[L][SP], SA[L][SP];                     // [t][i]
    float S[NH][SP];                                         // state [i][j]
    float T[L][TP], AbT[L][TP], Rb[L][TP], Ak[L][TP], Rk[L][TP];  // AbT [t][s], the others [s][t]
    double tot[NW][NH];
    float D15[NH];
    alignas(16) int slow[NW];
};

// TRAIN, CARRY, segs, seg_m, seg_n, s_init, ckpt, sa_out: as wkv7_chunk2_kernel (wkv7_chunk.hip)
template <bool TRAIN, bool CARRY>
__global__ __launch_bounds__(TH) void wkv7_fwd32_kernel(
    int H, int T_uniform, const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ slot_idx, int pool_slots,
    int total_tokens, WkvSegs segs, float* seg_m, float* seg_n, float* state, const float* __restrict__ r,
    const float* __restrict__ w, const float* __restrict__ k, const float* __restrict__ v,
    const float* __restrict__ a, const float* __restrict__ b, float* __restrict__ y, const float* s_init,
    float* __restrict__ ckpt, float* __restrict__ sa_out)
{
    __shared__ FwdLds sm;
    const int tid = threadIdx.x, lane0 = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int unit = blockIdx.x, h = unit % H;
    int s = unit / H, seg = 0, nsg = 1;
    const bool ident = CARRY && blockIdx.y == 0;
    if (segs.cps > 0) {
        if (!wkvseg::locate(segs, unit / H, s, seg, nsg)) return;
        if (CARRY && (seg == nsg - 1 || (ident && seg == 0))) return;
    }
    const int tb = cu_seqlens != nullptr ? cu_seqlens[s] : s * T_uniform;
    const int te = cu_seqlens != nullptr ? cu_seqlens[s + 1] : tb + T_uniform;
    if (tb < 0 || te < tb || te > total_tokens || te == tb) return;  // malformed or empty: untouched
    const int slot = slot_idx != nullptr ? slot_idx[s] : s;
    if (slot < 0 || slot >= pool_slots) return;
    const int C = H * NH;
    float* gS = state != nullptr ? state + ((size_t)slot * H + h) * (NH * NH) : nullptr;
    const int nck = TRAIN ? (T_uniform + 15) / 16 : 0;
    float* gCk = TRAIN ? ckpt + (size_t)(s * H + h) * nck * (NH * NH) : nullptr;

    // S: waves 0 .. 3 hold the tile of rows si .. and columns sj .., element (row, l % 32)
    const int si = 32 * ((wave >> 1) & 1), sj = 32 * (wave & 1);
    f32x16 S = {0.f};
    auto each = [&](auto f) {
#pragma unroll
        for (int q = 0; q < 16; ++q) f(q, (si + acc_row(q, lane0)) * NH + sj + (lane0 & 31));
    };
    if (wave < 4) {
        const float* src = s_init != nullptr ? s_init + ((size_t)s * H + h) * (NH * NH) : TRAIN ? nullptr : gS;
        if (seg > 0 || (nsg > 1 && !CARRY))
            src = seg > 0 ? seg_n + (size_t)(unit - H) * (NH * NH) : seg_m + (size_t)unit * (NH * NH);
        if (src != nullptr && !(CARRY && seg > 0)) each([&](int q, int o) { S[q] = src[o]; });
        if (CARRY && seg == 0) each([&](int q, int o) { seg_m[(size_t)unit * (NH * NH) + o] = S[q]; });
        if (ident) each([&](int q, int o) { S[q] = o / NH == o % NH ? 1.f : 0.f; });
        put<false>(&sm.S[0][0], SP, si, sj, S, lane0);
    }

    const uint32_t stride = (uint32_t)C * 4u;
    Raw<float, 2> qr, qw, qk, qv, qa, qb;
    auto rows = [&](const float* p, int t0) {
        return Rows(p + (size_t)t0 * C + h * NH, min(L, te - t0), stride, 4);
    };
    auto fetch = [&](int t0, int id) {
        const uint32_t o = (uint32_t)(id >> 5) * stride + 8u * (id & 31);
        qw.load(rows(w, t0), o);
        if constexpr (!CARRY) qr.load(rows(r, t0), o);
        qa.load(rows(a, t0), o);
        qb.load(rows(b, t0), o);
        qk.load(rows(k, t0), o);
        qv.load(rows(v, t0), o);
    };
    const int t_lo = tb + seg * segs.cps * L, t_hi = nsg > 1 ? min(te, t_lo + segs.cps * L) : te;
    fetch(t_lo, tid);

    for (int t0 = t_lo; t0 < t_hi; t0 += L) {
        const int id = opaque(tid), lane = id & 63;
        const int tk = id >> 5, j0 = 2 * (id & 31);
        const int n = min(L, te - t0);
        [[maybe_unused]] const int ci = (t0 - tb) / L;
        // ---- log2-decay prefix (two tokens per wave, the waves' totals through LDS) ------------------
        float xr[2] = {0.f, 0.f}, xw[2], xk[2], xv[2], xa[2], xb[2];  // zero past the sequence
        if constexpr (!CARRY) qr.get(xr);
        qw.get(xw);
        qk.get(xk);
        qv.get(xv);
        qa.get(xa);
        qb.get(xb);
        if (ident) xv[0] = xv[1] = 0.f;
        double lw2[2], before[2];
        bool slow = false;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            lw2[e] = tk < n ? -(double)expf(xw[e]) * 1.4426950408889634 : 0.0;
            slow |= !(lw2[e] >= (double)kLog2DecayFloor);
            const double p = xor32(lw2[e]);
            before[e] = lane >= 32 ? p : 0.0;
            if (lane >= 32) sm.tot[wave][j0 + e] = p + lw2[e];
        }
        const bool wave_slow = __ballot(slow) != 0;
        if (lane == 0) sm.slow[wave] = wave_slow ? 1 : 0;
        lds_barrier();
        int any_slow = 0;
#pragma unroll
        for (int q = 0; q < NW; q += 4) {
            const int4 x = *reinterpret_cast<const int4*>(&sm.slow[q]);
            any_slow |= x.x | x.y | x.z | x.w;
        }

        if (any_slow) {
            // ---- exact token-serial update: 16 threads per state row, four columns each --------------
            float dec[2] = {ex2(lw2[0]), ex2(lw2[1])};
            put_ch<false, 2>(&sm.Rt[tk][j0], xr);
            put_ch<false, 2>(&sm.At[tk][j0], xa);
            put_ch<false, 2>(&sm.Kh[tk][j0], xk);
            put_ch<false, 2>(&sm.Bh[tk][j0], xb);
            put_ch<false, 2>(&sm.V[tk][j0], xv);
            put_ch<false, 2>(&sm.X[tk][j0], dec);
            lds_barrier();
            const int i = id >> 4, q0 = 4 * (id & 15);
            f32x4 x = *reinterpret_cast<const f32x4*>(&sm.S[i][q0]);
#pragma unroll 1
            for (int t = 0; t < n; ++t) {
                const f32x4 at = *reinterpret_cast<const f32x4*>(&sm.At[t][q0]);
                const f32x4 kt = *reinterpret_cast<const f32x4*>(&sm.Kh[t][q0]);
                const f32x4 bt = *reinterpret_cast<const f32x4*>(&sm.Bh[t][q0]);
                const f32x4 dt = *reinterpret_cast<const f32x4*>(&sm.X[t][q0]);
                const f32x4 rt = *reinterpret_cast<const f32x4*>(&sm.Rt[t][q0]);
                const float sa = row16_sum(fast_dot4(at, x)), vi = sm.V[t][i];
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = x[e] * dt[e] + kt[e] * vi + sa * bt[e];
                const size_t o = (size_t)(t0 + t) * C + h * NH + i;
                if constexpr (!CARRY) {
                    const float yi = row16_sum(fast_dot4(rt, x));
                    if ((id & 15) == 0) y[o] = yi;
                }
                if constexpr (TRAIN) {
                    if ((id & 15) == 0) sa_out[o] = sa;
                    if (t == 15 || t == n - 1)
                        *reinterpret_cast<f32x4*>(gCk + (size_t)(2 * ci + (t >= 16 ? 1 : 0)) * (NH * NH) + i * NH + q0) = x;
                }
            }
            *reinterpret_cast<f32x4*>(&sm.S[i][q0]) = x;
            if (t0 + L < t_hi) fetch(t0 + L, id);
            lds_barrier();
            if (wave < 4) {
#pragma unroll
                for (int q = 0; q < 16; ++q) S[q] = sm.S[si + acc_row(q, lane)][sj + (lane & 31)];
            }
            continue;
        }

        // ---- scaled operands -----------------------------------------------------------------------
        // (all reads first: a branch around each would wait for them one by one)
        double tots[NW - 1][2];
#pragma unroll
        for (int q = 0; q < NW - 1; ++q) {
            tots[q][0] = sm.tot[q][j0];
            tots[q][1] = sm.tot[q][j0 + 1];
        }
#pragma unroll
        for (int q = 0; q < NW - 1; ++q) {
            before[0] += q < wave ? tots[q][0] : 0.0;
            before[1] += q < wave ? tots[q][1] : 0.0;
        }
        float D15[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const double ld = before[e] + lw2[e];
            const float D = ex2(ld), iD = ex2(-ld);
            xr[e] *= D;
            xa[e] *= ex2(before[e]);
            xk[e] *= iD;
            xb[e] *= iD;
            D15[e] = D;
        }
        if constexpr (!CARRY) put_ch<false, 2>(&sm.Rt[tk][j0], xr);
        put_ch<false, 2>(&sm.At[tk][j0], xa);
        put_ch<false, 2>(&sm.Kh[tk][j0], xk);
        put_ch<false, 2>(&sm.Bh[tk][j0], xb);
        put_ch<false, 2>(&sm.V[tk][j0], xv);
        if (TRAIN && tk == 15) put_ch<false, 2>(&sm.D15[j0], D15);
        float DL = 0.f;  // decay of the chunk for the column of this lane's state elements
        if (wave < 4) {
            double all = 0.0;
#pragma unroll
            for (int q = 0; q < NW; ++q) all += sm.tot[q][sj + (lane & 31)];
            DL = ex2(all);
        }
        if (t0 + L < t_hi) fetch(t0 + L, id);
        lds_barrier();

        const Mat<false> Rt{&sm.Rt[0][0], SP}, At{&sm.At[0][0], SP}, Kh{&sm.Kh[0][0], SP}, Bh{&sm.Bh[0][0], SP};
        const Mat<false> V{&sm.V[0][0], SP}, X{&sm.X[0][0], SP}, SA{&sm.SA[0][0], SP}, Sm{&sm.S[0][0], SP};
        const Mat<false> Tm{&sm.T[0][0], TP}, Rb{&sm.Rb[0][0], TP}, Ak{&sm.Ak[0][0], TP}, Rk{&sm.Rk[0][0], TP};
        const int tile = 32 * (wave & 1);
        f32x16 acc = {0.f};
        // tokens 0 .. 15 / 16 .. 31 of M^T V-like updates of S: rows of V or SA against rows of k^ or b^
        auto state_half = [&](const Mat<false>& P, const Mat<false>& Q, int t1) {
            mm<true, true, true, 16>(S, Mat<false>{P.p + t1 * SP, SP}, si, Mat<false>{Q.p + t1 * SP, SP}, sj, lane);
        };

        // ---- P0: the intra-chunk matrices, S a~^T, S r~^T, V^T k^ ----------------------------------------
        if (wave < 4) {
            state_half(V, Kh, 0);
            if constexpr (!TRAIN) state_half(V, Kh, 16);
        } else if (wave == 4) {
            mm<true, false, false, NH>(acc, At, 0, Bh, 0, lane);  // A_ab^T [t][s]
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[q] = (lane & 31) < acc_row(q, lane) ? acc[q] : 0.f;
            put<false>(&sm.AbT[0][0], TP, 0, 0, acc, lane);
        } else if (wave == 5) {
            mm<true, false, false, NH>(acc, Kh, 0, At, 0, lane);
            mask_upper<true>(acc, lane);
            put<false>(&sm.Ak[0][0], TP, 0, 0, acc, lane);
        } else if (wave < 8) {
            mm<true, false, false, NH>(acc, Sm, tile, At, 0, lane);  // X [i][t]
        } else if constexpr (!CARRY) {
            if (wave < 10) {
                mm<true, false, false, NH>(acc, Sm, tile, Rt, 0, lane);  // Y [i][t]
            } else if (wave == 10) {
                mm<true, false, false, NH>(acc, Bh, 0, Rt, 0, lane);
                mask_upper<false>(acc, lane);
                put<false>(&sm.Rb[0][0], TP, 0, 0, acc, lane);
            } else if (wave == 11) {
                mm<true, false, false, NH>(acc, Kh, 0, Rt, 0, lane);
                mask_upper<false>(acc, lane);
                put<false>(&sm.Rk[0][0], TP, 0, 0, acc, lane);
            }
        }
        lds_barrier();

        // ---- P1: T on two waves; X and Y take V's terms --------------------------------------------------
        if (wave == 4 || wave == 5) {
            unit_upper_inverse<false>(&sm.AbT[0][0], &sm.T[0][0], id - 256);
        } else if (wave == 6 || wave == 7) {
            mm<true, true, true, L>(acc, V, tile, Ak, 0, lane);
            put_t<false>(&sm.X[0][0], SP, 0, tile, acc, lane);
        } else if (!CARRY && (wave == 8 || wave == 9)) {
            mm<true, true, true, L>(acc, V, tile, Rk, 0, lane);
        }
        lds_barrier();

        // ---- P2: SA = X T ----------------------------------------------------------------------------
        if (wave == 6 || wave == 7) {
            acc = f32x16{0.f};
            mm<true, true, true, L>(acc, X, tile, Tm, 0, lane);  // [i][t]
            put_t<false>(&sm.SA[0][0], SP, 0, tile, acc, lane);
            if constexpr (TRAIN) {
                const Rows out = rows(sa_out, t0);
                const uint32_t o = (uint32_t)(lane & 31) * stride + 4u * (tile + 4 * (lane >> 5));
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float x[4] = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
                    store_ch<float, 4>(out, o + 32u * g, x);
                }
            }
        }
        lds_barrier();

        // ---- P3: y; S' -----------------------------------------------------------------------------------
        if (wave < 4) {
            state_half(SA, Bh, 0);
            if constexpr (TRAIN) {
                // the state after token 15 (after the last one when n <= 16: later tokens add nothing)
                const float d = sm.D15[sj + (lane & 31)];
                float* p = gCk + (size_t)(2 * ci) * (NH * NH);
                each([&](int q, int o) { p[o] = S[q] * d; });
                state_half(V, Kh, 16);
            }
            state_half(SA, Bh, 16);
#pragma unroll
            for (int q = 0; q < 16; ++q) S[q] *= DL;
            if (TRAIN && n > 16) {
                float* p = gCk + (size_t)(2 * ci + 1) * (NH * NH);
                each([&](int q, int o) { p[o] = S[q]; });
            }
            put<false>(&sm.S[0][0], SP, si, sj, S, lane);
        } else if (!CARRY && (wave == 8 || wave == 9)) {
            mm<true, true, true, L>(acc, SA, tile, Rb, 0, lane);
            const Rows out = rows(y, t0);
            const uint32_t o = (uint32_t)(lane & 31) * stride + 4u * (tile + 4 * (lane >> 5));
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float x[4] = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
                store_ch<float, 4>(out, o + 32u * g, x);
            }
        }
        // no barrier: the next chunk's first LDS writes (tot, slow) touch nothing read in P3, the others
        // come after its first barrier
    }
    if (wave < 4) {
        if constexpr (CARRY) {
            float* p = (ident ? seg_m : seg_n) + (size_t)unit * (NH * NH);
            each([&](int q, int o) { p[o] = S[q]; });
        } else {
            if (gS != nullptr && seg == nsg - 1) each([&](int q, int o) { gS[o] = S[q]; });
        }
    }
}

}  // namespace

// m.cps > 0: in segments, with ws for m.gmax * H * 2 states
hipError_t launch_wkv7_fwd32(const WkvSegs& m, int H, int T_uniform, const int32_t* cu, const int32_t* slot_idx,
                             int pool_slots, int total, float* state, const float* r, const float* w, const float* k,
                             const float* v, const float* a, const float* b, float* y, const float* s0, float* ckpt,
                             float* sa, float* ws, hipStream_t stream)
{
    const unsigned groups = m.cps > 0 ? (unsigned)m.gmax : (unsigned)m.nseq;
    float *sm = ws, *sn = m.cps > 0 ? ws + (size_t)m.gmax * H * NH * NH : nullptr;
    auto launch = [&](auto kern, dim3 grid, float* st, float* ck, float* sa_) -> hipError_t {
        hipLaunchKernelGGL(kern, grid, dim3(TH), 0, stream, H, T_uniform, cu, slot_idx, pool_slots, total,
                           m, sm, sn, st, r, w, k, v, a, b, y, s0, ck, sa_);
        return hipGetLastError();
    };
    if (m.cps > 0) {
        hipError_t e = launch(wkv7_fwd32_kernel<false, true>, dim3(groups * (unsigned)H, 2),
                              ckpt != nullptr ? nullptr : state, nullptr, nullptr);
        if (e == hipSuccess) e = launch_wkv7_scan_forward(m, H, sm, sn, stream);
        if (e != hipSuccess) return e;
    }
    const dim3 grid(groups * (unsigned)H);
    return ckpt != nullptr ? launch(wkv7_fwd32_kernel<true, false>, grid, state, ckpt, sa)
                           : launch(wkv7_fwd32_kernel<false, false>, grid, state, nullptr, nullptr);
}
