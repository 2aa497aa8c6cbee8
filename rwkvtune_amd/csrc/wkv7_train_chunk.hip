// WKV7 training backward in chunked (matrix) form on gfx950.
//
// The token-serial backward (wkv7_train.hip) is one chain of T dependent steps per
// (sequence, head).  Here 32 tokens are one set of contractions.  With the chunk
// algebra of wkv7_chunk.hip (S the state at the chunk start, D the cumulative
// decay, r~ = r D, a~ = a D_{t-1}, k^ = k / D, b^ = b / D, token rows),
//   SA = (S a~^T + V^T A_ak) T,  T = (I - A_ab)^-1
//   Y  = S r~^T + SA B_rb + V^T B_rk
//   S' = (S + SA b^ + V^T k^) diag(D_L)
// the gradients of one chunk, given G = dL/dS' and G^ = G diag(D_L), are
//   X = dY B_rb^T + G^ b^^T,  Z = X T^T          (dL/dsa before / after the solve)
//   dV^T = G^ k^^T + dY B_rk^T + Z A_ak^T
//   dA_ab = SA^T Z, dA_ak = V Z, dB_rb = SA^T dY, dB_rk = V dY   (masked as A, B)
//   dr~ = dY^T S + dB_rb^T b^ + dB_rk^T k^,   da~ = Z^T S + dA_ab^T b^ + dA_ak^T k^
//   db^ = SA^T G^ + dB_rb r~ + dA_ab a~,      dk^ = V G^ + dB_rk r~ + dA_ak a~
//   dL/dS = G^ + dY r~ + Z a~
// and the log-decay's gradient is a suffix sum over the chunk of
// r~ dr~ - k^ dk^ - b^ db^ (own token on) + a~ da~ (next token on), plus
// sum_i G S' per key.  SA and the chunk start states come from the forward.
//
// Layout: a 1024-thread block walks the chunks of one (sequence, head) segment from
// the last to the first (~150 KB of LDS, one block per CU, four waves per SIMD); every
// wave owns one 32 x 32 output tile per phase, and G stays in the float32 accumulators
// of four of them.  Products behind float32 results (G when the initial state's gradient
// is wanted, every product of float32 inputs) run on v_mfma_f32_32x32x2_f32; the others
// end in 16-bit gradients and take bf16 hi + lo operand parts (wkv7_mm.hpp, ~2^-16 per
// product, far inside the 16-bit output rounding).
//
// A launch with fewer (sequence, head) units than CUs cuts each sequence into
// segments: a first pass walks every segment with G = 0 and with G = I (only the
// G recurrence), which gives G_start = G_end Q + H per segment, a short scan turns
// these into every segment's G_end, and the gradient pass walks all segments at once.
//
// Measured against the token-serial kernel (bf16): B = 8, T = 4096, H = 32 (256 units, no
// segments) 3.15 -> 1.23 ms; B = 1, T = 512, H = 12 (16 segments) 370 -> 36 us in three
// launches; B = 2, T = 1000, H = 32 with the initial state's gradient 740 -> 180 us.  What
// bounds it: VALU issue (about two thirds of the cycles, 16k wave instructions per chunk of
// which the element-wise phases are the larger half) and LDS operand reads (a third),
// with no bank conflicts; the matrix cores are busy 13%.  Four waves per SIMD with packed
// operands took 1.23 ms where two waves per SIMD that split operands at each read took 1.5.
#include "wkv7_mm.hpp"
#include "wkv7_seg.hpp"

#include <type_traits>

namespace {

using namespace wkvmm;

constexpr int NH = 64;
constexpr int L = 32;
constexpr int CK = 16;  // the forward's checkpoint interval (tokens)
constexpr float kLog2e = 1.4426950408889634f;
// the matrix form's log-decay floor, as in the chunked forward (wkv7_chunk.hip)
constexpr float kLog2DecayFloor = -1.25f * kLog2e;

// sum over the 8 lanes of a state row (token-serial fallback)
__device__ __forceinline__ float sum8(float x) {
    x += dpp_xor1(x);
    x += dpp_xor2(x);
    return x + dpp_xor7(x);
}

// DT: type of the log2-decay sums (double for float32 inputs)
template <bool GRADS, typename DT>
struct __attribute__((aligned(16))) BwdLds {
    float Rt[L][SP], At[L][SP], Bh[L][SP];  // scaled operands [t][j]
    float DY[L][SP], X[L][SP];              // [t][i]
    float G[NH][SP];                        // G^ of the chunk [i][j]
    float T[L][TP], AbT[L][TP], Rb[L][TP];  // T [s][t], A_ab^T [t][s], B_rb [s][t]
    DT tot[GRADS ? 16 : 8][NH];
    alignas(16) int slow[16];
    struct Grads {
        float Z[L][SP], Kh[L][SP], V[L][SP], SA[L][SP], S[NH][SP];
        float Ak[L][TP], Rk[L][TP], dAb[L][TP], dAk[L][TP], dRb[L][TP], dRk[L][TP];
        float cpart[3][NH];  // sum_i G S' per key, one partial sum per 32 rows; [2] scratch
    };
    struct None {};
    typename std::conditional<GRADS, Grads, None>::type g;
};
static_assert(sizeof(BwdLds<true, double>) <= 160 * 1024, "one block per CU");
static_assert(sizeof(BwdLds<false, double>) <= 80 * 1024, "two blocks per CU");

template <bool GRADS>
constexpr int kBwdThreads = GRADS ? 1024 : 512;

// One block: the chunks [seg * cps, ...) of unit (sequence, head), last to first.
// GRADS: G_end of the segment comes from seg_h (the last segment: ds_in or zero), all gradients
// are written and segment 0 leaves ds0.  Otherwise blockIdx.y picks the walk that starts from
// G = I without dY (Q) or from G = 0 (the last segment: ds_in) with dY (H), and only the segment's
// start value is written; segment 0 and the last segment's Q are not needed.
template <typename IO, bool GRADS, bool EXACT>
__global__ __launch_bounds__(kBwdThreads<GRADS>) void wkv7_train_bwd_chunk_kernel(
    int T, int H, int nseg, int cps, const IO* __restrict__ r, const IO* __restrict__ w, const IO* __restrict__ k,
    const IO* __restrict__ v, const IO* __restrict__ a, const IO* __restrict__ b, const IO* __restrict__ dy,
    const float* __restrict__ ckpt, const float* __restrict__ sa_in, const float* __restrict__ ds_in,
    const float* __restrict__ s0, int start_known, float* __restrict__ seg_q, float* __restrict__ seg_h,
    IO* __restrict__ dr, IO* __restrict__ dw, IO* __restrict__ dk, IO* __restrict__ dv, IO* __restrict__ da,
    IO* __restrict__ db, float* __restrict__ ds0)
{
    typedef io_traits<IO> tr;
    constexpr bool FI = sizeof(IO) == 4;                  // float32 inputs: every product in float32
    constexpr bool FG = FI || EXACT;                      // the products behind G
    constexpr bool PI = !FI, PG = !FG;                    // words of the operands: packed parts unless float32
    constexpr bool XV = std::is_same<IO, bf16_t>::value;  // dY and V are exact bf16 operands
    constexpr int NW = kBwdThreads<GRADS> / 64;
    constexpr int CH = NH * L / kBwdThreads<GRADS>;       // channels per thread of the element-wise phases
    constexpr int TPW = L / NW;                           // tokens per wave there
    typedef typename std::conditional<FI, double, float>::type DT;
    __shared__ BwdLds<GRADS, DT> sm;
    const int tid = threadIdx.x, lane0 = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int unit = blockIdx.x / nseg;
    const int seg = blockIdx.x - unit * nseg;
    const bool ident = !GRADS && blockIdx.y == 0;  // the walk from G = I
    if (!GRADS && (seg == 0 || (ident && seg == nseg - 1))) return;
    const int bb = unit / H, hh = unit - bb * H;
    const int C = H * NH;
    const size_t row0 = (size_t)bb * T;
    const int nck = (T + CK - 1) / CK;
    const float* gCk = ckpt + (size_t)unit * nck * (NH * NH);
    const int nchunk = (T + L - 1) / L;
    const int c_lo = seg * cps, c_hi = min(nchunk, c_lo + cps);

    // G: waves 0 .. 3 hold the 32 x 32 tile of rows gi .. and columns gj .. in accumulator layout,
    // through the whole walk
    const int gi = 32 * ((wave >> 1) & 1), gj = 32 * (wave & 1);
    f32x16 G = {0.f};
    if (wave < 4) {
        const float* src = nullptr;
        if (seg == nseg - 1)
            src = ds_in != nullptr ? ds_in + (size_t)unit * (NH * NH) : nullptr;
        else if (GRADS)
            src = seg_h + ((size_t)unit * nseg + seg + 1) * (NH * NH);  // scanned: G at the next segment's start
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int i = gi + acc_row(q, lane0), j = gj + (lane0 & 31);
            if (src != nullptr) G[q] = src[i * NH + j];
            if (ident) G[q] = i == j ? 1.f : 0.f;
        }
    }

    // inputs of a chunk: one token x CH channels per thread, four elements of the start state
    Raw<IO, CH> qr, qw, qk, qv, qa, qb, qy;
    Raw<float, CH> qs;
    f32x4 xs;
    const uint32_t stride = (uint32_t)C * (uint32_t)sizeof(IO);
    // the chunk's rows of the head in a tensor
    auto rows = [&](const auto* p, int c) {
        constexpr int es = (int)sizeof(*p);
        return Rows(p + (row0 + (size_t)c * L) * C + hh * NH, min(L, T - c * L), (uint32_t)C * es, es);
    };
    auto fetch = [&](int c, int id) {
        const uint32_t o = (uint32_t)(id / (NH / CH)) * stride + CH * (id & (NH / CH - 1)) * sizeof(IO);
        qw.load(rows(w, c), o);
        qr.load(rows(r, c), o);
        qa.load(rows(a, c), o);
        qb.load(rows(b, c), o);
        if (!ident) qy.load(rows(dy, c), o);
        if constexpr (GRADS) {
            qk.load(rows(k, c), o);
            qv.load(rows(v, c), o);
            qs.load(rows(sa_in, c), o * (4 / sizeof(IO)));
            const float* sp = c > 0 ? gCk + (size_t)(2 * c - 1) * (NH * NH)
                                    : start_known ? (s0 != nullptr ? s0 + (size_t)unit * (NH * NH) : nullptr)
                                                  : gCk;  // unknown start: the state after token 15, stepped back
            xs = sp != nullptr ? *reinterpret_cast<const f32x4*>(sp + 4 * (uint32_t)id) : f32x4{0.f, 0.f, 0.f, 0.f};
        }
    };
    if (ident) {
#pragma unroll
        for (int e = 0; e < Raw<IO, CH>::N; ++e) qy.u[e] = 0;
    }
    fetch(c_hi - 1, tid);
    // sum_i G S' per key: G and S' (the state after the chunk) meet where the chunk after it ends, for the
    // segment's last chunk here
    auto key_sums = [&](auto&& state, int lane) {
        if constexpr (GRADS) {
            float p = 0.f;
#pragma unroll
            for (int q = 0; q < 16; ++q) p = fmaf(G[q], state(gi + acc_row(q, lane), gj + (lane & 31)), p);
            p += lane_xor32(p);
            if (lane < 32) sm.g.cpart[gi >> 5][gj + lane] = p;
        }
    };
    if constexpr (GRADS) {
        if (wave < 4) {
            const float* p = gCk + (size_t)(min(2 * c_hi, nck) - 1) * (NH * NH);
            key_sums([&](int i, int j) { return p[i * NH + j]; }, lane0);
        }
    }

    for (int c = c_hi - 1; c >= c_lo; --c) {
        // element-wise phases: token tk, channels j0 .. j0 + CH - 1 (grp: the token within its wave);
        // the start state: row sr, columns sc .. sc + 3
        const int id = opaque(tid), lane = id & 63;
        const int tk = id / (NH / CH), j0 = CH * (id & (NH / CH - 1)), grp = tk & (TPW - 1);
        [[maybe_unused]] const int sr = id >> 4, sc = 4 * (id & 15);
        const int n = min(L, T - c * L);
        float xr[CH], xw[CH], xk[CH], xv[CH], xa[CH], xb[CH], xdy[CH], xsa[CH];  // zero past the sequence
        qr.get(xr);
        qw.get(xw);
        qa.get(xa);
        qb.get(xb);
        qy.get(xdy);
        if constexpr (GRADS) {
            qk.get(xk);
            qv.get(xv);
            qs.get(xsa);
        }
        DT lw2[CH], pre[CH];
        bool slow = false;
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            const DT x = tk < n ? -(DT)(FI ? expf(xw[e]) : ex2(xw[e] * kLog2e)) * (DT)1.4426950408889634 : (DT)0;
            slow |= !(x >= (DT)kLog2DecayFloor);
            lw2[e] = x;
            if constexpr (TPW == 4) {
                const DT p1 = xor16(x), p2 = xor32(x + p1);
                pre[e] = (grp >= 2 ? p2 : (DT)0) + ((grp & 1) ? p1 : (DT)0);  // tokens of the wave before this one
            } else {
                const DT p = xor32(x);
                pre[e] = grp ? p : (DT)0;
            }
        }
        if (grp == TPW - 1) {
#pragma unroll
            for (int e = 0; e < CH; ++e) sm.tot[wave][j0 + e] = pre[e] + lw2[e];
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
            // ---- exact token-serial update of the chunk.  Half 0 (512 threads): rows of G, thread (i, q)
            // elements 8q .. 8q + 7; half 1 (GRADS): columns of G and S, stepped back from the 16-token
            // checkpoints as in the token-serial kernel
            float dec[CH];
#pragma unroll
            for (int e = 0; e < CH; ++e) {
                dec[e] = ex2(lw2[e]);
            }
            put_ch<false, CH>(&sm.Rt[tk][j0], xr);
            put_ch<false, CH>(&sm.At[tk][j0], xa);
            put_ch<false, CH>(&sm.Bh[tk][j0], xb);
            put_ch<false, CH>(&sm.DY[tk][j0], xdy);
            float(*Dc)[SP] = sm.X;          // decays
            float* dsa = &sm.AbT[0][0];     // dsa of two tokens
            if constexpr (GRADS) {
                put_ch<false, CH>(&sm.g.Kh[tk][j0], xk);
                put_ch<false, CH>(&sm.g.V[tk][j0], xv);
                put_ch<false, CH>(&sm.g.SA[tk][j0], xsa);
            }
            put_ch<false, CH>(&Dc[tk][j0], dec);
            if (wave < 4) put<false>(&sm.G[0][0], SP, gi, gj, G, lane);
            lds_barrier();
            const bool col = GRADS && wave >= 8;
            const int i = (id & 511) >> 3, q0 = 8 * (id & 7);
            float g[8], sT[8];  // G[i][q0 ..] or G[q0 ..][i], S[q0 ..][i]
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                g[e] = col ? sm.G[q0 + e][i] : sm.G[i][q0 + e];
                sT[e] = 0.f;
            }
#pragma unroll 1
            for (int t = n - 1; t >= 0; --t) {
                float* ds = dsa + NH * (t & 1);
                const size_t o = (row0 + (size_t)c * L + t) * C + hh * NH + i;
                const float wi = Dc[t][i], ai = sm.At[t][i];
                float gsa = 0.f;
                if (!col) {
                    const float dyi = sm.DY[t][i];
                    float gv = 0.f;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        g[e] = fmaf(dyi, sm.Rt[t][q0 + e], g[e]);
                        gsa = fmaf(g[e], sm.Bh[t][q0 + e], gsa);
                        if constexpr (GRADS) gv = fmaf(g[e], sm.g.Kh[t][q0 + e], gv);
                    }
                    gsa = sum8(gsa);
                    ds[i] = gsa;
                    if constexpr (GRADS) {
                        gv = sum8(gv);
                        if ((id & 7) == 0) dv[o] = tr::from_f32(gv);
                    }
                } else if constexpr (GRADS) {
                    if (t == n - 1 || t == CK - 1) {
                        const float* p = gCk + (size_t)(2 * c + (t >= CK ? 1 : 0)) * (NH * NH);
#pragma unroll
                        for (int e = 0; e < 8; ++e) sT[e] = p[(q0 + e) * NH + i];
                    }
                    const float ri = sm.Rt[t][i], ki = sm.g.Kh[t][i], bi = sm.Bh[t][i], iwi = 1.0f / wi;
                    float o_r = 0.f, o_w = 0.f, o_k = 0.f, o_b = 0.f;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float dyj = sm.DY[t][q0 + e], vj = sm.g.V[t][q0 + e], sj = sm.g.SA[t][q0 + e];
                        o_r = fmaf(sT[e], dyj, o_r);
                        sT[e] = (sT[e] - ki * vj - bi * sj) * iwi;
                        g[e] = fmaf(ri, dyj, g[e]);
                        o_w = fmaf(g[e], sT[e], o_w);
                        o_k = fmaf(g[e], vj, o_k);
                        o_b = fmaf(g[e], sj, o_b);
                    }
                    o_r = sum8(o_r);
                    o_w = sum8(o_w);
                    o_k = sum8(o_k);
                    o_b = sum8(o_b);
                    if ((id & 7) == 0) {
                        dr[o] = tr::from_f32(o_r);
                        dw[o] = tr::from_f32(o_w * wi * -expf(tr::to_f32(w[o])));
                        dk[o] = tr::from_f32(o_k);
                        db[o] = tr::from_f32(o_b);
                    }
                }
                lds_barrier();  // dsa of the token; the next token writes the other buffer
                if (!col) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) g[e] = fmaf(g[e], Dc[t][q0 + e], gsa * sm.At[t][q0 + e]);
                } else if constexpr (GRADS) {
                    float o_a = 0.f;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        o_a = fmaf(sT[e], ds[q0 + e], o_a);
                        g[e] = fmaf(g[e], wi, ai * ds[q0 + e]);
                    }
                    o_a = sum8(o_a);
                    if ((id & 7) == 0) da[o] = tr::from_f32(o_a);
                }
            }
            lds_barrier();
            if (!col) {
#pragma unroll
                for (int e = 0; e < 8; ++e) sm.G[i][q0 + e] = g[e];
            }
            if (c > c_lo) fetch(c - 1, id);
            lds_barrier();
            if (wave < 4) {
#pragma unroll
                for (int q = 0; q < 16; ++q) G[q] = sm.G[gi + acc_row(q, lane)][gj + (lane & 31)];
                if constexpr (GRADS) {
                    if (c > c_lo) {
                        const float* p = gCk + (size_t)(2 * c - 1) * (NH * NH);
                        key_sums([&](int i, int j) { return p[i * NH + j]; }, lane);
                    }
                }
            }
            continue;
        }

        // ---- scaled operands -----------------------------------------------------------------------
        DT before[CH];  // log2 D before this token
#pragma unroll
        for (int e = 0; e < CH; ++e) before[e] = pre[e];
        // (all reads first: a branch around each would wait for them one by one)
        DT tots[NW - 1][CH];
#pragma unroll
        for (int q = 0; q < NW - 1; ++q)
#pragma unroll
            for (int e = 0; e < CH; ++e) tots[q][e] = sm.tot[q][j0 + e];
#pragma unroll
        for (int q = 0; q < NW - 1; ++q)
#pragma unroll
            for (int e = 0; e < CH; ++e) before[e] += q < wave ? tots[q][e] : (DT)0;
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            const DT ld = before[e] + lw2[e];
            const float iD = ex2(-ld);
            xr[e] *= ex2(ld);
            xa[e] *= ex2(before[e]);
            xb[e] *= iD;
            if constexpr (GRADS) xk[e] *= iD;
        }
        put_ch<PG, CH>(&sm.Rt[tk][j0], xr);
        put_ch<PG, CH>(&sm.At[tk][j0], xa);
        put_ch<PG, CH>(&sm.Bh[tk][j0], xb);
        put_ch<PG && !XV, CH>(&sm.DY[tk][j0], xdy);  // an exact bf16 value is its own packed word
        if constexpr (GRADS) {
            put_ch<PI, CH>(&sm.g.Kh[tk][j0], xk);
            put_ch<PI && !XV, CH>(&sm.g.V[tk][j0], xv);
            put_ch<PI, CH>(&sm.g.SA[tk][j0], xsa);
            if (c == 0 && !start_known) {
                // S = S_15 / D_15 - (k^^T v + b^^T sa)^T over the first 16 tokens
                if (tk == min(CK, n) - 1) {
                    float iD[CH];
#pragma unroll
                    for (int e = 0; e < CH; ++e) iD[e] = ex2(-(before[e] + lw2[e]));
                    put_ch<false, CH>(&sm.g.cpart[2][j0], iD);
                }
                lds_barrier();
                f32x4 x = xs * *reinterpret_cast<const f32x4*>(&sm.g.cpart[2][sc]);
#pragma unroll 1
                for (int t = 0; t < CK; ++t) {
                    const float vi = value<PI>(sm.g.V[t][sr]), si = value<PI>(sm.g.SA[t][sr]);
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        x[e] -= value<PI>(sm.g.Kh[t][sc + e]) * vi + value<PG>(sm.Bh[t][sc + e]) * si;
                }
                xs = x;
                lds_barrier();
            }
            *reinterpret_cast<f32x4*>(&sm.g.S[sr][sc]) = words4<PI>(xs);
        }
        float cj[CH];  // sum_i G S' per key
        if constexpr (GRADS) {
            float x[CH];
            get_ch<CH>(&sm.g.cpart[0][j0], cj);
            get_ch<CH>(&sm.g.cpart[1][j0], x);
#pragma unroll
            for (int e = 0; e < CH; ++e) cj[e] += x[e];
        }
        if (wave < 4) {  // G^ = G diag(D_L)
            DT all = 0;
#pragma unroll
            for (int q = 0; q < NW; ++q) all += sm.tot[q][gj + (lane & 31)];
            const float DL = ex2(all);
#pragma unroll
            for (int q = 0; q < 16; ++q) G[q] *= DL;
            put<PG>(&sm.G[0][0], SP, gi, gj, G, lane);
        }
        if (c > c_lo) fetch(c - 1, id);
        lds_barrier();

        const Mat<PG> Rt{&sm.Rt[0][0], SP}, At{&sm.At[0][0], SP}, Bh{&sm.Bh[0][0], SP}, X{&sm.X[0][0], SP};
        const Mat<PG> Gm{&sm.G[0][0], SP}, Tm{&sm.T[0][0], TP}, Rb{&sm.Rb[0][0], TP};
        const Mat<PG, XV> DY{&sm.DY[0][0], SP};
        float* zp;  // without gradients Z lies over dY, whose last readers are in P1
        if constexpr (GRADS) zp = &sm.g.Z[0][0];
        else zp = &sm.DY[0][0];
        const Mat<PG> Z{zp, SP};
        const f32x16 zero16 = {0.f};
        const int tile = 32 * (wave & 1);  // the 32-wide half of the wave's outputs
        f32x16 acc = zero16;

        // ---- P0: the intra-chunk matrices and the products with G^ and S; one 64-term tile per wave ----
        if (wave == 4) {
            mm<FG, false, false, NH>(acc, At, 0, Bh, 0, lane);  // A_ab^T [t][s]
#pragma unroll
            for (int q = 0; q < 16; ++q) acc[q] = (lane & 31) < acc_row(q, lane) ? acc[q] : 0.f;
            put<false>(&sm.AbT[0][0], TP, 0, 0, acc, lane);
        } else if (wave == 5) {
            if (!ident) {
                mm<FG, false, false, NH>(acc, Bh, 0, Rt, 0, lane);
                mask_upper<false>(acc, lane);
                put<PG>(&sm.Rb[0][0], TP, 0, 0, acc, lane);
            }
        } else if (wave >= 6 && wave < 8) {
            mm<FG, false, false, NH>(acc, Gm, tile, Bh, 0, lane);  // G^ b^^T [i][s]
        } else if constexpr (GRADS) {
            const Mat<PI> Kh{&sm.g.Kh[0][0], SP}, SA{&sm.g.SA[0][0], SP}, S{&sm.g.S[0][0], SP};
            const Mat<PI, XV> V{&sm.g.V[0][0], SP};
            if (wave == 0) {
                mm<FI, false, false, NH>(acc, Kh, 0, At, 0, lane);
                mask_upper<true>(acc, lane);
                put<PI>(&sm.g.Ak[0][0], TP, 0, 0, acc, lane);
            } else if (wave == 1) {
                mm<FI, false, false, NH>(acc, Kh, 0, Rt, 0, lane);
                mask_upper<false>(acc, lane);
                put<PI>(&sm.g.Rk[0][0], TP, 0, 0, acc, lane);
            } else if (wave == 2) {
                mm<FI, false, false, NH>(acc, SA, 0, DY, 0, lane);
                mask_upper<false>(acc, lane);
                put<PI>(&sm.g.dRb[0][0], TP, 0, 0, acc, lane);
            } else if (wave == 3) {
                mm<FI, false, false, NH>(acc, V, 0, DY, 0, lane);
                mask_upper<false>(acc, lane);
                put<PI>(&sm.g.dRk[0][0], TP, 0, 0, acc, lane);
            } else if (wave < 10) {
                mm<FI, false, false, NH>(acc, Gm, tile, Kh, 0, lane);  // dV [i][s]
            } else if (wave < 12) {
                mm<FI, false, true, NH>(acc, DY, 0, S, tile, lane);  // dr~ [t][j]
            } else if (wave < 14) {
                mm<FI, false, true, NH>(acc, V, 0, Gm, tile, lane);  // dk^ [s][j]
            } else {
                mm<FI, false, true, NH>(acc, SA, 0, Gm, tile, lane);  // db^ [s][j]
            }
        }
        lds_barrier();

        // ---- P1: T; X; everything else that needs only the matrices -----------------------------------
        if (wave < 4) {
            if (!ident) mm<FG, true, true, L>(G, DY, gi, Rt, gj, lane);  // G^ + dY r~
        } else if (wave < 6) {
            unit_upper_inverse<PG>(&sm.AbT[0][0], &sm.T[0][0], id - 256);
        } else if (wave < 8) {
            if (!ident) mm<FG, true, false, L>(acc, DY, tile, Rb, 0, lane);
            put_t<PG>(&sm.X[0][0], SP, 0, tile, acc, lane);
        } else if constexpr (GRADS) {
            const Mat<PI> Kh{&sm.g.Kh[0][0], SP};
            const Mat<PI> dRb{&sm.g.dRb[0][0], TP}, dRk{&sm.g.dRk[0][0], TP}, Rk{&sm.g.Rk[0][0], TP};
            if (wave < 10) {
                mm<FI, true, false, L>(acc, DY, tile, Rk, 0, lane);
            } else if (wave < 12) {
                mm<FI, true, true, L>(acc, dRb, 0, Bh, tile, lane);
                mm<FI, true, true, L>(acc, dRk, 0, Kh, tile, lane);
            } else if (wave < 14) {
                mm<FI, false, true, L>(acc, dRk, 0, Rt, tile, lane);
            } else {
                mm<FI, false, true, L>(acc, dRb, 0, Rt, tile, lane);
            }
        }
        lds_barrier();

        // ---- P2: Z = X T^T --------------------------------------------------------------------------
        if (wave >= 6 && wave < 8) {
            acc = zero16;
            mm<FG, true, false, L>(acc, X, tile, Tm, 0, lane);  // [i][t]
            put_t<PG>(zp, SP, 0, tile, acc, lane);
        }
        lds_barrier();

        // ---- P3: what needs Z alone -------------------------------------------------------------------
        if (wave < 4) {
            mm<FG, true, true, L>(G, Z, gi, At, gj, lane);  // G of the chunk start
        } else if constexpr (GRADS) {
            const Mat<PI> SA{&sm.g.SA[0][0], SP}, S{&sm.g.S[0][0], SP}, Ak{&sm.g.Ak[0][0], TP};
            const Mat<PI, XV> V{&sm.g.V[0][0], SP};
            if (wave == 4) {
                acc = zero16;
                mm<FI, false, false, NH>(acc, SA, 0, Z, 0, lane);
                mask_upper<true>(acc, lane);
                put<PI>(&sm.g.dAb[0][0], TP, 0, 0, acc, lane);
            } else if (wave == 5) {
                acc = zero16;
                mm<FI, false, false, NH>(acc, V, 0, Z, 0, lane);
                mask_upper<true>(acc, lane);
                put<PI>(&sm.g.dAk[0][0], TP, 0, 0, acc, lane);
            } else if (wave < 8) {
                acc = zero16;
                mm<FI, false, true, NH>(acc, Z, 0, S, tile, lane);  // da~ [t][j]
            } else if (wave < 10) {
                mm<FI, true, false, L>(acc, Z, tile, Ak, 0, lane);
                const Rows out = rows(dv, c);
                const uint32_t o = (uint32_t)(lane & 31) * stride + (tile + 4 * (lane >> 5)) * sizeof(IO);
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float x[4] = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
                    store_ch<IO, 4>(out, o + 8 * g * sizeof(IO), x);
                }
            }
        }

        if constexpr (GRADS) {
            lds_barrier();
            // ---- P4: the A_ab / A_ak terms; the four [t][j] gradients to LDS (over V, SA, dY, Z) --------
            const Mat<PI> Kh{&sm.g.Kh[0][0], SP}, dAb{&sm.g.dAb[0][0], TP}, dAk{&sm.g.dAk[0][0], TP};
            // (waves 0 .. 3: the key sums of the chunk before this one)
            if (wave < 4) {
                key_sums([&](int i, int j) { return value<PI>(sm.g.S[i][j]); }, lane);
            } else if (wave >= 6 && wave < 8) {
                mm<FI, true, true, L>(acc, dAb, 0, Bh, tile, lane);
                mm<FI, true, true, L>(acc, dAk, 0, Kh, tile, lane);
                put<false>(&sm.g.SA[0][0], SP, 0, tile, acc, lane);
            } else if (wave >= 10 && wave < 12) {
                put<false>(&sm.g.V[0][0], SP, 0, tile, acc, lane);
            } else if (wave >= 12 && wave < 14) {
                mm<FI, false, true, L>(acc, dAk, 0, At, tile, lane);
                put<false>(&sm.g.Z[0][0], SP, 0, tile, acc, lane);
            } else if (wave >= 14) {
                mm<FI, false, true, L>(acc, dAb, 0, At, tile, lane);
                put<false>(&sm.DY[0][0], SP, 0, tile, acc, lane);
            }
            lds_barrier();

            // ---- epilogue: scale back, the decay's suffix sums ---------------------------------------
            float gr[CH], ga[CH], gb[CH], gk[CH], suf[CH], ya[CH];
            get_ch<CH>(&sm.g.V[tk][j0], gr);
            get_ch<CH>(&sm.g.SA[tk][j0], ga);
            get_ch<CH>(&sm.DY[tk][j0], gb);
            get_ch<CH>(&sm.g.Z[tk][j0], gk);
            {
                float rt[CH], at[CH], bh[CH], kh[CH];
                get_ch<CH>(&sm.Rt[tk][j0], rt);
                get_ch<CH>(&sm.At[tk][j0], at);
                get_ch<CH>(&sm.Bh[tk][j0], bh);
                get_ch<CH>(&sm.g.Kh[tk][j0], kh);
#pragma unroll
                for (int e = 0; e < CH; ++e) {
                    ya[e] = value<PG>(at[e]) * ga[e];
                    const float x = value<PG>(rt[e]) * gr[e] - value<PI>(kh[e]) * gk[e] - value<PG>(bh[e]) * gb[e] + ya[e];
                    const float p = lane_xor32(x);  // two tokens per wave
                    suf[e] = x + (grp ? 0.f : p);
                }
            }
            if (grp == 0) {
#pragma unroll
                for (int e = 0; e < CH; ++e) sm.tot[wave][j0 + e] = suf[e];
            }
            lds_barrier();
            float sums[NW][CH];
#pragma unroll
            for (int q = 1; q < NW; ++q)
#pragma unroll
                for (int e = 0; e < CH; ++e) sums[q][e] = (float)sm.tot[q][j0 + e];
#pragma unroll
            for (int q = 1; q < NW; ++q)
#pragma unroll
                for (int e = 0; e < CH; ++e) suf[e] += q > wave ? sums[q][e] : 0.f;
            const uint32_t o = (uint32_t)tk * stride + j0 * sizeof(IO);
#pragma unroll
            for (int e = 0; e < CH; ++e) {
                const DT ld = before[e] + lw2[e];
                const float iD = ex2(-ld);
                gr[e] *= ex2(ld);
                ga[e] *= ex2(before[e]);
                gk[e] *= iD;
                gb[e] *= iD;
                suf[e] = (suf[e] + cj[e] - ya[e]) * (float)(lw2[e] * (DT)0.6931471805599453);  // log-decay -exp(w)
            }
            store_ch<IO, CH>(rows(dr, c), o, gr);
            store_ch<IO, CH>(rows(da, c), o, ga);
            store_ch<IO, CH>(rows(dk, c), o, gk);
            store_ch<IO, CH>(rows(db, c), o, gb);
            store_ch<IO, CH>(rows(dw, c), o, suf);
        }
        lds_barrier();
    }

    float* out = nullptr;
    if constexpr (GRADS) {
        if (seg == 0 && ds0 != nullptr) out = ds0 + (size_t)unit * (NH * NH);
    } else {
        out = (ident ? seg_q : seg_h) + ((size_t)unit * nseg + seg) * (NH * NH);
    }
    if (out != nullptr && wave < 4) {
#pragma unroll
        for (int q = 0; q < 16; ++q) out[(gi + acc_row(q, lane0)) * NH + gj + (lane0 & 31)] = G[q];
    }
}

// Segments per unit, by the cost (us) of a walk's chunk: 9.6 in the gradient pass (one block per CU, rounds of
// 256), 5.5 in the G pass (8 with two blocks on a CU; 2 n - 3 blocks per unit), 0.6 per step of the scan, and 30
// for two more launches (12 on the device; the rest is what they cost a caller that enqueues as fast as it
// can).  Measured (bf16, one segment -> split): 12 units of 96 tokens 33 -> 32 and not split,
// of 512 tokens 158 -> 36, 64 units of 1,000 tokens 310 -> 140.
int bwd_segments(int64_t units, int T, int* cps) {
    const int nchunk = (T + L - 1) / L;
    *cps = nchunk;
    if (units >= 256) return 1;
    float best = 9.6f * nchunk;
    for (int n = 2; n <= 64 && n <= nchunk; ++n) {
        const int c = (nchunk + n - 1) / n, nn = (nchunk + c - 1) / c;
        const int64_t b1 = units * (2 * nn - 3);
        const float pass1 = b1 <= 256 ? 5.5f : 8.f * (float)((b1 + 511) / 512);
        const float cost = c * (pass1 + 9.6f * (float)((units * nn + 255) / 256)) + 0.6f * nn + 30.f;
        if (cost < best) {
            best = cost;
            *cps = c;
        }
    }
    return (nchunk + *cps - 1) / *cps;
}

}  // namespace

// floats of workspace launch_wkv7_train_bwd_chunk needs
int64_t wkv7_train_bwd_chunk_ws(int B, int T, int H) {
    int cps;
    const int nseg = bwd_segments((int64_t)B * H, T, &cps);
    return nseg > 1 ? (int64_t)B * H * nseg * 2 * NH * NH : 0;
}

template <typename IO>
hipError_t launch_wkv7_train_bwd_chunk(int B, int T, int H, const void* r, const void* w, const void* k,
                                       const void* v, const void* a, const void* b, const void* dy,
                                       const float* ckpt, const float* sa, const float* ds_in, const float* s0,
                                       int start_known, void* dr, void* dw, void* dk, void* dv, void* da, void* db,
                                       float* ds0, float* ws, hipStream_t st)
{
    const int64_t units = (int64_t)B * H;
    int cps;
    const int nseg = bwd_segments(units, T, &cps);
    float* q = ws;
    float* h = nseg > 1 ? ws + units * nseg * (NH * NH) : nullptr;
    auto launch = [&](auto kern, dim3 grid, int threads) -> hipError_t {
        hipLaunchKernelGGL(kern, grid, dim3(threads), 0, st, T, H, nseg, cps, (const IO*)r, (const IO*)w, (const IO*)k,
                           (const IO*)v, (const IO*)a, (const IO*)b, (const IO*)dy, ckpt, sa, ds_in, s0, start_known,
                           q, h, (IO*)dr, (IO*)dw, (IO*)dk, (IO*)dv, (IO*)da, (IO*)db, ds0);
        return hipGetLastError();
    };
    const dim3 full((unsigned)(units * nseg)), two((unsigned)(units * nseg), 2);
    auto passes = [&](auto exact) -> hipError_t {
        constexpr bool EX = decltype(exact)::value;
        if (nseg > 1) {
            hipError_t e = launch(wkv7_train_bwd_chunk_kernel<IO, false, EX>, two, kBwdThreads<false>);
            if (e == hipSuccess && nseg > 2) e = launch_wkv7_scan_backward(units, nseg, q, h, st);
            if (e != hipSuccess) return e;
        }
        return launch(wkv7_train_bwd_chunk_kernel<IO, true, EX>, full, kBwdThreads<true>);
    };
    if constexpr (sizeof(IO) == 4) return passes(std::true_type());
    else return ds0 != nullptr ? passes(std::true_type()) : passes(std::false_type());
}

#define RWKV7_INST(IO)                                                                                              \
    template hipError_t launch_wkv7_train_bwd_chunk<IO>(int, int, int, const void*, const void*, const void*,       \
                                                        const void*, const void*, const void*, const void*,         \
                                                        const float*, const float*, const float*, const float*,     \
                                                        int, void*, void*, void*, void*, void*, void*, float*,      \
                                                        float*, hipStream_t);
RWKV7_INST(float)
RWKV7_INST(bf16_t)
RWKV7_INST(f16_t)
