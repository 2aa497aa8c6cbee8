// Chunked WKV7 prefill on gfx950 MFMA.
//
// The reference prefills by running its token-serial kernel over each chunk
// (rwkvtune/models/rwkv7/operators/cuda/wkv7s.cu:22-53 via
// grpo_batch_generator.py:353-456): T dependent steps per (sequence, head).
// Here a chunk of L = 32 tokens is one set of dense contractions.  Per head,
// with S the [value i][key j] state at the chunk start and, per key j, the
// cumulative log-decay logD_t = sum_{u<=t} -exp(w_raw_u):
//   r~_t = r_t * D_t,  a~_t = a_t * D_{t-1},  k^_s = k_s / D_s,  b^_s = b_s / D_s,
//   kbar_s = k_s * D_L / D_s,  bbar_s = b_s * D_L / D_s
//   A_ab[s,t] = b^_s . a~_t, A_ak[s,t] = k^_s . a~_t     (s < t)
//   B_rb[s,t] = b^_s . r~_t, B_rk[s,t] = k^_s . r~_t     (s <= t)
//   SA = S a~^T + V^T A_ak + SA A_ab    (column t of SA is sa_t = S_{t-1} a_t;
//                                        A_ab strictly upper: a triangular solve)
//   Y  = S r~^T + SA B_rb + V^T B_rk    (column t is y_t)
//   S' = S diag(D_L) + SA bbar + V^T kbar
// which is the recurrence S_t = S_{t-1} (diag(w_t) + a_t b_t^T) + v_t k_t^T,
// y_t = S_t r_t (wkv7s.cu:33-48) summed in closed form over the chunk.
//
// This file: the kernel of the 16-bit types (float32 inputs: wkv7_fwd32.hip) and the dispatch of both.  A
// chunk whose per-token log-decay drops below kLogDecayFloor runs the exact token-serial update instead, so
// every input gives the recurrence's result.
#include "common.hpp"
#include "wkv7_seg.hpp"

#include <type_traits>

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr int NH = 64;   // head size
constexpr int L = 32;    // chunk length
constexpr int SP = 68;   // padded row stride (floats) of [*][64] LDS matrices
constexpr int TP = 36;   // padded row stride (floats) of [*][32] LDS matrices
// Per-token log-decay floor of the matrix form.  32 tokens * -1.25 bound every
// scaled operand (r~, a~, k^, b^) to e^+-40, far from float overflow and from the
// denormal range, where the bf16 lo parts would lose precision.  Trained RWKV-7
// layers compute w = -softplus(..) - 0.5 (rwkvtune/models/rwkv7/model.py:147), so
// their log-decay -exp(w) >= -e^-0.5 ~ -0.61 and never reaches the fallback.
constexpr float kLogDecayFloor = -1.25f;

// ===========================================================================
// bf16 / fp16 I/O: the chunk algebra with every MFMA operand stored once,
// at production, as bf16 hi + lo planes in LDS (x = hi + lo + e, |e| <= 2^-17 |x|),
// and three v_mfma_f32_32x32x16_bf16 per product step (hi.hi + hi.lo + lo.hi;
// two for the products with V when the inputs are bf16, exact as bf16 operands).
// The per-product error (~2^-16) leaves y ~5e-5 of its rms from the exact
// recurrence and the state ~5e-6 relative, well inside the bf16 / fp16 output
// rounding.
//
// One 256-thread block per (sequence, head), two blocks per CU for bf16 inputs
// (~78 KB of LDS each; the float32 state in registers, one 32 x 32 tile per wave).
// The state update is taken as S' = (S + SA b^ + V^T k^) diag(D_L), which equals
// the form with bbar and kbar above and lets the transposed planes of k^ and b^
// reuse the hi/lo words already split for their token-major planes.
// Per chunk: phase A turns the prefetched inputs into the scaled operand planes
// (log-decay prefix in registers, one barrier); phase B gives each wave one
// state product (X or Y of a value tile) and one intra-chunk matrix; phase C
// adds V^T A_ak to X (waves 0/1) and V^T B_rk to Y (waves 2/3); the
// right-looking triangular solve (quad broadcasts) runs with each wave's
// state-tile MFMAs interleaved; phase D finishes Y and S.
//
// 32x32x16 operand layout: lane l supplies row (l % 32) of A (and of B^T) at
// k = 8*(l/32) .. +7; accumulator q of lane l is C[8*(q/4) + 4*(l/32) + q%4][l%32].
// Products whose result is stored are computed transposed where that gives each
// lane 4 consecutive elements of a stored row.
// ===========================================================================
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));

constexpr int KP = 72;  // bf16 row stride of planes whose K is 64 (144 B)
constexpr int TQ = 40;  // bf16 row stride of planes whose K is 32 (80 B)

// LDS of the 16-bit kernel, under 80 KB for bf16 inputs so that two blocks share
// a CU (each SIMD then runs two waves, which hide each other's VALU and LDS
// latencies and barrier waits).  The float32 state lives in the waves' registers
// (one 32 x 32 tile per wave); the operand planes of phase A and the products of
// phase B share one region (the planes are dead once phase B has read them); the
// planes of S and SA are unpadded with XOR-swizzled 16-byte groups.
template <bool V_LO>
struct __attribute__((aligned(16))) ChunkLds2 {
    union {
        struct {  // phase A -> B
            uint16_t Rt[2][L][KP], At[2][L][KP], Kh[2][L][KP], Bh[2][L][KP];  // rows t, K = key j
        } pa;
        struct {  // phase B -> D
            float AT[L][TP];                                          // A_ab^T [t][s], 0 for s >= t
            uint16_t AakT[2][L][TQ], BrbT[2][L][TQ], BrkT[2][L][TQ];  // rows t, K = s
            float XT[L][NH];                                          // S a~^T + V^T A_ak, [t][i] (xtswz)
            uint16_t SA[2][NH][L];                                    // rows i, K = t (saswz)
        } pb;
        float Sf[NH][SP];   // float32 state [i][j] while a chunk runs token-serially
        int lens[256];      // sequence lengths while ranking them
    } u;
    uint16_t VT[V_LO ? 2 : 1][NH][TQ], BhT[2][NH][TQ], KhT[2][NH][TQ];  // rows i (VT) / j, K = t (tswz)
    uint16_t Sp[2][NH][NH];   // state hi / lo planes, rows i, K = j (spswz)
    float tot[4][NH];   // per wave: log2-decay sums over its 8 tokens  [w][j]
    float DL[NH];       // decay over the whole chunk
    float D15[NH];      // decay over the chunk's first 16 tokens (training checkpoints)
    alignas(16) int slow[4];  // per wave: a token of the chunk decays below the floor
    int pick;                 // the block's sequence (ragged batches, longest first)
};

// Swizzled offsets (elements).  A fragment read covers 32 rows x one 16-byte group
// and a stored accumulator 32 rows x one group; with these layouts any 16
// consecutive rows of one group fall on 16 distinct 16-byte bank slots of the
// 256-byte bank space, as the padded strides did.
// Sp: 64 bf16 per row (8 groups), group ^= row bits 1-3
__device__ __forceinline__ int spswz(int row, int col) {
    return row * NH + ((((col >> 3) ^ (row >> 1)) & 7) << 3) + (col & 7);
}
// XT: 64 floats per row, columns XOR 8 * (row % 4): the solve's 4-byte reads
// (8 consecutive columns for each of 4 consecutive rows per half-wave) reach 32
// distinct banks (measured conflict-free on gfx950; XOR 16 * (row % 4) is not)
__device__ __forceinline__ int xtswz(int row, int col) { return row * NH + (col ^ ((row & 3) << 3)); }
// SA: 32 bf16 per row (4 groups), group ^= row bits 2-3
__device__ __forceinline__ int saswz(int row, int col) {
    return row * L + ((((col >> 3) ^ (row >> 2)) & 3) << 3) + (col & 7);
}

__device__ __forceinline__ void split2(float x0, float x1, uint32_t& hi, uint32_t& lo) {
    const f32x2 v = {x0, x1};
    hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
    const f32x2 r = {x0 - __uint_as_float(hi << 16), x1 - __uint_as_float(hi & 0xffff0000u)};
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2_t));
}

// hi / lo planes of 4 consecutive values, as two 8-byte words
__device__ __forceinline__ void split4(float x0, float x1, float x2, float x3, uint2& hi, uint2& lo) {
    split2(x0, x1, hi.x, lo.x);
    split2(x2, x3, hi.y, lo.y);
}

template <typename IO> __device__ __forceinline__ f32x4 unpack4(uint2 u);
template <> __device__ __forceinline__ f32x4 unpack4<bf16_t>(uint2 u) {
    f32x4 o;
    o.x = __uint_as_float(u.x << 16);
    o.y = __uint_as_float(u.x & 0xffff0000u);
    o.z = __uint_as_float(u.y << 16);
    o.w = __uint_as_float(u.y & 0xffff0000u);
    return o;
}
template <> __device__ __forceinline__ f32x4 unpack4<f16_t>(uint2 u) {
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    const h4 h = __builtin_bit_cast(h4, u);
    f32x4 o;
    o.x = (float)h.x; o.y = (float)h.y; o.z = (float)h.z; o.w = (float)h.w;
    return o;
}

// 4 consecutive outputs as one 8-byte word, rounded to nearest-even (the
// hardware conversions)
template <typename IO> __device__ __forceinline__ uint2 pack4(float x0, float x1, float x2, float x3);
template <> __device__ __forceinline__ uint2 pack4<bf16_t>(float x0, float x1, float x2, float x3) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    const f32x2 p = {x0, x1}, q = {x2, x3};
    return make_uint2(__builtin_bit_cast(uint32_t, __builtin_convertvector(p, b2)),
                      __builtin_bit_cast(uint32_t, __builtin_convertvector(q, b2)));
}
template <> __device__ __forceinline__ uint2 pack4<f16_t>(float x0, float x1, float x2, float x3) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const f32x2 p = {x0, x1}, q = {x2, x3};
    return make_uint2(__builtin_bit_cast(uint32_t, __builtin_convertvector(p, h2)),
                      __builtin_bit_cast(uint32_t, __builtin_convertvector(q, h2)));
}

// 8 bf16 of plane row (row0 + l%32) at k0 + 8*(l/32)
__device__ __forceinline__ bf16x8_t frag(const uint16_t* plane, int stride, int row0, int k0, int lane) {
    return *reinterpret_cast<const bf16x8_t*>(plane + (row0 + (lane & 31)) * stride + k0 + 8 * (lane >> 5));
}

// Token-major planes ([row][t] with TQ stride: VT, KhT, BhT) keep their 16-byte
// groups of 8 tokens XOR-swizzled by row bits 4-5.  Phase A's transposing stores
// (a wave writes 4 consecutive words into each of 16 rows 4 apart) then reach 64
// distinct banks instead of 16; a fragment read covers 16 consecutive rows with
// one swizzle, so reads stay conflict-free.
__device__ __forceinline__ int tswz(int row, int t) { return row * TQ + ((((t >> 3) ^ (row >> 4)) & 3) << 3) + (t & 7); }

__device__ __forceinline__ bf16x8_t fragT(const uint16_t* plane, int row0, int k0, int lane) {
    return *reinterpret_cast<const bf16x8_t*>(plane + tswz(row0 + (lane & 31), k0 + 8 * (lane >> 5)));
}

__device__ __forceinline__ f32x16 mfma3(f32x16 acc, bf16x8_t a0, bf16x8_t a1, bf16x8_t b0, bf16x8_t b1) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b0, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b1, acc, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b0, acc, 0, 0, 0);
}

// mfma3 with a B operand that has no lo part when V_HI_ONLY (the skipped term is 0)
template <bool V_HI_ONLY>
__device__ __forceinline__ f32x16 mfma_v(f32x16 acc, bf16x8_t a0, bf16x8_t a1, bf16x8_t b0, bf16x8_t b1) {
    if constexpr (V_HI_ONLY) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, b0, acc, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b0, acc, 0, 0, 0);
    } else {
        return mfma3(acc, a0, a1, b0, b1);
    }
}

// mfma3 with an A operand that has no lo part when V_HI_ONLY
template <bool V_HI_ONLY>
__device__ __forceinline__ f32x16 mfma_av(f32x16 acc, bf16x8_t a0, bf16x8_t a1, bf16x8_t b0, bf16x8_t b1) {
    if constexpr (V_HI_ONLY) {
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b1, acc, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, b0, acc, 0, 0, 0);
    } else {
        return mfma3(acc, a0, a1, b0, b1);
    }
}

// Store accumulator C (= M^T of the stored matrix M) as hi/lo planes of M:
// lane l holds M[l%32][8g + 4*(l/32) + 0..3] in acc[4g .. 4g+3].
__device__ __forceinline__ void store_planes_T(uint16_t* P, int stride, int plane, int row0, int col0,
                                               const f32x16& acc, int lane) {
    const int row = row0 + (lane & 31);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        uint2 hi, lo;
        split4(acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3], hi, lo);
        const int col = col0 + 8 * g + 4 * (lane >> 5);
        *reinterpret_cast<uint2*>(P + row * stride + col) = hi;
        *reinterpret_cast<uint2*>(P + plane + row * stride + col) = lo;
    }
}

constexpr int RT_PLANE = L * KP, S_PLANE = NH * NH, T32_PLANE = L * TQ, SA_PLANE = NH * L;

// fragments of the swizzled S and SA planes (row0 + l%32, k0 + 8*(l/32))
__device__ __forceinline__ bf16x8_t fragSp(const uint16_t* plane, int row0, int k0, int lane) {
    return *reinterpret_cast<const bf16x8_t*>(plane + spswz(row0 + (lane & 31), k0 + 8 * (lane >> 5)));
}
__device__ __forceinline__ bf16x8_t fragSA(const uint16_t* plane, int row0, int k0, int lane) {
    return *reinterpret_cast<const bf16x8_t*>(plane + saswz(row0 + (lane & 31), k0 + 8 * (lane >> 5)));
}

// A wave's state tile (rows 32*ir + l%32, columns 32*jt + 8g + 4*(l/32) + 0..3 in
// acc[4g .. 4g+3]) stored as the hi/lo planes of S
__device__ __forceinline__ void store_state_planes(uint16_t* Sp, int ir, int jt, const f32x16& acc, int lane) {
    const int row = 32 * ir + (lane & 31);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        uint2 hi, lo;
        split4(acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3], hi, lo);
        const int o = spswz(row, 32 * jt + 8 * g + 4 * (lane >> 5));
        *reinterpret_cast<uint2*>(Sp + o) = hi;
        *reinterpret_cast<uint2*>(Sp + S_PLANE + o) = lo;
    }
}

// The 16-bit kernel keeps log-decays in base 2, so every exponential is one
// v_exp_f32 (about 1 ulp for the arguments here, all >= -58).  Their accuracy is
// bounded anyway by the float32 prefix sum of up to 32 log-decays.
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLog2DecayFloor = kLogDecayFloor * kLog2e;
__device__ __forceinline__ float ex2(float x) { return __builtin_amdgcn_exp2f(x); }

// lane e of each quad, to all four lanes (quad_perm eeee); e is a constant after unrolling
__device__ __forceinline__ float quad_bcast(float x, int e) {
    switch (e) {
    case 0: return __builtin_amdgcn_mov_dpp(x, 0x00, 0xf, 0xf, false);
    case 1: return __builtin_amdgcn_mov_dpp(x, 0x55, 0xf, 0xf, false);
    case 2: return __builtin_amdgcn_mov_dpp(x, 0xaa, 0xf, 0xf, false);
    default: return __builtin_amdgcn_mov_dpp(x, 0xff, 0xf, 0xf, false);
    }
}

// Block barrier for data exchanged through LDS.  __syncthreads() also waits for every global load and store
// of the wave: the loads issued a chunk ahead, y and the training checkpoints.  Training forward at
// B = 8, T = 4096, H = 32 (bf16, one block per CU): 0.88 -> 0.73 ms.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <bool LDS_ONLY>
__device__ __forceinline__ void block_sync()
{
    if constexpr (LDS_ONLY) lds_barrier();
    else __syncthreads();
}

// hi / lo bf16 parts of one value (hardware round-to-nearest-even)
__device__ __forceinline__ void split1(float x, uint16_t& hi, uint16_t& lo) {
    uint32_t h, l;
    split2(x, 0.f, h, l);
    hi = (uint16_t)h;
    lo = (uint16_t)l;
}

// TRAIN: the training operator's forward over B uniform sequences of T_uniform
// tokens (cu_seqlens and slot_idx null): the initial state comes from s_init (zero
// when null) and the final one goes to `state` (skipped when null), and the
// kernel also writes every token's sa_t = S_{t-1} a_t (float32, [tokens][H][64])
// and the state after every 16th token of a sequence and after its last one
// (ckpt [B][H][ceil(T/16)][64][64]), the layout the training backward reads.
//
// SEG: the sequences are walked in segments (wkv7_seg.hpp), block group g taking segment g (a template
// argument, and the initial state's choice compiled only where there is one: the unsplit kernel lost 0.4 us a launch
// to them).  CARRY is the pass before the scan: only the state is walked, blockIdx.y = 0 from the identity without values (M),
// 1 from zero, or from the sequence's initial state in its first segment (N); the first segment's M place
// keeps a copy of that initial state, since the last segment's block of the full pass writes the final state
// where the first one's may still have to be read.
template <typename IO, bool TRAIN, bool SEG, bool CARRY>
__global__ __launch_bounds__(256, (std::is_same<IO, bf16_t>::value ? 2 : 1)) void wkv7_chunk2_kernel(
    int H, int T_uniform, const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ slot_idx, int pool_slots,
    int total_tokens, WkvSegs segs, float* seg_m, float* seg_n, float* state, const IO* __restrict__ r, const IO* __restrict__ w,
    const IO* __restrict__ k, const IO* __restrict__ v, const IO* __restrict__ a, const IO* __restrict__ b,
    IO* __restrict__ y, const float* s_init, float* __restrict__ ckpt, float* __restrict__ sa_out)
{
    typedef io_traits<IO> tr;
    // bf16 inputs are exact as bf16 MFMA operands: V (unscaled) has no lo plane, and
    // the products with V skip their hi.lo term
    constexpr bool kVExact = std::is_same<IO, bf16_t>::value;
    // The next chunk's loads: with the training stores in flight, early and behind barriers that wait for LDS only;
    // the prefill kernel (two blocks per CU) is 0.5-1 % faster with them late (27 ragged sequences, H = 16:
    // 39.1 -> 38.6 us; 16 x 300, H = 32: 67.1 -> 66.9).
    constexpr bool kFetchB = TRAIN;
    constexpr int kVLo = kVExact ? 0 : 1;  // plane of V's lo part (none for bf16)
    __shared__ ChunkLds2<!kVExact> sm;
    const int unit = blockIdx.x;
    const int h = unit % H;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;

    // Ragged batches of up to 256 sequences run longest sequence first: block
    // group r takes the r-th longest sequence (ties by index, so every sequence
    // is taken once), and the longest chains of chunks start earliest instead of
    // stretching the launch's tail.  The lengths are ranked from LDS: one length
    // per thread against all nseq, so at most 256 LDS reads per thread.  Larger
    // batches keep their order (the ranking would cost more than the tail it
    // shortens).
    int s = unit / H;
    int seg = 0, nsg = 1;  // segment of the sequence
    const bool ident = CARRY && blockIdx.y == 0;
    if constexpr (SEG) {
        if (!wkvseg::locate(segs, unit / H, s, seg, nsg)) return;
        if (CARRY && (seg == nsg - 1 || (ident && seg == 0))) return;
    } else if (cu_seqlens != nullptr) {
        const int nseq = (int)(gridDim.x / (unsigned)H);
        if (nseq <= 256) {
            int* lens = sm.u.lens;
            for (int c = tid; c < nseq; c += 256) lens[c] = cu_seqlens[c + 1] - cu_seqlens[c];
            block_sync<kFetchB>();
            for (int c = tid; c < nseq; c += 256) {
                const int len = lens[c];
                int rank = 0;
                for (int d = 0; d < nseq; ++d) {
                    const int l2 = lens[d];
                    rank += (l2 > len || (l2 == len && d < c)) ? 1 : 0;
                }
                if (rank == s) sm.pick = c;
            }
            block_sync<kFetchB>();
            s = sm.pick;
        }
    }

    const int tb = cu_seqlens != nullptr ? cu_seqlens[s] : s * T_uniform;
    const int te = cu_seqlens != nullptr ? cu_seqlens[s + 1] : tb + T_uniform;
    if (tb < 0 || te < tb || te > total_tokens || te == tb) return;  // malformed or empty: untouched
    const int slot = slot_idx != nullptr ? slot_idx[s] : s;
    if (slot < 0 || slot >= pool_slots) return;

    const int C = H * NH;
    float* gS = state != nullptr ? state + ((size_t)slot * H + h) * (NH * NH) : nullptr;
    // training checkpoints of this (sequence, head): ceil(T / 16) states of 64 x 64
    const int nck = TRAIN ? (T_uniform + 15) / 16 : 0;
    float* gCk = TRAIN ? ckpt + (size_t)(s * H + h) * nck * (NH * NH) : nullptr;

    // The float32 state: wave w holds the tile of value rows 32*ir_t .. and keys
    // 32*jt_t .. (ir_t = w / 2, jt_t = w % 2), lane l row 32*ir_t + l%32 and keys
    // 32*jt_t + 8g + 4*(l/32) + 0..3 in tile[4g .. 4g+3] (the accumulator layout of
    // the products that update it); the hi/lo planes in LDS are the MFMA operand.
    const int ir_t = wave >> 1, jt_t = wave & 1;
    f32x16 tile;
    auto tile_io = [&](float* base, int ld, bool store) {
        const int i = 32 * ir_t + (lane & 31);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            f32x4* p = reinterpret_cast<f32x4*>(base + i * ld + 32 * jt_t + 8 * g + 4 * (lane >> 5));
            if (store) {
                *p = f32x4{tile[4 * g], tile[4 * g + 1], tile[4 * g + 2], tile[4 * g + 3]};
            } else {
                const f32x4 x = *p;
#pragma unroll
                for (int e = 0; e < 4; ++e) tile[4 * g + e] = x[e];
            }
        }
    };
    if constexpr (!SEG && !TRAIN) {
        tile_io(gS, NH, false);
    } else {
        // the initial state of the sequence: the pool slot's, or (training) s_init
        const float* gInit = s_init != nullptr ? s_init + ((size_t)s * H + h) * (NH * NH) : TRAIN ? nullptr : gS;
        if (SEG && (seg > 0 || (nsg > 1 && !CARRY)))  // found by the passes before (unused in CARRY)
            gInit = seg > 0 ? seg_n + (size_t)(unit - H) * (NH * NH) : seg_m + (size_t)unit * (NH * NH);
        if (gInit == nullptr || (CARRY && seg > 0))
            tile = f32x16{0.f};
        else
            tile_io(const_cast<float*>(gInit), NH, false);
    }
    if (CARRY && seg == 0) tile_io(seg_m + (size_t)unit * (NH * NH), NH, true);
    if (ident) {
#pragma unroll
        for (int q = 0; q < 16; ++q)
            tile[q] = 32 * ir_t + (lane & 31) == 32 * jt_t + 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3) ? 1.f : 0.f;
    }
    store_state_planes(&sm.Sp[0][0][0], ir_t, jt_t, tile, lane);
    // a 64 x 64 state in the tiles' layout, one 16-byte store per group
    auto put_state = [&](float* base, const f32x16& x) {
        const int i = 32 * ir_t + (lane & 31);
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<f32x4*>(base + i * NH + 32 * jt_t + 8 * g + 4 * (lane >> 5)) =
                f32x4{x[4 * g], x[4 * g + 1], x[4 * g + 2], x[4 * g + 3]};
    };

    // phase-A mapping: tokens 2*tp, 2*tp+1 of the chunk, channels 4*c4 .. +3; the 16
    // lanes of a row read one 128-byte token row of the head
    const int tp = tid >> 4, c4 = tid & 15, j0 = 4 * c4;
    uint2 raw[6][2];  // r, w, k, v, a, b of this thread's two tokens (zero past the end)
    // Buffer loads: one resource per input, based at the chunk's first row of the
    // head and ending after its last row in the sequence, so each load is one
    // per-lane offset (the same for all six inputs) and rows past the sequence read
    // as zero (the hardware range check) without any select.
    auto fetch = [&](int t0c) {
        const uint32_t bytes = (uint32_t)min(L, te - t0c) * (uint32_t)C * (uint32_t)sizeof(IO);
        const size_t base = (size_t)t0c * C + h * NH;
        const IO* src[6] = {r, w, k, v, a, b};
#pragma unroll
        for (int q = CARRY ? 1 : 0; q < 6; ++q) {  // (r is for y only)
            const __amdgpu_buffer_rsrc_t rs =
                __builtin_amdgcn_make_buffer_rsrc(const_cast<IO*>(src[q] + base), 0, (int)bytes, 0x00020000);
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int off = ((2 * tp + e) * C + j0) * (int)sizeof(IO);
                const auto u = __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0);
                raw[q][e] = make_uint2((uint32_t)u[0], (uint32_t)u[1]);
            }
        }
        if (ident) raw[3][0] = raw[3][1] = make_uint2(0, 0);
    };
    // the tokens this block walks
    const int t_lo = SEG ? tb + seg * segs.cps * L : tb, t_hi = SEG && nsg > 1 ? min(te, t_lo + segs.cps * L) : te;
    fetch(t_lo);

    for (int t0 = t_lo; t0 < t_hi; t0 += L) {
        const int n = min(L, te - t0);
        [[maybe_unused]] const int ci = (t0 - tb) / L;  // chunk of the sequence: checkpoints 2 ci, 2 ci + 1
        // ---- A1: log2-decays of the thread's two tokens, their prefix over the chunk
        // (pair sums scanned over the wave's 4 lane rows = tokens 8w .. 8w+7 by lane
        // swaps, then the four wave totals through LDS), strong-decay test ---------
        bool slow = false;
        f32x4 lw[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int t = 2 * tp + e;
            const f32x4 wv = unpack4<IO>(raw[1][e]);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const float x = t < n ? -ex2(wv[c] * kLog2e) * kLog2e : 0.f;
                slow |= !(x >= kLog2DecayFloor);
                lw[e][c] = x;
            }
        }
        f32x4 inc, exc;  // inclusive / exclusive prefix of the pair sums over the wave's 4 rows
        const int g = lane >> 4;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float x = lw[0][c] + lw[1][c];
            const float p1 = lane_xor16(x);  // row g ^ 1
            const float p2 = lane_xor32(x + p1);  // rows (g ^ 2) & 2 and + 1
            exc[c] = (g >= 2 ? p2 : 0.f) + ((g & 1) ? p1 : 0.f);
            inc[c] = exc[c] + x;
        }
        if (g == 3) *reinterpret_cast<f32x4*>(&sm.tot[wave][j0]) = inc;
        const bool wave_slow = __ballot(slow) != 0;
        if (lane == 0) sm.slow[wave] = wave_slow ? 1 : 0;
        block_sync<kFetchB>();
        const int4 sl = *reinterpret_cast<const int4*>(sm.slow);
        const bool any_slow = (sl.x | sl.y | sl.z | sl.w) != 0;

        if (!any_slow) {
            // ---- A2: scaled operands as hi/lo planes ------------------------------
            {
                f32x4 base = {0.f, 0.f, 0.f, 0.f}, all = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const f32x4 tq = *reinterpret_cast<const f32x4*>(&sm.tot[q][j0]);
                    if (q < wave) base += tq;
                    all += tq;
                }
                const f32x4 DLv = {ex2(all.x), ex2(all.y), ex2(all.z), ex2(all.w)};  // D_L
                if (tp == 0) *reinterpret_cast<f32x4*>(&sm.DL[j0]) = DLv;
                const f32x4 ld_before = base + exc;  // log2 D of the token before 2tp
                const f32x4 ld_first = ld_before + lw[0];
                f32x4 vv[2], Dprev;
                uint2 kw[2][2], bw[2][2];  // hi / lo words of k^ and b^ for the two tokens
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const int t = 2 * tp + e;
                    const f32x4 ld = e == 0 ? ld_first : ld_first + lw[1];
                    const f32x4 rv = CARRY ? f32x4{} : unpack4<IO>(raw[0][e]), kv = unpack4<IO>(raw[2][e]);
                    const f32x4 av = unpack4<IO>(raw[4][e]), bv = unpack4<IO>(raw[5][e]);
                    vv[e] = unpack4<IO>(raw[3][e]);
                    f32x4 rt, at, kh, bh;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const float Dt = ex2(ld[c]), iD = ex2(-ld[c]);
                        const float Dtm1 = e == 0 ? ex2(ld_before[c]) : Dprev[c];
                        Dprev[c] = Dt;
                        rt[c] = rv[c] * Dt;
                        at[c] = av[c] * Dtm1;
                        kh[c] = kv[c] * iD;
                        bh[c] = bv[c] * iD;
                    }
                    uint2 hi, lo;
                    if constexpr (!CARRY) {
                        split4(rt.x, rt.y, rt.z, rt.w, hi, lo);
                        *reinterpret_cast<uint2*>(&sm.u.pa.Rt[0][t][j0]) = hi;
                        *reinterpret_cast<uint2*>(&sm.u.pa.Rt[1][t][j0]) = lo;
                    }
                    split4(at.x, at.y, at.z, at.w, hi, lo);
                    *reinterpret_cast<uint2*>(&sm.u.pa.At[0][t][j0]) = hi;
                    *reinterpret_cast<uint2*>(&sm.u.pa.At[1][t][j0]) = lo;
                    split4(kh.x, kh.y, kh.z, kh.w, kw[e][0], kw[e][1]);
                    *reinterpret_cast<uint2*>(&sm.u.pa.Kh[0][t][j0]) = kw[e][0];
                    *reinterpret_cast<uint2*>(&sm.u.pa.Kh[1][t][j0]) = kw[e][1];
                    split4(bh.x, bh.y, bh.z, bh.w, bw[e][0], bw[e][1]);
                    *reinterpret_cast<uint2*>(&sm.u.pa.Bh[0][t][j0]) = bw[e][0];
                    *reinterpret_cast<uint2*>(&sm.u.pa.Bh[1][t][j0]) = bw[e][1];
                }
                if constexpr (TRAIN) {
                    // D after token 15 (decay 1 past the chunk's last token)
                    if (tp == 7) *reinterpret_cast<f32x4*>(&sm.D15[j0]) = Dprev;
                }
                // channel c of tokens 2tp, 2tp+1 as one word, from the two tokens' words
                auto tword = [](const uint2& w0, const uint2& w1, int c) -> uint32_t {
                    const uint32_t a = c < 2 ? w0.x : w0.y, b = c < 2 ? w1.x : w1.y;
                    return (c & 1) ? ((a >> 16) | (b & 0xffff0000u)) : ((a & 0xffffu) | (b << 16));
                };
                // transposed planes: key / value j, tokens 2tp and 2tp+1 in one word
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int j = j0 + c;
                    uint32_t hi, lo;
                    if constexpr (kVExact) {
                        // the raw bf16 bits of channel j for tokens 2tp, 2tp+1 (no lo plane)
                        *reinterpret_cast<uint32_t*>(&sm.VT[0][0][0] + tswz(j, 2 * tp)) = tword(raw[3][0], raw[3][1], c);
                    } else {
                        split2(vv[0][c], vv[1][c], hi, lo);
                        *reinterpret_cast<uint32_t*>(&sm.VT[0][0][0] + tswz(j, 2 * tp)) = hi;
                        *reinterpret_cast<uint32_t*>(&sm.VT[1][0][0] + tswz(j, 2 * tp)) = lo;
                    }
                    *reinterpret_cast<uint32_t*>(&sm.KhT[0][0][0] + tswz(j, 2 * tp)) = tword(kw[0][0], kw[1][0], c);
                    *reinterpret_cast<uint32_t*>(&sm.KhT[1][0][0] + tswz(j, 2 * tp)) = tword(kw[0][1], kw[1][1], c);
                    *reinterpret_cast<uint32_t*>(&sm.BhT[0][0][0] + tswz(j, 2 * tp)) = tword(bw[0][0], bw[1][0], c);
                    *reinterpret_cast<uint32_t*>(&sm.BhT[1][0][0] + tswz(j, 2 * tp)) = tword(bw[0][1], bw[1][1], c);
                }
            }
        }
        block_sync<kFetchB>();

        if (any_slow) {
            // ---- exact token-serial update on a float32 copy of the state in LDS ----
            tile_io(&sm.u.Sf[0][0], SP, true);
            block_sync<kFetchB>();
            const int i = tid >> 2, q = tid & 3;
            for (int t = 0; t < n; ++t) {
                const size_t off = (size_t)(t0 + t) * C + h * NH;
                float sa = 0.f;
#pragma unroll
                for (int c = 0; c < 16; ++c) sa += tr::to_f32(a[off + q * 16 + c]) * sm.u.Sf[i][q * 16 + c];
                sa += __shfl_xor(sa, 1, 64);
                sa += __shfl_xor(sa, 2, 64);
                const float vi = ident ? 0.f : tr::to_f32(v[off + i]);
                float yi = 0.f;
#pragma unroll
                for (int c = 0; c < 16; ++c) {
                    const int jj = q * 16 + c;
                    const float wd = expf(-expf(tr::to_f32(w[off + jj])));
                    const float sv = sm.u.Sf[i][jj] * wd + tr::to_f32(k[off + jj]) * vi + sa * tr::to_f32(b[off + jj]);
                    sm.u.Sf[i][jj] = sv;
                    if constexpr (!CARRY) yi += sv * tr::to_f32(r[off + jj]);
                }
                if constexpr (!CARRY) {
                    yi += __shfl_xor(yi, 1, 64);
                    yi += __shfl_xor(yi, 2, 64);
                    if (q == 0) y[off + i] = tr::from_f32(yi);
                }
                if constexpr (TRAIN) {
                    if (q == 0) sa_out[off + i] = sa;
                    if (t == 15 || t == n - 1) {  // checkpoint 2 ci (after token 15) or 2 ci + 1
                        float* ck = gCk + (size_t)(2 * ci + (t >= 16 ? 1 : 0)) * (NH * NH) + i * NH + q * 16;
#pragma unroll
                        for (int c = 0; c < 16; ++c) ck[c] = sm.u.Sf[i][q * 16 + c];
                    }
                }
            }
            block_sync<kFetchB>();
            // back to the registers, and the hi/lo planes
            tile_io(&sm.u.Sf[0][0], SP, false);
            store_state_planes(&sm.Sp[0][0][0], ir_t, jt_t, tile, lane);
            if (t0 + L < t_hi) fetch(t0 + L);
            // the next chunk writes the region that holds Sf after its first barrier
            continue;
        }

        // the raw registers are free from here to the next phase A
        if (kFetchB && t0 + L < t_hi) fetch(t0 + L);

        // ---- B: two 32x32 tiles per wave, K = 64 over keys, sharing one operand:
        //   wave 0: X (value tile 0) and A_ab,   wave 1: X (value tile 1) and A_ak,
        //   wave 2: Y (value tile 0) and B_rb,   wave 3: Y (value tile 1) and B_rk,
        // where X[i][t] = S_i . a~_t, Y[i][t] = S_i . r~_t (lane l holds value rows
        // 32*vt + 8g + 4*(l/32) + 0..3 of token l%32), A_ab[s][t] = b^_s . a~_t,
        // A_ak[s][t] = k^_s . a~_t (s < t), B_rb[s][t] = b^_s . r~_t, B_rk[s][t] = k^_s . r~_t (s <= t)
        const f32x16 zero16 = {0.f};
        const int vt = wave & 1;                  // value tile of X / Y
        f32x16 accXY = zero16;                    // waves 0/1: X, waves 2/3: Y
        {
            const uint16_t* Q = wave < 2 ? &sm.u.pa.At[0][0][0] : &sm.u.pa.Rt[0][0][0];
            const uint16_t* P = (wave & 1) ? &sm.u.pa.Kh[0][0][0] : &sm.u.pa.Bh[0][0][0];
            f32x16 c1 = zero16;
            if constexpr (CARRY) {
                // the state only: X on waves 0 / 1, A_ab and A_ak on waves 2 / 3
                for (int k0 = 0; k0 < NH; k0 += 16) {
                    const uint16_t* At = &sm.u.pa.At[0][0][0];
                    const bf16x8_t q0 = frag(At, KP, 0, k0, lane), q1 = frag(At + RT_PLANE, KP, 0, k0, lane);
                    if (wave < 2)
                        accXY = mfma3(accXY, fragSp(&sm.Sp[0][0][0], 32 * vt, k0, lane),
                                      fragSp(&sm.Sp[1][0][0], 32 * vt, k0, lane), q0, q1);
                    else
                        c1 = mfma3(c1, frag(P, KP, 0, k0, lane), frag(P + RT_PLANE, KP, 0, k0, lane), q0, q1);
                }
            } else {
                for (int k0 = 0; k0 < NH; k0 += 16) {
                    const bf16x8_t s0 = fragSp(&sm.Sp[0][0][0], 32 * vt, k0, lane);
                    const bf16x8_t s1 = fragSp(&sm.Sp[1][0][0], 32 * vt, k0, lane);
                    const bf16x8_t q0 = frag(Q, KP, 0, k0, lane), q1 = frag(Q + RT_PLANE, KP, 0, k0, lane);
                    const bf16x8_t p0 = frag(P, KP, 0, k0, lane), p1 = frag(P + RT_PLANE, KP, 0, k0, lane);
                    accXY = mfma3(accXY, s0, s1, q0, q1);
                    c1 = mfma3(c1, p0, p1, q0, q1);
                }
            }
            constexpr int kA = CARRY ? 2 : 0;  // the wave with A_ab; the next one has A_ak
            // lane holds [s = 8g + 4(l/32) + e][t = l%32]
            const int tcol = lane & 31;
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int srow = 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3);
                const bool keep = CARRY || wave < 2 ? srow < tcol : srow <= tcol;
                c1[q] = keep ? c1[q] : 0.f;
            }
            // the products overwrite the planes they were computed from
            block_sync<kFetchB>();
            if (wave == kA) {
                float* AT = &sm.u.pb.AT[0][0];
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *reinterpret_cast<f32x4*>(AT + tcol * TP + 8 * g + 4 * (lane >> 5)) =
                        f32x4{c1[4 * g], c1[4 * g + 1], c1[4 * g + 2], c1[4 * g + 3]};
            } else if (!CARRY || wave == kA + 1) {
                uint16_t* out = wave == kA + 1 ? &sm.u.pb.AakT[0][0][0] : wave == 2 ? &sm.u.pb.BrbT[0][0][0]
                                                                               : &sm.u.pb.BrkT[0][0][0];
                store_planes_T(out, TQ, T32_PLANE, 0, 0, c1, lane);
            }
        }
        block_sync<kFetchB>();

        // ---- C: X += V^T A_ak (waves 0/1), stored as X^T; Y += V^T B_rk (waves 2/3) --
        if (!CARRY || wave < 2) {
            const uint16_t* M = wave < 2 ? &sm.u.pb.AakT[0][0][0] : &sm.u.pb.BrkT[0][0][0];
            for (int k0 = 0; k0 < L; k0 += 16) {
                const bf16x8_t a0 = frag(M, TQ, 0, k0, lane), a1 = frag(M + T32_PLANE, TQ, 0, k0, lane);
                const bf16x8_t v0 = fragT(&sm.VT[0][0][0], 32 * vt, k0, lane);
                const bf16x8_t v1 = kVExact ? v0 : fragT(&sm.VT[kVLo][0][0], 32 * vt, k0, lane);
                accXY = mfma_av<kVExact>(accXY, v0, v1, a0, a1);
            }
        }
        if (wave < 2) {
            // XT[t][i]: lane holds t = l%32, i = 32*wave + 8g + 4(l/32) + 0..3
            const int t = lane & 31;
            float* XT = &sm.u.pb.XT[0][0];
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<f32x4*>(XT + xtswz(t, 32 * wave + 8 * g + 4 * (lane >> 5))) =
                    f32x4{accXY[4 * g], accXY[4 * g + 1], accXY[4 * g + 2], accXY[4 * g + 3]};
        }
        block_sync<kFetchB>();

        // ---- triangular solve: SA[i][t] = X[i][t] + sum_{u<t} SA[i][u] A_ab[u][t] -----
        // Right-looking: lane q of row i keeps running sums for its targets t = 4m + q.
        // At step t the owner lane (q = t % 4) finishes sa_t, a quad broadcast hands it
        // to the other three lanes, and every lane pushes sa_t A_ab[t][4m + q] into its
        // later sums (which start from X); the dependency chain per step is one DPP
        // move and one FMA, the other FMAs fill its gaps.  Operands are read before the chain: the
        // lane's 8 X values up front, the transposed A_ab rows one group of 4 tokens
        // ahead as 16-byte reads.  Every wave also issues its state tile's k^^T V
        // products on the matrix cores (straight-line code in the same block as the
        // solve, so its MFMAs overlap the chain): the tile becomes S + (k^^T V)^T.
        bf16x8_t tv[2][2], tk[2][2];  // v and k^ fragments of the tile's two k steps (hi, lo)
        {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                tv[ks][0] = fragT(&sm.VT[0][0][0], 32 * ir_t, 16 * ks, lane);
                tv[ks][1] = kVExact ? tv[ks][0] : fragT(&sm.VT[kVLo][0][0], 32 * ir_t, 16 * ks, lane);
                tk[ks][0] = fragT(&sm.KhT[0][0][0], 32 * jt_t, 16 * ks, lane);
                tk[ks][1] = fragT(&sm.KhT[1][0][0], 32 * jt_t, 16 * ks, lane);
            }
        }
        // the tile's six MFMAs, one per group of the solve, in mfma3's order per k step
        // (lo.hi, hi.lo, hi.hi); the scheduling barrier keeps each in its group
        auto tile_mfma = [&](int m) {
            const int ks = m / 3, part = m % 3;
            if (kVExact && part == 1) return;  // hi(k^) . lo(v) = 0
            const bf16x8_t a = part == 0 ? tk[ks][1] : tk[ks][0];
            const bf16x8_t b = part == 1 ? tv[ks][1] : tv[ks][0];
            tile = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, tile, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        {
            const int i = tid >> 2, q = tid & 3;
            const float* XT = &sm.u.pb.XT[0][0];
            const float* AT = &sm.u.pb.AT[0][0];
            // pq[m]: X[i][4m + q] plus the terms pushed so far; it is SA[i][4m + q] from the
            // step of token 4m + q on (later pushes into it multiply A_ab entries that are 0)
            float pq[8];
#pragma unroll
            for (int m = 0; m < 8; ++m) pq[m] = XT[xtswz(4 * m + q, i)];
            f32x4 av[L / 4], nx[L / 4];  // AT[4m + q][4g .. 4g+3] for m >= g: this group / the next
#pragma unroll
            for (int m = 0; m < L / 4; ++m) av[m] = *reinterpret_cast<const f32x4*>(AT + (4 * m + q) * TP);
#pragma unroll
            for (int g = 0; g < L / 4; ++g) {
                if (g + 1 < L / 4) {
#pragma unroll
                    for (int m = g + 1; m < L / 4; ++m)
                        nx[m] = *reinterpret_cast<const f32x4*>(AT + (4 * m + q) * TP + 4 * (g + 1));
                }
                // (TRAIN: only the first 16 tokens' three here; phase D takes the
                // rest after it has stored the state after token 15)
                if (g >= 1 && g <= (TRAIN ? 3 : 6)) tile_mfma(g - 1);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float sat = quad_bcast(pq[g], e);  // sa_t, t = 4g + e, from lane e
#pragma unroll
                    for (int m = g; m < L / 4; ++m) pq[m] = fmaf(sat, av[m][e], pq[m]);
                }
#pragma unroll
                for (int m = g + 1; m < L / 4; ++m) av[m] = nx[m];
            }
            uint16_t* SA = &sm.u.pb.SA[0][0][0];
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const int o = saswz(i, 4 * m + q);
                split1(pq[m], SA[o], SA[SA_PLANE + o]);
            }
            if constexpr (TRAIN) {
#pragma unroll
                for (int m = 0; m < 8; ++m)
                    if (4 * m + q < n) sa_out[(size_t)(t0 + 4 * m + q) * C + h * NH + i] = pq[m];
            }
        }
        block_sync<kFetchB>();

        if (!kFetchB && t0 + L < t_hi) fetch(t0 + L);

        // ---- D: every wave: its state tile += (b^^T SA)^T, scaled by D_L and stored as the next chunk's
        //         planes; waves 2/3 also Y += SA B_rb (value tile wave - 2) and store y
        const uint16_t* SA = &sm.u.pb.SA[0][0][0];
        auto d_step = [&](int k0) {  // tokens k0 .. k0 + 15 of b^^T SA
            const bf16x8_t sa0 = fragSA(SA, 32 * ir_t, k0, lane), sa1 = fragSA(SA + SA_PLANE, 32 * ir_t, k0, lane);
            const bf16x8_t b0 = fragT(&sm.BhT[0][0][0], 32 * jt_t, k0, lane);
            const bf16x8_t b1 = fragT(&sm.BhT[1][0][0], 32 * jt_t, k0, lane);
            tile = mfma3(tile, b0, b1, sa0, sa1);
        };
        d_step(0);
        if constexpr (TRAIN) {
            // the state after token 15 (or after the chunk's last token when n <= 16, the later
            // tokens adding nothing): (S + the first 16 tokens' k^^T V + b^^T SA) diag(D_15)
            f32x16 mid;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 dv = *reinterpret_cast<const f32x4*>(&sm.D15[32 * jt_t + 8 * g + 4 * (lane >> 5)]);
#pragma unroll
                for (int e = 0; e < 4; ++e) mid[4 * g + e] = tile[4 * g + e] * dv[e];
            }
            put_state(gCk + (size_t)(2 * ci) * (NH * NH), mid);
            tile_mfma(3);
            tile_mfma(4);
            tile_mfma(5);
        }
        d_step(16);
        // S' = (S + k^^T V + b^^T SA) diag(D_L)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 dv = *reinterpret_cast<const f32x4*>(&sm.DL[32 * jt_t + 8 * g + 4 * (lane >> 5)]);
#pragma unroll
            for (int e = 0; e < 4; ++e) tile[4 * g + e] *= dv[e];
        }
        if constexpr (TRAIN) {
            if (n > 16) put_state(gCk + (size_t)(2 * ci + 1) * (NH * NH), tile);  // after the chunk's last token
        }
        store_state_planes(&sm.Sp[0][0][0], ir_t, jt_t, tile, lane);
        if (!CARRY && wave >= 2) {
            for (int k0 = 0; k0 < L; k0 += 16) {
                const bf16x8_t p0 = frag(&sm.u.pb.BrbT[0][0][0], TQ, 0, k0, lane);
                const bf16x8_t p1 = frag(&sm.u.pb.BrbT[1][0][0], TQ, 0, k0, lane);
                const bf16x8_t s0 = fragSA(SA, 32 * vt, k0, lane), s1 = fragSA(SA + SA_PLANE, 32 * vt, k0, lane);
                accXY = mfma3(accXY, s0, s1, p0, p1);
            }
            // y[t0 + l%32][32*vt + 8g + 4(l/32) + 0..3]: one 8-byte store per g
            const int t = lane & 31;
            if (t < n) {
                IO* yr = y + (size_t)(t0 + t) * C + h * NH + 32 * vt + 4 * (lane >> 5);
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *reinterpret_cast<uint2*>(yr + 8 * g) =
                        pack4<IO>(accXY[4 * g], accXY[4 * g + 1], accXY[4 * g + 2], accXY[4 * g + 3]);
            }
        }
        // No barrier here: the next chunk's first LDS writes (tot, slow) touch nothing
        // read in phase D, and its barriers precede every other write (the next phase B
        // reads the state planes written here after two of them).
    }
    // the final state, straight from the registers
    if constexpr (CARRY) {
        tile_io((ident ? seg_m : seg_n) + (size_t)unit * (NH * NH), NH, true);
    } else {
        if ((!TRAIN || gS != nullptr) && (!SEG || seg == nsg - 1)) tile_io(gS, NH, true);
    }
}

// Cost of a launch per chunk of its walk, in microseconds: a block alone on its CU takes 4.55 us per chunk
// (bf16, H = 32), two on a CU 6.2 us for both (float16 and float32 have one block per CU); more blocks run in
// rounds.
float walk_cost(int64_t blocks, bool two_per_cu)
{
    if (blocks <= 256) return 4.55f;
    return two_per_cu ? 6.2f * (float)((blocks + 511) / 512) : 4.55f * (float)((blocks + 255) / 256);
}

}  // namespace

hipError_t launch_wkv7_fwd32(const WkvSegs& m, int H, int T_uniform, const int32_t* cu, const int32_t* slot_idx,
                             int pool_slots, int total, float* state, const float* r, const float* w, const float* k,
                             const float* v, const float* a, const float* b, float* y, const float* s0, float* ckpt,
                             float* sa, float* ws, hipStream_t stream);

// Segments of a launch; cps = 0 (unsplit) where that is not slower.  n segments per sequence cost the state
// pass (0.75 of a full walk per chunk; 2 n - 3 blocks per unit), the scan (0.5 us a step), two more launches and
// the full pass over n segments, against one block per unit over the whole sequence.  Two launches are 9 us on the
// device; in the training operator, where a call this small waits for its caller (110 us of autograd for 20 of
// kernels), also what they cost the caller, 18 us.  Ragged sequences count with their average length, and unsplit
// with a quarter more: the launch ends with its longest one.  Measured (us, bf16, unsplit -> split): 12 units
// 128 tokens 22 -> 20, 12 x 512 76 -> 31, 32 x 1000 148 -> 54, 32 x 4096 580 -> 150, 64 x 256 40 -> 35,
// 64 x 2048 291 -> 146, 128 x 1000 148 -> 131, 60 ragged of 83 - 322 49 -> 41; not split by the model and slower
// split: 32 x 64 13 -> 18, 64 x 160 27 -> 30, 128 x 384 58 -> 60, 192 x 4096 583 -> 679, 256 x 4096 588 -> 744.
static WkvSegs plan_segments(int nseq, int H, int T_uniform, const int32_t* cu, int total, bool two_per_cu, bool train)
{
    WkvSegs m = {nseq, 0, 0, T_uniform, total, cu};
    const int64_t units = (int64_t)nseq * H;
    const int per_seq = cu == nullptr ? (T_uniform + L - 1) / L : (int)(((int64_t)total + nseq * L - 1) / ((int64_t)nseq * L));
    if (units >= 256) return m;
    float best = (cu == nullptr || nseq == 1 ? 1.f : 1.25f) * per_seq * walk_cost(units, two_per_cu);
    for (int n = 2; n <= 32 && n <= per_seq; ++n) {
        const int cps = (per_seq + n - 1) / n, nn = (per_seq + cps - 1) / cps;
        const float cost = cps * (0.75f * walk_cost(units * (2 * nn - 3), two_per_cu) +
                                  walk_cost(units * nn, two_per_cu)) + 0.5f * nn + (train ? 18.f : 9.f);
        if (cost < best) {
            best = cost;
            m.cps = cps;
        }
    }
    if (m.cps > 0)
        m.gmax = cu == nullptr ? nseq * ((per_seq + m.cps - 1) / m.cps) : total / (m.cps * L) + nseq;
    return m;
}

// floats of workspace with which a launch of these sizes may run in segments; without it, it runs unsplit
int64_t wkv7_chunk_ws(int nseq, int H, int T_uniform, bool ragged, int total, bool two_per_cu, bool train)
{
    static const int32_t some = 0;
    const WkvSegs m = plan_segments(nseq, H, T_uniform, ragged ? &some : nullptr, total, two_per_cu, train);
    return (int64_t)m.gmax * H * 2 * NH * NH;
}

template <typename IO, bool TRAIN>
static hipError_t launch_chunk2(int nseq, int H, int T_uniform, const int32_t* cu_seqlens, const int32_t* slot_idx,
                                int pool_slots, int total, float* state, const void* r, const void* w, const void* k,
                                const void* v, const void* a, const void* b, void* y, const float* s0, float* ckpt,
                                float* sa, float* ws, int64_t ws_floats, hipStream_t stream)
{
    WkvSegs m = plan_segments(nseq, H, T_uniform, cu_seqlens, total, std::is_same<IO, bf16_t>::value, TRAIN);
    const int64_t half = (int64_t)m.gmax * H * NH * NH;
    if (m.cps > 0 && (ws == nullptr || ws_floats < 2 * half)) m.cps = 0;
    float *sm = ws, *sn = ws + half;
    const unsigned groups = m.cps > 0 ? (unsigned)m.gmax : (unsigned)nseq;
    auto walk = [&](auto kern, dim3 grid, float* st, float* ck, float* sa_) -> hipError_t {
        hipLaunchKernelGGL(kern, grid, dim3(256), 0, stream, H, T_uniform, cu_seqlens, slot_idx, pool_slots, total, m,
                           sm, sn, st, (const IO*)r, (const IO*)w, (const IO*)k, (const IO*)v, (const IO*)a,
                           (const IO*)b, (IO*)y, s0, ck, sa_);
        return hipGetLastError();
    };
    const dim3 grid(groups * (unsigned)H);
    if (m.cps == 0) return walk(wkv7_chunk2_kernel<IO, TRAIN, false, false>, grid, state, ckpt, sa);
    hipError_t e = walk(wkv7_chunk2_kernel<IO, false, true, true>, dim3(grid.x, 2), TRAIN ? nullptr : state, nullptr,
                        nullptr);
    if (e == hipSuccess) e = launch_wkv7_scan_forward(m, H, sm, sn, stream);
    if (e != hipSuccess) return e;
    return walk(wkv7_chunk2_kernel<IO, TRAIN, true, false>, grid, state, ckpt, sa);
}

template <typename IO>
hipError_t launch_wkv7_chunk(int nseq, int H, int T_uniform, const int32_t* cu_seqlens, const int32_t* slot_idx,
                             int pool_slots, int total_tokens, float* state, const void* r, const void* w,
                             const void* k, const void* v, const void* a, const void* b, void* y, float* ws,
                             int64_t ws_floats, hipStream_t stream)
{
    if constexpr (sizeof(IO) == 4) {
        WkvSegs m = plan_segments(nseq, H, T_uniform, cu_seqlens, total_tokens, false, false);
        if (ws == nullptr || ws_floats < (int64_t)m.gmax * H * 2 * NH * NH) m.cps = 0;
        return launch_wkv7_fwd32(m, H, T_uniform, cu_seqlens, slot_idx, pool_slots, total_tokens, state,
                                 (const float*)r, (const float*)w, (const float*)k, (const float*)v, (const float*)a,
                                 (const float*)b, (float*)y, nullptr, nullptr, nullptr, ws, stream);
    } else {
        return launch_chunk2<IO, false>(nseq, H, T_uniform, cu_seqlens, slot_idx, pool_slots, total_tokens, state, r,
                                        w, k, v, a, b, y, nullptr, nullptr, nullptr, ws, ws_floats, stream);
    }
}

// The training operator's forward in chunked form: B sequences of T
// tokens, initial state s0 (zero when null), final state s_out (not written when
// null), checkpoints and sa as the token-serial training forward writes them.
template <typename IO>
hipError_t launch_wkv7_chunk_train(int B, int T, int H, const void* r, const void* w, const void* k, const void* v,
                                   const void* a, const void* b, void* y, const float* s0, float* s_out, float* ckpt,
                                   float* sa, float* ws, int64_t ws_floats, hipStream_t stream)
{
    if constexpr (sizeof(IO) == 4) {
        WkvSegs m = plan_segments(B, H, T, nullptr, B * T, false, true);
        if (ws == nullptr || ws_floats < (int64_t)m.gmax * H * 2 * NH * NH) m.cps = 0;
        return launch_wkv7_fwd32(m, H, T, nullptr, nullptr, B, B * T, s_out, (const float*)r, (const float*)w,
                                 (const float*)k, (const float*)v, (const float*)a, (const float*)b, (float*)y, s0,
                                 ckpt, sa, ws, stream);
    } else {
        return launch_chunk2<IO, true>(B, H, T, nullptr, nullptr, B, B * T, s_out, r, w, k, v, a, b, y, s0, ckpt, sa,
                                       ws, ws_floats, stream);
    }
}

#define RWKV7_INST(IO)                                                                                               \
    template hipError_t launch_wkv7_chunk<IO>(int, int, int, const int32_t*, const int32_t*, int, int, float*,       \
                                              const void*, const void*, const void*, const void*, const void*,      \
                                              const void*, void*, float*, int64_t, hipStream_t);
#define RWKV7_INST_TRAIN(IO)                                                                                         \
    template hipError_t launch_wkv7_chunk_train<IO>(int, int, int, const void*, const void*, const void*,            \
                                                    const void*, const void*, const void*, void*, const float*,     \
                                                    float*, float*, float*, float*, int64_t, hipStream_t);
RWKV7_INST(float)
RWKV7_INST(bf16_t)
RWKV7_INST(f16_t)
RWKV7_INST_TRAIN(float)
RWKV7_INST_TRAIN(bf16_t)
RWKV7_INST_TRAIN(f16_t)
