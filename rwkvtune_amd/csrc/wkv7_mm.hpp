// 32-wide matrix products on LDS operands for the chunked WKV7 kernels that keep
// every operand once, in either orientation, as one 32-bit word per element.
//
// A word is a float, or ("packed") the element's bf16 hi and lo parts in its upper
// and lower half (x = hi + lo + e, |e| <= 2^-17 |x|).  Packed operands go to the
// bf16 matrix cores with two byte permutes per pair of elements; the split is done
// once, by the writer, where splitting at each read cost three times as many VALU
// instructions.  Products of two float operands can run on the float32 MFMA instead.
#pragma once

#include "common.hpp"

#include <type_traits>

namespace wkvmm {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int SP = 68;  // row stride of [*][64] matrices: 16 consecutive rows on distinct 16-byte bank groups
constexpr int TP = 36;  // row stride of [*][32] matrices

// bf16 parts of two values as the words hi(x1) hi(x0) and lo(x1) lo(x0)
__device__ __forceinline__ void split2(float x0, float x1, uint32_t& hi, uint32_t& lo) {
    const f32x2 v = {x0, x1};
    hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
    const f32x2 r = {x0 - __uint_as_float(hi << 16), x1 - __uint_as_float(hi & 0xffff0000u)};
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf16x2_t));
}

// two elements as words of a matrix
template <bool PK>
__device__ __forceinline__ f32x2 words2(float x0, float x1) {
    if constexpr (!PK) {
        return f32x2{x0, x1};
    } else {
        uint32_t h, l;
        split2(x0, x1, h, l);
        return f32x2{__uint_as_float(__builtin_amdgcn_perm(h, l, 0x05040100u)),
                     __uint_as_float(__builtin_amdgcn_perm(h, l, 0x07060302u))};
    }
}
template <bool PK>
__device__ __forceinline__ f32x4 words4(f32x4 x) {
    const f32x2 a = words2<PK>(x.x, x.y), b = words2<PK>(x.z, x.w);
    return f32x4{a.x, a.y, b.x, b.y};
}
// the value of a word
template <bool PK>
__device__ __forceinline__ float value(float w) {
    if constexpr (!PK) return w;
    const uint32_t u = __float_as_uint(w);
    return __uint_as_float(u & 0xffff0000u) + __uint_as_float(u << 16);
}

struct F8 {
    float v[8];
};

// Operand of a 32-wide tile for 16 contraction terms: lane l holds index l % 32 at terms
// 8 (l / 32) + 0..7.  Not TR: index = row, terms along the row; TR: index = column, terms down the rows.
template <bool TR>
__device__ __forceinline__ F8 operand(const float* P, int ld, int x0, int k0, int lane) {
    F8 o;
    const int c = lane & 31, k = k0 + 8 * (lane >> 5);
    if constexpr (TR) {
#pragma unroll
        for (int e = 0; e < 8; ++e) o.v[e] = P[(k + e) * ld + x0 + c];
    } else {
        const f32x4* p = reinterpret_cast<const f32x4*>(P + (x0 + c) * ld + k);
        const f32x4 a = p[0], b = p[1];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            o.v[e] = a[e];
            o.v[4 + e] = b[e];
        }
    }
    return o;
}

// hi / lo bf16 vectors of an operand (LO: the lo part is wanted)
template <bool PK, bool LO>
__device__ __forceinline__ void parts(const F8& x, bf16x8_t& hi, bf16x8_t& lo) {
    uint32_t h[4], l[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if constexpr (PK) {
            const uint32_t d0 = __float_as_uint(x.v[2 * q]), d1 = __float_as_uint(x.v[2 * q + 1]);
            h[q] = __builtin_amdgcn_perm(d1, d0, 0x07060302u);
            l[q] = LO ? __builtin_amdgcn_perm(d1, d0, 0x05040100u) : 0;
        } else {
            split2(x.v[2 * q], x.v[2 * q + 1], h[q], l[q]);
        }
    }
    hi = __builtin_bit_cast(bf16x8_t, make_uint4(h[0], h[1], h[2], h[3]));
    lo = __builtin_bit_cast(bf16x8_t, make_uint4(l[0], l[1], l[2], l[3]));
}

// How a matrix is stored: float words or packed ones, and whether its values are exact in bf16
template <bool PK, bool EX = false>
struct Mat {
    const float* p;
    int ld;
    static constexpr bool packed = PK, exact = EX;
};

// acc[4g + e] (lane l) += sum_k A[8g + 4 (l / 32) + e][k] B[k][l % 32] over K terms, the tile at index
// a0 of A and b0 of B.  F32: float32 MFMAs (both operands float words); otherwise bf16 parts,
// lo.hi + hi.lo + hi.hi (the terms with the lo part of an exact operand are 0 and left out).
//
// 32 terms of a float32 product are summed by themselves and added to acc once: one rounding on acc, which a recurrence
// carries along, instead of one for each term (final state after 2,000 tokens: 2.5e-7 -> 2.0e-7 from float64).
template <bool F32, bool TA, bool TB, int K, class MA, class MB>
__device__ __forceinline__ void mm(f32x16& acc, MA A, int a0, MB B, int b0, int lane) {
    if constexpr (F32) {
        static_assert(!MA::packed && !MB::packed, "float operands");
        constexpr int KB = K < 32 ? K : 32;
#pragma unroll
        for (int k1 = 0; k1 < K; k1 += KB) {
            f32x16 t = {0.f};
#pragma unroll
            for (int k0 = k1; k0 < k1 + KB; k0 += 16) {
                const F8 a = operand<TA>(A.p, A.ld, a0, k0, lane), b = operand<TB>(B.p, B.ld, b0, k0, lane);
#pragma unroll
                for (int e = 0; e < 8; ++e) t = __builtin_amdgcn_mfma_f32_32x32x2f32(a.v[e], b.v[e], t, 0, 0, 0);
            }
            acc += t;
        }
    } else {
#pragma unroll
        for (int k0 = 0; k0 < K; k0 += 16) {
            const F8 a = operand<TA>(A.p, A.ld, a0, k0, lane), b = operand<TB>(B.p, B.ld, b0, k0, lane);
            bf16x8_t ah, al, bh, bl;
            parts<MA::packed, !MA::exact>(a, ah, al);
            parts<MB::packed, !MB::exact>(b, bh, bl);
            if constexpr (!MA::exact) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bh, acc, 0, 0, 0);
            if constexpr (!MB::exact) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bl, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bh, acc, 0, 0, 0);
        }
    }
}

// row of accumulator element q in a lane
__device__ __forceinline__ int acc_row(int q, int lane) { return 8 * (q >> 2) + 4 * (lane >> 5) + (q & 3); }

// acc as a tile of a matrix: M[r0 + row][c0 + l % 32]
template <bool PK>
__device__ __forceinline__ void put(float* M, int ld, int r0, int c0, const f32x16& acc, int lane) {
#pragma unroll
    for (int q = 0; q < 16; q += 2) {
        const f32x2 x = words2<PK>(acc[q], acc[q + 1]);
        float* p = M + (r0 + acc_row(q, lane)) * ld + c0 + (lane & 31);
        p[0] = x.x;
        p[ld] = x.y;
    }
}
// the transpose: M[r0 + l % 32][c0 + row], four columns per store
template <bool PK>
__device__ __forceinline__ void put_t(float* M, int ld, int r0, int c0, const f32x16& acc, int lane) {
#pragma unroll
    for (int g = 0; g < 4; ++g)
        *reinterpret_cast<f32x4*>(M + (r0 + (lane & 31)) * ld + c0 + 8 * g + 4 * (lane >> 5)) =
            words4<PK>(f32x4{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]});
}
// keep the elements with row < col (row <= col unless STRICT)
template <bool STRICT>
__device__ __forceinline__ void mask_upper(f32x16& acc, int lane) {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int s = acc_row(q, lane), t = lane & 31;
        acc[q] = (STRICT ? s < t : s <= t) ? acc[q] : 0.f;
    }
}

// lane e of each quad, to all four lanes; e is a constant after unrolling
__device__ __forceinline__ float quad_bcast(float x, int e) {
    switch (e) {
    case 0: return __builtin_amdgcn_mov_dpp(x, 0x00, 0xf, 0xf, false);
    case 1: return __builtin_amdgcn_mov_dpp(x, 0x55, 0xf, 0xf, false);
    case 2: return __builtin_amdgcn_mov_dpp(x, 0xaa, 0xf, 0xf, false);
    default: return __builtin_amdgcn_mov_dpp(x, 0xff, 0xf, 0xf, false);
    }
}

// T = (I - A)^-1 of a strictly upper 32 x 32 matrix by 128 threads (id = 0 .. 127): thread (s, q) keeps
// the running sums x_t = e_s[t] + sum_{u < t} x_u A[u][t] of row s for its targets t = 4m + q; at step u
// the owner lane hands x_u to its quad by DPP.  At: A transposed, [t][u], float words.
template <bool PK>
__device__ __forceinline__ void unit_upper_inverse(const float* At, float* Tm, int id) {
    const int s = id >> 2, q = id & 3;
    float pq[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) pq[m] = 4 * m + q == s ? 1.f : 0.f;
#pragma unroll
    for (int g = 0; g < 8; ++g) {
        f32x4 av[8];
#pragma unroll
        for (int m = g; m < 8; ++m) av[m] = *reinterpret_cast<const f32x4*>(At + (4 * m + q) * TP + 4 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float x = quad_bcast(pq[g], e);
#pragma unroll
            for (int m = g; m < 8; ++m) pq[m] = fmaf(x, av[m][e], pq[m]);
        }
    }
#pragma unroll
    for (int m = 0; m < 8; m += 2) {
        const f32x2 x = words2<PK>(pq[m], pq[m + 1]);
        Tm[s * TP + 4 * m + q] = x.x;
        Tm[s * TP + 4 * m + 4 + q] = x.y;
    }
}

// The value, unknown to the compiler: keeps it from computing every phase's LDS addresses ahead of a
// chunk loop and holding them in (spilled) registers.
__device__ __forceinline__ int opaque(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// Block barrier for data exchanged through LDS.  __syncthreads() also waits for every global load and store
// of the wave, which puts the latency of loads issued a chunk ahead back into the phase they were issued in.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ float ex2(float x) { return __builtin_amdgcn_exp2f(x); }

// The log2-decay sums of float32 inputs are kept in double: a float32 sum of 32 of them is off by up to 2e-7,
// which the scaled operands would carry as their relative error.
__device__ __forceinline__ float ex2(double x) {
    const float hi = (float)x, lo = (float)(x - (double)hi);
    return __builtin_amdgcn_exp2f(hi) * fmaf(lo, 0.6931471805599453f, 1.f);
}
__device__ __forceinline__ float xor32(float x) { return lane_xor32(x); }
__device__ __forceinline__ double xor32(double x) {
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __float_as_uint(lane_xor32(__uint_as_float((uint32_t)u)));
    const uint32_t hi = __float_as_uint(lane_xor32(__uint_as_float((uint32_t)(u >> 32))));
    return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}
__device__ __forceinline__ double xor16(double x) {
    const uint64_t u = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __float_as_uint(lane_xor16(__uint_as_float((uint32_t)u)));
    const uint32_t hi = __float_as_uint(lane_xor16(__uint_as_float((uint32_t)(u >> 32))));
    return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}
__device__ __forceinline__ float xor16(float x) { return lane_xor16(x); }

// Two floats as two adjacent 16-bit values (round to nearest even, the hardware conversions)
template <typename IO>
__device__ __forceinline__ uint32_t pack2(float x0, float x1) {
    const f32x2 v = {x0, x1};
    if constexpr (std::is_same<IO, bf16_t>::value) {
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
    } else {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, h2));
    }
}

// A chunk's rows of one head: `rows` rows of 64 values, `stride` bytes apart, as a buffer resource that
// ends after the last row.  Loads past it read zero and stores past it are dropped, without a select, and
// the same 32-bit lane offset serves every tensor of the chunk.
struct Rows {
    __amdgpu_buffer_rsrc_t rs;
    __device__ __forceinline__ Rows(const void* p, int rows, uint32_t stride, int es)
        : rs(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)((rows - 1) * stride + 64 * es),
                                               0x00020000)) {}
};

// CH consecutive values of one token (CH = 2 or 4) as loaded: converted only where they are used, so
// that a load issued ahead of its use is not waited for at once
template <typename IO, int CH>
struct Raw {
    static constexpr int N = CH * (int)sizeof(IO) / 4;
    uint32_t u[N];
    __device__ __forceinline__ void load(const Rows& r, uint32_t off) {
        if constexpr (N == 4) {
            const auto x = __builtin_amdgcn_raw_buffer_load_b128(r.rs, (int)off, 0, 0);
            u[0] = x[0]; u[1] = x[1]; u[2] = x[2]; u[3] = x[3];
        } else if constexpr (N == 2) {
            const auto x = __builtin_amdgcn_raw_buffer_load_b64(r.rs, (int)off, 0, 0);
            u[0] = x[0]; u[1] = x[1];
        } else {
            u[0] = __builtin_amdgcn_raw_buffer_load_b32(r.rs, (int)off, 0, 0);
        }
    }
    __device__ __forceinline__ void get(float (&x)[CH]) const {
        typedef io_traits<IO> tr;
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            if constexpr (sizeof(IO) == 4) x[e] = __uint_as_float(u[e]);
            else x[e] = tr::to_f32(__builtin_bit_cast(IO, (uint16_t)(u[e / 2] >> (16 * (e & 1)))));
        }
    }
};
template <typename IO, int CH>
__device__ __forceinline__ void store_ch(const Rows& r, uint32_t off, const float (&x)[CH]) {
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    if constexpr (sizeof(IO) == 4) {
#pragma unroll
        for (int q = 0; q < CH; q += 2)
            __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(x[q]), __float_as_uint(x[q + 1])}, r.rs,
                                                  (int)off + 4 * q, 0, 0);
    } else if constexpr (CH == 2) {
        __builtin_amdgcn_raw_buffer_store_b32(pack2<IO>(x[0], x[1]), r.rs, (int)off, 0, 0);
    } else {
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack2<IO>(x[0], x[1]), pack2<IO>(x[2], x[3])}, r.rs, (int)off, 0,
                                              0);
    }
}
// CH words of a matrix row
template <bool PK, int CH>
__device__ __forceinline__ void put_ch(float* p, const float (&x)[CH]) {
    if constexpr (CH == 4) {
        *reinterpret_cast<f32x4*>(p) = words4<PK>(f32x4{x[0], x[1], x[2], x[3]});
    } else {
        *reinterpret_cast<f32x2*>(p) = words2<PK>(x[0], x[1]);
    }
}
template <int CH>
__device__ __forceinline__ void get_ch(const float* p, float (&x)[CH]) {
#pragma unroll
    for (int q = 0; q < CH; q += 2) {
        const f32x2 v = *reinterpret_cast<const f32x2*>(p + q);
        x[q] = v.x;
        x[q + 1] = v.y;
    }
}

}  // namespace wkvmm
