// One decode step of a bf16 model in one call: the launches of every layer (row kernels, grouped projection
// GEMMs, fused time-mix) and of the final norm, enqueued from native code.
//
// A layer is eight launches of a few microseconds; issued one by one through the Python binding they cost
// ~130 us of host time per layer (argument conversion, workspace queries, about ten allocations), several
// times the GPU's.  Here the layers' pointers are read from a table the caller lays out with the packed
// weights, the activations are slices of one scratch buffer, and a launch costs its enqueueing.  One token of
// a 12-layer, 768-wide model (forward_with_state, with the parameter check and the state copies also
// shortened): 1,810 -> 572 us; two 2,048-wide layers at 200 rows are bound by the GPU (334 -> 333 us).
#include <stdint.h>

#include "rwkv7_hip.h"

int capi_invalid(const char* msg);  // sets the library's error message (capi.hip)

namespace {

constexpr int kBf16 = RWKV7_DTYPE_BF16;

struct Layout {
    // byte offsets of the scratch sections
    int64_t x_res, x_mid, v_first, mixes, xk, rkv, up, o, hk, h, total;
    int64_t rank;  // row stride of the LoRA hidden rows
};

int64_t take(int64_t& at, int64_t bytes) {
    const int64_t here = at;
    at += (bytes + 255) / 256 * 256;
    return here;
}

Layout layout_of(int64_t M, int64_t C, int64_t FF, int n_layer, const rwkv7_layer* layers) {
    Layout l;
    l.rank = 8;
    for (int i = 0; i < n_layer; ++i)
        for (int q = 0; q < 4; ++q)
            if (layers[i].rank[q] > l.rank) l.rank = layers[i].rank[q];
    l.rank = (l.rank + 7) / 8 * 8;
    int64_t at = 0;
    l.x_res = take(at, 4 * M * C);
    l.x_mid = take(at, 4 * M * C);
    l.v_first = take(at, 4 * M * C);
    l.mixes = take(at, 2 * 7 * M * C);
    l.xk = take(at, 2 * M * C);
    l.rkv = take(at, 2 * 3 * M * C);
    l.up = take(at, 2 * 4 * M * C);
    l.o = take(at, 2 * M * C);
    l.hk = take(at, 2 * M * FF);
    l.h = take(at, 2 * 4 * M * l.rank);
    l.total = at;
    return l;
}

// one grouped GEMM launch under construction
struct Group {
    const void* A[8];
    const void* B[8];
    void* C[8];
    int64_t lda[8], ldc[8];
    int N[8], K[8], epi[8], n = 0;

    void add(const void* a, int64_t la, const void* b, void* c, int64_t lc, int64_t N_, int64_t K_, int e) {
        A[n] = a;
        B[n] = b;
        C[n] = c;
        lda[n] = la;
        ldc[n] = lc;
        N[n] = (int)N_;
        K[n] = (int)K_;
        epi[n] = e;
        ++n;
    }
    int run(int64_t M, float* ws, int64_t ws_floats, void* st) const {
        return rwkv7_gemm_decode(M, n, A, B, C, lda, ldc, N, K, epi, ws, ws_floats, st);
    }
};

// r, k, v and the LoRA downs (tanh on w, sigmoid on g) of a layer
Group downs_of(const rwkv7_layer& l, int64_t M, int64_t C, uint16_t* mixes, uint16_t* rkv, uint16_t* h, int64_t rank) {
    Group g;
    const void* w[3] = {l.r, l.k, l.v};
    for (int q = 0; q < 3; ++q) g.add(mixes + q * M * C, C, w[q], rkv + q * M * C, C, C, C, 0);
    const int src[4] = {3, 4, 5, 2}, epi[4] = {2, 0, 3, 0};  // xw, xa, xg, xv
    for (int q = 0; q < 4; ++q)
        if (l.down[q] != nullptr)
            g.add(mixes + src[q] * M * C, C, l.down[q], h + q * M * rank, rank, l.rank[q], C, epi[q]);
    return g;
}

Group ups_of(const rwkv7_layer& l, int64_t M, int64_t C, uint16_t* h, uint16_t* up, int64_t rank) {
    Group g;
    for (int q = 0; q < 4; ++q)
        if (l.up[q] != nullptr) g.add(h + q * M * rank, rank, l.up[q], up + q * M * C, C, C, l.rank[q], 0);
    return g;
}

Group key_of(const rwkv7_layer& l, int64_t M, int64_t C, int64_t FF, uint16_t* xk, uint16_t* hk) {
    Group g;
    g.add(xk, C, l.fk, hk, FF, FF, C, 1);  // relu^2
    return g;
}

}  // namespace

extern "C" int64_t rwkv7_decode_layers_scratch(int64_t M, int64_t C, int64_t FF, int n_layer,
                                               const rwkv7_layer* layers) {
    if (M <= 0 || C <= 0 || FF <= 0 || n_layer < 0 || (n_layer > 0 && layers == nullptr)) return -1;
    return layout_of(M, C, FF, n_layer, layers).total;
}

extern "C" int64_t rwkv7_decode_layers_ws_floats(int64_t M, int64_t C, int64_t FF, int n_layer,
                                                 const rwkv7_layer* layers) {
    if (M <= 0 || C <= 0 || FF <= 0 || n_layer < 0 || (n_layer > 0 && layers == nullptr)) return -1;
    int64_t need = 0;
    auto most = [&](int64_t n) {
        if (n < 0 || need < 0) need = -1;
        else if (n > need) need = n;
    };
    for (int i = 0; i < n_layer; ++i) {
        const Group d = downs_of(layers[i], M, C, nullptr, nullptr, nullptr, 0);
        const Group u = ups_of(layers[i], M, C, nullptr, nullptr, 0);
        const Group f = key_of(layers[i], M, C, FF, nullptr, nullptr);
        most(rwkv7_gemm_decode_workspace(M, d.n, d.N, d.K));
        most(rwkv7_gemm_decode_workspace(M, u.n, u.N, u.K));
        most(rwkv7_gemm_decode_workspace(M, f.n, f.N, f.K));
        const int po = rwkv7_gemm_decode_partial_count(M, (int)C, (int)C);
        const int pf = rwkv7_gemm_decode_partial_count(M, (int)C, (int)FF);
        if (po < 1 || pf < 1) return -1;
        most((int64_t)po * M * C);
        most((int64_t)pf * M * C);
    }
    return need;
}

extern "C" int rwkv7_decode_layers(int64_t M, int64_t C, int64_t FF, int n_layer, const rwkv7_layer* layers,
                                   const int64_t* tokens, const void* emb, int64_t vocab, const int32_t* row_slot,
                                   const int32_t* row_last, float* kv, float* att_x, float* ffn_x,
                                   int64_t pool_slots, const float* ln_w, const float* ln_b,
                                   const int32_t* logit_rows, int64_t n_out, void* out, void* scratch,
                                   int64_t scratch_bytes, float* ws, int64_t ws_floats, void* stream) {
    const int64_t need = rwkv7_decode_layers_scratch(M, C, FF, n_layer, layers);
    // (the sub-calls check everything that reaches them; these are the ones read here)
    if (need < 0 || n_layer < 1 || !scratch || scratch_bytes < need || (((uintptr_t)scratch) & 255) || !kv || !att_x ||
        !ffn_x || pool_slots < 0)
        return capi_invalid("rwkv7_decode_layers: bad sizes, a null pointer, or a scratch buffer too small or not "
                            "256-byte aligned");
    const Layout l = layout_of(M, C, FF, n_layer, layers);
    char* base = (char*)scratch;
    float *x_res = (float*)(base + l.x_res), *x_mid = (float*)(base + l.x_mid), *v_first = (float*)(base + l.v_first);
    uint16_t *mixes = (uint16_t*)(base + l.mixes), *xk = (uint16_t*)(base + l.xk), *rkv = (uint16_t*)(base + l.rkv);
    uint16_t *up = (uint16_t*)(base + l.up), *o = (uint16_t*)(base + l.o), *hk = (uint16_t*)(base + l.hk);
    uint16_t* h = (uint16_t*)(base + l.h);
    const int64_t row = M * C;
    int32_t parts = 0;  // partial planes of the last FFN value product, in ws
    for (int i = 0; i < n_layer; ++i) {
        const rwkv7_layer& L = layers[i];
        float* ax = att_x + (size_t)i * pool_slots * C;
        float* fx = ffn_x + (size_t)i * pool_slots * C;
        float* S = kv + (size_t)i * pool_slots * C * 64;
        int rc;
        if (i == 0)
            rc = rwkv7_shift_mix(kBf16, M, C, nullptr, nullptr, 0, 0, tokens, emb, vocab, L.ln0_w, L.ln0_b, x_res,
                                 L.ln1_w, L.ln1_b, ax, pool_slots, row_slot, row_last, 7, L.mix7, mixes, stream);
        else
            rc = rwkv7_shift_mix(kBf16, M, C, x_mid, ws, parts, row, nullptr, nullptr, 0, nullptr, nullptr, x_res,
                                 L.ln1_w, L.ln1_b, ax, pool_slots, row_slot, row_last, 7, L.mix7, mixes, stream);
        if (rc != RWKV7_OK) return rc;
        if ((rc = downs_of(L, M, C, mixes, rkv, h, l.rank).run(M, ws, ws_floats, stream)) != RWKV7_OK) return rc;
        if ((rc = ups_of(L, M, C, h, up, l.rank).run(M, ws, ws_floats, stream)) != RWKV7_OK) return rc;
        rc = rwkv7_tmix_decode(kBf16, M, C / 64, i == 0, rkv, rkv + row, rkv + 2 * row, up, up + row,
                               i == 0 ? nullptr : up + 3 * row, up + 2 * row, v_first, L.tparams, S, pool_slots,
                               row_slot, o, stream);
        if (rc != RWKV7_OK) return rc;
        // the output projection's K-range partials, summed by the next row kernel
        rc = rwkv7_gemm_decode_partials(M, o, L.o, C, (int)C, (int)C, ws, ws_floats, &parts, stream);
        if (rc != RWKV7_OK) return rc;
        rc = rwkv7_shift_mix(kBf16, M, C, x_res, ws, parts, row, nullptr, nullptr, 0, nullptr, nullptr, x_mid, L.ln2_w,
                             L.ln2_b, fx, pool_slots, row_slot, row_last, 1, L.mixk, xk, stream);
        if (rc != RWKV7_OK) return rc;
        if ((rc = key_of(L, M, C, FF, xk, hk).run(M, ws, ws_floats, stream)) != RWKV7_OK) return rc;
        rc = rwkv7_gemm_decode_partials(M, hk, L.fv, FF, (int)C, (int)FF, ws, ws_floats, &parts, stream);
        if (rc != RWKV7_OK) return rc;
    }
    return rwkv7_final_norm(kBf16, n_out, C, x_mid, ws, parts, row, logit_rows, ln_w, ln_b, out, stream);
}
