// Segments of a chunked WKV7 walk: each sequence's 32-token chunks in runs of `cps`, numbered g = 0, 1, ...
// over the batch.  A launch with fewer (sequence, head) units than the chip has room for walks the segments
// side by side: the state recurrence is linear in the state (S_end = S_start M + N per segment), so one pass
// finds M and N of every segment (from S = I without values, and from S = 0), a scan over the segments
// turns them into every segment's start state, and the last pass runs all segments in full.
#pragma once

#include "common.hpp"

struct WkvSegs {
    int nseq;           // sequences
    int cps;            // chunks per segment; 0: sequences are not split
    int gmax;           // segments the launch has blocks (and workspace) for
    int T;              // tokens of every sequence when cu is null
    int total;          // packed rows
    const int32_t* cu;  // [nseq + 1] row offsets, or null
};

namespace wkvseg {

constexpr int kChunk = 32;

// segments of sequence s (0 when its range is empty or malformed)
__device__ __forceinline__ int count(const WkvSegs& m, int s) {
    const int tb = m.cu != nullptr ? m.cu[s] : s * m.T, te = m.cu != nullptr ? m.cu[s + 1] : tb + m.T;
    if (tb < 0 || te <= tb || te > m.total) return 0;
    return ((te - tb + kChunk - 1) / kChunk + m.cps - 1) / m.cps;
}

// More segments than the launch has blocks for: only offsets that decrease somewhere and then cover
// rows twice; such a batch runs unsplit, block group g taking sequence g.
__device__ __forceinline__ bool overfull(const WkvSegs& m) {
    if (m.cu == nullptr) return false;
    int n = 0;
    for (int s = 0; s < m.nseq; ++s) n += count(m, s);
    return n > m.gmax;
}

// first segment and number of segments of sequence s
__device__ __forceinline__ void range(const WkvSegs& m, int s, int& g0, int& n) {
    if (m.cu == nullptr) {
        n = count(m, 0);
        g0 = s * n;
        return;
    }
    if (overfull(m)) {
        g0 = s;
        n = 1;
        return;
    }
    g0 = 0;
    for (int q = 0; q < s; ++q) g0 += count(m, q);
    n = count(m, s);
}

// the sequence of segment g, its place there and the sequence's number of segments; false: no such segment
__device__ __forceinline__ bool locate(const WkvSegs& m, int g, int& s, int& seg, int& n) {
    if (m.cu == nullptr) {
        n = count(m, 0);
        s = g / n;
        seg = g - s * n;
        return s < m.nseq;
    }
    if (overfull(m)) {
        s = g;
        seg = 0;
        n = 1;
        return g < m.nseq;
    }
    int left = g;
    for (s = 0; s < m.nseq; ++s) {
        n = count(m, s);
        if (left < n) {
            seg = left;
            return true;
        }
        left -= n;
    }
    return false;
}

}  // namespace wkvseg

// Scan over the segments' maps q (M) and offsets h (N), each [64][64] at index * 4096; see wkv7_scan.hip.
// forward: index g H + head; the state at the end of segments 1 .. n - 2 of every sequence, over h.
hipError_t launch_wkv7_scan_forward(const WkvSegs& m, int H, const float* q, float* h, hipStream_t st);
// backward: index unit nseg + segment; the gradient at the start of segments nseg - 2 .. 1, over h.
hipError_t launch_wkv7_scan_backward(int64_t units, int nseg, const float* q, float* h, hipStream_t st);
