// Sums of point-source and receiver taps in their listed order, spread over
// a block.
//
// A receiver off the nodes is a sum of 9, 81 (2D) or 729 (3D) taps, and one
// cell of a dense adjoint source collects the taps of every receiver near
// it.  The reference adds them one after another, and FP32 sums keep that order
// here, so one thread per sum is a chain of dependent loads: it is bound by
// memory latency, not by bytes.  The block therefore forms all products of
// its sums at once (independent loads, up to 8 in flight per thread),
// leaves them in LDS, and then one thread per sum adds its own run of LDS
// values in order.  Bit-identical to the serial loop.
//
// Measured on one MI355X with receivers off the nodes, us per launch, one
// thread per sum -> this form: 2D acoustic, 391 receivers of one shot 31 ->
// 4.0, of 32 shots 42 -> 6.5; 2D elastic, 8 shots 27 -> 5.0; FSG, 32 shots
// 79 -> 18 (with 8-byte taps); 3D elastic, 144 x 3 components of 8 shots
// 146 -> 19; 3D acoustic, 144 receivers of 2 shots 37 -> 6.8.  It did not
// help the sparse adjoint sources of the elastic solvers (one to three taps
// a cell: 5.6 us per thread, 22 us here), which keep one thread per cell.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

namespace owl {

constexpr int kOrderedThreads = 256;
constexpr int kOrderedTaps = 2048;  // products a block holds (8 KB of LDS)

// The block's n products, U per thread with all their loads in flight (the
// index is clamped rather than the load skipped).
template <int U, class Product>
__device__ __forceinline__ void ordered_terms(float* term, int k0, int n, Product product) {
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = product(k0 + min(int(threadIdx.x) + u * kOrderedThreads, n - 1));
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int k = int(threadIdx.x) + u * kOrderedThreads;
        if (k < n) term[k] = v[u];
    }
}

// Sums r0 .. r1-1 (at most kOrderedThreads of them): the terms of sum r are
// first(r) .. first(r+1)-1, term k is product(k) * scale(r); init(r) starts
// sum r, store(r, acc) takes the result.  Called by every thread of the
// block.
template <class First, class Product, class Init, class Scale, class Store>
__device__ __forceinline__ void ordered_sums(int r0, int r1, First first, Product product, Init init, Scale scale,
                                             Store store) {
    constexpr int kRun = 16;  // LDS values read ahead of the chain of additions
    __shared__ float term[kOrderedTaps];
    if (r0 >= r1) return;  // the whole block
    const int k0 = first(r0), n = first(r1) - k0;
    const int r = r0 + int(threadIdx.x);
    // the sum's own start, scale and range, in flight with the terms
    const bool mine = r < r1;
    float acc = mine ? init(r) : 0.0f;
    const float sc = mine ? scale(r) : 0.0f;
    const int b = mine ? first(r) : k0, e = mine ? first(r + 1) : k0;
    if (n <= kOrderedTaps) {
        if (n > 4 * kOrderedThreads) ordered_terms<8>(term, k0, n, product);
        else if (n > 2 * kOrderedThreads) ordered_terms<4>(term, k0, n, product);
        else if (n > kOrderedThreads) ordered_terms<2>(term, k0, n, product);
        else if (n > 0) ordered_terms<1>(term, k0, n, product);
        __syncthreads();
        int k = b - k0;
        for (; k + kRun <= e - k0; k += kRun) {
            float v[kRun];
#pragma unroll
            for (int u = 0; u < kRun; ++u) v[u] = term[k + u];
#pragma unroll
            for (int u = 0; u < kRun; ++u) acc = acc + v[u] * sc;
        }
        if (k < e - k0) {
            float v[kRun];
#pragma unroll
            for (int u = 0; u < kRun; ++u) v[u] = term[min(k + u, e - k0 - 1)];
#pragma unroll
            for (int u = 0; u < kRun; ++u) acc = k + u < e - k0 ? acc + v[u] * sc : acc;
        }
    } else {
        // more terms than the block holds (one sum of that many)
        for (int k = b; k < e; ++k) acc = acc + product(k) * sc;
    }
    if (mine) store(r, acc);
}

// Sums one block takes: as many as leave every block's terms within its LDS
// (`beg` holds the running term counts, beg[r] .. beg[r+1] is sum r).  A
// receiver line off the nodes takes 16 sums of 81 terms, one on the nodes
// 256 single ones.
inline int ordered_group(const std::vector<int>& beg) {
    const size_t n = beg.empty() ? 0 : beg.size() - 1;
    for (int g = kOrderedThreads; g > 1; g /= 2) {
        bool fits = true;
        for (size_t r = 0; r < n && fits; ++r) fits = beg[std::min(n, r + size_t(g))] - beg[r] <= kOrderedTaps;
        if (fits) return g;
    }
    return 1;
}

}  // namespace owl
