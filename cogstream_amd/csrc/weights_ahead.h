// Weights of the next mid-size product read into the L2 caches by workgroups of the launch in front of it, on CUs that this launch leaves idle.
//
// One image in the vision encoder is a chain of launches of 5 to 12 us of which none fills the chip: the attention has 32 workgroups of 256 CUs, the
// output and second feed-forward products 144. Their weights (30 MB a layer) come from HBM, and a tile's loop waits for the first of them at the
// start of every launch; the L2 caches hold one layer's, 4 MB an XCD. Each XCD reads the panel of columns that its own tiles will read (gemm_mid.hip
// hands out tiles in runs per XCD, rows fastest), one dword of every 128-byte line; nothing waits for it and nothing is kept. The query, key and value
// product reads the output product's, the attention the first feed-forward product's, and so on round the layer: one image 1372 -> 1313 us (its weights in
// the Infinity Cache, layers made to share them: 1242). A CU asks for 40 to 55 B/ns, so all CUs that are left over take part, and none reads its own
// launch's weights any more.
#pragma once
#include "kernels.h"

struct AheadPanel { const char* W; long ldw; int lo, hi, cols, KT; };
__device__ __forceinline__ AheadPanel ahead_panel(const CogsWeightsAhead& d, int xcd) {
    AheadPanel p{d.W, d.ldw, 0, 0, 0, d.KT};
    if (!d.W) return p;
    const int tiles = d.nbm * d.nbn, q = tiles >> 3, r = tiles & 7;
    const int x0 = xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q, x1 = x0 + q + (xcd < r);
    if (x0 >= x1) return p;
    p.lo = x0 / d.nbm * d.tn;
    p.hi = min(((x1 - 1) / d.nbm + 1) * d.tn, d.N);
    p.cols = (p.hi - p.lo + 63) >> 6;
    return p;
}
// two products' panels (or one) as one run of 64-line pieces, slabs in order like the loop that will read them; me of `of` waves on this XCD
__device__ __forceinline__ void read_weights_ahead(const CogsWeightsAhead& d0, const CogsWeightsAhead& d1, int xcd, int me, int of, int lane) {
    const AheadPanel a = ahead_panel(d0, xcd), b = ahead_panel(d1, xcd);
    const int na = a.cols * a.KT, n = na + b.cols * b.KT;
    constexpr int U = 6;                         // pieces on their way
    for (int i0 = me; i0 < n; i0 += of * U) {
        unsigned v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = min(i0 + u * of, n - 1);
            const AheadPanel& p = i < na ? a : b;
            const int j = i < na ? i : i - na, k = j / p.cols, c = j - k * p.cols;
            v[u] = *reinterpret_cast<const unsigned*>(p.W + (long)min(p.lo + 64 * c + lane, p.hi - 1) * p.ldw + (long)k * 128);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) asm volatile("" ::"v"(v[u]));
    }
}
