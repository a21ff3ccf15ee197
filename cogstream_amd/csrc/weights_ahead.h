// Weights of the next mid-size product read into the L2 caches by workgroups of the launch in front of it, on CUs that this launch leaves idle.
//
// One image in the vision encoder is a chain of launches of 5 to 12 us of which none fills the chip: the attention has 32 workgroups of 256 CUs, the
// output and second feed-forward products 144. Their weights (30 MB a layer) come from HBM, and a tile's loop waits for the first of them at the
// start of every launch; the L2 caches hold one layer's, 4 MB an XCD. Each XCD reads the panel of columns that its own tiles will read (gemm_mid.hip
// hands out tiles in runs per XCD, rows fastest), one dword of every 128-byte line; nothing waits for it and nothing is kept. The query, key and value
// product reads the output product's, the attention the first feed-forward product's, and so on round the layer; a launch whose own weights were read has
// its CUs free for the next one's, and one whose were not reads its own. One image, one encoder by itself 1372 -> 1313 us (its weights in
// the Infinity Cache, layers made to share them: 1242). A CU asks for 40 to 55 B/ns, so all CUs that are left over take part.
#pragma once
#include "kernels.h"

// a workgroup's share at the most: what takes as long as a short launch. 10 MB on the 40 CUs that the output product of 384 rows leaves made its 6.9 us 10.1, on 72
// (320 rows) 6.8 to 7.8, and the product behind gained 0 and 0.4 us. Encoder alone, one by itself, us, without / all that is left over / up to here: 240 rows
// 1338 / 1283 / 1280, 336 1470 / 1455 / 1436, 384 1478 / 1499 / 1451, 2 x 192 1435 / 1458 / 1411, 480 1693 / 1637 / 1640, 576 1766 / 1706 / 1702
constexpr long WEIGHTS_AHEAD_BYTES = 160 * 1000;
inline long ahead_bytes(const CogsWeightsAhead& d) { return d.W ? (long)d.N * d.KT * 128 : 0; }

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
