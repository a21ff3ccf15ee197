// A new row's latents, shared by the kernel of their own (mla.hip) and the few-row query product that norms its rows itself (gemm_skinny.hip).
#pragma once
#include "common.h"
#include "kernels.h"

// sums of up to two values over a 256-thread workgroup, result in every thread; `red` holds 8 floats
__device__ __forceinline__ void block_sum2(float& a, float& b, float* red) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    a = wave_sum(a);
    b = wave_sum(b);
    if (lane == 0) { red[wid] = a; red[4 + wid] = b; }
    __syncthreads();
    a = (red[0] + red[1]) + (red[2] + red[3]);
    b = (red[4] + red[5]) + (red[6] + red[7]);
    __syncthreads();
}

// One row by a workgroup of 256 threads: RMS norm of the query latent (QUERY), RMS norm of the kv latent and rotation of the shared key part
// (both straight into the sequence's cache row), sigmoid of the gate logits. red: 8 floats. Squares are fused in the order of the columns, here and
// in the query product: a row's norm has the same bits by either
template <typename T, bool QUERY>
__device__ __forceinline__ void latent_row(const CogsMlaLatent& p, int row, int tid, float* red) {
    const float* t = p.t + (long)row * p.ldt;
    float sq = 0.f, skv = 0.f;
    if constexpr (QUERY)
        for (int i = tid * 4; i < p.qrp; i += 1024) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(t + i);
#pragma unroll
            for (int e = 0; e < 4; ++e) sq = fmaf(v[e], v[e], sq);
        }
    const float* tk = t + p.qrp;
    if (p.own_kv)
        for (int i = tid * 4; i < p.kvp; i += 1024) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(tk + i);
#pragma unroll
            for (int e = 0; e < 4; ++e) skv = fmaf(v[e], v[e], skv);
        }
    block_sum2(sq, skv, red);
    if constexpr (QUERY) {
        const float rq = 1.f / sqrtf(sq / (float)p.qr + p.eps);
        T* cq = reinterpret_cast<T*>(p.cq) + (long)row * p.qrp;
        for (int i = tid * 4; i < p.qrp; i += 1024) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(t + i), g = *reinterpret_cast<const f32x4*>(p.q_norm + i);
            st4_f<T>(cq + i, f32x4{v[0] * rq * g[0], v[1] * rq * g[1], v[2] * rq * g[2], v[3] * rq * g[3]});
        }
    }
    if (p.own_kv) {
        const CogsSeq s = p.seqs[p.rowseq[row]];
        const int kvw = p.kvp + p.krc;
        T* c = reinterpret_cast<T*>(s.cache) + p.layer_off * s.max_len + (long)p.rowpos[row] * kvw;
        const float rk = 1.f / sqrtf(skv / (float)p.kvr + p.eps);
        for (int i = tid * 4; i < p.kvp; i += 1024) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(tk + i), g = *reinterpret_cast<const f32x4*>(p.kv_norm + i);
            st4_f<T>(c + i, f32x4{v[0] * rk * g[0], v[1] * rk * g[1], v[2] * rk * g[2], v[3] * rk * g[3]});
        }
        const float* tr = tk + p.kvp;
        const float* cs = p.rope + ((long)row * p.rope_pairs + p.rope_first) * 2;
        for (int i = tid * 2; i < p.krc; i += 512) {
            float a = 0.f, b = 0.f;
            if (i < p.dr) {
                const float u = tr[i], v = tr[i + 1], co = cs[i], si = cs[i + 1];
                a = fmaf(-v, si, u * co);
                b = fmaf(u, si, v * co);
            }
            st_f<T>(c + p.kvp + i, a);
            st_f<T>(c + p.kvp + i + 1, b);
        }
    }
    if (p.gate_col >= 0)
        for (int i = tid; i < p.heads; i += 256) p.gate[(long)row * p.heads + i] = 1.f / (1.f + expf(-t[p.gate_col + i]));
}
