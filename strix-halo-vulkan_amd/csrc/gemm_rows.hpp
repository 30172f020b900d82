// What the matrix-core projections share about their activation rows: the prologue of a quad of columns and where a row goes.
#pragma once
#include "shv_device.hpp"
#include "shv_internal.hpp"

namespace shv_gemm {

using namespace shv;

// pro(x) of the four columns c..c+3 of activation row t; `scale` is the row's RMSNorm factor.
// Every lane of a wave calls it for the same row (the gated norm adds up across lanes).
__device__ __forceinline__ void pro_quad(const shv_gemv_q4k_args &a, int t, int c, float scale, float (&x)[4]) {
    const int sl = a.seq_len > 0 ? a.seq_len : a.n_tok;
    const float4 v = *reinterpret_cast<const float4 *>(a.x + static_cast<size_t>(t) * a.x_stride + c);
    x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
    if (a.prologue == SHV_PRO_RMSNORM) {
        const float4 g = *reinterpret_cast<const float4 *>(a.gamma + c);
        x[0] *= scale * g.x; x[1] *= scale * g.y; x[2] *= scale * g.z; x[3] *= scale * g.w;
    } else if (a.prologue == SHV_PRO_GATED_NORM || a.prologue == SHV_PRO_MUL_SIGMOID) {
        const float *z = a.z + static_cast<size_t>(t) * a.z_stride;
        if (a.z_ring) {
            const int s = t / sl, k = t % sl;
            const int p = a.pos ? a.pos[s] : 0;
            const int slot = a.slot ? a.slot[s] : s;
            z = a.z + (static_cast<size_t>(slot) * a.ring_slots + (p + k) % a.ring_slots) * a.ring_stride;
        }
        const int zi = a.prologue == SHV_PRO_MUL_SIGMOID && a.head_dim > 0 ? (c & ~(a.head_dim - 1)) * 2 + a.head_dim + (c & (a.head_dim - 1)) : c;
        const float4 zq = *reinterpret_cast<const float4 *>(z + zi);
        const float zz[4] = {zq.x, zq.y, zq.z, zq.w};
        if (a.prologue == SHV_PRO_GATED_NORM) {
            float ss = fmaf(x[0], x[0], fmaf(x[1], x[1], fmaf(x[2], x[2], x[3] * x[3])));
            const int span = a.head_dim / 4;  // lanes a head spans: a power of two up to 64
            for (int off = 1; off < span; off <<= 1) ss += __shfl_xor(ss, off, 64);
            const float scale = 1.f / sqrtf(ss / static_cast<float>(a.head_dim) + a.eps);
            const float4 g4 = *reinterpret_cast<const float4 *>(a.gamma + (c & (a.head_dim - 1)));
            const float gg[4] = {g4.x, g4.y, g4.z, g4.w};
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = x[j] * scale * gg[j] * sigmoid_fast(zz[j]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] *= sigmoid_fast(zz[j]);
        }
    }
}

// Where activation row t of the pass writes its outputs: the DeltaNet projection ring, or plain rows.
__device__ __forceinline__ size_t out_offset(const shv_gemv_q4k_args &a, int t) {
    if (a.ring_slots > 0 && !a.z_ring) {
        const int sl = a.seq_len > 0 ? a.seq_len : a.n_tok;
        const int s = t / sl, i = t % sl;
        const int p = a.pos ? a.pos[s] : 0;
        const int slot = a.slot ? a.slot[s] : s;
        return (static_cast<size_t>(slot) * a.ring_slots + (p + i) % a.ring_slots) * a.ring_stride;
    }
    return static_cast<size_t>(t) * a.y_stride;
}

}  // namespace shv_gemm
