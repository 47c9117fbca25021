// RMSNorm, RoPE, fp16 KV append and embedding gather for gfx950.
// Elementwise arithmetic uses the _rn intrinsics so no multiply-add is fused:
// every element rounds exactly as the reference's CPU loops do.
#pragma once
#include "common.h"

// Block-wide sum of one float per thread (NW waves); every thread receives
// the total.  Waves are combined in fixed order.
template <int NW>
RFP4_DEV float block_sum(float v, float *red /* >= NW floats */)
{
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float t = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; w++) t += red[w];
    __syncthreads();
    return t;
}

// y = x * (1/sqrt(sum(x^2)/d + eps)) * w   (llama_run/src/main.rs:79-116,
// order (x*rms)*w as llama_rmsnorm/src/main.rs:77).  One workgroup of 1024.
// Latency bound: with XV elements per thread in registers (dim <= 1024 XV),
// the x and w loads are all issued at once and x is read once; XV = 0 loops.
// Same sums in the same order.  Workgroup size as a constant: read from the
// dispatch packet it is one more dependent load.  dim 4096: 3.2 -> 2.0 us.
template <int W_F16, int XV>
RFP4_DEV void rmsnorm_regs(const RmsnormArgs &a, float *red)
{
    const auto weight = [&](uint32_t i) { return W_F16 ? f16_bits_to_f32(((const uint16_t *)a.w)[i]) : ((const float *)a.w)[i]; };
    float ss = 0.0f, x[XV > 0 ? XV : 1], w[XV > 0 ? XV : 1];
    if (XV > 0) {
#pragma unroll
        for (int j = 0; j < XV; j++) x[j] = a.x[min(threadIdx.x + 1024u * j, a.dim - 1u)];
#pragma unroll
        for (int j = 0; j < XV; j++) w[j] = weight(min(threadIdx.x + 1024u * j, a.dim - 1u));
#pragma unroll
        for (int j = 0; j < XV; j++) {
            const float t = __fadd_rn(ss, __fmul_rn(x[j], x[j]));
            ss = threadIdx.x + 1024u * j < a.dim ? t : ss;
        }
    } else {
        for (uint32_t i = threadIdx.x; i < a.dim; i += 1024u) ss = __fadd_rn(ss, __fmul_rn(a.x[i], a.x[i]));
    }
    const float total = block_sum<16>(ss, red);
    const float rms = __fdiv_rn(1.0f, __fsqrt_rn(__fadd_rn(__fdiv_rn(total, (float)a.dim), a.eps)));
    if (XV > 0) {
#pragma unroll
        for (int j = 0; j < XV; j++)
            if (threadIdx.x + 1024u * j < a.dim) a.y[threadIdx.x + 1024u * j] = __fmul_rn(__fmul_rn(x[j], rms), w[j]);
    } else {
        for (uint32_t i = threadIdx.x; i < a.dim; i += 1024u) a.y[i] = __fmul_rn(__fmul_rn(a.x[i], rms), weight(i));
    }
}

template <int W_F16>
RFP4_DEV void rmsnorm_body(const RmsnormArgs &a)
{
    __shared__ float red[16];
    if (a.dim <= 2048u) rmsnorm_regs<W_F16, 2>(a, red);
    else if (a.dim <= 4096u) rmsnorm_regs<W_F16, 4>(a, red);
    else if (a.dim <= 8192u) rmsnorm_regs<W_F16, 8>(a, red);
    else rmsnorm_regs<W_F16, 0>(a, red);
}

// Rotate-half RoPE on one (head, j) pair: llama_run/src/main.rs:118-138.
RFP4_DEV void rope_pair(float *b, uint32_t j, uint32_t half, float c, float s)
{
    float x0 = b[j], x1 = b[j + half];
    b[j] = __fsub_rn(__fmul_rn(x0, c), __fmul_rn(x1, s));
    b[j + half] = __fadd_rn(__fmul_rn(x1, c), __fmul_rn(x0, s));
}

RFP4_DEV void rope_body(const RopeArgs &a)
{
    uint32_t half = a.head_dim / 2;
    uint32_t gid = blockIdx.x * 256u + threadIdx.x;
    if (gid >= a.num_heads * half) return;
    uint32_t head = gid / half, j = gid % half;
    rope_pair(a.q + (size_t)head * a.head_dim, j, half, a.cosv[a.cos_base + j], a.sinv[a.cos_base + j]);
}


// x[i] = embed[ids[step]][i] (fp16 or bf16 -> f32): llama_run/src/main.rs:509-510,
// but gathered on the device so no per-token host upload is needed.
RFP4_DEV void embed_body(const EmbedArgs &a)
{
    uint32_t tok = a.ids[a.state->step];
    if (tok >= a.vocab) tok = 0;
    const uint16_t *row = a.embed + (size_t)tok * a.dim;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < a.dim; i += gridDim.x * 256u)
        a.x[i] = half_bits_to_f32(row[i], a.bf16 != 0);
}
