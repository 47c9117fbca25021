// Causal GQA attention for the batched prefill (gfx950 matrix cores).
//
// Semantics as attn.h for every prompt row r (absolute position pos0 + r):
//   out[r][h] = softmax over t <= pos0 + r of (q_h . k_t) / sqrt(HD), times v_t
// (llama_run/src/main.rs:148-242 applied row by row), with the prompt's own
// rows already appended to the fp16 caches.
//
// A workgroup of NW waves per key group takes BQ = max(16, 16 NW / GT) prompt
// rows and every query head of one KV head (GT heads, G <= GT real), i.e. NT =
// (BQ/16) * GT tiles of 16 (row, head) pairs, MT = NT / NW per wave, and walks
// the keys 0 .. last row's position in blocks of 64 keys (head dim 64) or 32
// (128).  K and V rows are staged in LDS by DMA as they lie in the cache
// (chunks XOR-swizzled, no bank conflicts: SQ_LDS_BANK_CONFLICT 0); V^T
// operands come out of the row-major rows through the transposing LDS read.
// Every product is transposed so that the scores' accumulator is the next
// product's operand as it lies in the registers:
//   S^T (32 x 16) = K (32 x HD) . Q^T         -- B = q as two fp16 terms
//   online softmax per row (base 2, f32)      -- a row lives in the 4 lanes
//                                                l % 16 = row of the wave
//   O^T (HD x 16) += V^T (HD x 32) . P^T      -- B = p as two fp16 terms
// Lane (q4 = l / 16, row l % 16) holds the scores of keys 4 q4 .. +3 and
// 16 + 4 q4 .. +3 of each 32-key half of a block, which are the 8 K values
// of its P^T operand for that half; the V^T operand takes the same 8 keys of
// each dimension (two transposing reads), so P never leaves the registers.
//
// What bounds it: matrix and vector instructions of 4 waves per SIMD.  At 2048
// rows after 2048 keys of the 8B heads (206 GFLOP with the hi + lo terms, 191
// us) the matrix cores are busy 57 % of the cycles and the vector ALU about as
// much; LDS reads take 29 %.  Staging through registers (V transposed by 2-byte
// LDS writes, two register sets of loads) needed 141 registers, so a CU held
// one workgroup of 8 waves: 1531 rows after 517 keys 146 us, by DMA 93 us, with
// two key groups of 4 waves 81 us, with the rarely raised maximum, uniform DMA
// bases and two interleaved score chains 75 us (267 -> 191 us at 2048 + 2048,
// 33 -> 20.5 us at 700 rows).  The kernels of 8 and 16 waves take at most 127
// registers, which keeps 4 waves per SIMD; the one-group kernels of 4 waves,
// planned for contexts of two key blocks only, take 120 to 152.
//
// q and p enter as hi + lo (hi = fp16(x), lo = fp16(x - hi): about 2^-22
// relative, two MFMAs per product; K and V are fp16 already), products exact
// and f32 accumulation, so the output matches the f32 decode kernel's to
// about 1e-6: one fp16 rounding of q and p (2^-11) moves enough of the O
// projection's MXFP4 input codes across rounding boundaries to shift the
// logits by percent.  Operand
// layout (pinned by the fp16 layout test): lane l holds A row / B column
// l % 16 and K = 8 (l / 16) .. +7; accumulator r of lane l is D[4 (l/16) + r][l % 16].
#pragma once
#include "common.h"
#include "misc.h"

typedef __attribute__((address_space(3))) uint8_t pf_lds_u8;
typedef __attribute__((address_space(1))) void pf_glb_void;
#define PF_VMCNT(V) (((V) & 0xFu) | (((V) >> 4) << 14) | (0x7u << 4) | (0xFu << 8)) // s_waitcnt vmcnt(V)

// Chunk swizzles of the staged rows (the physical chunk of logical chunk q of
// row r is q ^ swizzle(r)).  K rows are read 16 at a time, one chunk of each:
// 16 rows of 256 bytes (HD 128), or 16 of 128 (HD 64, two rows per 256-byte
// bank line), fall on 16 distinct chunks of a bank line.  V rows are read 8
// at a time (by half a wave), 32 bytes of each: the swizzle moves pairs of
// chunks, so 8 rows cover a bank line once.
template <int HD>
RFP4_DEV uint32_t pf_kswz(uint32_t r)
{
    return HD == 128 ? r & 15u : (r ^ ((r >> 3) & 1u)) & 7u;
}
template <int HD>
RFP4_DEV uint32_t pf_vswz(uint32_t r)
{
    return HD == 128 ? (r & 7u) << 1 : ((r >> 1) & 3u) << 1;
}

// LDS reads in inline asm: the compiler treats every LDS read after an LDS DMA
// as a possible alias of it and would wait for every DMA in flight.  Each asm
// waits for its own reads, so no register of a read in flight is ever visible
// outside it.
// pf_read_k: four K operands, rows 16 h + l16 and chunk 4 k + q4 of the block
// (a step of k is an XOR of 4 chunks on the address, a step of h 16 rows): HD
// 128 k = k0, k0 + 1 of both 16-key quarters (ka[2 i + h]), HD 64 k = k0 of all
// four (ka[h]).  pf_read_v: the V^T operands of dimension tiles n0 .. n0 + 3
// for one 32-key chunk (two transposing reads each, 16 rows apart).
template <int HD>
RFP4_DEV void pf_read_k(f16x8 (&ka)[4], uint32_t addr, uint32_t k0)
{
    if constexpr (HD == 128)
        asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:4096\n\t"
                     "ds_read_b128 %2, %5\n\tds_read_b128 %3, %5 offset:4096\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(ka[0]), "=&v"(ka[1]), "=&v"(ka[2]), "=&v"(ka[3])
                     : "v"(addr ^ (k0 << 6)), "v"(addr ^ ((k0 + 1u) << 6)));
    else
        asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:2048\n\t"
                     "ds_read_b128 %2, %4 offset:4096\n\tds_read_b128 %3, %4 offset:6144\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(ka[0]), "=&v"(ka[1]), "=&v"(ka[2]), "=&v"(ka[3])
                     : "v"(addr ^ (k0 << 6)));
}
template <uint32_t RB>
RFP4_DEV void pf_read_v(f16x8 (&va)[4], uint32_t addr, uint32_t n0)
{
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    u32x2 lo[4], hi[4];
    asm volatile("ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %1, %8 offset:%12\n\t"
                 "ds_read_b64_tr_b16 %2, %9\n\tds_read_b64_tr_b16 %3, %9 offset:%12\n\t"
                 "ds_read_b64_tr_b16 %4, %10\n\tds_read_b64_tr_b16 %5, %10 offset:%12\n\t"
                 "ds_read_b64_tr_b16 %6, %11\n\tds_read_b64_tr_b16 %7, %11 offset:%12\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(lo[0]), "=&v"(hi[0]), "=&v"(lo[1]), "=&v"(hi[1]), "=&v"(lo[2]), "=&v"(hi[2]), "=&v"(lo[3]),
                   "=&v"(hi[3])
                 : "v"(addr ^ (n0 << 5)), "v"(addr ^ ((n0 + 1u) << 5)), "v"(addr ^ ((n0 + 2u) << 5)),
                   "v"(addr ^ ((n0 + 3u) << 5)), "n"(16u * RB));
#pragma unroll
    for (int i = 0; i < 4; i++) {
        typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));
        va[i] = __builtin_bit_cast(f16x8, (u32x4v){lo[i].x, lo[i].y, hi[i].x, hi[i].y});
    }
}

// One query tile: prompt rows r0 .. r0 + BQ of KV head kvh.  QO: the
// kernel variant that can quantize its output rows (AttnPrefillArgs::q_codes;
// a separate instantiation: the epilogue's code changes how the compiler
// schedules the main loop's LDS reads in the same function).
// KSP: key groups.  KSP groups of NW waves take the same query tiles and
// alternate key blocks (group g blocks g, g + KSP, ...; each staging step
// brings KSP blocks into LDS), then merge their softmax states through LDS
// (m the maximum, l and O rescaled by 2^(m_g - m) and summed): the serial
// chain of blocks of a tile is KSP times shorter.
//
// Grid (n_kv_heads, tiles): consecutive workgroups take the same query tile of
// every KV head, the longest causal range first, so that the short ones fill
// the end of the launch; with 8 KV heads each XCD (workgroup id % 8) keeps one
// head's K/V in its L2.
template <int HD, int GT, int NW, bool QO = false, int KSP = 1>
RFP4_DEV void attn_prefill_body(const AttnPrefillArgs &a)
{
    const uint32_t pos0 = a.pos0, nrows = a.rows;
    constexpr int BQ = attn_prefill_rows(GT, NW);    // prompt rows per workgroup
    constexpr int NT = (BQ / 16) * GT;               // 16-row tiles per workgroup
    constexpr int MT = NT / NW;                      // tiles per wave
    constexpr int KS = HD / 32;                      // K steps of S = Q K^T
    constexpr int NN = HD / 16;                      // 16-wide column tiles of O
    // keys per block: 64 for head dim 64, 32 for 128 (measured: 8B 2048-row
    // kernel 96.4 us with 32, 103.2 with 64; TinyLlama 41.2 -> 37.8 us)
    constexpr int PF_BK = HD == 64 ? 64 : 32;
    constexpr uint32_t RB = 2u * HD;                 // bytes per K/V row
    constexpr uint32_t LPR = HD / 8;                 // 16-byte chunks per row
    constexpr int NWV = NW * KSP;                    // waves
    constexpr uint32_t PB = PF_BK * RB / 1024u;      // 1 KB pieces of a block's K (and V)
    constexpr uint32_t BLOCK = 2u * PF_BK * RB, STAGE = KSP * BLOCK;
    constexpr int NI = (int)(STAGE / 1024u) / NWV;   // DMA instructions per wave and step
    // stages: two steps of DMA lookahead with one block per step; two blocks per step leave the LDS for
    // two workgroups per CU with one
    constexpr uint32_t NST = KSP == 1 || NW == 8 ? 3 : 2;
    static_assert(NT % NW == 0 && MT >= 1, "tiles per wave");
    static_assert(NI * NWV * 1024 == (int)STAGE, "every wave copies the same number of pieces");
    __shared__ __attribute__((aligned(1024))) uint8_t lds_raw[NST * STAGE];
    pf_lds_u8 *lds = (pf_lds_u8 *)lds_raw;

    const uint32_t kvh = blockIdx.x, r0 = (a.tile - blockIdx.y) * BQ;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    // key group; wave within it (KSP = 1: the plain kernel's code, group 0)
    const int kgrp = KSP > 1 ? wid / NW : 0, wave = KSP > 1 ? wid % NW : wid;
    const uint32_t l16 = (uint32_t)lane & 15u, q4 = (uint32_t)lane >> 4;
    const uint32_t G = a.group;
    const uint16_t *kc = a.kc + (size_t)kvh * a.hs;
    const uint16_t *vc = a.vc + (size_t)kvh * a.hs;
    // keys of this workgroup: 0 .. position of its last row
    const uint32_t last_row = min(r0 + (uint32_t)BQ, nrows) - 1u;
    const uint32_t nk = pos0 + last_row + 1u;
    const uint32_t nblk = (nk + PF_BK - 1) / PF_BK;
    const uint32_t niter = KSP > 1 ? (nblk + KSP - 1) / KSP : nblk; // staging steps
    // The softmax scale log2(e) / sqrt(HD) in two factors: 4 times it goes into
    // q, so that a score's exponent is a quarter of it, a power of two: score
    // times factor minus maximum is then exact to one rounding, and 0 for the
    // maximum itself.  (With the whole scale as the fma's factor the difference
    // carries the rounding error of the subtracted maximum: 2^-24 of it, which
    // for finite scores from about 2^30 on made the exponential infinite.)
    const float qscale = 4.0f * __fmul_rn(1.4426950408889634f, __fdiv_rn(1.0f, __fsqrt_rn((float)HD)));
    constexpr float quarter = 0.25f;

    // ---- Q tiles of this wave as fp16 A operands (rows past the prompt or heads past G: zero)
    f16x8 qa[MT][KS], ql[MT][KS];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const uint32_t t = (uint32_t)(wave * MT + mt), g = t % GT, row = r0 + 16u * (t / GT) + l16;
        const bool in = row < nrows && g < G;
        const float *qp = a.q + (size_t)min(row, nrows - 1u) * a.q_rs + (size_t)(kvh * G + min(g, G - 1u)) * HD + 8u * q4;
#pragma unroll
        for (int k = 0; k < KS; k++) {
            float v[8];
            const float4 x0 = *(const float4 *)(qp + 32 * k), x1 = *(const float4 *)(qp + 32 * k + 4);
            v[0] = x0.x; v[1] = x0.y; v[2] = x0.z; v[3] = x0.w;
            v[4] = x1.x; v[5] = x1.y; v[6] = x1.z; v[7] = x1.w;
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = in ? __fmul_rn(v[i], qscale) : 0.0f;
            split_hi_lo8(v, qa[mt][k], ql[mt][k]);
        }
    }

    // O^T tile n: accumulator r of lane l is dimension 16 n + 4 q4 + r of row l16;
    // the running max (finite, also while every key so far is masked) and sum
    // are the lane's row's
    f32x4 o[MT][NN];
    float mrun[MT], lrun[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        mrun[mt] = -3.402823466e38f;
        lrun[mt] = 0.0f;
#pragma unroll
        for (int n = 0; n < NN; n++) o[mt][n] = {0.0f, 0.0f, 0.0f, 0.0f};
    }

    // ---- K / V staging: DMA (global_load_lds), no registers.  A step's stage
    // holds KSP blocks, each PF_BK K rows then PF_BK V rows of HD halves, row
    // major, the 16-byte chunks of a row XOR-swizzled (pf_kswz, pf_vswz).  One
    // DMA instruction fills 1 KB (64 / LPR rows of LPR chunks): lane l's chunk
    // goes to physical chunk l % LPR, so it fetches logical chunk l % LPR ^
    // swizzle(row).  Keys past the last one re-read it (finite values, masked
    // scores), so every wave issues the same DMAs in every step.
    // Steps inside the context use 32-bit lane offsets from a uniform base (one
    // scalar add per step instead of a 64-bit address per lane and copy); the
    // last ones, and strides past 4 GB, clamp each row.
    constexpr uint32_t RPI = 64u / LPR; // rows per DMA instruction
    static_assert((NWV * RPI) % 16u == 0u && (NWV % PB == 0u || PB % NWV == 0u), "the same swizzle for every copy of a lane");
    const uint32_t row0 = ((uint32_t)wid % PB) * RPI + (uint32_t)lane / LPR, ch = (uint32_t)lane % LPR;
    const uint32_t lck = ch ^ pf_kswz<HD>(row0), lcv = ch ^ pf_vswz<HD>(row0);
    const uint32_t voffk = 2u * (row0 * (uint32_t)a.ts + 8u * lck), voffv = 2u * (row0 * (uint32_t)a.ts + 8u * lcv);
    const bool small = a.ts < (1ull << 24); // PF_BK rows of ts halves stay under 4 GB
    auto stage_dma = [&](uint32_t step, uint32_t buf) {
        const bool whole = small && (step + 1u) * (KSP * PF_BK) <= nk;
#pragma unroll
        for (int j = 0; j < NI; j++) {
            const uint32_t c = (uint32_t)wid + (uint32_t)(NWV * j); // 1 KB piece of the stage
            const uint32_t slot = c / (2u * PB), isv = (c / PB) & 1u;
            const uint32_t k0 = (step * KSP + slot) * PF_BK + ((uint32_t)(NWV * j) % PB) * RPI; // row0's first key
            const uint16_t *base = isv ? vc : kc;
            pf_lds_u8 *dst = lds + buf * STAGE + 1024u * c;
            if (whole) {
                const uint8_t *src = (const uint8_t *)(base + (size_t)k0 * a.ts);
                __builtin_amdgcn_global_load_lds((pf_glb_void *)(src + (isv ? voffv : voffk)), dst, 16, 0, 0);
            } else {
                const uint16_t *src = base + (size_t)min(k0 + row0, nk - 1u) * a.ts + 8u * (isv ? lcv : lck);
                __builtin_amdgcn_global_load_lds((pf_glb_void *)src, dst, 16, 0, 0);
            }
        }
    };
    // this lane's LDS byte addresses inside a stage.  K: row l16 of the first
    // 16 keys, chunk q4; key quarter h and dimension step k are 16 rows and an
    // XOR of 4 k chunks away.  V: the transposing read (ds_read_b64_tr_b16:
    // lane j of 16 gives the address of 4 halves, row j / 4 of a 4 x 16 block,
    // columns 4 (j % 4) .. +3, and receives column j of its 4 rows) of keys
    // 4 q4 .. +3 and dimensions 0 .. 15; dimension tile n is an XOR of 2 n
    // chunks away, the chunk's other 16 keys 16 rows.
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds + (uint32_t)kgrp * BLOCK;
    const uint32_t kaddr = lds0 + l16 * RB + ((q4 ^ pf_kswz<HD>(l16)) << 4);
    const uint32_t vrow = 4u * q4 + (l16 >> 2);
    const uint32_t vaddr = lds0 + PF_BK * RB + vrow * RB + ((((l16 & 3u) >> 1) ^ pf_vswz<HD>(vrow)) << 4) + 8u * (l16 & 1u);
#pragma unroll
    for (uint32_t i = 0; i + 1u < NST; i++)
        if (KSP > 1 || i < niter) stage_dma(i, i);

    // the block's scores, softmax and P V from the stage at byte sb (this key
    // group's block b of the step in slot kgrp; none past the last block)
    auto block = [&](uint32_t b, uint32_t sb) {
        if (KSP > 1 && b >= nblk) return; // the same for the whole key group
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            const uint32_t t = (uint32_t)(wave * MT + mt);
            // ---- S^T = K Q^T for the block's 16-key quarters h: accumulator r
            // of lane l is key 16 h + 4 q4 + r of row l16
            constexpr int NQ = PF_BK / 16;
            static_assert(NQ * KS == 8 && 4 % NQ == 0, "pf_read_k");
            f32x4 s[NQ];
#pragma unroll
            for (int h = 0; h < NQ; h++) s[h] = {0.0f, 0.0f, 0.0f, 0.0f};
            constexpr int KB = 4 / NQ; // dimension steps per read
#pragma unroll
            for (int k0 = 0; k0 < KS; k0 += KB) {
                f16x8 ka[4];
                pf_read_k<HD>(ka, kaddr + sb, (uint32_t)k0);
#pragma unroll
                for (int i = 0; i < KB; i++) {
#pragma unroll
                    for (int h = 0; h < NQ; h++)
                        s[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka[i * NQ + h], qa[mt][k0 + i], s[h], 0, 0, 0);
#pragma unroll
                    for (int h = 0; h < NQ; h++)
                        s[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka[i * NQ + h], ql[mt][k0 + i], s[h], 0, 0, 0);
                }
            }
            // ---- causal mask (only in blocks that reach past the tile's first row)
            const uint32_t row0t = r0 + 16u * (t / GT);
            const bool masked = (b + 1u) * PF_BK > pos0 + min(row0t, nrows - 1u) + 1u; // the same for the whole wave
            float p[4 * NQ];
#pragma unroll
            for (int h = 0; h < NQ; h++)
#pragma unroll
                for (int r = 0; r < 4; r++) p[4 * h + r] = s[h][r];
            if (masked) {
                const uint32_t qpos = pos0 + min(row0t + l16, nrows - 1u);
#pragma unroll
                for (int h = 0; h < NQ; h++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const uint32_t key = b * PF_BK + 16u * h + 4u * q4 + (uint32_t)r;
                        if (key > qpos) p[4 * h + r] = -INFINITY; // p is 0 whatever maximum is subtracted
                    }
            }
            // ---- online softmax (base 2) of the lane's row.  The subtracted
            // maximum is raised only when a score of the row exceeds it by
            // more than 8 (p is at most 2^8 and keeps its relative precision
            // in hi + lo; l and O are f32): in the common block there is no
            // cross-lane step and no O rescale (32 of 150 VALU instructions),
            // and the sum stays per lane until the end.
            float mx = p[0];
#pragma unroll
            for (int i = 1; i < 4 * NQ; i++) mx = fmaxf(mx, p[i]);
            mx *= quarter;
            if (__any(mx > mrun[mt] + 8.0f)) {
                const float rowmax = xor32_max(xor16_max(mx));
                const float mnew = rowmax > mrun[mt] + 8.0f ? rowmax : mrun[mt]; // a row's own choice, whatever its wave holds
                const float alpha = __builtin_amdgcn_exp2f(mrun[mt] - mnew);
                mrun[mt] = mnew;
                lrun[mt] *= alpha;
#pragma unroll
                for (int n = 0; n < NN; n++) o[mt][n] *= alpha;
            }
#pragma unroll
            for (int i = 0; i < 4 * NQ; i++) {
                p[i] = __builtin_amdgcn_exp2f(fmaf(p[i], quarter, -mrun[mt]));
                lrun[mt] += p[i];
            }
            // ---- O^T += V^T P^T per 32-key chunk c (quarters 2c, 2c + 1): P^T as
            // hi + lo operands straight from the registers; V^T dimension row
            // 16 n + l16 at the lane's 8 keys of the chunk
#pragma unroll
            for (int c = 0; c < NQ / 2; c++) {
                f16x8 pb, pl;
                split_hi_lo8_mix(p + 8 * c, pb, pl);
#pragma unroll
                for (int n0 = 0; n0 < NN; n0 += 4) {
                    f16x8 va[4];
                    pf_read_v<RB>(va, vaddr + sb + (uint32_t)c * 32u * RB, (uint32_t)n0);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        o[mt][n0 + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[i], pb, o[mt][n0 + i], 0, 0, 0);
                        o[mt][n0 + i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[i], pl, o[mt][n0 + i], 0, 0, 0);
                    }
                }
            }
        }
    };
    // Step i: wait for this wave's DMAs of step i (those of the NST - 2 steps
    // behind it may be in flight), then the barrier: every wave's copies of
    // step i are in LDS and every wave is past its reads of step i - 1, whose
    // buffer the DMAs of step i + NST - 1 then overwrite.  With one key group
    // (contexts of a few blocks) no DMA is issued past the last block, and the
    // last step waits for all: the copies that nothing reads were 0.2 to 0.3
    // of the 5.6 us of 51 rows of TinyLlama's heads.  With more groups the
    // branch around the DMAs costs more than the copies (100 rows after 4000
    // keys of the 8B heads 55.9 us without it, 58.2 with).
    uint32_t buf = 0;
    for (uint32_t it = 0; it < niter; it++) {
        if (KSP > 1 || it + 1u < niter) __builtin_amdgcn_s_waitcnt(PF_VMCNT(NI * (NST - 2u)));
        else __builtin_amdgcn_s_waitcnt(PF_VMCNT(0));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (KSP > 1 || it + NST - 1u < niter) stage_dma(it + NST - 1u, buf == 0u ? NST - 1u : buf - 1u);
        block(it * KSP + (uint32_t)kgrp, buf * STAGE);
        buf = buf + 1u == NST ? 0u : buf + 1u;
    }
    if (KSP > 1) { // the last DMAs (past the end) land before the merge uses the LDS again
        __builtin_amdgcn_s_waitcnt(PF_VMCNT(0));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    }

    // the row's sum over its four lanes
#pragma unroll
    for (int mt = 0; mt < MT; mt++) lrun[mt] = xor32_sum(xor16_sum(lrun[mt]));

    if constexpr (KSP > 1) {
        // ---- the key groups' states merged into group 0's: groups 1.. put
        // (O, m, l) in LDS (lane-contiguous words), group 0 combines
        // (in the stages, free after the loop)
        typedef float pf_mg[NW][MT][NN * 4 + 2][64];
        static_assert(sizeof(pf_mg) * (KSP - 1) <= NST * STAGE, "the merged states in the stages");
        pf_mg *mg = (pf_mg *)lds_raw;
        if (kgrp > 0) {
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                float(*w)[64] = mg[kgrp - 1][wave][mt];
#pragma unroll
                for (int n = 0; n < NN; n++)
#pragma unroll
                    for (int r = 0; r < 4; r++) w[4 * n + r][lane] = o[mt][n][r];
                w[NN * 4][lane] = mrun[mt];
                w[NN * 4 + 1][lane] = lrun[mt];
            }
        }
        __syncthreads();
        if (kgrp > 0) return; // group 0 writes the output
#pragma unroll
        for (int g2 = 0; g2 < KSP - 1; g2++)
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                const float(*w)[64] = mg[g2][wave][mt];
                const float m2 = w[NN * 4][lane], l2 = w[NN * 4 + 1][lane];
                const float m = fmaxf(mrun[mt], m2);
                const float a0 = __builtin_amdgcn_exp2f(mrun[mt] - m), a1 = __builtin_amdgcn_exp2f(m2 - m);
                mrun[mt] = m;
                lrun[mt] = fmaf(lrun[mt], a0, l2 * a1);
#pragma unroll
                for (int n = 0; n < NN; n++)
#pragma unroll
                    for (int r = 0; r < 4; r++) o[mt][n][r] = fmaf(o[mt][n][r], a0, w[4 * n + r][lane] * a1);
            }
    }

    // ---- out[row][head][dim] = O / l for rows in the prompt and heads < G
    // (lane: row l16, dimensions 16 n + 4 q4 .. +3 of each tile n)
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const uint32_t t = (uint32_t)(wave * MT + mt), g = t % GT;
        if (g >= G) continue; // the same for the whole wave
        const uint32_t row = r0 + 16u * (t / GT) + l16, head = kvh * G + g;
        if (a.out && row < nrows) {
            float *op = a.out + (size_t)row * a.out_rs + (size_t)head * HD + 4u * q4;
#pragma unroll
            for (int n = 0; n < NN; n++)
                *(float4 *)(op + 16 * n) = make_float4(__fdiv_rn(o[mt][n][0], lrun[mt]), __fdiv_rn(o[mt][n][1], lrun[mt]),
                                                       __fdiv_rn(o[mt][n][2], lrun[mt]), __fdiv_rn(o[mt][n][3], lrun[mt]));
        }
        if (QO && a.q_codes) {
            // MXFP4 per 32 dimensions (quant_block32's arithmetic): block b of
            // the head is tiles 2b, 2b + 1, i.e. this lane's 8 values and those
            // of lanes ^16, ^32, ^48 (the same row); the maximum first over all
            // four, then each lane codes its two runs of 4 dimensions.  One
            // block at a time, each value formed as the f32 rows would hold it.
            const uint32_t qd = a.n_heads * HD, qd32 = qd / 32u;
#pragma unroll
            for (int b = 0; b < HD / 32; b++) {
                float y[8];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    y[r] = __fdiv_rn(o[mt][2 * b][r], lrun[mt]);
                    y[4 + r] = __fdiv_rn(o[mt][2 * b + 1][r], lrun[mt]);
                }
                float amax = 0.0f;
#pragma unroll
                for (int i = 0; i < 8; i++) amax = fmaxf(amax, fabsf(y[i]));
                amax = xor32_max(xor16_max(amax));
                int se = 0;
                uint32_t sbyte = 0;
                if (amax != 0.0f) {
                    se = floor_log2_pos(amax) - 2;
                    se = se < -127 ? -127 : (se > 127 ? 127 : se);
                    sbyte = (uint32_t)(se + 127);
                }
                const float sc = ldexpf(1.0f, se); // 1 where amax is 0 (se = 0)
                const uint32_t lo = fp4_pack2<1>(fp4_pack2<0>(0u, y[0], y[1], sc), y[2], y[3], sc);
                const uint32_t hi = fp4_pack2<1>(fp4_pack2<0>(0u, y[4], y[5], sc), y[6], y[7], sc);
                if (row < nrows) {
                    uint8_t *cp = a.q_codes + (size_t)row * (qd / 2u) + (size_t)head * (HD / 2) + 16u * b + 2u * q4;
                    *(uint16_t *)cp = (uint16_t)lo;
                    *(uint16_t *)(cp + 8) = (uint16_t)hi;
                    if (q4 == 0u) {
                        const uint32_t blk = head * (HD / 32) + (uint32_t)b;
                        a.q_scales[(size_t)row * qd32 + blk] = (uint8_t)sbyte;
                        if (a.q_scales_t) a.q_scales_t[mx_st_offset(row, blk, qd / 256u)] = (uint8_t)sbyte;
                    }
                }
            }
        }
    }
}
