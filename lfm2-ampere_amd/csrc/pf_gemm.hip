// pf_gemm.hip - the consumer of the prefill attention output for gfx950: the
// Q4_0 weight x planar Q8_1 activation GEMM that applies attn_output.weight to
// the chunk's attention rows (as lk_pf_attn8_q81 emits them) and adds the
// residual, and the same GEMM for any dense Q4_0 matrix of that format.
//
// Reference behaviour: k_pf_mmq with the plain epilogue (EPI 0) for one dense
// weight tensor (/root/reference/src/prefill.cu:173-490, driven by
// pf_gemm_dense, prefill.cu:818-826; PfGemm / PfAct, prefill.cuh:33-69),
// launched for the attention output at engine.cu:1128-1131.  With PF_EPI2 (its
// default, prefill.cu:131-141), per output (token t, row r):
//     acc = 0; for each 32-element block b in order:
//         F   = float bits of (0x4B400000 + sumi)  = 1.5*2^23 + sumi exactly
//               (sumi = the exact int32 sum of nibble * q8 over the block)
//         c   = fma(d8, 1.5*2^23, s8)              (s8 = 8 * fp16 sum, from the sc plane)
//         acc = fma(d4, fma(d8, F, -c), acc)
//     a = acc * scale[t] (scale NULL: 1);  out[t][r] = add ? out[t][r] + a : a
// Every step is an explicit fma or a separately rounded product or sum
// (contraction off), so this kernel and the CPU oracle produce the same bits;
// so does the reference's main loop.  Its nvcc build may contract the
// epilogue's acc * scale + out into one fma, a difference of one rounding.
//
// MI355X design: one 32-element Q4_0 block per MFMA, because the scales change
// from block to block.  A wave covers MT weight rows x MT*NT tokens, MT = 32
// (v_mfma_i32_32x32x32_i8) or 16 (16x16x32).  The accumulator is seeded with
// 0x4B400000 so the integer sum arrives as the float F.  The row scale d4 of
// the second fma is the same for every lane of a result row group: each lane
// holds one row's d4 and the fma takes it by DPP (row_newbcast), so a block's
// 16 row scales cost one LDS dword per lane and two blocks instead of 32
// bytes per lane and block.
// All operands reach LDS by LDS DMA (16 bytes per lane; the row scales 4), in
// two stages of KC blocks, one barrier per stage.  A DMA instruction covers
// whole runs of memory, a row's KC blocks side by side: with one row per lane
// (64 cache lines per instruction) the address unit was the limit of every
// launch under 4096 tokens.
// What bounds it: the two fmas per output and block.  A step (one MFMA, its
// 16 + 16 fmas, about 12 other VALU) measured 131 cycles per SIMD with 4
// waves and everything in registers (v_fmac by DPP and v_fma_mix 4.3 cycles,
// plain v_fma 2.7 as two waves issue together, the MFMA under them), 33 us
// for 4096 tokens x 2048 x 2048; that launch takes 51-52 us (56-59 us in
// the form before, whose d4 took 16 bytes more of LDS reads per lane and
// block), about 7 of them the first stage's latency and the final stores of
// 33.5 MB.  The blocks of an output are accumulated in order, so K cannot be
// split: a launch of few tokens is a chain of bpr steps, and the shapes at the
// launch below trade operand reuse for shorter chains.
// Workgroups are mapped to tiles XCD by XCD (each XCD's L2 holds a few token
// tiles' activations with every row tile).  The output tile is written as
// float4 (4 consecutive rows of one token).  Needs N % 128 == 0 and bpr % 8
// == 0, as the reference's pf_gemm_dense does (PF_BM = 128).
#include "lk_common.h"

typedef int lk_i4g __attribute__((ext_vector_type(4)));
typedef int lk_i16g __attribute__((ext_vector_type(16)));
typedef float lk_f16g __attribute__((ext_vector_type(16)));

// The shape of a launch: MT x MT MFMA tiles, NT of them along the tokens per
// wave, WM x WN waves, KC blocks per stage.
template <int MT_, int WM_, int WN_, int NT_, int KC_>
struct PfgShape {
    static constexpr int MT = MT_, WM = WM_, WN = WN_, NT = NT_, KC = KC_;
    static constexpr int NW = WM * WN, BM = MT * WM, BN = MT * NT * WN;
    // one stage in LDS, as 16-byte slots: a[row][block] (the 16 quant bytes of
    // a weight block), b[token][2*block + half] (activation elements 16*half ..
    // +15), s[token][block pair] (the (d8, 8 sum) of two blocks), then the
    // dwords d[row][block pair] (two fp16 weight scales).  A row's blocks of a
    // stage are contiguous here as in memory, so that a DMA instruction reads
    // whole runs of 32 to 256 bytes.
    static constexpr int OB = KC * BM * 16, OS = OB + KC * 2 * BN * 16, OD = OS + KC / 2 * BN * 16;
    static constexpr int BYTES = OD + KC / 2 * BM * 4;
    // DMA instructions per stage: a, b, s, d
    static constexpr int NA = KC * BM / 64, NB = KC * 2 * BN / 64, NS = KC / 2 * BN / 64, ND = KC / 2 * BM / 64;
    static constexpr int NI = NA + NB + NS + ND, PW = (NI + NW - 1) / NW;
    static_assert(KC * BM % 64 == 0 && KC / 2 * BN % 64 == 0 && KC / 2 * BM % 64 == 0, "whole DMA instructions");
    static_assert(8 % KC == 0, "a stage is whole for every accepted bpr");
};

// Slot of piece x (0 .. n-1, n dividing 16) of a row of n slots: the pieces are
// XOR-permuted within the row so that the same piece of 16 consecutive rows
// lies in 16 different slots modulo 256 bytes (all LDS banks).  DMA writes
// slots in lane order; the permutation is applied to its source addresses.
__device__ __forceinline__ constexpr int pfg_slot(int n, int row, int x) { return row * n + (x ^ (row / (16 / n) % n)); }

// 4-byte LDS DMA (lane l's dword to lds + 4*l), wave-uniform base and per-lane offset.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void pfg_dma4(const void * sbase, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1"
                 :: "v"(voff), "s"(sbase), "s"(lds) : "memory", "m0");
}
#pragma clang diagnostic pop

// acc[e] = fma(d4 of lane e of the 16-lane row, t[e], acc[e]) for 4 or 8 results from E0 on.
// The s_nop covers the wait states between a VALU write of d and its DPP read,
// which the compiler does not see inside the asm.
#define PFG_FD(o, v, n) "v_fmac_f32_dpp %" #o ", %[d], %" #v " row_newbcast:%c" #n " row_mask:0xf bank_mask:0xf\n\t"
template <int E0>
__device__ __forceinline__ void pfg_fmac4(float * a, float d, const float * t) {
#ifdef __HIP_DEVICE_COMPILE__
    asm("s_nop 1\n\t" PFG_FD(0, 4, [e0]) PFG_FD(1, 5, [e1]) PFG_FD(2, 6, [e2]) PFG_FD(3, 7, [e3])
        : "+v"(a[E0]), "+v"(a[E0 + 1]), "+v"(a[E0 + 2]), "+v"(a[E0 + 3])
        : "v"(t[E0]), "v"(t[E0 + 1]), "v"(t[E0 + 2]), "v"(t[E0 + 3]), [d] "v"(d),
          [e0] "n"(E0), [e1] "n"(E0 + 1), [e2] "n"(E0 + 2), [e3] "n"(E0 + 3));
#endif
}
template <int E0>
__device__ __forceinline__ void pfg_fmac8(float * a, float d, const float * t) {
#ifdef __HIP_DEVICE_COMPILE__
    asm("s_nop 1\n\t" PFG_FD(0, 8, [e0]) PFG_FD(1, 9, [e1]) PFG_FD(2, 10, [e2]) PFG_FD(3, 11, [e3])
        PFG_FD(4, 12, [e4]) PFG_FD(5, 13, [e5]) PFG_FD(6, 14, [e6]) PFG_FD(7, 15, [e7])
        : "+v"(a[E0]), "+v"(a[E0 + 1]), "+v"(a[E0 + 2]), "+v"(a[E0 + 3]),
          "+v"(a[E0 + 4]), "+v"(a[E0 + 5]), "+v"(a[E0 + 6]), "+v"(a[E0 + 7])
        : "v"(t[E0]), "v"(t[E0 + 1]), "v"(t[E0 + 2]), "v"(t[E0 + 3]),
          "v"(t[E0 + 4]), "v"(t[E0 + 5]), "v"(t[E0 + 6]), "v"(t[E0 + 7]), [d] "v"(d),
          [e0] "n"(E0), [e1] "n"(E0 + 1), [e2] "n"(E0 + 2), [e3] "n"(E0 + 3),
          [e4] "n"(E0 + 4), [e5] "n"(E0 + 5), [e6] "n"(E0 + 6), [e7] "n"(E0 + 7));
#endif
}
#undef PFG_FD

// Bounded to the registers of 4 waves per SIMD, which the LDS of each shape admits
// (29, 58 and 38 KB a workgroup of 4, 16 and 4 waves, in the order of the table at
// the launch).  128 x 64 needs 129 registers: one is spilled, before and after the
// loop only.  Compiled for 3 waves it had the registers but an order of the pipeline
// that was slower (4096 tokens 51.5 -> 58.9 us).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wpass-failed"
template <class SH, bool ADD>
__global__ void __launch_bounds__(64 * SH::NW, 4)
lk_k_pf_gemm_q4_0(const uint8_t * __restrict__ qs, const _Float16 * __restrict__ d, int N, int bpr,
                  const int8_t * __restrict__ aqs, const float2 * __restrict__ asc, int ntok,
                  const float * __restrict__ scale, float * __restrict__ out, int out_ld) {
#pragma clang fp contract(off)
    constexpr int MT = SH::MT, NT = SH::NT, KC = SH::KC, NW = SH::NW, BM = SH::BM, BN = SH::BN, PW = SH::PW;
    constexpr int NE = MT == 32 ? 16 : 4;              // results per lane and MFMA tile
    __shared__ __attribute__((aligned(16))) uint8_t stg[2][SH::BYTES];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // XCD-aware tile order: workgroups are dispatched round-robin over the 8
    // XCDs (id % 8), so consecutive tile indices L are given to one XCD and L
    // runs over the row tiles first: an XCD holds a few token tiles with all
    // row tiles, and its L2 fetches each activation row once instead of every
    // XCD fetching all of them.
    const int nrt = N / BM, ntile = gridDim.x;
    const int id = blockIdx.x, x8 = id & 7, rem = ntile & 7;
    const int L = x8 * (ntile >> 3) + (x8 < rem ? x8 : rem) + (id >> 3);
    const int row0 = (L % nrt) * BM, tok0 = (L / nrt) * BN;
    const int wr = (w % SH::WM) * MT, wt = (w / SH::WM) * (MT * NT);   // the wave's sub-tile
    const int lm = lane & (MT - 1), h = lane / MT;     // MT 32: half 0/1; MT 16: lane group 0..3
    constexpr float MAGIC = 12582912.0f;               // 1.5 * 2^23 = float bits 0x4B400000

    // ---- staging: DMA instruction j = i*NW + w of a stage, i < PW, in the
    // order a, b, s, d.  Its lanes' byte offsets from the stage's first block
    // are formed once; a stage advances the uniform base only.
    auto below = [&](int i, int n) -> bool {           // instruction i*NW + w < n; known at compile time unless the kinds meet in i
        return i * NW + NW <= n || (i * NW < n && i * NW + w < n);
    };
    uint32_t voff[PW];
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        const int j = i * NW + w;
        if (below(i, SH::NA)) {
            const int slot = 64 * j + lane, r = slot / KC;
            voff[i] = (uint32_t) (r * bpr * 16 + (pfg_slot(KC, r, slot % KC) % KC) * 16);
        } else if (below(i, SH::NA + SH::NB)) {
            const int slot = 64 * (j - SH::NA) + lane, r = slot / (2 * KC), t = tok0 + r;
            voff[i] = (uint32_t) (t < ntok ? t : ntok - 1) * (uint32_t) (bpr * 32)             // clamped: in bounds
                      + (uint32_t) (pfg_slot(2 * KC, r, slot % (2 * KC)) % (2 * KC) * 16);
        } else if (below(i, SH::NA + SH::NB + SH::NS)) {
            const int slot = 64 * (j - SH::NA - SH::NB) + lane, r = slot / (KC / 2), t = tok0 + r;
            voff[i] = (uint32_t) (t < ntok ? t : ntok - 1) * (uint32_t) (bpr * 8)
                      + (uint32_t) (pfg_slot(KC / 2, r, slot % (KC / 2)) % (KC / 2) * 16);
        } else {
            const int slot = 64 * (j - SH::NA - SH::NB - SH::NS) + lane, r = slot / (KC / 2);
            voff[i] = (uint32_t) (r * bpr * 2 + slot % (KC / 2) * 4);
        }
    }
    const uint8_t * a_base = qs + (size_t) row0 * bpr * 16;
    const _Float16 * d_base = d + (size_t) row0 * bpr;
    const uint32_t lds0 = lk_lds_addr(&stg[0][0]);
    auto fetch = [&](int ck) {
        const uint32_t sb = lds0 + (uint32_t) ((ck & 1) * SH::BYTES);
        const int kb0 = ck * KC;
#pragma unroll
        for (int i = 0; i < PW; ++i) {
            const int j = i * NW + w;                  // wave-uniform
            if (below(i, SH::NA)) lk_dma16c_so(a_base + 16 * kb0, voff[i], sb + (uint32_t) (1024 * j));
            else if (below(i, SH::NA + SH::NB)) lk_dma16c_so(aqs + 32 * kb0, voff[i], sb + (uint32_t) (SH::OB + 1024 * (j - SH::NA)));
            else if (below(i, SH::NA + SH::NB + SH::NS))
                lk_dma16c_so(asc + kb0, voff[i], sb + (uint32_t) (SH::OS + 1024 * (j - SH::NA - SH::NB)));
            else if (below(i, SH::NI)) pfg_dma4(d_base + kb0, voff[i], sb + (uint32_t) (SH::OD + 256 * (j - SH::NA - SH::NB - SH::NS)));
        }
    };

    const int mb = 0x4B400000;
    // the row whose d4 this lane holds: result e of the lane's row group, e = lane % 16 (MT 16: % 4)
    const int c16 = lane & 15;
    const int drow = wr + (MT == 32 ? 8 * (c16 >> 2) + 4 * h + (c16 & 3) : 4 * h + (c16 & 3));
    float acc[NT][NE];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < NE; ++e) acc[j][e] = 0.0f;

    // The DMA of stage ck + 1 is issued after the barrier of stage ck, which
    // every wave reaches only when done reading stage ck - 1 (the same buffer).
    // (Rings of three and four stages were slower: their LDS costs co-resident
    // workgroups, 640 tokens 14.9 -> 18.6 and 21.1 us.)
    const int nck = bpr / KC;
    fetch(0);
    for (int ck = 0; ck < nck; ++ck) {
        lk_wait_vm<0>();
        __syncthreads();
        if (ck + 1 < nck) fetch(ck + 1);
        const uint8_t * S = stg[ck & 1];
        // The stage's NI = KC*NT MFMAs in the order block, token tile, as a
        // pipeline: operands are asked for two steps ahead and the MFMA of step
        // i + 1 is issued before the fmas of step i, so that it runs under
        // them (the sched_barriers keep only MFMAs from moving).  The compiler,
        // short of registers, sinks most reads of 128 x 64 to right before their
        // MFMA, with a wait for all of them in between.
        constexpr int NI = KC * NT;
        lk_i4g av[2], bv[2];                           // operands of the step's block / step, by parity
        uint32_t d2[2];
        float4 sv[2][NT];
        lk_f16g F[2];
        auto load = [&](int i) {
            const int b = i / NT, j = i % NT;
            if (j == 0) {
                if (b % 2 == 0) {
                    d2[(b / 2) & 1] = *(const uint32_t *) (S + SH::OD + (drow * (KC / 2) + b / 2) * 4);
#pragma unroll
                    for (int jj = 0; jj < NT; ++jj)
                        sv[(b / 2) & 1][jj] = *(const float4 *) (S + SH::OS + pfg_slot(KC / 2, wt + MT * jj + lm, b / 2) * 16);
                }
                const uint8_t * ap = S + pfg_slot(KC, wr + lm, b) * 16;
                if constexpr (MT == 32) av[b & 1] = *(const lk_i4g *) ap;
                else { const int2 q = *(const int2 *) (ap + 8 * (h & 1)); av[b & 1] = (lk_i4g){ q.x, q.y, 0, 0 }; }
            }
            const uint8_t * bp = S + SH::OB + pfg_slot(2 * KC, wt + MT * j + lm, 2 * b + (MT == 32 ? h : h >> 1)) * 16;
            if constexpr (MT == 32) bv[i & 1] = *(const lk_i4g *) bp;
            else { const int2 q = *(const int2 *) (bp + 8 * (h & 1)); bv[i & 1] = (lk_i4g){ q.x, q.y, 0, 0 }; }
        };
        lk_i4g a;                                      // nibbles of the block, low or high by lane half
        auto mfma = [&](int i) {
            const int b = i / NT;
            if (i % NT == 0) {
                const int nsh = MT == 32 ? 4 * h : 4 * (h >> 1);
#pragma unroll
                for (int k = 0; k < (MT == 32 ? 4 : 2); ++k) a[k] = (int) (((uint32_t) av[b & 1][k] >> nsh) & 0x0F0F0F0Fu);
            }
            if constexpr (MT == 32) {
                const lk_i16g seed = { mb, mb, mb, mb, mb, mb, mb, mb, mb, mb, mb, mb, mb, mb, mb, mb };
                F[i & 1] = __builtin_bit_cast(lk_f16g, __builtin_amdgcn_mfma_i32_32x32x32_i8(a, bv[i & 1], seed, 0, 0, 0));
            } else {
                const lk_i4g seed = { mb, mb, mb, mb };
                const int2 a2 = make_int2(a[0], a[1]), b2 = make_int2(bv[i & 1][0], bv[i & 1][1]);
                const lk_f4 f = __builtin_bit_cast(lk_f4, __builtin_amdgcn_mfma_i32_16x16x32_i8(
                    __builtin_bit_cast(long, a2), __builtin_bit_cast(long, b2), seed, 0, 0, 0));
#pragma unroll
                for (int e = 0; e < 4; ++e) F[i & 1][e] = f[e];
            }
        };
        load(0);
        if (NI > 1) load(1);
        mfma(0);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int b = i / NT, j = i % NT, u = b & 1;
            // the scales of this step, before load(i + 2) may replace them
            const uint32_t dd = d2[(b / 2) & 1];
            const float4 ss = sv[(b / 2) & 1][j];
            __builtin_amdgcn_sched_barrier(0x7F7);
            if (i + 1 < NI) mfma(i + 1);
            __builtin_amdgcn_sched_barrier(0x7F7);
            if (i + 2 < NI) load(i + 2);
            const float d4 = (float) __builtin_bit_cast(_Float16, (unsigned short) (u ? dd >> 16 : dd & 0xffff));
            const float d8 = u ? ss.z : ss.x, s8 = u ? ss.w : ss.y;
            const float c = __builtin_fmaf(d8, MAGIC, s8);
            float t[NE];
#pragma unroll
            for (int e = 0; e < NE; ++e) t[e] = __builtin_fmaf(d8, F[i & 1][e], -c);   // row 8(e/4) + 4h + e%4
            if constexpr (MT == 32) { pfg_fmac8<0>(acc[j], d4, t); pfg_fmac8<8>(acc[j], d4, t); }
            else pfg_fmac4<0>(acc[j], d4, t);
        }
    }
    // epilogue: lane holds, per token tile, 4 consecutive rows NE/4 times
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int t = tok0 + wt + MT * j + lm;
        if (t >= ntok) continue;
        const float sc = scale ? scale[t] : 1.0f;
#pragma unroll
        for (int a4 = 0; a4 < NE / 4; ++a4) {
            float4 * p = (float4 *) (out + (size_t) t * out_ld + row0 + wr + 8 * a4 + 4 * h);
            float4 v = make_float4(acc[j][4 * a4] * sc, acc[j][4 * a4 + 1] * sc,
                                   acc[j][4 * a4 + 2] * sc, acc[j][4 * a4 + 3] * sc);
            if (ADD) {
                const float4 o = *p;
                v = make_float4(o.x + v.x, o.y + v.y, o.z + v.z, o.w + v.w);
            }
            *p = v;
        }
    }
}
#pragma clang diagnostic pop

template <class SH>
static void pfg_launch(const uint8_t * qs, const _Float16 * d, int N, int bpr, const int8_t * aqs, const float2 * asc,
                       int ntok, const float * scale, float * out, int out_ld, int add, hipStream_t st) {
    const dim3 grid((N / SH::BM) * ((ntok + SH::BN - 1) / SH::BN));
    if (add)
        hipLaunchKernelGGL((lk_k_pf_gemm_q4_0<SH, true>), grid, dim3(64 * SH::NW), 0, st, qs, d, N, bpr, aqs, asc, ntok, scale, out, out_ld);
    else
        hipLaunchKernelGGL((lk_k_pf_gemm_q4_0<SH, false>), grid, dim3(64 * SH::NW), 0, st, qs, d, N, bpr, aqs, asc, ntok, scale, out, out_ld);
}

extern "C" int lk_pf_gemm_q4_0(const void * qs, const void * d, int N, int bpr, const int8_t * aqs,
                               const float * asc, int ntok, const float * scale, float * out, int out_ld,
                               int add, void * stream) {
    if (N < 0 || ntok < 0 || bpr < 1)
        return lk_fail(hipErrorInvalidValue, "lk_pf_gemm_q4_0: N %d / ntok %d / bpr %d", N, ntok, bpr);
    if (N == 0 || ntok == 0) return 0;
    if (N % 128 != 0 || bpr % 8 != 0 || out_ld % 4 != 0 || out_ld < N)
        return lk_fail(hipErrorInvalidValue, "lk_pf_gemm_q4_0: N %d must be a multiple of %d, bpr %d of %d, out_ld %d a multiple of 4 and >= N",
                       N, 128, bpr, 8, out_ld);
    // the kernel addresses activation rows with 32-bit byte offsets
    if ((size_t) ntok * bpr * 32 > 0xFFFFFFFFull)
        return lk_fail(hipErrorInvalidValue, "lk_pf_gemm_q4_0: ntok %d x bpr %d activations exceed 4 GiB", ntok, bpr);
    if (!qs || !d || !aqs || !asc || !out)
        return lk_fail(hipErrorInvalidValue, "lk_pf_gemm_q4_0: null pointer argument");
    // the widths the kernel loads and stores at: qs, aqs, asc and out 16 bytes, d 8 bytes, scale 4
    if (((uintptr_t) qs & 15) || ((uintptr_t) d & 7) || ((uintptr_t) aqs & 15) || ((uintptr_t) asc & 15) ||
        ((uintptr_t) out & 15) || ((uintptr_t) scale & 3))
        return lk_fail(hipErrorInvalidValue, "lk_pf_gemm_q4_0: misaligned argument (qs, aqs, asc, out 16 B; d 8 B; scale 4 B)");
    const hipStream_t st = lk_stream(stream);
    auto go = [&](auto sh) {
        pfg_launch<decltype(sh)>((const uint8_t *) qs, (const _Float16 *) d, N, bpr, aqs, (const float2 *) asc, ntok,
                                 scale, out, out_ld, add, st);
    };
    // The shape (2048 x 2048 weights, us per launch in a hipGraph; old: the one
    // shape of 128 x 128 in 8 waves with whole-line-per-lane staging that
    // served every size before):
    //   tokens       1    77   201   333   640   896   960  1024  1100  1536  2048  2999  4096
    //   old       25.6  27.5  29.5  30.2  30.2  30.8  30.8  30.6  31.3  32.2  33.7  49.1  56.3
    //   32 x 32    6.3   6.6   8.0  10.0  14.6  18.7  21.5  22.2  23.9  30.6  39.9  57.1  75.7
    //   128 x 128 21.4  22.4  22.9  23.5  23.5  23.8  23.9  24.4  24.2  24.9  28.4  48.2  53.5
    //   128 x 64  17.0  17.9  18.0  18.3  18.3  18.9  19.2  19.1  26.7  27.0  29.3  40.5  51.4
    // A launch takes a whole chain of bpr blocks per round of workgroups.  Up to
    // 7 tiles of 32 x 32 per CU (256 of them) the shortest chain wins; then 128 x
    // 128 in 16 waves while one round of the chip holds all of its tiles; past
    // that 128 x 64, four workgroups per CU, whose rounds end less ragged.
    // Between the first two, while the tiles of 128 x 64 fit one per CU (897 to
    // 1024 tokens here; 1793 to 2048 for 1024 rows, 598 to 640 for 3072), 128 x 64
    // would be shorter by 5 us: the lines do not give it that range.
    const long t32 = (long) (N / 32) * ((ntok + 31) / 32), t128 = (long) (N / 128) * ((ntok + 127) / 128);
    if (t32 <= 7 * 256)    go(PfgShape<16, 2, 2, 1, 8>{});
    else if (t128 <= 256)  go(PfgShape<32, 4, 4, 1, 4>{});
    else                   go(PfgShape<32, 4, 1, 2, 4>{});
    return lk_launch_status("lk_pf_gemm_q4_0");
}
