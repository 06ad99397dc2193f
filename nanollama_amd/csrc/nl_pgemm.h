// nl_pgemm.h -- the multi-token GEMM of long token runs and of K-quant files: Y[n][row] = sum_k W[row][k] X[n][k], every block format.
//
// Tile: a workgroup of four wavefronts owns RT 16-row weight tiles x 4 NTW / WR 16-token tiles.  Its threads expand the weights of a
// 128-column chunk ONCE into fp16 MFMA fragments in LDS (two buffers); every wavefront multiplies them against its own NTW token
// tiles, whose hi / lo activation fragments go straight from the fragment store into its registers.
//
// What bounds a launch of these sizes is not a pipe but latency: an activation fragment is an L2 or fabric round trip (500-2000
// cycles) away, a block of a 64 x 64 tile is 128 cycles of matrix work, and a prompt's narrow matrices give a compute unit one or two
// workgroups.  So the fragments of a WHOLE chunk are in flight -- block b's registers are requested again for the next chunk right
// behind block b's last MFMA --, raw weights are requested two chunks ahead, and the barrier between chunks orders LDS only
// (__syncthreads() also waits for every global load in flight, i.e. for exactly that prefetch).
//
// The activation fragment is the MFMA's A operand: D[token][row], a lane holds four tokens of ONE row, so a block's scale is one
// register (a chunk's four scales one ds_read_b128 per row tile) instead of four.  The accumulators go through LDS once at the end and
// the epilogues read whole rows of a token: coalesced stores, and fragments in either k-slot order.
//
// Arithmetic: weights as exact integers in fp16, x = hi + lo in fp16 (2^-22 of it; 2^-25 where it is below 2^-3, and finite below 65520),
// float32 accumulation, then
//   Q4_0 / Q8_0 (/ Q5_0)  acc += d_block * z                      per 32-column block (go/quant.go:74-94, :149-165)
//   F16                   its own operand, accumulated in the MFMA
// Files with K-quant matrices (PG_EXACT, every matrix of such a file): what the single-token plan computes in float32 stays that -- x as
// three bf16 parts (all 24 bits, all exponents), every product exact, sums in float32 with their rounding carried on:
//   Q4_0 / Q8_0           as above
//   Q4_K                  z over q - 8; acc += d * scale * z and acc -= (dmin * min - 8 d * scale) * sum(x) per block, sum(x) by MFMAs against ones (go/quant.go:296-323)
//   Q6_K                  scale * (q - 32) has 13 bits, two bf16 parts: six MFMAs; acc += d * z per block
//
// Measured (us a launch inside a model, profiled; Q|K|V, gate and up, mean of WO and down; in brackets the kernels that these launches ran on
// before): Q4_0, 2047 tokens, 768 columns: 18.9 (21.8), 37.2 (40.5), 18.5 (23.5); F16, 993 tokens, 1536 columns: 27.6 (35.6), 53.5 (85.0), 28.3
// (43.2), Q|K|V of both with the attention's images; Q4_K, 333 tokens, 768 columns, PG_EXACT: 9.9, 20.7, 12.0.  A 64 x 64 tile's block costs a
// wavefront about 310 cycles: 128 on the matrix pipe, the rest vector instructions (16 scalings, its share of the expansion, addresses).  Those
// overlap with the MFMAs of the SIMD's other wavefronts (1.47 PFLOP/s beside four vector instructions an MFMA) and not with its own, and a SIMD
// holds two or three; larger tiles share the expansion and the LDS reads.  A Q4_K prompt of 333 tokens (173M parameters) used to
// be 333 single-token steps: 151 ms, now 1.47 ms (1.92 at first, 1.49 then with two fp16 parts an activation, whose error was 1.59e-7 against 1.32e-7 of those
// steps and 1.19e-7 now, and whose range ends at 65504).
#pragma once
#include "nl_qgemm.h"
#include <type_traits>

namespace nl {

// LDS-only workgroup barrier
__device__ __forceinline__ void pg_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// raw buffer loads: a base in scalar registers, a lane's and a scalar 32-bit offset
typedef unsigned pg_u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned pg_u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t pg_rsrc(const void *p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, 0xffffffff, 0x00020000);       // (raw, 32-bit elements)
}
__device__ __forceinline__ uint4 pg_load16(__amdgpu_buffer_rsrc_t r, unsigned lane_off, unsigned off) {
    return __builtin_bit_cast(uint4, (pg_u32x4)__builtin_amdgcn_raw_buffer_load_b128(r, lane_off, off, 0));
}

enum { PG_NONE = 0, PG_BLOCK = 1 };   // when a sum is multiplied by its scale

// (1024 + b) for the bytes b of u as packed fp16: the two halves of four bytes
__device__ __forceinline__ h2_t pg_bytes_lo(uint32_t u) { return bits_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)); }
__device__ __forceinline__ h2_t pg_bytes_hi(uint32_t u) { return bits_h2(__builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)); }
__device__ __forceinline__ h2_t pg_h2(float v) { return h2_t{(_Float16)v, (_Float16)v}; }
__device__ __forceinline__ half8_t pg_join(h2_t a, h2_t b, h2_t c, h2_t d) {
    const uint4 u = make_uint4(h2_bits(a), h2_bits(b), h2_bits(c), h2_bits(d));
    return __builtin_bit_cast(half8_t, u);
}

// one (row, 32-column block) of the tile layout: NC 16-byte chunks and SW scale words; part w of its fragment; its scales
template <int WT> struct PgFmt;
template <> struct PgFmt<WT_Q4_0> {
    static constexpr int CPP = 2, NC = 1, SW = 1, SC = PG_BLOCK, FR = 1;
    static __device__ __forceinline__ int chunk(int h, int) { return h; }
    static __device__ __forceinline__ void part(const uint4 (&c)[1], const uint32_t (&)[1], int, int w, half8_t (&f)[1]) {
        f[0] = WFrag<WT_Q4_0>::expand(w == 0 ? c[0].x : w == 1 ? c[0].y : w == 2 ? c[0].z : c[0].w);
    }
    static __device__ __forceinline__ float scale(const uint32_t (&s)[1], int h) { return h2f_bits((s[0] >> (16 * h)) & 0xffff); }
    static __device__ __forceinline__ float least(const uint32_t (&)[1], int) { return 0.f; }
};
template <> struct PgFmt<WT_Q8_0> {
    static constexpr int CPP = 4, NC = 2, SW = 1, SC = PG_BLOCK, FR = 1;
    static __device__ __forceinline__ int chunk(int h, int i) { return 2 * h + i; }
    static __device__ __forceinline__ void part(const uint4 (&c)[2], const uint32_t (&)[1], int, int w, half8_t (&f)[1]) {
        const uint4 &v = c[w >> 1];
        const uint32_t a = ((w & 1) ? v.z : v.x) ^ 0x80808080u, b = ((w & 1) ? v.w : v.y) ^ 0x80808080u;   // 1024 + 128 + q, exact
        const h2_t off = pg_h2(1152.f);
        f[0] = pg_join(pg_bytes_lo(a) - off, pg_bytes_hi(a) - off, pg_bytes_lo(b) - off, pg_bytes_hi(b) - off);
    }
    static __device__ __forceinline__ float scale(const uint32_t (&s)[1], int h) { return h2f_bits((s[0] >> (16 * h)) & 0xffff); }
    static __device__ __forceinline__ float least(const uint32_t (&)[1], int) { return 0.f; }
};
template <> struct PgFmt<WT_F16> {
    static constexpr int CPP = 8, NC = 4, SW = 0, SC = PG_NONE, FR = 1;
    static __device__ __forceinline__ int chunk(int h, int i) { return 4 * h + i; }
    static __device__ __forceinline__ void part(const uint4 (&c)[4], const uint32_t (&)[1], int, int w, half8_t (&f)[1]) { f[0] = __builtin_bit_cast(half8_t, c[w]); }
    static __device__ __forceinline__ float scale(const uint32_t (&)[1], int) { return 1.f; }
    static __device__ __forceinline__ float least(const uint32_t (&)[1], int) { return 0.f; }
};
// Files with K-quant matrices (PG_EXACT): x in three bf16 parts, weights as integers that bf16 holds exactly, so every product is exact
__device__ __forceinline__ half8_t pg_bf16(const float (&v)[8]) {       // values of at most eight bits
    uint32_t u[8];
#pragma unroll
    for (int i = 0; i < 8; i++) u[i] = __float_as_uint(v[i]);
    return __builtin_bit_cast(half8_t, pack_bf16(u));
}
template <int WT> struct PgExact;
template <> struct PgExact<WT_Q4_0> : PgFmt<WT_Q4_0> {
    static __device__ __forceinline__ void part(const uint4 (&c)[1], const uint32_t (&)[1], int, int w, half8_t (&f)[1]) {
        const uint32_t u = w == 0 ? c[0].x : w == 1 ? c[0].y : w == 2 ? c[0].z : c[0].w;
        float v[8];                                                   // (k-slot order: load_x_slots)
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = (float)((u >> (8 * ((j & 1) * 2 + ((j >> 1) & 1)) + 4 * (j >> 2))) & 0xf) - 8.f;
        f[0] = pg_bf16(v);
    }
};
template <> struct PgExact<WT_Q8_0> : PgFmt<WT_Q8_0> {
    static __device__ __forceinline__ void part(const uint4 (&c)[2], const uint32_t (&)[1], int, int w, half8_t (&f)[1]) {
        const uint4 &q = c[w >> 1];
        const uint32_t u[2] = {(w & 1) ? q.z : q.x, (w & 1) ? q.w : q.y};
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = (float)(int)(int8_t)(u[j >> 2] >> (8 * (j & 3)));
        f[0] = pg_bf16(v);
    }
};
template <> struct PgExact<WT_Q4_K> {
    // pair p's 32 bytes: low nibbles = block 2p, high nibbles = block 2p + 1; words d | dmin and scale0 | min0 | scale1 | min1.
    // q - 8 and min - 8 scale: the sums of q x and of x would mostly cancel (relative error of a 512-column model 1.06e-7 instead of 7.6e-8)
    static constexpr int CPP = 2, NC = 2, SW = 2, SC = PG_BLOCK, FR = 1;
    static __device__ __forceinline__ int chunk(int, int i) { return i; }
    static __device__ __forceinline__ void part(const uint4 (&c)[2], const uint32_t (&)[2], int h, int w, half8_t (&f)[1]) {
        const uint4 &q = c[w >> 1];
        const uint32_t u[2] = {(w & 1) ? q.z : q.x, (w & 1) ? q.w : q.y};
        // the nibbles where they are, in the mantissa of fp16 numbers: 1024 + q or 1024 + 16 q, and q - 8 by one v_fma_mix_f32 each, exactly.  (A field extraction,
        // a subtraction and a conversion a value: 223 vector instructions a chunk beside its 24 MFMAs, now 175.  us a launch: 1536 x 1536 and x 4096, 33 tokens, the
        // mean 18.4 -> 16.7, 768 x 768 and x 2048, 100 tokens 12.0 -> 10.8, gate and up there 12.2 -> 11.6.  Q6_K's products by a scale gain nothing by it: 20.6, 20.8)
        const uint32_t mask = h ? 0x00f000f0u : 0x000f000fu;
        const float mul = h ? 0.0625f : 1.f, add = h ? -72.f : -1032.f;
        float v[8];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const h2_t n = bits_h2(((u[j >> 1] >> (8 * (j & 1))) & mask) | 0x64006400u);      // bytes j & 1 and (j & 1) + 2
            v[4 * (j >> 1) + (j & 1)] = fmaf((float)n[0], mul, add);
            v[4 * (j >> 1) + (j & 1) + 2] = fmaf((float)n[1], mul, add);
        }
        f[0] = pg_bf16(v);
    }
    static __device__ __forceinline__ float scale(const uint32_t (&s)[2], int h) { return h2f_bits(s[0] & 0xffff) * (float)((s[1] >> (16 * h)) & 0xff); }     // (17 bits)
    static __device__ __forceinline__ float least(const uint32_t (&s)[2], int h) { return h2f_bits(s[0] >> 16) * (float)((s[1] >> (16 * h + 8)) & 0xff) - 8.f * scale(s, h); }
};
template <> struct PgExact<WT_Q6_K> {
    // int8 (q - 32); words d and four int8 scales of 16 columns each.  scale * (q - 32) has 13 bits: two parts
    static constexpr int CPP = 4, NC = 2, SW = 2, SC = PG_BLOCK, FR = 2;
    static __device__ __forceinline__ int chunk(int h, int i) { return 2 * h + i; }
    static __device__ __forceinline__ void part(const uint4 (&c)[2], const uint32_t (&s)[2], int h, int w, half8_t (&f)[2]) {
        const uint4 &q = c[w >> 1];
        const float sc = (float)(int)(int8_t)(s[1] >> (8 * (2 * h + (w >> 1))));
        const uint32_t u[2] = {(w & 1) ? q.z : q.x, (w & 1) ? q.w : q.y};
        float hi[8], lo[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float v = (float)(int)(int8_t)(u[j >> 2] >> (8 * (j & 3))) * sc;
            hi[j] = __uint_as_float(__float_as_uint(v) & 0xffff0000u);
            lo[j] = v - hi[j];
        }
        f[0] = pg_bf16(hi);
        f[1] = pg_bf16(lo);
    }
    static __device__ __forceinline__ float scale(const uint32_t (&s)[2], int) { return h2f_bits(s[0] & 0xffff); }
    static __device__ __forceinline__ float least(const uint32_t (&)[2], int) { return 0.f; }
};
typedef __bf16 pg_bf16x8 __attribute__((ext_vector_type(8)));
template <bool BF16>
__device__ __forceinline__ f32x4_t pg_mma(const uint4 &x, const half8_t &w, f32x4_t c) {
    if constexpr (BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(pg_bf16x8, x), __builtin_bit_cast(pg_bf16x8, w), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, x), w, c, 0, 0, 0);
}
enum { PG_HILO = 0, PG_HI = 1, PG_EXACT = 2 };

// WR: the wavefronts of a set split the rows WR ways and share 64 NTW / WR tokens.
// EPI: QG_EPI_PLAIN (out / resid / bias; optionally the folded norm's fragments and sums of squares), QG_EPI_SWIGLU
// (RT / 2 tiles of gate, the same of up), QG_EPI_ROPE (a layer's packed Q|K|V).  PREC: PG_HILO; PG_HI, the single-product precision mode of
// Q4_0 prompts (block scales multiplied into the fp16 weights, only the hi half of every activation); PG_EXACT.
// Wavefronts per SIMD: a plain 64 x 64 Q4_0 tile is held to 168 registers, three workgroups a compute unit (172 without the bound, since the
// loads are buffer loads: two.  WO and down of 2112 x 2112 and 2112 x 5632, 1000 tokens, 528 workgroups, mean of both: 63.4 us two at a time,
// 53.9 three).  What it spills is a value of the epilogue's, around the K loop.
// KWR: sets + 16 (WR - 1)
template <int WT, int RT, int NTW, int KWR, int EPI, int PREC = PG_HILO>
__global__ void __launch_bounds__(256 * (KWR & 15), ((KWR & 15) > 1 ? 1 : WT == WT_Q4_0 && RT == 4 && NTW == 1 && PREC == PG_HILO ? 3 : 2)) pgemm_kernel(QGemmParams P) {
    constexpr int KW = KWR & 15, WR = (KWR >> 4) + 1;
    constexpr bool X1 = PREC == PG_HI, EXACT = PREC == PG_EXACT;
    using F = typename std::conditional_t<EXACT, PgExact<WT>, PgFmt<WT>>;
    static_assert(!X1 || WT == WT_Q4_0, "the single-product mode is Q4_0's");
    static_assert(RT >= 4 || (EXACT && NTW == 1 && WR <= RT && KW == 2 && RT == (EPI == QG_EPI_SWIGLU ? 2 : 1)), "slim tiles");
    constexpr int NP = X1 ? 1 : EXACT ? 3 : 2, PS = EXACT ? 3 : 2;      // parts of an activation that are read, and that are stored
    constexpr int KB = 4;                                   // blocks per chunk
    constexpr int RTW = RT / WR, TTW = 4 * NTW / WR;        // row tiles of a wavefront, token tiles of a workgroup
    // tiles of one or two row tiles (pg_slim): four or two wavefronts share a block's expansion, one or two of its four parts each
    constexpr int SPL = RT >= 4 ? 1 : 4 / RT, NPT = 4 / SPL;
    constexpr int ROWS = RT * TR, TOK = TTW * 16, IPT = RT >= 4 ? ROWS * KB / 256 : 1, LD = ROWS + 4, SWN = F::SW ? F::SW : 1;
    constexpr int SC = X1 ? PG_NONE : F::SC;
    constexpr bool MINS = WT == WT_Q4_K, PAIRS = EXACT || WT == WT_Q4_0;
    // The bounded tile whose epilogue spills makes the scales' offset of the weights' (52 bytes of scratch otherwise: 2112 columns, 1000 tokens, all of its
    // GEMMs 804 us, now 798; tiles that have the registers lose 0.5 to 1.5 % by it)
    constexpr bool TIGHT = WT == WT_Q4_0 && RT == 4 && NTW == 1 && KW == 1 && EPI == QG_EPI_PLAIN && PREC == PG_HILO;
    // a block's plane of fragments is padded by 64 bytes: the two pairs' expansions of a wavefront land on different banks
    constexpr int PLANE = F::FR * RT * 1024 + 64, BUF = KB * PLANE, SCP = ROWS + 16, SCB = SCP * KB * 4, WBYTES = 2 * (BUF + (SC ? SCB : 0) + (MINS ? SCB : 0));
    constexpr int SBYTES = TOK * LD * 4, SET = WBYTES > SBYTES ? WBYTES : SBYTES, NTHR = 256 * KW;
    __shared__ __attribute__((aligned(16))) char smem_all[KW * SET];
    __shared__ float s_tok[TOK];                            // consumer of a folded norm: 1 / rms per token; producer: the fragments' pre-scale
    __shared__ __attribute__((aligned(16))) float s_gain[EPI == QG_EPI_PLAIN ? ROWS : 4];
    // KW sets of four wavefronts take every KW-th chunk each, with weight buffers of their own; the epilogue adds their sums in set order
    const int kset = KW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    char *const smem = smem_all + kset * SET;
    const int tid = threadIdx.x & 255, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, li = lane & 15, lq = lane >> 4;
    const int nblocks = P.cols / 32, nchunks = P.npairs / KL * 2 + ((P.npairs % KL) + 1) / 2;
    constexpr bool FUSED = EPI == QG_EPI_SWIGLU;
    constexpr int TPW = FUSED ? RT / 2 : RT;                // row tiles of a matrix per workgroup
    const int nrb = (P.ntiles + TPW - 1) / TPW, ntb = (P.n_tokens + TOK - 1) / TOK, total = nrb * ntb, per = (total + 7) / 8;
    // blocks b, b + 8, ... run on one XCD, which takes a contiguous range of the tiles: of the operand that runs along the range each XCD
    // reads an eighth, the other one it streams whole -- the smaller one (fragments are 2 PS bytes a value, weights 16 CPP bytes a pair and row)
    const int id = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (((int)blockIdx.x >> 3) >= per || id >= total) return;
    const bool by_rows = (long long)P.ntiles * TR * (FUSED ? 2 : 1) * F::CPP > (long long)P.n_tokens * 8 * PS;
    const int tb = by_rows ? id % ntb : id / nrb, rbk = by_rows ? id / ntb : id % nrb, tile0 = rbk * TPW, row0 = tile0 * TR, tok0 = tb * TOK, wt0 = wave % (4 / WR) * NTW, ttile0 = tb * TTW + wt0, wr0 = wave / (4 / WR) * RTW;

    // F16 and Q8_0: a group of four pairs is two chunks, the even blocks of its pairs, then the odd ones.  A wavefront's load is then one 16-byte plane of
    // all four pairs over a tile's rows, a whole KiB; two pairs with both their blocks (PAIRS) are half of every 64-byte run, twice the sectors.  Profiled
    // inside a model, Q|K|V / gate and up / mean of WO and down: F16, 993 tokens, 1536 columns 29.9 / 57.0 / 30.8 us, now 27.6 / 53.5 / 28.3; Q8_0, 700 tokens
    // 20.9 / 53.3 / 28.5, now 20.8 / 50.4 / 26.4 (and Q|K|V writes the attention's images now).  Q4_0's blocks are one plane, K-quants' two share their bytes:
    // nothing to gain (Q|K|V 17.3 and 17.6, 11.8 and 11.9).
    // A last group of one or two pairs is one chunk of both their blocks.
    // staging items: block kk of the chunk, row r, row tile
    const int i_kk = PAIRS ? 2 * (tid & 1) + ((tid >> 5) & 1) : tid & 3, i_r = (PAIRS ? tid >> 1 : tid >> 2) & 15, i_t = SPL == 1 ? wave : wave % RT, i_w = SPL == 1 ? 0 : wave / RT * NPT;
    struct Raw { uint4 c[F::NC]; uint32_t s[SWN]; };
    // Weights as raw buffer loads from the workgroup's first tile: the wavefront's row tile and the chunk are scalar arithmetic, the lane's part is a
    // register that changes in the last group only.  (With a 64-bit address per load a chunk's staging was 100 of a wavefront's 224 vector
    // instructions beside 128 MFMAs: 841M F16, 993 tokens 5456 us against 5400; 173M Q4_K, 333 tokens 1961 against 1911)
    constexpr unsigned QG = F::CPP * TR * 16, SG = TR * F::SW * 4;      // bytes of a pair over a tile's rows
    const __amdgpu_buffer_rsrc_t rq0 = pg_rsrc(P.q + (size_t)tile0 * P.npairs * QG), rq1 = pg_rsrc((FUSED ? P.q1 : P.q) + (size_t)tile0 * P.npairs * QG);
    [[maybe_unused]] const __amdgpu_buffer_rsrc_t rs0 = pg_rsrc(reinterpret_cast<const char *>(P.s) + (size_t)tile0 * P.npairs * SG),
                                                  rs1 = pg_rsrc(reinterpret_cast<const char *>(FUSED ? P.s1 : P.s) + (size_t)tile0 * P.npairs * SG);
    const int last_g = (P.npairs - 1) / KL, last_sz = P.npairs - last_g * KL;
    // a chunk's group; whether it holds both blocks of two pairs
    auto group_of = [&](int chunk) __attribute__((always_inline)) { return min(chunk, nchunks - 1) >> 1; };
    auto paired = [&](int g) __attribute__((always_inline)) { return PAIRS || (g == last_g && last_sz <= 2); };
    const unsigned lane_s = (unsigned)(i_r * KL + (PAIRS ? i_kk >> 1 : i_kk)), lane_q = (lane_s + (PAIRS ? (unsigned)F::chunk(i_kk & 1, 0) * (TR * KL) : 0u)) * 16u;
    auto stage_load = [&](int chunk, Raw (&r)[IPT]) __attribute__((always_inline)) {
        const int c = min(chunk, nchunks - 1), g = c >> 1;      // (a chunk past the end: the last one's, never used)
        unsigned lq_ = lane_q, ls_ = lane_s * F::SW * 4u, step = TR * KL * 16u;          // plane F::chunk(h, j): j steps on
        const unsigned k0 = PAIRS ? (unsigned)(c & 1) * 2u : 0u;
        if (PAIRS ? min(KL, P.npairs - g * KL) != KL : last_sz != KL && g == last_g) {
            const bool both = paired(g);
            const unsigned row_pair = (unsigned)(i_r * last_sz + min(both ? i_kk >> 1 : i_kk, last_sz - 1 - (int)k0));
            step = (unsigned)(TR * last_sz) * 16u;
            lq_ = row_pair * 16u + (both ? (unsigned)F::chunk(i_kk & 1, 0) * step : 0u);
            ls_ = row_pair * F::SW * 4u;
        }
        if constexpr (TIGHT) ls_ = (lq_ - (unsigned)F::chunk(i_kk & 1, 0) * step) / 4u * F::SW;
        const unsigned first = k0 * 16u + (paired(g) ? 0u : (unsigned)F::chunk(c & 1, 0) * step);
#pragma unroll
        for (int i = 0; i < IPT; i++) {
            const int rt = i_t + 4 * i, dt = min(FUSED ? rt % TPW : rt, P.ntiles - 1 - tile0);
            const bool second = FUSED && rt >= TPW;
            const unsigned gp = (unsigned)(dt * P.npairs + g * KL);
#pragma unroll
            for (int j = 0; j < F::NC; j++) r[i].c[j] = pg_load16(second ? rq1 : rq0, lq_, gp * QG + first + j * step);
            if constexpr (F::SW > 0) {
                const unsigned so = gp * SG + k0 * 4u * F::SW;
                if constexpr (F::SW == 2) {
                    const pg_u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(second ? rs1 : rs0, ls_, so, 0);
                    r[i].s[0] = v[0];
                    r[i].s[SWN - 1] = v[1];
                } else r[i].s[0] = __builtin_amdgcn_raw_buffer_load_b32(second ? rs1 : rs0, ls_, so, 0);
            } else r[i].s[0] = 0;
        }
    };
    char *const s_sc = smem + 2 * BUF, *const s_mn = s_sc + 2 * SCB;
    // block b of a chunk
    auto block_of = [&](int chunk, int b) __attribute__((always_inline)) {
        if (PAIRS) return chunk * KB + b;
        const int g = group_of(chunk);
        return g * 2 * KL + (paired(g) ? b : 2 * b + (chunk & 1));
    };
    auto stage_expand = [&](int chunk, int buf, int w, const Raw (&r)[IPT]) __attribute__((always_inline)) {
        const int g = group_of(chunk), i_h = paired(g) ? i_kk & 1 : chunk & 1, b = i_kk;
        const bool live = (PAIRS || chunk < nchunks) && block_of(chunk, i_kk) < nblocks;     // a block past the end of K contributes nothing
#pragma unroll
        for (int i = 0; i < IPT; i++) {
            const int rt = i_t + 4 * i;
            half8_t f[F::FR];
            F::part(r[i].c, r[i].s, i_h, w, f);
            if constexpr (X1) {
                const _Float16 d = (_Float16)(live ? F::scale(r[i].s, i_h) : 0.f);      // (an fp16 value: exact)
#pragma unroll
                for (int e = 0; e < 8; e++) f[0][e] = f[0][e] * d;
            }
            if constexpr (SC == PG_NONE && !X1) if (!live) f[0] = half8_t{};
#pragma unroll
            for (int p = 0; p < F::FR; p++)
                *reinterpret_cast<uint4 *>(smem + buf * BUF + b * PLANE + ((p * RT + rt) * 64 + w * 16 + i_r) * 16) = __builtin_bit_cast(uint4, f[p]);
            if constexpr (SC != PG_NONE)
                if (w == 0) *reinterpret_cast<float *>(s_sc + buf * SCB + (b * SCP + rt * 16 + i_r) * 4) = live ? F::scale(r[i].s, i_h) : 0.f;
            if constexpr (MINS)
                if (w == 0) *reinterpret_cast<float *>(s_mn + buf * SCB + (b * SCP + rt * 16 + i_r) * 4) = live ? F::least(r[i].s, i_h) : 0.f;
        }
    };
    auto stage_part = [&](int chunk, int buf, int w, const Raw (&r)[IPT]) __attribute__((always_inline)) {
        if constexpr (SPL == 1) stage_expand(chunk, buf, w, r);
        else switch (i_w + w) {                             // (the wavefront's: constants inside)
            case 0: stage_expand(chunk, buf, 0, r); break;
            case 1: stage_expand(chunk, buf, 1, r); break;
            case 2: stage_expand(chunk, buf, 2, r); break;
            default: stage_expand(chunk, buf, 3, r); break;
        }
    };
    // activation fragments [block][token tile][part][lane] x 16 bytes: kernel argument + 32-bit offset, the block part wave-uniform
    const __amdgpu_buffer_rsrc_t rx = pg_rsrc(P.xf);
    unsigned xtile[NTW];
#pragma unroll
    for (int t = 0; t < NTW; t++) xtile[t] = (unsigned)min(ttile0 + t, P.nt16 - 1) * (unsigned)(PS * QG_FRAG * 16);
    const unsigned xblock = (unsigned)P.nt16 * (unsigned)(PS * QG_FRAG) * 16u, xlane = (unsigned)lane * 16u;
    uint4 xp[NP][KB][NTW];
    auto xload = [&](int chunk, int b) __attribute__((always_inline)) {
        const unsigned uo = (unsigned)min(block_of(chunk, b), nblocks - 1) * xblock;
#pragma unroll
        for (int t = 0; t < NTW; t++)
#pragma unroll
            for (int k = 0; k < NP; k++) xp[k][b][t] = pg_load16(rx, xlane, uo + xtile[t] + k * QG_FRAG * 16);
    };
    f32x4_t acc[RTW][NTW];
#pragma unroll
    for (int rt = 0; rt < RTW; rt++)
#pragma unroll
        for (int t = 0; t < NTW; t++) acc[rt][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // PG_EXACT: the sums of two chunks are kept apart and join the accumulators with what the addition drops carried on (Kahan): a plain
    // chain over K / 32 blocks is further off than the single-token plan's lanes and trees (relative error at K = 10752 1.8e-7 against 1.1e-7)
    [[maybe_unused]] f32x4_t part[EXACT ? RTW : 1][NTW] = {}, lost[EXACT ? RTW : 1][NTW] = {};

    const int niter = (nchunks + KW - 1) / KW;               // (every set runs as many chunks; past the end of K: zeros)
    int chunk = kset;
    Raw rb[2][IPT];                                         // raw weights of the next chunk and of the one after it
    stage_load(chunk, rb[1]);
#pragma unroll
    for (int b = 0; b < KB; b++) xload(chunk, b);
    stage_load(chunk + KW, rb[0]);
    // folded RMSNorm, consumer side: 1 / rms of this workgroup's tokens from the producer's partial sums of squares, 256 / TOK threads a token
    if constexpr (EPI != QG_EPI_PLAIN)
        if (P.nrm_in.ssq) {
            constexpr int TPT = 256 / TOK;
            const int t = tid / TPT, n = min(tok0 + t, P.n_tokens - 1), p0 = tid % TPT;
            const double *sp = P.nrm_in.ssq + (size_t)n * P.nrm_in.nrb;
            double tot = 0.0;
            for (int r0 = p0; r0 < P.nrm_in.nrb; r0 += 8 * TPT) {
                double v[8];
#pragma unroll
                for (int j = 0; j < 8; j++) v[j] = sp[min(r0 + j * TPT, P.nrm_in.nrb - 1)];
#pragma unroll
                for (int j = 0; j < 8; j++) tot += r0 + j * TPT < P.nrm_in.nrb ? v[j] : 0.0;
            }
#pragma unroll
            for (int m = 1; m < TPT; m *= 2) tot += __shfl_xor(tot, m);
            float inv = (float)(1.0 / sqrt(tot / (double)P.nrm_in.dim + (double)P.nrm_in.eps));
            if (P.nrm_in.scale) {        // the producer's power-of-two pre-scale (norm_prescale, nl_qgemm.h), undone exactly
                if (rbk == 0 && p0 == 0) P.nrm_in.scale_next[n] = norm_prescale(inv);
                inv *= 1.0f / P.nrm_in.scale[n];
            }
            if (p0 == 0) s_tok[t] = inv;
        }
    // producer: what its epilogue needs is requested here, ahead of the K loop -- behind it, every dependent fetch is a round trip of its own
    constexpr int RQ = ROWS / 4, NIT = TOK * RQ > NTHR ? TOK * RQ / NTHR : 1, NRES = EPI == QG_EPI_PLAIN && NIT <= 4 && !(EXACT && KW == 1) ? NIT : 1;    // (EXACT, one set: no registers for it)
    [[maybe_unused]] f32x4_t res[NRES];
    [[maybe_unused]] const bool vec = (P.ldo & 3) == 0;
    [[maybe_unused]] const float *const resid = P.resid;
    [[maybe_unused]] auto load_res = [&](int i) {
        const int it = i * NTHR + (int)threadIdx.x, a = it % RQ, n = min(tok0 + it / RQ, P.n_tokens - 1), row = row0 + 4 * a;
        return resid && vec && row + 3 < P.rows ? *reinterpret_cast<const f32x4_t *>(resid + (size_t)n * P.ldo + row) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    };
    if constexpr (EPI == QG_EPI_PLAIN) {
        if (NRES == NIT)
#pragma unroll
            for (int i = 0; i < NRES; i++) res[i] = load_res(i);
        if (P.nrm_out.w) {
            for (int i = threadIdx.x; i < ROWS; i += NTHR) s_gain[i] = P.nrm_out.w[min(row0 + i, P.rows - 1)];
            for (int i = threadIdx.x; i < TOK; i += NTHR) s_tok[i] = P.nrm_out.scale ? P.nrm_out.scale[min(tok0 + i, P.n_tokens - 1)] : 1.0f;
        }
    }
#pragma unroll
    for (int w = 0; w < NPT; w++) stage_part(chunk, 0, w, rb[1]);
    stage_load(chunk + 2 * KW, rb[1]);
    // The K loop is a pipeline of groups (RG row tiles x NTW token tiles: four independent MFMA chains): while group i is on the matrix
    // cores, group i + 1's weight fragments leave LDS and group i - 1's sums are scaled.  One barrier per chunk, in front of its last
    // group: the next chunk's fragments are then complete (all parts were stored by block 2) and the last group's are already in
    // registers, so the buffer that the next chunk's stores will overwrite has no reader left.
    constexpr int RG = RTW == 1 ? 1 : NTW == 1 && !EXACT && RTW >= 4 ? 4 : 2, NG = RTW / RG, STEPS = KB * NG;
    static_assert(STEPS % 2 == 0, "ping-pong");
    half8_t wf[2][F::FR][RG];
    f32x4_t z[2][RG][NTW], xs[2][NTW];
    [[maybe_unused]] f32x4_t zs[2][RG][NTW];      // PG_EXACT: sums of the products with a second or third part
    float dv[4][RG], mv[4][RG];         // of groups idx - 1 .. idx + 1
    auto read_w = [&](int bf, int idx) {
        const int b = idx / NG, r0 = (idx % NG) * RG;
#pragma unroll
        for (int p = 0; p < F::FR; p++)
#pragma unroll
            for (int q = 0; q < RG; q++)
                wf[idx & 1][p][q] = *reinterpret_cast<const half8_t *>(smem + bf * BUF + b * PLANE + (p * RT + wr0 + r0 + q) * 1024 + lane * 16);
#pragma unroll
        for (int q = 0; q < RG; q++) {
            if constexpr (SC != PG_NONE) dv[idx & 3][q] = *reinterpret_cast<const float *>(s_sc + bf * SCB + (b * SCP + (wr0 + r0 + q) * 16 + li) * 4);
            if constexpr (MINS) mv[idx & 3][q] = *reinterpret_cast<const float *>(s_mn + bf * SCB + (b * SCP + (wr0 + r0 + q) * 16 + li) * 4);
        }
    };
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    // the sums of group idx into the accumulators
    auto scale_sums = [&](int idx) {
        const int b = idx / NG, g = idx % NG;
#pragma unroll
        for (int q = 0; q < RG; q++)
#pragma unroll
            for (int t = 0; t < NTW; t++) {
                const int rt = g * RG + q;
                f32x4_t &to = EXACT ? part[EXACT ? rt : 0][t] : acc[rt][t];
                if constexpr (EXACT) {
                    // (as many roundings as possible at the size of a block's sum instead of the running one's)
                    const f32x4_t all = z[idx & 1][q][t] + zs[idx & 1][q][t];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        if constexpr (MINS) to[j] += fmaf(all[j], dv[idx & 3][q], -mv[idx & 3][q] * xs[b & 1][t][j]);
                        else to[j] = fmaf(all[j], dv[idx & 3][q], to[j]);
                    }
                } else if constexpr (SC == PG_BLOCK) {
#pragma unroll
                    for (int j = 0; j < 4; j++) to[j] = fmaf(z[idx & 1][q][t][j], dv[idx & 3][q], to[j]);
                }
                asm volatile("" : "+v"(to));     // (hipcc otherwise sinks the scalings of a chunk below its MFMAs: 4 x the live registers)
            }
    };
    pg_barrier();
    read_w(0, 0);
    // one chunk; PAR: its parity (which buffer and which raw registers)
    auto do_chunk = [&](auto par_tag) {
        constexpr int PAR = decltype(par_tag)::value;
        const int nxt = chunk + KW;
#pragma unroll
        for (int idx = 0; idx < STEPS; idx++) {
            const int b = idx / NG, g = idx % NG;
            if (idx == STEPS - 1) pg_barrier();
            if (idx + 1 < STEPS) read_w(PAR, idx + 1);
            else read_w(PAR ^ 1, 0);
            if constexpr (MINS)
                if (g == 0) {
                    const half8_t ones = __builtin_bit_cast(half8_t, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));
#pragma unroll
                    for (int t = 0; t < NTW; t++) {
                        const f32x4_t less = pg_mma<EXACT>(xp[1][b][t], ones, pg_mma<EXACT>(xp[2][b][t], ones, zero));
                        xs[b & 1][t] = pg_mma<EXACT>(xp[0][b][t], ones, zero) + less;
                    }
                }
            // part k of the activations times part p of the weights
            auto mul = [&](int p, int k, f32x4_t (&sum)[2][RG][NTW], bool start) {
#pragma unroll
                for (int q = 0; q < RG; q++)
#pragma unroll
                    for (int t = 0; t < NTW; t++) {
                        f32x4_t &to = SC == PG_BLOCK ? sum[idx & 1][q][t] : acc[g * RG + q][t];
                        to = pg_mma<EXACT>(xp[k][b][t], wf[idx & 1][p][q], SC == PG_BLOCK && start ? zero : to);
                    }
            };
            if constexpr (EXACT) {
                // An MFMA rounds the sum with its C operand down, not to nearest: the large products have C = 0, and their sum meets the small
                // ones' in scale_sums (all in one chain: mean error -1.9e-8 of the result at K = 2048, and 1.3e-7 instead of 1e-7 for Q6_K)
#pragma unroll
                for (int k = F::FR + 1; k > 0; k--)
#pragma unroll
                    for (int p = F::FR - 1; p >= 0; p--)
                        if (k - p >= 0 && k - p < 3) mul(p, k - p, zs, k == F::FR + 1);
                mul(0, 0, z, true);
            } else {
                if constexpr (!X1) mul(0, 1, z, true);
                mul(0, 0, z, X1);
            }
            if (idx) scale_sums(idx - 1);
            if (g == NG - 1) {
                xload(nxt, b);
                if (b < KB - 1 && b < NPT) stage_part(nxt, PAR ^ 1, b, rb[PAR]);
                if (b == KB - 2) {
                    if constexpr (NPT == 4) stage_part(nxt, PAR ^ 1, KB - 1, rb[PAR]);
                    stage_load(nxt + 2 * KW, rb[PAR]);
                }
            }
        }
        scale_sums(STEPS - 1);
        chunk = nxt;
    };
    for (int i = 0; i < niter; i += 2) {
        do_chunk(std::integral_constant<int, 0>{});
        if (i + 1 < niter) do_chunk(std::integral_constant<int, 1>{});
        if constexpr (EXACT) {
#pragma unroll
            for (int rt = 0; rt < RTW; rt++)
#pragma unroll
                for (int t = 0; t < NTW; t++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float y = part[rt][t][j] - lost[rt][t][j], to = acc[rt][t][j] + y;
                        const float l = (to - acc[rt][t][j]) - y;
                        lost[rt][t][j] = l == l ? l : 0.f;       // (an infinity stays one)
                        acc[rt][t][j] = to;
                        part[rt][t][j] = 0.f;
                    }
        }
    }

    // accumulators -> LDS [token][row], then whole rows of a token
    __syncthreads();
    float *const S = reinterpret_cast<float *>(smem);
#pragma unroll
    for (int rt = 0; rt < RTW; rt++)
#pragma unroll
        for (int t = 0; t < NTW; t++)
#pragma unroll
            for (int j = 0; j < 4; j++) S[((wt0 + t) * 16 + 4 * lq + j) * LD + (wr0 + rt) * 16 + li] = acc[rt][t][j];
    __syncthreads();
    const int et = threadIdx.x;
    const float *const S0 = reinterpret_cast<const float *>(smem_all);
    float *const SW = reinterpret_cast<float *>(smem_all);
    auto sum4 = [&](int off) {
        f32x4_t v = *reinterpret_cast<const f32x4_t *>(S0 + off);
#pragma unroll
        for (int k = 1; k < KW; k++) v += *reinterpret_cast<const f32x4_t *>(S0 + k * (SET / 4) + off);
        return v;
    };
    const bool folded_in = EPI != QG_EPI_PLAIN && P.nrm_in.ssq != nullptr;

    if constexpr (EPI == QG_EPI_SWIGLU) {
        // h = SiLU(gate) * up (go/quant.go:629-631, go/model.go:604-606), stored as the down projection's fragments (RT = 2: half of a block's k-slots)
#pragma unroll
        for (int it0 = 0; it0 < TOK * RT; it0 += NTHR) {
            const int it = it0 + et, w = RT == 2 ? (tile0 & 1) * 2 + (lq & 1) : lane >> 4, tt = RT == 2 ? it >> 5 : (it >> 6) % TTW, hb = RT == 2 ? 0 : (it >> 6) / TTW, t = tt * 16 + li, n = tok0 + t;
            const int hblk = tile0 / 2 + hb;
            if (NTHR > TOK * RT && (RT == 2 ? tt >= TTW : hb >= RT / 4)) break;     // (more threads than items of 32 rows)
            int oa, ob;
            slot_offsets(RT == 2 ? 0 : P.out_q4, RT == 2 ? lq & 1 : w, oa, ob);
            const int sg = t * LD + hb * 32, su = sg + ROWS / 2;
            f32x4_t ga = sum4(sg + oa), gb = sum4(sg + ob);
            f32x4_t ua = sum4(su + oa), ub = sum4(su + ob);
            if (folded_in) {
                const float inv = s_tok[t];
                ga *= inv; gb *= inv; ua *= inv; ub *= inv;
            }
            float4 a, b;
            float *pa = &a.x, *pb = &b.x;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                pa[j] = (ga[j] / (1.0f + exp_f64_as_f32(-ga[j]))) * ua[j];
                pb[j] = (gb[j] / (1.0f + exp_f64_as_f32(-gb[j]))) * ub[j];
            }
            float v[8];
            slots_from(P.out_q4, a, b, v);
            if (n < P.n_tokens && hblk * 32 < P.rows) store_frag(P.xf_out, P.nt16, n, hblk, w, v, EXACT ? FRAG_EXACT : 0);
        }
        return;
    }
    if constexpr (EPI == QG_EPI_ROPE) {
        // RoPE (go/model.go:449-477), attention biases (:525-527), KV store (:552-554): rows 0-7 of a tile hold elements i, rows 8-15
        // elements i + hd / 2 of one head (ROWMAP_HEADPERM)
        const QGemmParams::Rope &R = P.rope;
        const int hd = R.head_dim, half = hd >> 1, tph = hd / 16, nq = R.n_q_heads * hd;
#pragma unroll 2
        for (int it0 = 0; it0 < TOK * RT * 2; it0 += NTHR) {
            const int it = it0 + et, u = it % (RT * 2), t = it / (RT * 2), rt = u >> 1, grp = u & 1, n = tok0 + t, nn = min(n, P.n_tokens - 1);
            if (NTHR > TOK * RT * 2 && t >= TOK) break;
            const int tile = min(tile0 + rt, P.ntiles - 1), head = tile / tph, i0 = (tile % tph) * 8 + 4 * grp;
            const bool is_q = head < R.n_q_heads, is_k = !is_q && head < R.n_q_heads + R.n_kv_heads;
            const int kvh = head - R.n_q_heads - (is_k ? 0 : R.n_kv_heads);
            const long long at = R.tkv[nn];       // stream and position, resolved once per token by the embedding launch
            f32x4_t x0 = sum4(t * LD + rt * 16 + 4 * grp), x1 = sum4(t * LD + rt * 16 + 8 + 4 * grp);
            if (folded_in) {
                const float inv = s_tok[t];
                x0 *= inv; x1 *= inv;
            }
            if (R.bias_q) {
                const float *bp = (is_q ? R.bias_q + head * hd : is_k ? R.bias_k + kvh * hd : R.bias_v + kvh * hd) + i0;
                x0 += *reinterpret_cast<const f32x4_t *>(bp);
                x1 += *reinterpret_cast<const f32x4_t *>(bp + half);
            }
            f32x4_t o0 = x0, o1 = x1;
            if (is_q || is_k) {
                const f32x4_t c = *reinterpret_cast<const f32x4_t *>(R.tcos + (long long)nn * half + i0), s = *reinterpret_cast<const f32x4_t *>(R.tsin + (long long)nn * half + i0);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float a0 = x0[j] * c[j], b0 = x1[j] * s[j], a1 = x0[j] * s[j], b1 = x1[j] * c[j];
                    o0[j] = R.conj ? a0 + b0 : a0 - b0;
                    o1[j] = R.conj ? b1 - a1 : a1 + b1;
                }
            }
            if (n >= P.n_tokens || tile0 + rt >= P.ntiles) continue;
            float *dst = is_q ? R.q + ((long long)n * nq + head * hd + i0)
                              : (is_k ? R.kcache : R.vcache) + (at + (long long)kvh * R.seq_len * hd + i0);
            *reinterpret_cast<f32x4_t *>(dst) = o0;
            *reinterpret_cast<f32x4_t *>(dst + half) = o1;
            if (R.kv16 && is_k) {
                // ... and as the attention's image: elements i0 .. + 3 and the same of the other half, hi and lo (position = token)
                typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
                typedef Kv16Image<64> Img;
                _Float16 *const K = reinterpret_cast<_Float16 *>(R.kv16 + ((long long)kvh * R.kv16_chunks + n / ATT_CH) * (Img::BYTES / 16));
                half4_t h0, l0, h1, l1;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    _Float16 a, b;
                    split_hi_lo(o0[j], a, b);
                    h0[j] = a; l0[j] = b;
                    split_hi_lo(o1[j], a, b);
                    h1[j] = a; l1[j] = b;
                }
                const int k0 = Img::k_off(n % ATT_CH, i0 >> 3) + (i0 & 4), k1 = Img::k_off(n % ATT_CH, (i0 >> 3) + 4) + (i0 & 4);
                *reinterpret_cast<half4_t *>(K + k0) = h0;
                *reinterpret_cast<half4_t *>(K + ATT_CH * Img::KS + k0) = l0;
                *reinterpret_cast<half4_t *>(K + k1) = h1;
                *reinterpret_cast<half4_t *>(K + ATT_CH * Img::KS + k1) = l1;
            }
        }
        if (R.kv16) {
            // V^T: eight keys of one element per item, one 16-byte segment of hi and of lo; keys past the prompt up to the chunk's end are zeros (their
            // probabilities are, too, and must meet finite values).  A head is four tiles.
            typedef Kv16Image<64> Img;
            const bool last = tok0 + TOK >= P.n_tokens;
            const int keys = last ? (tok0 + TOK + ATT_CH - 1) / ATT_CH * ATT_CH - tok0 : TOK;      // (a last 64-token tile may be half of its chunk)
#pragma unroll
            for (int hh = 0; hh < RT / 4; hh++) {
                const int kvh = (tile0 >> 2) + hh - R.n_q_heads - R.n_kv_heads;
                if (kvh < 0 || tile0 + 4 * hh >= P.ntiles) continue;
                for (int it = et; it < 8 * keys; it += NTHR) {
                    constexpr int SG = TOK % 64 ? 4 : 8;                // segments of an element: a tile's keys, or 64
                    const int sg = it % SG, d = (it / SG) & 63, t0 = it / (SG * 64) * (SG * 8) + (sg >> 2) * 32 + (sg & 3) * 4, n0 = tok0 + t0;
                    const int col = hh * 64 + ((d & 31) >> 3) * 16 + (d & 7) + 8 * (d >> 5);
                    const float bias = R.bias_v ? R.bias_v[kvh * 64 + d] : 0.f;
                    half8_t hi = {}, lo = {};
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const int t = t0 + (e >> 2) * 16 + (e & 3);
                        if (tok0 + t < P.n_tokens) {
                            float v = S0[t * LD + col];
#pragma unroll
                            for (int k = 1; k < KW; k++) v += S0[k * (SET / 4) + t * LD + col];
                            if (folded_in) v *= s_tok[t];
                            if (R.bias_v) v += bias;
                            _Float16 a, b;
                            split_hi_lo(v, a, b);
                            hi[e] = a; lo[e] = b;
                        }
                    }
                    _Float16 *const V = reinterpret_cast<_Float16 *>(R.kv16 + ((long long)kvh * R.kv16_chunks + n0 / ATT_CH) * (Img::BYTES / 16)) + Img::K_HALVES;
                    const int vo = Img::v_off(d, (n0 % ATT_CH) / 32 * 4 + (sg & 3));
                    *reinterpret_cast<half8_t *>(V + vo) = hi;
                    *reinterpret_cast<half8_t *>(V + 64 * Img::VS + vo) = lo;
                }
            }
        }
        return;
    }
    if constexpr (EPI == QG_EPI_PLAIN) {
        const float *const bias = P.bias;
        const bool fold = P.nrm_out.w != nullptr;
        constexpr int UN = NIT < 8 ? NIT : 8;
#pragma unroll 1
        for (int i0 = 0; i0 < NIT; i0 += UN) {
            f32x4_t v[UN], r[UN];
#pragma unroll
            for (int i = 0; i < UN; i++) r[i] = NRES == NIT ? res[i < NRES ? i : 0] : load_res(i0 + i);     // (a round's rows are requested together)
#pragma unroll
            for (int i = 0; i < UN; i++) {
                const int it = (i0 + i) * NTHR + et, a = it % RQ, t = it / RQ, n = tok0 + t, row = row0 + 4 * a;
                if (NTHR > TOK * RQ && t >= TOK) continue;
                v[i] = sum4(t * LD + 4 * a);
                const size_t off = (size_t)n * P.ldo + row;
                if (vec && row + 3 < P.rows) {
                    if (bias) v[i] += *reinterpret_cast<const f32x4_t *>(bias + row);
                    if (resid) v[i] += r[i];
                    if (n < P.n_tokens) *reinterpret_cast<f32x4_t *>(P.out + off) = v[i];
                } else if (n < P.n_tokens) {
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        if (row + j >= P.rows) continue;
                        float y = v[i][j] + (bias ? bias[row + j] : 0.f);
                        if (resid) y += resid[off + j];
                        P.out[off + j] = y;
                    }
                }
                if (fold) {
                    // folded RMSNorm, producer side (QGemmParams::NormOut): sum of squares of 64 rows (RT = 1: 16) of the new residual stream, in
                    // float64 and a fixed order; the values stay in LDS for the fragments below
                    constexpr int SL = RT == 1 ? 4 : 16;
                    *reinterpret_cast<f32x4_t *>(SW + t * LD + 4 * a) = v[i];
                    double ss = 0.0;
#pragma unroll
                    for (int j = 0; j < 4; j++) ss = fma((double)v[i][j], (double)v[i][j], ss);
#pragma unroll
                    for (int m = 1; m < SL; m *= 2) ss += __shfl_xor(ss, m);
                    if ((a & (SL - 1)) == 0 && n < P.n_tokens && row < P.rows) P.nrm_out.ssq[(size_t)n * (P.rows / (4 * SL)) + row / (4 * SL)] = ss;
                }
            }
        }
        if (!fold) return;
        __syncthreads();
#pragma unroll 2
        for (int it0 = 0; it0 < TOK * ROWS / 8; it0 += NTHR) {
            const int it = it0 + et, w = RT == 1 ? (rbk & 1) * 2 + (lq & 1) : lane >> 4, tt = RT == 1 ? it >> 5 : (it >> 6) % TTW, kb = RT == 1 ? 0 : (it >> 6) / TTW, t = tt * 16 + li, n = tok0 + t, c0 = row0 + kb * 32;
            if (NTHR > TOK * ROWS / 8 && (RT == 1 ? tt >= TTW : kb >= ROWS / 32)) break;
            if (n >= P.n_tokens || c0 >= P.rows) continue;
            int oa, ob;
            slot_offsets(RT == 1 ? 0 : P.out_q4, RT == 1 ? lq & 1 : w, oa, ob);
            const float psc = s_tok[t], *sp = S0 + t * LD + kb * 32, *gp = s_gain + kb * 32;
            const f32x4_t ya = (*reinterpret_cast<const f32x4_t *>(sp + oa) * *reinterpret_cast<const f32x4_t *>(gp + oa)) * psc;
            const f32x4_t yb = (*reinterpret_cast<const f32x4_t *>(sp + ob) * *reinterpret_cast<const f32x4_t *>(gp + ob)) * psc;
            float v[8];
            slots_from(P.out_q4, make_float4(ya[0], ya[1], ya[2], ya[3]), make_float4(yb[0], yb[1], yb[2], yb[3]), v);
            store_frag(P.nrm_out.xf, P.nt16, n, c0 / 32, w, v, EXACT ? FRAG_EXACT : 0);
        }
    }
}

template <int WT, int EPI, int PREC>
hipError_t pg_launch_as(const QGemmParams &P, hipStream_t st) {
    using std::integral_constant;
    auto go = [&](auto rt, auto ntw, auto kw, auto wr) {
        constexpr int RT = decltype(rt)::value, NTW = decltype(ntw)::value, KW = decltype(kw)::value, WR = decltype(wr)::value, TPW = EPI == QG_EPI_SWIGLU ? RT / 2 : RT, TOK = 64 * NTW / WR;
        const int total = ((P.ntiles + TPW - 1) / TPW) * ((P.n_tokens + TOK - 1) / TOK);
        hipLaunchKernelGGL((pgemm_kernel<WT, RT, NTW, KW + 16 * (WR - 1), EPI, PREC>), dim3((total + 7) / 8 * 8), dim3(256 * KW), 0, st, P);
        return hipGetLastError();
    };
    const integral_constant<int, 1> one{};
    const integral_constant<int, 2> two{};
    if constexpr (PREC == PG_EXACT && WT == WT_Q6_K)
        if (P.slim) {
            // (a row tile and all tokens a workgroup: a block's expansion is a quarter a wavefront, and four times as many units work.  us a launch, Q6_K, 17 tokens:
            //  the mean of 768 x 768 and x 2048 12.5 and 10.2, gate and up 11.6 and 9.7, in halves of the tokens while those find a unit each -- 1536 columns, 33 tokens,
            //  512 halves 25.7; prompts of 173M, 17 tokens 1035 and 897, of 841M, 17 and 33 tokens 2140 and 1919, 2197 and 2025.  Q4_K, whose expansion is two thirds of
            //  that: 173M 940 and 920, 841M 1880 and 1950: not there)
            if constexpr (EPI == QG_EPI_SWIGLU) return P.ntiles * ((P.n_tokens + 31) / 32) <= 256 ? go(two, one, two, two) : go(two, one, two, one);
            else return go(one, one, two, one);
        }
    const integral_constant<int, 4> four{};
    const integral_constant<int, 8> eight{};
    // Tiles by how many 64 x 64 ones there are.  Up to one per compute unit: eight wavefronts on each (K dealt to two sets), since the four
    // of one set leave every SIMD waiting on its own wavefront's instructions (Q4_0 768 x 2048 x 333 tokens, 72 tiles: 14.8 us one set,
    // 11.6 two; 64 x 128 tiles 20.3).  Up to two: 64 x 128 tiles of two sets (768 x 2048 x 2047: 17.7 us against 20.9 for 64 x 64, 22.0
    // for it with two sets).  Beyond, one set, and tiles that grow as the grid allows it (Q4_0 4096 x 768 x 2047, gate and up: 128 x 128
    // 31.8 us, 64 x 128 35.0, 64 x 64 37.0; Q8_0's expansion leaves no registers for 128 x 128: 68.9 us against 62.2).
    const long long tiles = (long long)((P.ntiles * (EPI == QG_EPI_SWIGLU ? 2 : 1) + 3) / 4) * ((P.n_tokens + 63) / 64);
    // Half or a quarter of a unit's tokens where that many workgroups still find a unit each: the wavefronts share the tokens and split the rows, a row
    // tile's scalings and products are half or a quarter a wavefront, the expansion of the weights is done two or four times over the chip.  The order of the
    // sums stays.  us a launch, 64 x 64 / x 32 / x 16: Q4_K 768 x 768 and x 2048, 333 tokens 11.3 / 8.9 / 8.3 and 22.0 / 16.7 / 15.1; 1152 x 768 11.6 / 9.3 / 14.3
    // (378 workgroups); Q6_K 12.5 / 9.6 and 24.7 / 18.4; Q4_0 7.2 / 5.9 / 5.6 and 12.0 / 9.7 / 9.3, 1536 x 4096 at 150 19.8 / 15.1 / 14.3, at 500 21.8 / 26.5 (384);
    // Q8_0 7.3 / 6.2 / 6.0 and 12.3 / 10.0 / 9.6; F16 6.6 / 6.0 / 5.9 and 10.7 / 9.6 / 9.6: no quarters.  (none either where V^T's image
    // is written: its segments hold keys of two 16-token tiles)
    const long long rb = (P.ntiles * (EPI == QG_EPI_SWIGLU ? 2 : 1) + 3) / 4;
    if constexpr (WT != WT_F16)
        if (rb * ((P.n_tokens + 15) / 16) <= 256 && !(EPI == QG_EPI_ROPE && P.rope.kv16)) return go(four, one, two, four);
    if (rb * ((P.n_tokens + 31) / 32) <= 256) return go(four, one, two, two);
    if (tiles <= 256) return go(four, one, two, one);
    // (three parts, the sums of a chunk pair and what their additions drop leave no registers for a second token tile: 46 to 150 spilled)
    if constexpr (PREC == PG_EXACT) {
        // (one token, the LM head of a prompt: 16 of them are multiplied, not 64.  Q6_K, us, 48000 x 1536 57.8 and 34.9, 32000 x 768 22.4 and
        //  12.8)
        if constexpr (EPI == QG_EPI_PLAIN)
            if (P.n_tokens <= 16) return go(four, one, one, four);
        return go(four, one, one, one);
    } else {
        if (tiles <= 512) return go(four, two, two, one);
        if (tiles < 1024 && !(WT == WT_F16 && EPI == QG_EPI_SWIGLU)) return go(four, one, one, one);
        if constexpr (WT == WT_Q4_0 || WT == WT_F16)
            if (tiles >= 1792) return go(eight, two, one, one);
        return go(four, two, one, one);
    }
}
template <int EPI>
hipError_t pg_launch(int wtype, const QGemmParams &P, hipStream_t st) {
    if (P.exact) {
        switch (wtype) {
        case WT_Q4_0: return pg_launch_as<WT_Q4_0, EPI, PG_EXACT>(P, st);
        case WT_Q8_0: return pg_launch_as<WT_Q8_0, EPI, PG_EXACT>(P, st);
        case WT_Q4_K: return pg_launch_as<WT_Q4_K, EPI, PG_EXACT>(P, st);
        case WT_Q6_K: return pg_launch_as<WT_Q6_K, EPI, PG_EXACT>(P, st);
        default: return hipErrorInvalidValue;
        }
    }
    switch (wtype) {
    case WT_Q4_0: return P.x1 ? pg_launch_as<WT_Q4_0, EPI, PG_HI>(P, st) : pg_launch_as<WT_Q4_0, EPI, PG_HILO>(P, st);
    case WT_Q8_0: return pg_launch_as<WT_Q8_0, EPI, PG_HILO>(P, st);
    case WT_F16: return pg_launch_as<WT_F16, EPI, PG_HILO>(P, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace nl
