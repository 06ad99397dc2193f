// nl_sgemm.h -- the GEMMs of a short multi-token step (decode batches, prompts and messages of a line) for every format and width that
// nl_dgemm.h does not take: Q8_0 and F16 files, Q4_0 ones whose widths are no whole 256-column groups.
//
// What bounds such a step is the number of its launches: 24 tokens against 89M Q8_0 parameters move 75 MB and were 10 launches a layer of 3 - 8 us
// (norm, Q|K|V in split-K slabs, slab sum + rotation, attention, merge, WO in slabs, slab sum + norm, gate || up in slabs, slab sum + SiLU,
// down in slabs).  Here the K splits of a tile are wavefronts of ONE workgroup, so their partial tiles meet in LDS and the rotation, SiLU and
// residual epilogues follow in the same launch; the norm is the prologue of the launch that consumes it: 5 launches a layer, 6 where the
// attention leaves partials (positions of 128 on).  Measured, profiled, us a launch -- a norm, a GEMM in slabs and what sums them; this kernel --, 89M
// Q8_0, 24 tokens: Q|K|V 3.5 + 4.7 + 4.6, 5.5; gate || up 3.5 + 4.8 + 4.0, 5.8; WO and down (mean) 4.6, 4.4.  A prompt of 24 / 64 tokens
// (its attention in one launch a layer as well, nl_batch.h) 703 -> 394 / 774 -> 434 us, 173M Q8_0 1092 -> 641 / 1227 -> 711, 841M 1766 -> 1255 / 2026 -> 1552,
// F16 1831 -> 1394 / 2074 -> 1742; a step of 64 streams at position 150: 89M 785 -> 604, 173M 1105 -> 823, 841M Q8_0 1923 -> 1750, F16 1968 -> 1934.
// What bounds a launch now is one workgroup's chain: requests, the norm (almost half of two launches), products at the vector pipe's rate
// (10 instructions an expansion, 4 a scaling), the meeting of the partial tiles.
//
// A workgroup owns 16 tokens x TW (x 2: gate and up) 16-row weight tiles; its KS x TW wavefronts are (split z, tile).  Split z multiplies the
// 128-column chunks z, z + KS, ... in order, exactly those that a split of qgemm_kernel takes (KS is qgemm_kernel's rule too), and the
// partial tiles are added in split order as the slabs' consumers add them, so the products are qgemm_kernel's bits.  The norm's factor is
// bnorm_kernel's to a few float64 ulps (its sum in another order, a reciprocal and Newton steps instead of a division and a square root), and
// the same float32 unless it lies that close to a rounding boundary, about one row in 10^8: none was seen.
//   * The weights of the first chunks (all of them where registers allow) are requested in the prologue, in front of the norm's round trip.
//   * NORM: the token tile's rows go to LDS once per workgroup as the fragments of all its wavefronts (up to 2112 columns fit), through the
//     same rounding as bnorm_kernel: 1 / rms is known before anything is rounded, so no range is lost.
//   * otherwise the fragments are read straight into registers, a chunk ring of DEP deep.
//   * Barriers order LDS only (pg_barrier): the weights in flight stay in flight.
#pragma once
#include "nl_dgemm.h"

namespace nl {

struct SGemmParams {
    const uint8_t *q, *q1;       // q1: up, where q is gate
    const uint32_t *s, *s1;
    const float *x, *normw;      // NORM: rows [N][cols] and the norm's gains
    const uint4 *xf;             // otherwise: fragments
    float *out;                  // PLAIN: out[n][row] += bias[row] + y
    const float *bias;
    uint4 *xf_out;               // SWIGLU: the next GEMM's fragments
    int rows, cols, npairs, ntiles, nt16, n_tokens;
    int ks, tw;                  // K splits, row tiles of a workgroup
    int out_form;                // k-slot order of xf_out
    float eps;
    double rcols;                // 1 / cols
    QGemmParams::Rope rope;
};

constexpr size_t SG_LDS_MAX = 160 * 1024;
inline size_t sg_lds_bytes(bool norm, int cols, int waves, int tpl) {
    return (norm ? (size_t)(cols / 32) * 2048 + (size_t)cols * 4 + (size_t)waves * 128 : 0) + (size_t)waves * tpl * 1024;
}

// A chunk (two pairs of blocks) of one 16-row tile, as raw buffer loads (pg_load16; skipping the vector L1, as nl_dgemm.h does, loses here: a token
// tile's rows and a row's second half of a sector are hits.  gate || up of 1536 x 4096 F16, 64 tokens: 18.2 us a launch through it, 22.8 past it),
// 16 bytes a lane and load: lane (row li, group lq) takes pair lq & 1, so that a row's two pairs
// (32 bytes) travel in one request, and the operand order -- each of the four groups an eighth of a block -- is made by swapping 16- and
// 32-lane rows between registers.  (Asked for in operand order, four or eight bytes a lane, every request moved a whole sector for a
// quarter of it or less: gate || up of 1536 x 4096, Q8_0, 33 tokens, 22.8 us a launch against 19.8.)
__device__ __forceinline__ void sg_swap16(uint32_t &a, uint32_t &b) {       // odd 16-lane rows of a <-> even ones of b
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0]; b = r[1];
}
__device__ __forceinline__ void sg_swap32(uint32_t &a, uint32_t &b) {       // upper half of a <-> lower half of b
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0]; b = r[1];
}
// NL loads a chunk; load i's bytes inside a group of gsz pairs, from the chunk's first pair on: lane() + uni(); block b = pair b >> 1, parity b & 1
template <int WT> struct SgW;
template <> struct SgW<WT_Q8_0> {
    static constexpr int NL = 2;
    static __device__ __forceinline__ unsigned lane(int li, int lq, int gsz, int second) { return (unsigned)(((lq >> 1) * TR + li) * gsz + (lq & second)) * 16u; }
    static __device__ __forceinline__ unsigned uni(int i, int gsz, int) { return (unsigned)(2 * i * TR * gsz) * 16u; }
    static __device__ __forceinline__ void order(uint4 (&v)[NL]) {
#pragma unroll
        for (int i = 0; i < NL; i++) { sg_swap16(v[i].x, v[i].z); sg_swap16(v[i].y, v[i].w); }
    }
    static __device__ __forceinline__ half8_t get(const uint4 (&v)[NL], int b) {
        const uint32_t u0 = (b >> 1 ? v[b & 1].z : v[b & 1].x) ^ 0x80808080u, u1 = (b >> 1 ? v[b & 1].w : v[b & 1].y) ^ 0x80808080u;      // 1024 + 128 + q, exact
        const h2_t o = pg_h2(1152.f);
        return pg_join(pg_bytes_lo(u0) - o, pg_bytes_hi(u0) - o, pg_bytes_lo(u1) - o, pg_bytes_hi(u1) - o);
    }
};
template <> struct SgW<WT_Q4_0> {
    static constexpr int NL = 1;
    static __device__ __forceinline__ unsigned lane(int li, int lq, int gsz, int second) { return (unsigned)(((lq >> 1) * TR + li) * gsz + (lq & second)) * 16u; }
    static __device__ __forceinline__ unsigned uni(int, int, int) { return 0u; }
    static __device__ __forceinline__ void order(uint4 (&v)[NL]) {          // (a 4 x 4 transpose)
        sg_swap16(v[0].x, v[0].y); sg_swap16(v[0].z, v[0].w);
        sg_swap32(v[0].x, v[0].z); sg_swap32(v[0].y, v[0].w);
    }
    static __device__ __forceinline__ half8_t get(const uint4 (&v)[NL], int b) { return WFrag<WT_Q4_0>::expand(b & 1 ? (b >> 1 ? v[0].w : v[0].z) : (b >> 1 ? v[0].y : v[0].x)); }
};
template <> struct SgW<WT_F16> {       // (eight values of a block are 16 bytes: already in order)
    static constexpr int NL = 4;
    static __device__ __forceinline__ unsigned lane(int li, int lq, int gsz, int) { return (unsigned)((lq * TR + li) * gsz) * 16u; }
    static __device__ __forceinline__ unsigned uni(int i, int gsz, int second) { return (unsigned)(4 * (i & 1) * TR * gsz + ((i >> 1) & second)) * 16u; }
    static __device__ __forceinline__ void order(uint4 (&)[NL]) {}
    static __device__ __forceinline__ half8_t get(const uint4 (&v)[NL], int b) { return __builtin_bit_cast(half8_t, v[b]); }
};

template <int WT, int EPI, int CPS, int NWV, int TPL>      // CPS: chunks a split walks at most; NWV: most wavefronts; TPL: row tiles of a wavefront (without NORM all of its workgroup's)
__global__ void __launch_bounds__(NWV * 64, NWV / 4) sgemm_kernel(SGemmParams P) {
    constexpr bool NORM = EPI != QG_EPI_PLAIN, FUSED = EPI == QG_EPI_SWIGLU;
    constexpr int MT = FUSED ? 2 : 1, FORM = WT == WT_Q4_0 ? FRAG_Q4_0 : 0;
    constexpr int NL = SgW<WT>::NL;
    // chunks in flight: registers of a chunk's weights and, without NORM, of its fragments
    constexpr int CHUNK_REGS = TPL * (NL * 4 + 1) + (NORM ? 0 : QG_KC * 8);
    constexpr int ROOM = NORM ? 64 : TPL == 1 ? 84 : 160, DEP = CPS * CHUNK_REGS <= ROOM ? CPS : ROOM / CHUNK_REGS;
    static_assert(DEP >= 1, "a chunk fits");
    static_assert(!NORM || TPL == 1, "a wavefront per tile and matrix");
    extern __shared__ __attribute__((aligned(16))) uint8_t sg_lds[];
    NL_KARGS8(P.q, P.s, P.x, P.normw, P.xf, P.out, P.bias, P.xf_out);
    NL_KARGS8(P.rows, P.cols, P.npairs, P.ntiles, P.nt16, P.n_tokens, P.ks, P.tw);
    if constexpr (NORM) NL_KARGS2(P.eps, P.rcols);
    if constexpr (FUSED) NL_KARGS4(P.q1, P.s1, P.out_form, P.eps);
    if constexpr (EPI == QG_EPI_ROPE) {
        NL_KARGS8(P.rope.tcos, P.rope.tsin, P.rope.tkv, P.rope.q, P.rope.kcache, P.rope.vcache, P.rope.bias_q, P.rope.bias_k);
        NL_KARGS8(P.rope.bias_v, P.rope.head_dim, P.rope.n_q_heads, P.rope.n_kv_heads, P.rope.seq_len, P.rope.conj, P.eps, P.s);
    }
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, nw = NORM ? NWV : (int)blockDim.x >> 6;      // (NORM: always that many)
    const int li = lane & 15, lq = lane >> 4;
    // wavefront: split, then (tile, matrix)
    const int ksl = 31 - __builtin_clz(P.ks), z = wv & (P.ks - 1), tw = (wv >> ksl) / MT, mat = MT == 1 ? 0 : (wv >> ksl) & 1;
    // the token tiles of a row group on one XCD, next to each other (dg_grid)
    const int rg = ((int)blockIdx.x & 7) + 8 * (int)blockIdx.y, tt = (int)blockIdx.x >> 3;
    if (rg * P.tw >= P.ntiles) return;                           // (padding of the row groups to a multiple of 8: the whole workgroup)
    const int tile0 = rg * P.tw + tw;                            // this wavefront's first (without NORM tw = 0)
    const int nblocks = P.cols >> 5, nchunks = (nblocks + QG_KC - 1) / QG_KC;
    uint4 *const xs = reinterpret_cast<uint4 *>(sg_lds);                                                        // NORM: [block][hi, lo][lane]
    float *const ws = reinterpret_cast<float *>(sg_lds + (NORM ? (size_t)nblocks * 2048 : 0));                  // NORM: gains
    double *const red = reinterpret_cast<double *>(sg_lds + (NORM ? (size_t)nblocks * 2048 + (size_t)P.cols * 4 : 0));
    float *const part = reinterpret_cast<float *>(sg_lds + (NORM ? (size_t)nblocks * 2048 + (size_t)P.cols * 4 + (size_t)nw * 128 : 0));    // [wavefront][token][row]

    // ---- requests, oldest first: the rows (NORM), then the weights ----
    [[maybe_unused]] const __amdgpu_buffer_rsrc_t rx = pg_rsrc(NORM ? (const void *)P.x : (const void *)P.xf);
    // (NORM: four lanes take 64 bytes of a row's 128-byte block, lane >> 2 is the row)
    const int xr = lane >> 2, xq = lane & 3;
    [[maybe_unused]] const unsigned xrow = (unsigned)min(tt * 16 + xr, P.n_tokens - 1) * (unsigned)P.cols * 4u + (unsigned)xq * 16u;
    constexpr int XB = 4;                                        // blocks a wavefront has in flight
    [[maybe_unused]] uint4 xa[XB], xb[XB], wn;
    [[maybe_unused]] const int nxb = (nblocks - wv + nw - 1) / nw;   // this wavefront's blocks wv, wv + nw, ... (may be 0)
    auto xload = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < XB; i++) {
            const unsigned o = (unsigned)min(wv + (i0 + i) * nw, nblocks - 1) * 128u;
            xa[i] = pg_load16(rx, xrow, o);
            xb[i] = pg_load16(rx, xrow, o + 64u);
        }
    };
    if constexpr (NORM) {
        xload(0);
        wn = *reinterpret_cast<const uint4 *>(P.normw + min(tid * 4, P.cols - 4));
        __builtin_amdgcn_s_barrier();        // no weight is asked for before all rows are: the norm waits for the slowest wavefront's (1536 columns: 2.5 us without)
    }
    asm volatile("" ::: "memory");
    const bool mul = !NORM || tw < P.tw;              // (NORM: the others bring rows and share the epilogue)
    uint4 wq[DEP][TPL][NL];
    [[maybe_unused]] uint32_t wd[DEP][TPL];                           // pair lq & 1's two scales
    [[maybe_unused]] uint4 xh[DEP][QG_KC], xl[DEP][QG_KC];
    [[maybe_unused]] const unsigned xblock = (unsigned)P.nt16 * (2 * QG_FRAG * 16), xtile = (unsigned)tt * (2 * QG_FRAG * 16);
    const __amdgpu_buffer_rsrc_t rw = pg_rsrc(FUSED && mat ? P.q1 : P.q), rs = pg_rsrc(FUSED && mat ? P.s1 : P.s);
    auto request = [&](int d, int c) __attribute__((always_inline)) {                           // chunk c of this split into ring place d (clamped past the last one, never used there)
        const int b0 = min(z + c * P.ks, nchunks - 1) * QG_KC, g = b0 >> 3, k0 = (b0 >> 1) & 3;
        const int gsz = min(KL, P.npairs - g * KL), second = k0 + 1 < gsz ? 1 : 0;
        if constexpr (!NORM) {
#pragma unroll
            for (int b = 0; b < QG_KC; b++) {
                const unsigned o = xtile + (unsigned)min(b0 + b, nblocks - 1) * xblock;
                xl[d][b] = pg_load16(rx, lane * 16u, o + QG_FRAG * 16);
                xh[d][b] = pg_load16(rx, lane * 16u, o);
            }
        }
        const unsigned lw = SgW<WT>::lane(li, lq, gsz, second), ls = (unsigned)(li * gsz + (lq & second)) * 4u;
#pragma unroll
        for (int t = 0; t < TPL; t++) {
            const unsigned gp = (unsigned)(min(tile0 + t, P.ntiles - 1) * P.npairs + g * KL);
            const unsigned gq = gp * (WFrag<WT>::CPP * TR * 16) + (unsigned)k0 * 16u;
#pragma unroll
            for (int i = 0; i < NL; i++) wq[d][t][i] = pg_load16(rw, lw, gq + SgW<WT>::uni(i, gsz, second));
            if constexpr (WTraits<WT>::SCALED) wd[d][t] = __builtin_amdgcn_raw_buffer_load_b32(rs, ls, gp * (TR * 4) + (unsigned)k0 * 4u, 0);
        }
    };
    // what the first round of the epilogue reads: unit u = wavefront, wavefront + all, ...: tile u >> 2 of the workgroup, its row li, token 4 (u & 3) + lq
    const int r = li, et0 = min(rg * P.tw + (wv >> 2), P.ntiles - 1), row0 = min(et0 * TR + r, P.rows - 1), nn0 = min(tt * 16 + (wv & 3) * 4 + lq, P.n_tokens - 1);
    [[maybe_unused]] float pre0 = 0.f, pre1 = 0.f;
    [[maybe_unused]] long long kvoff = 0;
    [[maybe_unused]] const int hd = P.rope.head_dim, half = hd >> 1, tsh = hd == 64 ? 2 : 1, ri0 = (et0 & ((1 << tsh) - 1)) * 8 + (r & 7);
    if constexpr (EPI == QG_EPI_ROPE) {
        pre0 = P.rope.tcos[(size_t)nn0 * half + ri0];
        pre1 = P.rope.tsin[(size_t)nn0 * half + ri0];
        kvoff = P.rope.tkv[nn0];
    } else if constexpr (EPI == QG_EPI_PLAIN) {
        pre0 = P.out[(size_t)nn0 * P.rows + row0];
        pre1 = P.bias ? P.bias[row0] : 0.f;
    }
    asm volatile("" ::: "memory");
    if (mul) {
#pragma unroll
        for (int c = 0; c < DEP; c++) request(c, c);
    }
    asm volatile("" ::: "memory");

    // ---- RMSNorm (go/quant.go:597-607) of the token tile into LDS: rows as they are, their sums of squares, then in place hi and lo ----
    if constexpr (NORM) {
        double ss = 0.0;
        auto xput = [&](int i0) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < XB; i++)
                if (i0 + i < nxb) {                              // (the same in all lanes)
                    const float4 a = __builtin_bit_cast(float4, xa[i]), b = __builtin_bit_cast(float4, xb[i]);
                    uint4 *const to = xs + (size_t)(wv + (i0 + i) * nw) * (2 * QG_FRAG) + xr * 8;
                    to[xq ^ (xr & 7)] = xa[i];                // (16-byte pieces of a row in an order of its own: no bank conflicts either way)
                    to[(xq + 4) ^ (xr & 7)] = xb[i];
                    double t = 0.0;
                    t = fma((double)a.x, (double)a.x, t); t = fma((double)a.y, (double)a.y, t); t = fma((double)a.z, (double)a.z, t); t = fma((double)a.w, (double)a.w, t);
                    t = fma((double)b.x, (double)b.x, t); t = fma((double)b.y, (double)b.y, t); t = fma((double)b.z, (double)b.z, t); t = fma((double)b.w, (double)b.w, t);
                    ss += t;
                }
        };
        xput(0);
        if (tid * 4 < P.cols) *reinterpret_cast<uint4 *>(ws + tid * 4) = wn;
        for (int i = (tid + nw * 64) * 4; i < P.cols; i += nw * 256) *reinterpret_cast<float4 *>(ws + i) = *reinterpret_cast<const float4 *>(P.normw + i);
        for (int i0 = XB; i0 < nxb; i0 += XB) { xload(i0); xput(i0); }     // (blocks past XB per wavefront: beyond 1024 columns of eight, 2048 of
                                                                             //  sixteen.  They are asked for behind the weights)
        ss += dpp_f64<DPP_QUAD_XOR1>(ss);
        ss += dpp_f64<DPP_QUAD_XOR2>(ss);
        if (xq == 0) red[wv * 16 + xr] = ss;
        pg_barrier();
        int offa, offb;
        slot_offsets(FORM, lq, offa, offb);
        double tot = 0.0, sq[NWV];
#pragma unroll
        for (int k = 0; k < NWV; k++) sq[k] = red[k * 16 + li];      // (in flight together)
#pragma unroll
        for (int k = 0; k < NWV; k++) tot += sq[k];
        const float inv = dg_inv_rms(tot, P.rcols, P.eps);       // (the division is the host's)
        for (int i = 0; i < nxb; i++) {
            const int blk = wv + i * nw;
            uint4 *const at = xs + (size_t)blk * (2 * QG_FRAG);
            const int pa = (FORM ? lq : 2 * lq) ^ (li & 7), pb = (FORM ? lq + 4 : 2 * lq + 1) ^ (li & 7);       // (slot_offsets, in pieces)
            float xv[8], gv[8];
            slots_from(FORM, __builtin_bit_cast(float4, at[li * 8 + pa]), __builtin_bit_cast(float4, at[li * 8 + pb]), xv);
            slots_from(FORM, *reinterpret_cast<const float4 *>(ws + blk * 32 + offa), *reinterpret_cast<const float4 *>(ws + blk * 32 + offb), gv);
            half8_t hi, lo;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                _Float16 h, l;
                split_hi_lo((xv[j] * inv) * gv[j], h, l);
                hi[j] = h; lo[j] = l;
            }
            at[lane] = __builtin_bit_cast(uint4, hi);             // (the block is this wavefront's alone, read before it is written: LDS keeps a wavefront's order)
            at[QG_FRAG + lane] = __builtin_bit_cast(uint4, lo);
        }
        pg_barrier();
    }

    // ---- the chunks of this split, in order: qgemm_kernel's arithmetic ----
    f32x4_t acc[TPL];
#pragma unroll
    for (int t = 0; t < TPL; t++) acc[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    dg_static_for<0, CPS>([&](auto c_) __attribute__((always_inline)) {
        constexpr int c = decltype(c_)::value, d = c % DEP;
        const int b0 = (z + c * P.ks) * QG_KC;
        if (mul && b0 < nblocks) {                               // (the same in all lanes.  Blocks past the last one of a begun chunk: its weights, scale 0,
            half8_t xhv[QG_KC], xlv[QG_KC];                      //  as in qgemm_kernel: straight-line code, four independent products a tile)
#pragma unroll
            for (int b = 0; b < QG_KC; b++) {
                if constexpr (NORM) {
                    const uint4 *const at = xs + (size_t)min(b0 + b, nblocks - 1) * (2 * QG_FRAG) + lane;
                    xlv[b] = __builtin_bit_cast(half8_t, at[QG_FRAG]);
                    xhv[b] = __builtin_bit_cast(half8_t, at[0]);
                } else {
                    xlv[b] = __builtin_bit_cast(half8_t, xl[d][b]);
                    xhv[b] = __builtin_bit_cast(half8_t, xh[d][b]);
                }
            }
#pragma unroll
            for (int t = 0; t < TPL; t++) {
                half8_t wf[QG_KC];
                SgW<WT>::order(wq[d][t]);
#pragma unroll
                for (int b = 0; b < QG_KC; b++) wf[b] = SgW<WT>::get(wq[d][t], b);
                if constexpr (WTraits<WT>::SCALED) {
                    uint32_t sw[2] = {wd[d][t], wd[d][t]};
                    sg_swap16(sw[0], sw[1]);
                    f32x4_t y[QG_KC];
#pragma unroll
                    for (int b = 0; b < QG_KC; b++) y[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xlv[b], wf[b], (f32x4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                    for (int b = 0; b < QG_KC; b++) y[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xhv[b], wf[b], y[b], 0, 0, 0);
#pragma unroll
                    for (int b = 0; b < QG_KC; b++) {
                        const float dsc = b0 + b < nblocks ? scale_of(sw[b >> 1], b) : 0.f;
#pragma unroll
                        for (int j = 0; j < 4; j++) acc[t][j] = fmaf(y[b][j], dsc, acc[t][j]);
                    }
                } else {
#pragma unroll
                    for (int b = 0; b < QG_KC; b++) {
                        if (b0 + b >= nblocks) wf[b] = __builtin_bit_cast(half8_t, make_uint4(0u, 0u, 0u, 0u));
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xlv[b], wf[b], acc[t], 0, 0, 0);
                        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xhv[b], wf[b], acc[t], 0, 0, 0);
                    }
                }
            }
        }
        if constexpr (c + DEP < CPS) if (mul) request(d, c + DEP);
    });

    // ---- partial tiles [token][row] meet in LDS; all wavefronts share the epilogue ----
    if (mul) {
#pragma unroll
        for (int t = 0; t < TPL; t++) {
            float *const mine = part + (size_t)((t << ksl) + wv) * 256;
#pragma unroll
            for (int j = 0; j < 4; j++) mine[(4 * lq + j) * 16 + li] = acc[t][j];
        }
    }
    pg_barrier();
    for (int u = wv; u < 4 * P.tw; u += nw) {
        const int q = u & 3, tile = rg * P.tw + (u >> 2), tile_c = min(tile, P.ntiles - 1), row = tile * TR + r;
        const float *const from = part + (size_t)(((u >> 2) * MT) << ksl) * 256 + q * 64 + lane;
        float y[MT];
#pragma unroll
        for (int m = 0; m < MT; m++) y[m] = from[(m << ksl) * 256];
        for (int k0 = 1; k0 < P.ks; k0 += 4) {                   // (four reads of a split at a time in flight, added in split order)
            float v[MT][4];
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int m = 0; m < MT; m++) v[m][k] = from[((m << ksl) + min(k0 + k, P.ks - 1)) * 256];
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int m = 0; m < MT; m++) y[m] += k0 + k < P.ks ? v[m][k] : 0.f;
        }
        const int n = tt * 16 + q * 4 + lq, nn = min(n, P.n_tokens - 1);
        const bool live = n < P.n_tokens && tile < P.ntiles && row < P.rows;
        if constexpr (FUSED) {
            // h = SiLU(gate) * up (go/quant.go:629-631, go/model.go:604-606)
            const float ex = exp_f64_as_f32(-y[0]), h = (y[0] / (1.0f + ex)) * y[1];
            const int e = (tile & 1) * 16 + r;                   // of the 32-column block
            const int w = P.out_form & FRAG_Q4_0 ? (e & 15) >> 2 : e >> 3;
            const int j = P.out_form & FRAG_Q4_0 ? (e >> 4) * 4 + ((e & 1) << 1 | ((e >> 1) & 1)) : e & 7;       // (slot_elem's inverse)
            _Float16 hi, lo;
            split_hi_lo(h, hi, lo);
            if (live) {
                _Float16 *const to = reinterpret_cast<_Float16 *>(P.xf_out + ((size_t)(tile >> 1) * P.nt16 + tt) * (2 * QG_FRAG) + w * 16 + (n & 15)) + j;
                to[0] = hi;
                to[QG_FRAG * 8] = lo;
            }
        } else if constexpr (EPI == QG_EPI_ROPE) {
            // RoPE (go/model.go:449-477) + attention biases (:525-527) + KV store (:552-554): rotation partners are rows r and r ^ 8
            const QGemmParams::Rope &R = P.rope;
            const int head = tile_c >> tsh, ri = (tile_c & ((1 << tsh) - 1)) * 8 + (r & 7), e = ri + (r >> 3) * half;
            const bool is_q = head < R.n_q_heads, is_k = !is_q && head < R.n_q_heads + R.n_kv_heads;
            const int kvh = head - R.n_q_heads - (is_k ? 0 : R.n_kv_heads);
            float v = y[0];
            if (R.bias_q) v += is_q ? R.bias_q[head * hd + e] : is_k ? R.bias_k[kvh * hd + e] : R.bias_v[kvh * hd + e];
            const float partner = __shfl_xor(v, 8);
            float c = pre0, s1 = pre1;
            long long ko = kvoff;
            if (u != wv) { c = R.tcos[(size_t)nn * half + ri]; s1 = R.tsin[(size_t)nn * half + ri]; ko = R.tkv[nn]; }
            float o = v;
            if (is_q || is_k) {
                const float x0 = r < 8 ? v : partner, x1 = r < 8 ? partner : v;
                if (!R.conj) o = r < 8 ? (x0 * c - x1 * s1) : (x0 * s1 + x1 * c);
                else o = r < 8 ? (x0 * c + x1 * s1) : (-x0 * s1 + x1 * c);
            }
            if (live) {
                if (is_q) R.q[(size_t)n * (R.n_q_heads * hd) + head * hd + e] = o;
                else (is_k ? R.kcache : R.vcache)[ko + (long long)kvh * R.seq_len * hd + e] = o;
            }
        } else {
            float v = y[0], res = pre0;
            if (u != wv) res = P.out[(size_t)nn * P.rows + min(row, P.rows - 1)];
            if (P.bias) v += u != wv ? P.bias[min(row, P.rows - 1)] : pre1;
            if (live) P.out[(size_t)n * P.rows + row] = v + res;
        }
    }
}

// ---- launches ----
// Which GEMMs: K splits of at most six chunks each, KS x TW wavefronts in a workgroup, the token tile in LDS (NORM)
inline int sg_cps(int cols, int ks) { return ((cols / 32 + QG_KC - 1) / QG_KC + ks - 1) / ks; }
// Row tiles of a workgroup: as few as one round of workgroups takes (16 tokens of gate || up of 1536 x 4096, Q8_0, on 64 compute units 14.4 us, on all 9.7;
// 64 tokens in two rounds 20.0 us, in one with twice the tiles 15.3).  NORM: at least eight wavefronts, since all of them bring and norm the token
// tile's rows, and sixteen only where there are tiles for more than eight (gate || up of 576 x 1536, 24 tokens: 5.5 us with eight, 6.3 with sixteen)
constexpr int SG_WAVES = 16, SG_ROUND = 256;
inline int sg_tw(bool norm, int mats, int ks, int ntiles, int n_tokens) {
    if (!norm) return ks <= 8 && (long long)ntiles * ((n_tokens + 15) / 16) > SG_ROUND ? 2 : 1;      // (two tiles of a wavefront: the fragments are read once for both)
    int tw = 1;
    while ((tw + 1) * mats * ks <= SG_WAVES && (long long)((ntiles + tw - 1) / tw) * ((n_tokens + 15) / 16) > SG_ROUND) tw++;
    return tw;
}
// rounds of workgroups of a launch, one a compute unit (their registers or LDS leave room for no second one where it matters)
inline int sg_rounds(bool norm, int mats, int ks, int ntiles, int n_tokens) {
    const int tw = sg_tw(norm, mats, ks, ntiles, n_tokens);
    return (int)(((long long)((ntiles + tw - 1) / tw) * ((n_tokens + 15) / 16) + SG_ROUND - 1) / SG_ROUND);
}
inline int sg_waves(bool norm, int mats, int ks, int tw) { return !norm ? ks : ks * mats * tw <= 8 ? 8 : SG_WAVES; }
inline bool sg_fits(bool norm, int mats, int cols, int ks) {
    if (cols % 32 || cols < 32 || ks < 1 || ks * mats > (norm ? SG_WAVES : 16) || (ks & (ks - 1)) || sg_cps(cols, ks) > 6) return false;
    return sg_lds_bytes(norm, cols, norm ? SG_WAVES : ks, norm ? 1 : 2) <= SG_LDS_MAX;
}
template <int WT, int EPI, int NWV, int TPL>
inline hipError_t sg_launch_w(const SGemmParams &P, int waves, hipStream_t st) {
    const dim3 grid = dg_grid(P.ntiles, P.tw, P.n_tokens), block((unsigned)(waves * 64));
    const size_t lds = sg_lds_bytes(EPI != QG_EPI_PLAIN, P.cols, waves, TPL);
    switch (sg_cps(P.cols, P.ks)) {
    case 1: hipLaunchKernelGGL((sgemm_kernel<WT, EPI, 1, NWV, TPL>), grid, block, lds, st, P); break;
    case 2: hipLaunchKernelGGL((sgemm_kernel<WT, EPI, 2, NWV, TPL>), grid, block, lds, st, P); break;
    case 3: hipLaunchKernelGGL((sgemm_kernel<WT, EPI, 3, NWV, TPL>), grid, block, lds, st, P); break;
    case 4: hipLaunchKernelGGL((sgemm_kernel<WT, EPI, 4, NWV, TPL>), grid, block, lds, st, P); break;
    case 5: case 6: hipLaunchKernelGGL((sgemm_kernel<WT, EPI, 6, NWV, TPL>), grid, block, lds, st, P); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
template <int WT, int EPI>
inline hipError_t sg_launch_t(const SGemmParams &P, int waves, hipStream_t st) {
    if (waves > 8) return sg_launch_w<WT, EPI, 16, 1>(P, waves, st);
    if constexpr (EPI == QG_EPI_PLAIN)
        if (P.tw == 2) return sg_launch_w<WT, EPI, 8, 2>(P, waves, st);
    return sg_launch_w<WT, EPI, 8, 1>(P, waves, st);
}
template <int EPI>
inline hipError_t sg_launch(int wtype, SGemmParams P, hipStream_t st) {
    constexpr bool NORM = EPI != QG_EPI_PLAIN;
    constexpr int MT = EPI == QG_EPI_SWIGLU ? 2 : 1;
    P.nt16 = ((P.n_tokens + 63) / 64) * 4;
    P.rcols = 1.0 / (double)P.cols;
    if (!sg_fits(NORM, MT, P.cols, P.ks)) return hipErrorInvalidValue;
    P.tw = sg_tw(NORM, MT, P.ks, P.ntiles, P.n_tokens);
    const int waves = sg_waves(NORM, MT, P.ks, P.tw);
    switch (wtype) {
    case WT_Q4_0: return sg_launch_t<WT_Q4_0, EPI>(P, waves, st);
    case WT_Q8_0: return sg_launch_t<WT_Q8_0, EPI>(P, waves, st);
    case WT_F16: return sg_launch_t<WT_F16, EPI>(P, waves, st);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace nl
