// nl_linattn.h -- gated linear attention (a decay per key channel), 32-bit throughout:
//
//   S_t = diag(alpha_t) S_{t-1} + k_t v_t^T        o_t = S_t^T q_t        alpha = sigmoid(a2 (a1 h) + bias)^(1 / tau)
//
// per head, S [dk][dv] float32, carried from token to token in the stream's state slot.  Behind the recurrence: RMS norm of o
// over dv, a plain weight, silu(gate), a branch scale; the result leaves as the output product's operand (nl_mfma.h).
//
// PROMPTS.  A run of tokens of one stream is cut into sub-chunks of 16 tokens and segments of LA_SEG tokens.  With
// l_t = sum of log alpha from the sub-chunk's first token to t (gla_decay_kernel, one pass over all tokens) a sub-chunk is
//
//   o_t = (q_t e^{l_t})^T S  +  sum_{s <= t} A_ts v_s        A_ts = sum_d q_td k_sd e^{l_td - l_sd}
//   S  <- diag(e^{l_16}) S   +  sum_s (k_s e^{l_16 - l_s}) v_s^T
//
// all of it on v_mfma_f32_16x16x4_f32.  A wavefront owns 16 value columns of S in its accumulators: the accumulator layout
// D[row = 4 g + i][col] is, taken as step i, a B operand whose k slot g is row 4 g + i, so S feeds the first product without
// moving.  A_ts = (q e^l)(k e^{-l}) while no channel of the sub-chunk decays by more than e^-LA_FACTOR_MAX (the products stay in
// range and only relative roundings are added); a sub-chunk beyond that takes the exponent of the difference per pair.
// Segments of a long prompt run in parallel: gla_seg_kernel<.., false> (state increments from zero), gla_scan_kernel (a scan over
// the segments: every segment's starting state), gla_seg_kernel<.., true> (outputs).  A run that fits one segment starts with the
// last of them and the stored state.
//
// DECODE.  One workgroup per (head, stream): the state is read, decayed, updated, multiplied and written back in one pass
// (gla_decode_block, called from the fused mixer launch of nl_winattn.h).
#pragma once
#include "nl_mfma.h"

namespace nl {

constexpr int LA_SUB = 16;               // tokens per sub-chunk
constexpr int LA_SEG = 64;               // tokens per segment
constexpr float LA_FACTOR_MAX = 40.f;
constexpr int LA_MAX_DIM = 256;          // key / value size per head (padded)

struct GlaSub { int tok0, len; };                                 // sub-chunk: tokens [tok0, tok0 + len) of the step
struct GlaSeg { int tok0, len, sub0, stream, pos0, nseg, index; };  // segment `index` of the `nseg` of its run; pos0: the run's first position

struct GlaParams {
    const float *proj;         // projections of the step [token][ldp]: q, k, v, g, a1 at the offsets below
    int ldp, off_q, off_k, off_v, off_g, off_a1;
    int heads, dk, dv, rank;
    int dkp, dvp;              // dk, dv rounded up to 16: the state's leading dimensions
    const float *a2, *a2b, *norm;   // [rank][heads * dk], [heads * dk], [dv]
    float tau, eps, qscale, oscale;
    float *state;              // this layer run, stream 0: [heads][dkp][dvp]
    long long state_stride;    // floats per stream
    void *y;                   // output operand, this branch's columns from y_k0
    int y_nks, y_k0;
    // prompts
    const GlaSub *subs;
    const GlaSeg *segs;
    float *ldec;               // [token][heads * dk] cumulated log decays
    float *inc;                // [segment][heads][dkp][dvp] state increments, then starting states
    float *totlog;             // [segment][heads][dkp]
    const int *runs;           // gla_scan_kernel: first segment of every run with more than one segment
};

// log sigmoid(z) / tau = (min(z, 0) - log1p(e)) / tau, e = exp(-|z|) in (0, 1]: log1p by the area-tangent series
// log(1 + e) = 2 (s + s^3 / 3 + s^5 / 5 + ...), s = e / (2 + e) <= 1 / 3, cut behind s^17 (relative error below 2e-9)
__device__ __forceinline__ float gla_log_alpha(float z, float inv_tau) {
    const float e = exp_f32(-fminf(fabsf(z), 1e4f)), s = e * rcp_f32(2.f + e), w = s * s;
    float p = 1.f / 17.f;
    p = fmaf(p, w, 1.f / 15.f);
    p = fmaf(p, w, 1.f / 13.f);
    p = fmaf(p, w, 1.f / 11.f);
    p = fmaf(p, w, 1.f / 9.f);
    p = fmaf(p, w, 1.f / 7.f);
    p = fmaf(p, w, 1.f / 5.f);
    p = fmaf(p, w, 1.f / 3.f);
    return (fminf(z, 0.f) - 2.f * fmaf(s * w, p, s)) * inv_tau;
}

// grid (sub-chunks, channels / 256)
__global__ void __launch_bounds__(256) gla_decay_kernel(GlaParams P) {
    extern __shared__ __align__(16) char lds[];
    float *a1 = reinterpret_cast<float *>(lds);                  // [rank][16]
    const GlaSub sc = P.subs[blockIdx.x];
    for (int i = threadIdx.x; i < LA_SUB * P.rank; i += 256) {
        const int t = i / P.rank, r = i - t * P.rank;
        a1[r * LA_SUB + t] = t < sc.len ? P.proj[(long long)(sc.tok0 + t) * P.ldp + P.off_a1 + r] : 0.f;
    }
    const int C = P.heads * P.dk, c = min((int)(blockIdx.y * 256 + threadIdx.x), C - 1);
    const float b = P.a2b[c];
    f32x4 z[LA_SUB / 4];
#pragma unroll
    for (int q = 0; q < LA_SUB / 4; q++) z[q] = f32x4{b, b, b, b};
    __syncthreads();
#pragma unroll 8
    for (int r = 0; r < P.rank; r++) {
        const float wr = P.a2[(long long)r * C + c];
#pragma unroll
        for (int q = 0; q < LA_SUB / 4; q++) {
            const f32x4 x = *reinterpret_cast<const f32x4 *>(a1 + r * LA_SUB + q * 4);
#pragma unroll
            for (int i = 0; i < 4; i++) z[q][i] = fmaf(wr, x[i], z[q][i]);
        }
    }
    const float it = 1.f / P.tau;
    float l = 0.f;
#pragma unroll
    for (int t = 0; t < LA_SUB; t++) {
        l += gla_log_alpha(z[t >> 2][t & 3], it);
        if (t < sc.len && (int)(blockIdx.y * 256 + threadIdx.x) < C) P.ldec[(long long)(sc.tok0 + t) * C + c] = l;
    }
}

// grid (segments, heads), max(dvp, dkp) / 16 wavefronts; wavefront w < dvp / 16 owns value columns 16 w .. 16 w + 15, all of them load.
// NE: operand elements per thread and sub-chunk, at least 16 dkp / threads (at most 4); WV: most wavefronts of a launch.
// What a workgroup spends is spread: matrix products (36 of 32 cycles per sub-chunk, wavefront and 64 channels, in float32), exponentials, sums over the
// value columns, and the wavefronts meeting.  The outputs of a head of at most 64 channels therefore take a whole segment a step: A's shared out over the
// wavefronts at once, S through all sub-chunks without a barrier, one meeting for all norms (three barriers a segment where a sub-chunk a step has
// fifteen); more channels have no registers for it, and the increments, which meet once a sub-chunk, are faster with the next sub-chunk's operands requested
// before the current one is multiplied (12.5 us, a whole segment at once 13.9).  Addresses are minima of byte offsets and the sums over 16 lanes are
// row operations.  The outputs of 2047 tokens, 64 channels, 128 values: twelve heads 32.5 -> 29.9 us, six 23.8 -> 19.4; that 384 workgroups are two for
// half of the 256 compute units is the difference between the two.
// Past 64 channels the registers bound it (the increments: past 128), so a thread keeps of its elements only which they are and makes offsets of that each time;
// held, those were sixteen registers through the products, and with them 104 and 228 bytes of scratch a lane at 128 and 256 channels.  The outputs of 2047
// tokens: twelve heads of 128 channels and values 63.5 -> 50.1 us, six of 256 values with 128 channels 65.6 -> 51.4, with 256 118 -> 94, with 64 (eight
// channel tiles, four elements a thread -> four and two) 48.3 -> 36.0.  Heads of 64 channels and fewer have them to spare (32: held 16.8, made 18.0).
constexpr int la_subs(int dkt, int wv, bool out) { return out && wv <= 8 && dkt <= 4 ? LA_SEG / LA_SUB : 1; }   // sub-chunks a step of longer runs
__host__ __device__ constexpr int la_parts(int subs, int nw) { return nw >= 4 * subs ? 4 : nw >= 2 * subs ? 2 : 1; }   // parts of one A
// t n, t <= 16, without a 32-bit product (four times an addition's time)
__device__ __forceinline__ unsigned la_rows(unsigned t, unsigned n) { return __umul24(t, n & 0xffff) + (__umul24(t, n >> 16) << 16); }
__host__ __device__ constexpr int la_ldk(int dkp) { return (dkp >> 4) & 1 ? dkp : dkp + 16; }   // rows g of k e^{l_end - l} in other banks
__host__ __device__ constexpr size_t gla_seg_lds(int dkp, int subs, int np, bool out) {
    const int rows = subs * LA_SUB;
    return (size_t)(rows * la_ldk(dkp) + subs * dkp + (out ? 2 * rows * (dkp + 4) + subs * np * 256 + 16 : 0)) * 4;
}
static_assert(gla_seg_lds(64, LA_SEG / LA_SUB, 2, true) <= 65536 && gla_seg_lds(256, 1, 4, true) <= 65536, "what a launch has without asking");

template <typename T, int DKT, int NE, int WV, bool OUT, int SUBS = la_subs(DKT, WV, OUT)>
__global__ void __launch_bounds__(WV * 64, WV > 8 || NE <= 2 || (OUT && DKT > 4) ? 4 : 2) gla_seg_kernel(GlaParams P) {
    extern __shared__ __align__(16) char lds[];
    constexpr int ROWS = SUBS * LA_SUB;
    const GlaSeg sg = P.segs[blockIdx.x];
    if (!OUT && (sg.nseg == 1 || sg.index + 1 == sg.nseg)) return;     // nobody starts from the state behind the last segment
    const int h = blockIdx.y, tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63, w = tid >> 6, nw = nthr >> 6, g = lane >> 4, c = lane & 15;
    const int dk = P.dk, dkp = P.dkp, nkt = dkp >> 4, ld = dkp + 4, ldk = la_ldk(dkp), C = P.heads * dk, dvc = w * 16 + c;
    const int nv = P.dvp >> 4, np = la_parts(la_subs(DKT, WV, OUT), nw);    // (short runs take the same parts: the same bits)
    const bool owner = w < nv, value = dvc < P.dv;
    float *ke = reinterpret_cast<float *>(lds);          // [ROWS][ldk] k e^{l_end - l}
    float *etot = ke + ROWS * ldk;                       // [SUBS][dkp] e^{l_end}
    float *qd = etot + SUBS * dkp;                       // [ROWS][ld]  q e^l
    float *ki = qd + ROWS * ld;                          // [ROWS][ld]  k e^-l
    float *part = ki + ROWS * ld;                        // [SUBS][np][256] partial A
    float *ssq = ki;                                     // [nw][ROWS] sums of squares, once the A's are made
    int *flag = reinterpret_cast<int *>(part + SUBS * np * 256);  // [16] sub-chunks in which the wavefront saw a decay beyond the factored range
    f32x4 S[DKT];
    const long long shead = (long long)dkp * P.dvp;
    float *stream_state = P.state + sg.stream * P.state_stride + h * shead;
    float *seg_state = P.inc + ((long long)blockIdx.x * P.heads + h) * shead;
    float rq[SUBS][NE] = {}, rk[SUBS][NE] = {}, rl[SUBS][NE] = {}, re[SUBS][NE] = {}, rv[SUBS][4] = {};
    // this thread's elements: token of the sub-chunk (16: none) and channel; where they lie: row t of the projections and of ldec, (t, d) of the LDS images
    struct Elem { int t, d, lk, lq; unsigned ep, el; };
    constexpr bool KEEP = OUT ? DKT <= 4 : DKT <= 8;     // (see above)
    unsigned elems[NE];
    Elem held[NE];
#pragma unroll
    for (int e = 0; e < NE; e++) {
        const int i = tid + e * nthr, t = min(i / dkp, LA_SUB), d = i - i / dkp * dkp;
        elems[e] = t << 16 | d;
        held[e] = Elem{t, d, t * ldk + d, t * ld + d, (unsigned)(t * P.ldp) * 4u, (unsigned)(t * C) * 4u};
    }
    auto elem = [&](int e, bool keep) __attribute__((always_inline)) {
        if (keep) return held[e];
        unsigned x = elems[e];
        asm volatile("" : "+v"(x));                      // (or hipcc keeps what is made of it)
        const int t = x >> 16, d = x & 0xffff;
        return Elem{t, d, (int)__umul24(t, ldk) + d, (int)__umul24(t, ld) + d, la_rows(t, P.ldp) * 4u, la_rows(t, C) * 4u};
    };
    const unsigned vrow = (unsigned)(g * P.ldp) * 4u, grow = 4 * vrow, prow = P.ldp * 4u;
    const unsigned vcol = (unsigned)(h * P.dv + min(dvc, P.dv - 1)) * 4u;
    const char *proj = reinterpret_cast<const char *>(P.proj + (long long)sg.tok0 * P.ldp), *ldec = reinterpret_cast<const char *>(P.ldec + (long long)sg.tok0 * C + h * dk);
    // (every address is clamped into the segment and the row, so that no load waits in a branch; what lies beyond is dropped below.  Row offsets are
    //  minima of byte offsets: a product per load costs four times an addition)
    auto fetch = [&](int u0) {
        const int last = sg.len - 1;
        const unsigned plast = last * prow;
#pragma unroll
        for (int s = 0; s < SUBS; s++) {
            const int us = u0 + s * LA_SUB, end = min(us + LA_SUB - 1, last);
            if (SUBS > 1 && us > last) break;                // (requests of all four by short runs among longer ones cost as much again as the first)
            const unsigned pend = end * prow, lend = (unsigned)(end * C) * 4u, p0 = us * prow, l0 = (unsigned)(us * C) * 4u;
#pragma unroll
            for (int e = 0; e < NE; e++) {
                const Elem E = elem(e, KEEP);
                const unsigned d = (unsigned)min(E.d, dk - 1) * 4u, at = min(E.ep + p0, pend) + h * dk * 4u + d;
                rk[s][e] = ld_off<float>(proj + P.off_k * 4ll, at);
                rl[s][e] = ld_off<float>(ldec, min(E.el + l0, lend) + d);
                re[s][e] = ld_off<float>(ldec, lend + d);
                if (OUT) rq[s][e] = ld_off<float>(proj + P.off_q * 4ll, at);
            }
            // value columns in B-operand order: step i holds token 4 i + g
#pragma unroll
            for (int i = 0; i < 4; i++) rv[s][i] = ld_off<float>(proj + P.off_v * 4ll, min(vrow + p0 + 4 * i * prow, plast) + vcol);
        }
    };
    fetch(0);
    {
        const float *from = !OUT || !owner ? nullptr : sg.nseg > 1 ? seg_state : sg.pos0 == 0 ? nullptr : stream_state;
#pragma unroll
        for (int dt = 0; dt < DKT; dt++) {
            S[dt] = f32x4{};
            if (from && dt < nkt)
#pragma unroll
                for (int i = 0; i < 4; i++) S[dt][i] = from[(long long)(dt * 16 + 4 * g + i) * P.dvp + dvc];
        }
    }
    const float inv_dv = 1.f / (float)P.dv;
    const int ycol = (int)op_index(0, P.y_k0 + h * P.dv + dvc, P.y_nks);
    const float nrm = OUT && value ? P.norm[dvc] * P.oscale : 0.f;
    float tot = 0.f;                                     // thread d < dkp: channel d's log decay up to here
    for (int u0 = 0; u0 < sg.len; u0 += ROWS) {
        const int left = sg.len - u0;                    // tokens from this step's first on
        if (ROWS < LA_SEG && u0) lds_barrier();          // the step before has been read
        // the step's operands; tokens beyond its length and channels beyond dk are zero
        int strong = 0;
        float v[SUBS][4] = {};
#pragma unroll
        for (int s = 0; s < SUBS; s++) {
            if (SUBS > 1 && s * LA_SUB >= left) break;
#pragma unroll
            for (int e = 0; e < NE; e++) {
                const Elem E = elem(e, KEEP || !OUT);
                const int t = E.t, d = E.d, row = s * LA_SUB + t, ak = s * LA_SUB * ldk + E.lk, aq = s * LA_SUB * ld + E.lq;
                const bool chan = d < dk && s * LA_SUB < left, live = d < dk && row < left;
                const float l = live ? rl[s][e] : 0.f, end = chan ? re[s][e] : 0.f, k = live ? rk[s][e] : 0.f;
                if (t < LA_SUB) {
                    ke[ak] = k * exp_f32(end - l);
                    if (OUT) {
                        strong |= end < -LA_FACTOR_MAX ? 1 << s : 0;
                        qd[aq] = (live ? rq[s][e] : 0.f) * P.qscale * exp_f32(l);
                        ki[aq] = k * exp_f32(fminf(-l, LA_FACTOR_MAX));
                    }
                    if (t == 0) {
                        etot[s * dkp + d] = exp_f32(end);
                        tot += end;                      // (only e == 0 has t == 0: nthr >= 4 dkp)
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) v[s][i] = value && s * LA_SUB + 4 * i + g < left ? rv[s][i] : 0.f;
            __builtin_amdgcn_sched_barrier(0);
        }
        if (OUT) {
            int any = 0;
#pragma unroll
            for (int s = 0; s < SUBS; s++) any |= __any(strong >> s & 1) ? 1 << s : 0;
            if (lane == 0) flag[w] = any;
        }
        lds_barrier();
        if (ROWS < LA_SEG && u0 + ROWS < sg.len) fetch(u0 + ROWS);
        if (OUT) {
            int slow = 0;
            for (int q = 0; q < nw; q++) slow |= flag[q];
            for (int task = w; task < SUBS * np; task += nw) {
                const int s = task % SUBS, p = task / SUBS;
                if (slow >> s & 1 || s * LA_SUB >= left) continue;
                f32x4 a = {};
                for (int ks = p; ks < dkp / 4; ks += np)
                    a = __builtin_amdgcn_mfma_f32_16x16x4f32(qd[(s * LA_SUB + c) * ld + 4 * ks + g], ki[(s * LA_SUB + c) * ld + 4 * ks + g], a, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < 4; i++) part[(s * np + p) * 256 + (4 * g + i) * 16 + c] = a[i];
            }
            if (slow)
                for (int i = tid; i < SUBS * 256; i += nthr) {
                    const int sub = i >> 8, t = i >> 4 & 15, s = i & 15;
                    if (!(slow >> sub & 1)) continue;
                    float a = 0.f;
                    if (s <= t && sub * LA_SUB + t < left) {
                        const int t0 = sg.tok0 + u0 + sub * LA_SUB;
                        const float *qp = P.proj + (long long)(t0 + t) * P.ldp + P.off_q + h * dk, *kp = P.proj + (long long)(t0 + s) * P.ldp + P.off_k + h * dk;
                        const float *lt = P.ldec + (long long)(t0 + t) * C + h * dk, *ls = P.ldec + (long long)(t0 + s) * C + h * dk;
#pragma unroll 1
                        for (int d = 0; d < dk; d++) a += qp[d] * P.qscale * kp[d] * exp_f32(lt[d] - ls[d]);
                    }
                    for (int p = 0; p < np; p++) part[(sub * np + p) * 256 + (i & 255)] = p == 0 ? a : 0.f;
                }
            lds_barrier();
        }
        f32x4 o[SUBS];
        float gz[SUBS][4];                               // gates, in accumulator order: token 4 g + i
        if (OUT)
#pragma unroll
            for (int s = 0; s < SUBS; s++) {
                if (SUBS > 1 && s * LA_SUB >= left) break;
#pragma unroll
                for (int i = 0; i < 4; i++) gz[s][i] = ld_off<float>(proj + P.off_g * 4ll, min(grow + (u0 + s * LA_SUB + i) * prow, (sg.len - 1) * prow) + vcol);
            }
        if (owner) {
#pragma unroll
            for (int s = 0; s < SUBS; s++) {
                __builtin_amdgcn_sched_barrier(0);       // (or the scheduler holds the next one's operands too, and half the wavefronts fit)
                o[s] = f32x4{};
                if (s * LA_SUB < left) {
                    if (OUT) {
#pragma unroll
                        for (int dt = 0; dt < DKT; dt++)
                            if (dt < nkt) {
                                const f32x4 qv = *reinterpret_cast<const f32x4 *>(qd + (s * LA_SUB + c) * ld + dt * 16 + 4 * g);
#pragma unroll
                                for (int i = 0; i < 4; i++) o[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[i], S[dt][i], o[s], 0, 0, 0);
                            }
                        float a[4];                      // row c, columns 4 i + g of A: nothing flows back in time
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const float *pa = part + s * np * 256 + c * 16 + 4 * i + g;
                            float x = pa[0];
                            for (int p = 1; p < np; p++) x += pa[p * 256];
                            a[i] = 4 * i + g <= c ? x : 0.f;
                        }
#pragma unroll
                        for (int i = 0; i < 4; i++) o[s] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], v[s][i], o[s], 0, 0, 0);
                    }
#pragma unroll
                    for (int dt = 0; dt < DKT; dt++)
                        if (dt < nkt) {
                            const f32x4 tl = *reinterpret_cast<const f32x4 *>(etot + s * dkp + dt * 16 + 4 * g);
#pragma unroll
                            for (int i = 0; i < 4; i++) S[dt][i] *= tl[i];
#pragma unroll
                            for (int i = 0; i < 4; i++) S[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(ke[(s * LA_SUB + 4 * i + g) * ldk + dt * 16 + c], v[s][i], S[dt], 0, 0, 0);
                        }
                }
            }
        }
        if (OUT) {
            // norm over the head's value columns: sums of squares over 16 lanes, then over the wavefronts
            if (owner)
#pragma unroll
                for (int s = 0; s < SUBS; s++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        float ss = o[s][i] * o[s][i];
                        ss += dpp_f32<DPP_QUAD_XOR1>(ss);
                        ss += dpp_f32<DPP_QUAD_XOR2>(ss);
                        ss += dpp_f32<DPP_HALF_MIRROR>(ss);
                        ss += dpp_f32<DPP_ROW_MIRROR>(ss);
                        if (c == 0) ssq[w * ROWS + s * LA_SUB + 4 * g + i] = ss;
                    }
            lds_barrier();
            T *y = reinterpret_cast<T *>(P.y);
            if (owner && value)
#pragma unroll
                for (int s = 0; s < SUBS; s++) {
                    if (s * LA_SUB >= left) continue;
                    f32x4 s2 = {};
                    for (int q0 = 0; q0 < nv; q0 += 4) {
                        f32x4 x[4];
#pragma unroll
                        for (int q = 0; q < 4; q++) x[q] = *reinterpret_cast<const f32x4 *>(ssq + min(q0 + q, nv - 1) * ROWS + s * LA_SUB + 4 * g);
#pragma unroll
                        for (int q = 0; q < 4; q++)
                            if (q0 + q < nv) s2 += x[q];
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int row = s * LA_SUB + 4 * g + i, t = sg.tok0 + u0 + row;
                        if (row < left)
                            put(y + (unsigned)((t >> 4) * P.y_nks * OPT + (t & 15) * 8 + ycol), o[s][i] * rsqrt_f32(s2[i] * inv_dv + P.eps) * nrm * (gz[s][i] * sigmoid_f32(gz[s][i])));
                    }
                }
        }
        if (ROWS >= LA_SEG) break;                       // (a segment is one step; a loop would keep its operands)
    }
    if (!OUT && tid < dkp) P.totlog[((long long)blockIdx.x * P.heads + h) * dkp + tid] = tot;      // (channels beyond dk: zero)
    if (owner && (!OUT || sg.index + 1 == sg.nseg)) {
        float *to = OUT ? stream_state : seg_state;
#pragma unroll
        for (int dt = 0; dt < DKT; dt++)
            if (dt < nkt)
#pragma unroll
                for (int i = 0; i < 4; i++) to[(long long)(dt * 16 + 4 * g + i) * P.dvp + dvc] = S[dt][i];
    }
}

// grid (state elements / 4 / 256, heads, runs): every segment's increment becomes its starting state
__global__ void __launch_bounds__(256) gla_scan_kernel(GlaParams P) {
    const int s0 = P.runs[blockIdx.z], h = blockIdx.y, e = blockIdx.x * 256 + threadIdx.x, per = P.dkp * P.dvp / 4;
    if (e >= per) return;
    const GlaSeg sg = P.segs[s0];
    const int d = e * 4 / P.dvp;
    f32x4 S = {};
    if (sg.pos0 > 0) S = *reinterpret_cast<const f32x4 *>(P.state + sg.stream * P.state_stride + (long long)h * P.dkp * P.dvp + e * 4);
    f32x4 *at = reinterpret_cast<f32x4 *>(P.inc) + ((long long)s0 * P.heads + h) * per + e;
    const float *tl = P.totlog + ((long long)s0 * P.heads + h) * P.dkp + d;
    const long long astep = (long long)P.heads * per, tstep = (long long)P.heads * P.dkp;
    constexpr int U = 8;
    for (int i0 = 0; i0 < sg.nseg; i0 += U) {
        f32x4 inc[U];
        float dec[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = min(i0 + u, sg.nseg - 1);
            inc[u] = at[i * astep];
            dec[u] = tl[i * tstep];
        }
#pragma unroll
        for (int u = 0; u < U; u++)
            if (i0 + u < sg.nseg) {
                at[(i0 + u) * astep] = S;
                S = S * exp_f32(dec[u]) + inc[u];           // (the last segment's increment was not computed and is not used)
            }
    }
}

// one (head, token of a decode batch) by a workgroup of 256; lds: see gla_decode_lds
__host__ __device__ inline size_t gla_decode_lds(int dkp, int dvp, int rank) { return (size_t)(3 * dkp + dvp + 1024 + 8 + rank) * 4; }

template <typename T>
__device__ __forceinline__ void gla_decode_block(const GlaParams &P, int h, int n, int stream, int pos, char *lds) {
    constexpr int U = 8, RU = 16;
    const int tid = threadIdx.x, dk = P.dk, dv = P.dv, C = P.heads * dk;
    float *q = reinterpret_cast<float *>(lds), *k = q + P.dkp, *al = k + P.dkp, *v = al + P.dkp, *part = v + P.dvp, *red = part + 1024, *a1 = red + 8;
    const float *pr = P.proj + (long long)n * P.ldp;
    const int nc = P.dvp >> 2, rp = 256 / nc, c4 = tid % nc, r0 = tid / nc;
    f32x4 *S = reinterpret_cast<f32x4 *>(P.state + stream * P.state_stride + (long long)h * P.dkp * P.dvp) + c4;
    // everything that does not depend on this step's arithmetic is requested up front (head sizes are at most 256: one element per
    // thread), what is needed first in front: loads return in order
    const bool kc = tid < dk, vc = tid < dv;
    const float rq = kc ? pr[P.off_q + h * dk + tid] : 0.f, rk = kc ? pr[P.off_k + h * dk + tid] : 0.f, rv = vc ? pr[P.off_v + h * dv + tid] : 0.f;
    const float ra = tid < P.rank ? pr[P.off_a1 + tid] : 0.f;
    const float *w2 = P.a2 + h * dk + min(tid, dk - 1);
    float w[RU];
#pragma unroll
    for (int r = 0; r < RU; r++) w[r] = w2[(long long)min(r, P.rank - 1) * C];
    const float bias = kc ? P.a2b[h * dk + tid] : 0.f, gz = vc ? pr[P.off_g + h * dv + tid] : 0.f, nrm = vc ? P.norm[tid] * P.oscale : 0.f;
    f32x4 s[U];
    // (rows past the last one repeat it, unused: each behind a branch of its own, the compiler waited for one row in front of the next where its registers fell
    // badly -- 64 streams of 28 layers of 1536 columns, a layer of both branches 15.6 or 16.9 us a launch; one stream of 20 layers of 768 472 a step, now 462)
    auto load = [&](int d0) {
#pragma unroll
        for (int u = 0; u < U; u++) s[u] = S[(long long)min(d0 + u * rp, dk - 1) * nc];
        if (pos == 0)
#pragma unroll
            for (int u = 0; u < U; u++) s[u] = f32x4{};
    };
    load(r0);
    if (tid < P.rank) a1[tid] = ra;
    for (int i = tid + 256; i < P.rank; i += 256) a1[i] = pr[P.off_a1 + i];
    if (kc) { q[tid] = rq * P.qscale; k[tid] = rk; }
    if (tid < P.dvp) v[tid] = rv;
    lds_barrier();
    if (kc) {
        float z = bias;
#pragma unroll
        for (int r = 0; r < RU; r++)
            if (r < P.rank) z = fmaf(w[r], a1[r], z);
        for (int r = RU; r < P.rank; r++) z = fmaf(w2[(long long)r * C], a1[r], z);
        al[tid] = exp_f32(gla_log_alpha(z, 1.f / P.tau));
    }
    lds_barrier();
    f32x4 o = {};
    if (r0 < rp) {
        const f32x4 vv = *reinterpret_cast<const f32x4 *>(v + c4 * 4);
        for (int d0 = r0; d0 < dk; d0 += U * rp) {
            if (d0 != r0) load(d0);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int d = d0 + u * rp;
                if (d < dk) {
                    const f32x4 x = s[u] * al[d] + vv * k[d];
                    S[(long long)d * nc] = x;
                    o += x * q[d];
                }
            }
        }
        *reinterpret_cast<f32x4 *>(part + r0 * P.dvp + c4 * 4) = o;
    }
    lds_barrier();
    float val = 0.f;                                     // dvp <= 256: one value column per thread
    if (vc)
        for (int r = 0; r < rp; r++) val += part[r * P.dvp + tid];
    const float ss = wave_sum(val * val);
    if ((tid & 63) == 0) red[tid >> 6] = ss;
    lds_barrier();
    if (vc) {
        const float inv = rsqrt_f32((red[0] + red[1] + red[2] + red[3]) / (float)dv + P.eps);
        put(reinterpret_cast<T *>(P.y) + op_index(n, P.y_k0 + h * dv + tid, P.y_nks), val * inv * nrm * (gz * sigmoid_f32(gz)));
    }
}

// longest: tokens of the longest run.  Up to one sub-chunk, the outputs are better off with a workgroup that holds one (64 channels, 128 values, 54 runs of
// 5 to 16 tokens: six heads 13.2 -> 12.4 us, twelve 19.8 -> 18.2; runs of 24, twelve heads: a sub-chunk a step 28.6, a segment 27.9)
template <typename T, bool OUT>
hipError_t launch_gla_seg(const GlaParams &P, int nsegs, int longest, hipStream_t st) {
    const int nw = std::max(P.dvp, P.dkp) / 16;
    auto go = [&](auto dkt, auto ne, auto wv, auto subs) {
        constexpr int DKT = decltype(dkt)::value, NE = decltype(ne)::value, WV = decltype(wv)::value, SUBS = decltype(subs)::value;
        hipLaunchKernelGGL((gla_seg_kernel<T, DKT, NE, WV, OUT, SUBS>), dim3(nsegs, P.heads), dim3(nw * 64), gla_seg_lds(P.dkp, SUBS, la_parts(la_subs(DKT, WV, OUT), nw), OUT), st, P);
        return hipGetLastError();
    };
    using std::integral_constant;
    const integral_constant<int, 1> one{};
    const integral_constant<int, 2> two{};
    const integral_constant<int, 4> four{};
    const integral_constant<int, 8> eight{};
    const integral_constant<int, 16> sixteen{};
    const bool half = 16 * P.dkp <= 2 * nw * 64;                 // two elements a thread
    if (nw <= 8) {
        if (P.dkp > 64) return go(eight, four, eight, one);      // (dkp <= 128)
        if constexpr (OUT)
            if (longest > LA_SUB) return half ? go(four, two, eight, four) : go(four, four, eight, four);
        return half ? go(four, two, eight, one) : go(four, four, eight, one);
    }
    if (P.dkp <= 64) return go(four, two, sixteen, one);         // (more than 128 values: two elements a thread)
    if (P.dkp <= 128) return go(eight, four, sixteen, one);
    return go(sixteen, four, sixteen, one);
}

// the recurrence of a ragged step: runs = streams' token runs with more than one segment (their first segments in P.runs)
template <typename T>
hipError_t launch_gla(const GlaParams &P, int nsubs, int nsegs, int nruns, int longest, hipStream_t st) {
    hipLaunchKernelGGL(gla_decay_kernel, dim3(nsubs, (P.heads * P.dk + 255) / 256), dim3(256), (size_t)LA_SUB * P.rank * 4, st, P);
    if (nruns > 0) {
        if (hipError_t s = launch_gla_seg<T, false>(P, nsegs, longest, st)) return s;
        hipLaunchKernelGGL(gla_scan_kernel, dim3((P.dkp * P.dvp / 4 + 255) / 256, P.heads, nruns), dim3(256), 0, st, P);
    }
    return launch_gla_seg<T, true>(P, nsegs, longest, st);
}

}  // namespace nl
