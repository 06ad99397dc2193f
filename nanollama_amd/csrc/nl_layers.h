// nl_layers.h -- every layer of a decode step in ONE launch, for the middle tiers (one GPU, one token).
//
// go/model.go:513-613 is, per layer, five matrix products and an attention that each need all of the one before.  As launches
// (nl_kernels.h) a layer of 1536 columns is 5 x 5.6 us, of which its 26 MB of Q8_0 weights explain 5.7 in all: a launch boundary, a
// cold fetch of weights and arguments, the reductions, five times over.  Here 256 workgroups stay for the whole step and hand the
// activations on as tagged 16-byte granules (nl_tp.h), while every weight is on its way into registers a phase or two before it is needed.
// Measured, 28 layers of 1536 / 4096 at position 733, Q8_0: 27.9 -> 21.5 us a layer; without the weights 18.8: what is left
// is the chain of five exchanges (1.5 - 2.8 us each) and five products (0.7 - 1.2 us).  Q4_K and Q6_K layers, us a token, 28 layers at 20 / 600: 756 -> 539 /
// 795 -> 625 and 749 -> 536 / 792 -> 618; 20 layers of 768 columns, Q4_K, at 20 / 400: 419 -> 320 / 442 -> 350.
//
// A workgroup is eight wavefronts that multiply and four that exchange.  Vector memory operations of a wavefront complete in order, so
// one that polls waits for every weight it has requested before; with the roles apart the weights stream while the others poll.
// Phases of a layer, two barriers each (the input comes into LDS | barrier | products | barrier | the first exchanging wavefront adds the
// partial sums and publishes, the multiplying ones request weights of a later phase):
//   1  x     -> RMSNorm -> this workgroup's 16-row tile of Q | K | V -> bias, RoPE         (go/quant.go:597-607, go/model.go:517-533, :449-477)
//   2  q k v -> attention of one unit: 128 positions of one kv head for some of its heads  (:552-587), a (max, sum, sum p v[64]) record a head;
//               the unit that holds the step's position merges a head's records
//   3  the heads' outputs -> half a tile of WO + residual                                  (:590-594)
//   4  x'    -> RMSNorm -> a tile of gate and the same of up -> SiLU(gate) * up            (:597-606)
//   5  h     -> half a tile of down + residual                                             (:609-612)
// Tile (or half) t of a matrix and unit u of the attention belong to workgroup t or u; half tiles, because 1536 rows are 96 tiles and 192
// workgroups read them in 2/3 of the time.  The heads' outputs and h are brought in by all twelve wavefronts, at places where the
// multiplying ones have little in flight (the other two inputs by all of them: 24.2).  A buffer per phase, reused by every layer under the layer's
// own tag: whoever writes the next layer's granules has, through the phases between, waited for everyone who reads this layer's.
// The K / V row of the step's position reaches the attention as granules; the unit that holds the position stores it.  Other units read rows
// that earlier launches wrote.
// Every poll is bounded; a give-up (some workgroup was not resident) sets the status words and the host redoes the step on the launch plans (and, up to
// three times, tries this launch again with the next call).
//
// Weights are requested by buffer loads whose range is empty where a wavefront has nothing to do: no branch around a load, so the compiler's
// count of loads in flight holds across the phases.  They go out a quarter of a microsecond apart: all at once they stand before
// the exchange that follows in every queue of the chip (22.5 us a layer; sleeps of 2, 4, 8: 22.1, 21.7, 21.85).
#pragma once
#include "nl_layers_map.h"
#include "nl_tp.h"

namespace nl {

constexpr int LY_CW = 8, LY_GW = 4, LY_WAVES = LY_CW + LY_GW, LY_THREADS = LY_WAVES * 64, LY_GT = LY_GW * 64;
constexpr int LY_PASS = 128;               // positions of a unit
constexpr int LY_MAX_REC = 16;             // records of a head
constexpr int LY_MAX_HPU = 8;              // heads of a unit
constexpr int LY_PER_XCD = 32;             // a launch is one workgroup a compute unit of a whole chip
static_assert(LY_TG == GPT, "granules of a tile");
constexpr int LY_RELAY = 1;                // the exchanging wavefront that relays
constexpr int LY_MAX_COLS = 2048, LY_MAX_FF = 4096;
constexpr int LY_CODES = 16;               // this launch's status codes are above those of the other launches on the same word

struct LayersEntry {                       // one layer: Q|K|V, WO, gate, up, down
    const uint8_t *q[5];
    const uint32_t *s[5];
    const float *norm[2], *bq, *bk, *bv, *bo;
};
constexpr int LY_ENTRY = sizeof(LayersEntry) / 8, LY_MAX_LAYERS = 64;
enum { LY_QP = 0, LY_SP = 5, LY_NORM = 10, LY_BQ = 12, LY_BO = 15 };      // places of an entry
struct LayersParams {
    const LayersEntry *layers;
    int L, D, H, KV, gqa, seq_len, rope_conj, single_stream;
    int np_d, np_o, np_i;                  // 64-column pairs of a row of Q|K|V and gate, of WO, of down
    int t_qkv, t_d, t_i;                   // 16-row tiles of Q|K|V, of WO and down, of gate
    float eps, scale;
    float *x;                              // the embedding row; the residual stream behind the last layer
    const float *rope_cos, *rope_sin;
    float *kcache, *vcache;                // layer 0, stream 0
    long long kv_layer_stride, kv_stream_stride;
    const int *ctl;
    const unsigned *tick;
    u32x4 *gq, *gr;                        // q|k|v tiles; records [H][rec_max][LY_REC]
    u32x4 *go, *gp, *gh, *gx;              // the heads' outputs [H][LY_REC] (values from 2 on); x' half tiles; h tiles; x half tiles
    u32x4 *loc;                            // [LY_XCDS] copies of gp | gh | gx, `loc_n` granules each
    int loc_n;
    unsigned *tickets;                     // [LY_XCDS], a line apart: workgroups that started on the XCD, ever
    int rec_max;
    unsigned *status, *host_status;
    int spin_limit;
};

template <int WT> struct LyUnit { uint4 c[WTraits<WT>::CPP]; uint2 s; };

typedef unsigned ly_u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t ly_rsrc(const void *p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void ly_barrier() {              // orders LDS only: weights in flight stay in flight
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ float ly_lane(float v, int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); }

// A wavefront's share u of a 16-row tile: the whole tile by 256 columns (lane = 4 row + pair) or, HALF, eight rows by 512 columns (lane = 8 row + pair).
// The lane's 64 columns, by buffer loads; none where !on.
template <int WT, bool HALF>
__device__ __forceinline__ void ly_load(LyUnit<WT> &v, const uint8_t *q, const uint32_t *s, int tile, int row0, int u, int npairs, bool on, int lane) {
    constexpr int CPP = WTraits<WT>::CPP, SW = scale_words(WT);
    const int pair = min(HALF ? 8 * u + (lane & 7) : 4 * u + (lane & 3), npairs - 1), g = pair / KL, gsz = min(KL, npairs - g * KL), row = row0 + (HALF ? lane >> 3 : lane >> 2);
    const unsigned at = (unsigned)(row * gsz + (pair - g * KL));
    const __amdgpu_buffer_rsrc_t rq = ly_rsrc(q + (size_t)tile * npairs * (CPP * TR * 16), on ? (unsigned)(npairs * CPP * TR * 16) : 0u);
#pragma unroll
    for (int j = 0; j < CPP; j++) {
        v.c[j] = __builtin_bit_cast(uint4, (u32x4)__builtin_amdgcn_raw_buffer_load_b128(rq, (int)(((unsigned)(g * KL * CPP * TR + j * TR * gsz) + at) * 16u), 0, 0));
        __builtin_amdgcn_s_sleep(4);
    }
    v.s = make_uint2(0u, 0u);
    if constexpr (WTraits<WT>::SCALED) {
        const __amdgpu_buffer_rsrc_t rs = ly_rsrc(reinterpret_cast<const char *>(s) + (size_t)tile * npairs * (TR * 4 * SW), on ? (unsigned)(npairs * TR * 4 * SW) : 0u);
        const int so = (int)(((unsigned)(g * KL * TR) + at) * (4u * SW));
        if constexpr (SW == 2) {
            const ly_u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(rs, so, 0, 0);
            v.s = make_uint2(w[0], w[1]);
        } else v.s.x = __builtin_amdgcn_raw_buffer_load_b32(rs, so, 0, 0);
    }
}
// its product with its columns' inputs -> the rows' partial sums
template <int WT, bool HALF>
__device__ __forceinline__ void ly_dot(const LyUnit<WT> &v, const float *xs, int u, int npairs, float *red, int lane) {
    const int pair = HALF ? 8 * u + (lane & 7) : 4 * u + (lane & 3);
    float a = pair_dot_lean<WT>(v.c, v.s, xs + min(pair, npairs - 1) * XS_PAIR, 0.f);
    a = quad_sum(pair < npairs ? a : 0.f);
    if constexpr (HALF) a += dpp_f32<DPP_HALF_MIRROR>(a);
    if ((lane & (HALF ? 7 : 3)) == 0) red[lane >> (HALF ? 3 : 2)] = a;
}

// pointer `place` of layer l, from the table in LDS (the table in memory is cold in the scalar cache every layer)
template <class T> __device__ __forceinline__ const T *ly_ptr(const uint2 *tab, int l, int place) {
    const uint2 v = tab[l * LY_ENTRY + place];
    return reinterpret_cast<const T *>(((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)v.y) << 32) | (unsigned)__builtin_amdgcn_readfirstlane((int)v.x));
}
struct LyPoll {
    unsigned *status, *host_status;
    int *lds_dead;
    int spin_limit;
    bool dead;
};
// another look?  (false: give up; wave-uniform)
__device__ __forceinline__ bool ly_again(LyPoll &Q, int &spins, unsigned code, int lane) {
    bool stop = ++spins >= Q.spin_limit || Q.dead;
    if ((spins & 63) == 63) stop = stop || __builtin_amdgcn_readfirstlane((int)__hip_atomic_load(Q.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0;
    if (stop) {
        Q.dead = true;
        if (lane == 0) { atomicOr(Q.status, code << LY_CODES); *Q.host_status = code << LY_CODES; *Q.lds_dead = 1; }
        return false;
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_sleep(1);
    return true;
}
// (sc1: past the L1, and past an L2 line that another XCD has written through)
__device__ __forceinline__ u32x4 ly_granule(__amdgpu_buffer_rsrc_t r, unsigned i) { return __builtin_amdgcn_raw_buffer_load_b128(r, (int)(i * 16u), 0, 16); }

// A record of R values is ceil(R / 3) granules (16: six, 8: three): granule g of an array of records -> its first value
template <int R> __device__ __forceinline__ int ly_first(int g, int &j) {
    constexpr int G = (R + 2) / 3;
    const int t = (int)(((unsigned)g * (65536u / G + 1)) >> 16);       // g / 6, g / 3 (g < 16384)
    j = g - t * G;
    return t * R + 3 * j;
}
// ng granules of records of R values by NT threads: f(granule of the thread, index of the first value, values 0, 1, 2; how many of them exist)
template <int R, int NR, int NT, class F>
__device__ __forceinline__ void ly_gather(const u32x4 *src, int ng, unsigned tag, LyPoll &Q, unsigned code, int gt, F f) {
    constexpr int LAST = R - (R - 1) / 3 * 3;
    const int lane = gt & 63;
    const __amdgpu_buffer_rsrc_t r = ly_rsrc(src, (unsigned)ng * 16u);
    u32x4 v[NR];
    if ((gt & ~63) < ng) {
        for (int spins = 0;;) {
            bool ok = true;
#pragma unroll
            for (int k = 0; k < NR; k++) v[k] = ly_granule(r, (unsigned)min(gt + k * NT, ng - 1));
#pragma unroll
            for (int k = 0; k < NR; k++) ok = ok && v[k].x == tag;
            if (__all(ok) || !ly_again(Q, spins, code, lane)) break;
        }
#pragma unroll
        for (int k = 0; k < NR; k++) {
            const int g = gt + k * NT;
            if (g < ng) {
                int j;
                const int i = ly_first<R>(g, j);
                f(k, i, __uint_as_float(v[k].y), __uint_as_float(v[k].z), __uint_as_float(v[k].w), j == (R - 1) / 3 ? LAST : 3);
            }
        }
    }
}
__device__ __forceinline__ int ly_at(int col) { return col + (col >> 6) * (XS_PAIR - PAIR); }     // LDS place of a column

// the norm's weights of the granules a thread will gather
struct LyNorm { float w[3][3]; };
__device__ __forceinline__ void ly_norm_weights(LyNorm &n, const float *normw, int ng, int gt) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
        int j;
        const int i = ly_first<8>(min(gt + k * LY_GT, ng - 1), j);
#pragma unroll
        for (int c = 0; c < 3; c++) n.w[k][c] = normw[i + (c < 2 || j < 2 ? c : 1)];
    }
}
// RMSNorm input, half tiles by the exchanging wavefronts: raw values to xr, x * g to xs, the thread's squares returned
__device__ __forceinline__ double ly_gather_norm(const u32x4 *src, int ng, unsigned tag, LyPoll &Q, unsigned code, int gt, const LyNorm &nw, float *xr, float *xs) {
    double ss = 0.0;
    ly_gather<8, 3, LY_GT>(src, ng, tag, Q, code, gt, [&](int k, int i, float a, float b, float c, int n) __attribute__((always_inline)) {
        xr[i] = a; xr[i + 1] = b;
        xs[ly_at(i)] = a * nw.w[k][0]; xs[ly_at(i + 1)] = b * nw.w[k][1];
        ss = fma((double)a, (double)a, ss);
        ss = fma((double)b, (double)b, ss);
        if (n == 3) {
            xr[i + 2] = c;
            xs[ly_at(i + 2)] = c * nw.w[k][2];
            ss = fma((double)c, (double)c, ss);
        }
    });
    return ss;
}
__device__ __forceinline__ void ly_store(u32x4 *p, unsigned tag, float a, float b, float c, int lane) {
    const u32x4 v = {tag, __float_as_uint(a), __float_as_uint(b), __float_as_uint(c)};
    __builtin_amdgcn_raw_buffer_store_b128(v, ly_rsrc(p, 16u * 64u), lane * 16, 0, 16 /* sc1: written through */);
}
// The records of a head, two splits to a load (N2 loads), merged by one wavefront and published as its output
template <int N2>
__device__ __forceinline__ void ly_merge_head(const u32x4 *rec, u32x4 *out, int nch, unsigned tag, LyPoll &Q, int lane) {
    const __amdgpu_buffer_rsrc_t r = ly_rsrc(rec, (unsigned)(nch * LY_REC) * 16u);
    const int half = lane >> 5, gj = min(lane & 31, LY_REC - 1), n2 = (nch + 1) / 2;
    u32x4 g[N2];
    for (int spins = 0;;) {
        bool ok = true;
#pragma unroll
        for (int k = 0; k < N2; k++) g[k] = ly_granule(r, (unsigned)(min(2 * k + half, nch - 1) * LY_REC + gj));        // (past the last split: it again)
#pragma unroll
        for (int k = 0; k < N2; k++) ok = ok && g[k].x == tag;
        if (__all(ok) || !ly_again(Q, spins, 64u, lane)) break;
    }
    float m[N2], M = -INFINITY;                                          // m: of the lane's half
#pragma unroll
    for (int k = 0; k < N2; k++) {
        const float ma = k < n2 ? ly_lane(__uint_as_float(g[k].y), 0) : -INFINITY, mb = 2 * k + 1 < nch ? ly_lane(__uint_as_float(g[k].y), 32) : -INFINITY;
        M = fmaxf(M, fmaxf(ma, mb));
        m[k] = half ? mb : ma;
    }
    float o0 = 0.f, o1 = 0.f, o2 = 0.f;                                  // (lane 0's o1: the sum)
#pragma unroll
    for (int k = 0; k < N2; k++) {
        const float w = __expf(m[k] - M);                                // (weights of splits are this engine's own construct: nl_kernels.h, PRO_ATTN)
        o0 = fmaf(w, __uint_as_float(g[k].y), o0);
        o1 = fmaf(w, __uint_as_float(g[k].z), o1);
        o2 = fmaf(w, __uint_as_float(g[k].w), o2);
    }
    o0 += __shfl_xor(o0, 32); o1 += __shfl_xor(o1, 32); o2 += __shfl_xor(o2, 32);
    const float il = 1.0f / ly_lane(o1, 0);
    if (lane < LY_REC) ly_store(out, tag, o0 * il, o1 * il, o2 * il, lane);
}
// Level two of an all-gather.  256 workgroups that each read a whole vector past their L2 are 2.4 MB a look for 1536 values, and every look
// competes with the weights: 2.4 - 2.8 us an exchange.  So one workgroup of an XCD reads a 32nd of the vector from the fabric and stores it
// into the XCD's own L2, where all 32 of them find it (24.4 -> 22.6 us a layer; not for the heads' outputs, where the wait is for the
// slowest unit and the second hop costs what it saves: 21.8 with, 21.5 without).
// (a later layer's granules of the same step: nobody on this XCD has read the vector, or it could not have been written again.  Of the same step
// only: the counter is shared with the other plans, so what this launch left may be any number of steps old, and "ahead of the tag" by a signed
// difference is also what a granule of 2^23 to 2^24 steps ago looks like)
__device__ __forceinline__ void ly_relay(const u32x4 *src, u32x4 *dst, int ng, int slot, unsigned tag, LyPoll &Q, int lane) {
    const int per = (ng + LY_PER_XCD - 1) / LY_PER_XCD, i = slot * per + lane, n = min(per, ng - slot * per);
    if (n <= 0) return;
    const __amdgpu_buffer_rsrc_t r = ly_rsrc(src, (unsigned)ng * 16u), w = ly_rsrc(dst, (unsigned)ng * 16u);
    u32x4 g;
    for (int spins = 0;;) {
        g = ly_granule(r, (unsigned)min(i, slot * per + n - 1));
        if (__all(g.x >> 8 == tag >> 8 && g.x >= tag) || !ly_again(Q, spins, 1024u, lane)) break;
    }
    if (lane < n) __builtin_amdgcn_raw_buffer_store_b128(g, w, i * 16, 0, 0);
}
// the heads' outputs, by all wavefronts
__device__ __forceinline__ void ly_gather_o(const u32x4 *src, int H, unsigned tag, LyPoll &Q, float *xs2, int tid) {
    const int ng = H * LY_REC, lane = tid & 63;
    if ((tid & ~63) >= ng) return;
    const __amdgpu_buffer_rsrc_t r = ly_rsrc(src, (unsigned)ng * 16u);
    u32x4 g;
    for (int spins = 0;;) {
        g = ly_granule(r, (unsigned)min(tid, ng - 1));
        if (__all(g.x == tag) || !ly_again(Q, spins, 512u, lane)) break;
    }
    if (tid < ng) {
        const int h = (int)(((unsigned)tid * 2979u) >> 16), j = tid - h * LY_REC;      // tid / 22
        float *o = xs2 + h * XS_PAIR + 3 * j;                            // (a head is a pair)
        if (j) { o[-2] = __uint_as_float(g.y); o[-1] = __uint_as_float(g.z); }
        o[0] = __uint_as_float(g.w);
    }
}
// h, by all wavefronts
__device__ __forceinline__ void ly_gather_h(const u32x4 *src, int ntile, unsigned tag, LyPoll &Q, float *xs2, int tid) {
    ly_gather<16, 2, LY_THREADS>(src, ntile * GPT, tag, Q, 256u, tid, [&](int, int i, float a, float b, float c, int n) __attribute__((always_inline)) {
        xs2[ly_at(i)] = a;
        if (n == 3) { xs2[ly_at(i + 1)] = b; xs2[ly_at(i + 2)] = c; }
    });
}
__device__ __forceinline__ float ly_inv_rms(const double *dred, int D, float eps) {
    double tot = 0.0;
#pragma unroll
    for (int w = 0; w < LY_GW; w++) tot += dred[w];
    const double m = tot / (double)D + (double)eps;
    double y = __builtin_amdgcn_rsq(m);                     // (v_rsq_f64 and two Newton steps: exact before the rounding to float32)
    y = y * fma(-0.5 * m * y, y, 1.5);
    y = y * fma(-0.5 * m * y, y, 1.5);
    return (float)y;
}
// sums of n shares' partials of row lane % 16, or of n <= 8 shares' of row lane % 8, in every lane
__device__ __forceinline__ float ly_row_sum(const float *red, int n, int lane) {
    float v = 0.f;
    for (int g = lane >> 4; g < n; g += 4) v += red[g * TR + (lane & 15)];
    return mf_rows4_sum(v);
}
__device__ __forceinline__ float ly_half_sum(const float *red, int n, int lane) {
    float v = lane >> 3 < n ? red[lane] : 0.f;
    v += dpp_f32<0x128 /* row_ror:8 */>(v);
    return mf_rows4_sum(v);
}
// a wavefront whose lanes hold value lane % R of a record publishes it
template <int R>
__device__ __forceinline__ void ly_publish(u32x4 *rec, unsigned tag, float v, int lane) {
    constexpr int G = (R + 2) / 3;
    const int j = min(lane, G - 1);
    const float a = __shfl(v, 3 * j), b = __shfl(v, min(3 * j + 1, R - 1)), c = __shfl(v, min(3 * j + 2, R - 1));
    if (lane < G) ly_store(rec, tag, a, b, c, lane);
}

template <int WT>
__global__ void __launch_bounds__(LY_THREADS) layers_kernel(LayersParams P0) {
    // (arguments are read again every layer through an opaque pointer: kept in scalar registers across the loop, with all that follows from
    //  them, they and their derivatives were 270 values spilled into vector lanes; 66 still are with Q8_0 and Q6_K weights, 78 with Q4_0 and Q4_K)
    typedef const __attribute__((address_space(4))) LayersParams *Args;
    Args pk = (Args)__builtin_amdgcn_kernarg_segment_ptr();
#define P (*pk)
    __shared__ __attribute__((aligned(16))) double dred[LY_GW];
    __shared__ __attribute__((aligned(16))) float xs[LY_MAX_COLS / PAIR * XS_PAIR];      // the norms' x * g
    __shared__ __attribute__((aligned(16))) float xs2[LY_MAX_FF / PAIR * XS_PAIR];       // the heads' outputs; h
    __shared__ __attribute__((aligned(16))) float xr[LY_MAX_COLS];                       // the residual stream
    __shared__ __attribute__((aligned(16))) float red[2 * LY_CW * TR];                   // partial sums
    __shared__ __attribute__((aligned(16))) float qs[(LY_MAX_HPU + 2) * 64];             // q of the unit's heads; k, v of the position
    __shared__ __attribute__((aligned(16))) float wpart[LY_MAX_HPU * LY_CW * 68];        // (max, sum, -, -, sum p v) a head and wavefront
    __shared__ __attribute__((aligned(16))) uint2 tab[LY_MAX_LAYERS * LY_ENTRY];
    __shared__ int lds_dead, lds_slot;
    float *const kcur = qs + LY_MAX_HPU * 64, *const vcur = kcur + 64;

    int wg = blockIdx.x;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane0 = tid & 63;
    int lane = lane0;
    unsigned xcd;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcd));
    xcd &= LY_XCDS - 1;
    if (tid == 0) {
        lds_dead = 0;
        lds_slot = (int)(atomicAdd(P.tickets + xcd * (LY_LINE * 4), 1u) % LY_PER_XCD);      // (32 of a launch have the 32 places, wherever the count stands)
    }
    for (int i = tid; i < P.L * LY_ENTRY; i += LY_THREADS) tab[i] = reinterpret_cast<const uint2 *>(P.layers)[i];
    const int pos = sload_i32(P.ctl + CTL_POS), strm = sload_i32(P.ctl + CTL_STREAM);
    const unsigned tag0 = (unsigned)sload_i32(reinterpret_cast<const int *>(P.tick)) << 8;
    const long long soff = P.single_stream ? 0 : (long long)strm * P.kv_stream_stride;

    // this workgroup's unit
    const int nch = pos / LY_PASS + 1;
    int hpu = 1, nhg = P.gqa;                                            // heads of a unit, units of a (kv head, pass)
    while (P.KV * nch * nhg > (int)gridDim.x && hpu < LY_MAX_HPU) { hpu *= 2; nhg = (P.gqa + hpu - 1) / hpu; }
    const bool unit = wg < P.KV * nch * nhg;
    const int ukv = wg % P.KV, urest = wg / P.KV, usplit = unit ? urest % nch : 0, uhg = unit ? urest / nch : 0;
    const int uh0 = ukv * P.gqa + uhg * hpu, unh = min(hpu, P.gqa - uhg * hpu);
    const int t0 = usplit * LY_PASS, un = min(LY_PASS, pos + 1 - t0);     // its first position, its positions
    const bool uown = unit && usplit == nch - 1;                         // it sees the step's own position
    LyPoll Q{P.status, P.host_status, &lds_dead, P.spin_limit, __builtin_amdgcn_readfirstlane((int)__hip_atomic_load(P.status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0};
#define LY_AGAIN() do { pk = (Args)__builtin_amdgcn_kernarg_segment_ptr(); wg = blockIdx.x; lane = lane0; asm volatile("" : "+s"(pk), "+s"(wg), "+v"(lane)); } while (0)
    // this workgroup's tiles; 256- and 512-column shares of a row
#define LY_Q (wg < P.t_qkv)
#define LY_D (wg < 2 * P.t_d)
#define LY_I (wg < P.t_i)
    // the XCD's copies of the vectors
#define LY_LOC (P.loc + (size_t)xcd * P.loc_n)
#define LY_NGD (P.t_d * 2 * LY_HG)
#define LY_NGI (P.t_i * GPT)
#define LY_ND ((P.np_d + KL - 1) / KL)
#define LY_NO ((P.np_o + 2 * KL - 1) / (2 * KL))
#define LY_NI ((P.np_i + 2 * KL - 1) / (2 * KL))

    if (wave < LY_CW) {
        // ================================================ products ================================================
        // wavefront w: share w of Q|K|V, WO and down; w and w + 8 of those of gate and, behind them, of up
        auto load_q = [&](int l, LyUnit<WT> &u) __attribute__((always_inline)) {
            const int ll = min(l, P.L - 1);
            ly_load<WT, false>(u, ly_ptr<uint8_t>(tab, ll, LY_QP), ly_ptr<uint32_t>(tab, ll, LY_SP), min(wg, P.t_qkv - 1), 0, wave, P.np_d, l < P.L && LY_Q && wave < LY_ND, lane);
        };
        auto load_o = [&](int l, LyUnit<WT> &u) __attribute__((always_inline)) {
            const int ll = min(l, P.L - 1);
            ly_load<WT, true>(u, ly_ptr<uint8_t>(tab, ll, LY_QP + 1), ly_ptr<uint32_t>(tab, ll, LY_SP + 1), min(wg >> 1, P.t_d - 1), (wg & 1) * 8, wave, P.np_o, l < P.L && LY_D && wave < LY_NO, lane);
        };
        auto load_g = [&](int l, int g, LyUnit<WT> &u) __attribute__((always_inline)) {
            const int ll = min(l, P.L - 1);
            const int m = g >= LY_ND;
            ly_load<WT, false>(u, ly_ptr<uint8_t>(tab, ll, LY_QP + 2 + m), ly_ptr<uint32_t>(tab, ll, LY_SP + 2 + m), min(wg, P.t_i - 1), 0, g - m * LY_ND, P.np_d, LY_I && g < 2 * LY_ND, lane);
        };
        auto load_d = [&](int l, LyUnit<WT> &u) __attribute__((always_inline)) {
            const int ll = min(l, P.L - 1);
            ly_load<WT, true>(u, ly_ptr<uint8_t>(tab, ll, LY_QP + 4), ly_ptr<uint32_t>(tab, ll, LY_SP + 4), min(wg >> 1, P.t_d - 1), (wg & 1) * 8, wave, P.np_i, LY_D && wave < LY_NI, lane);
        };
        LyUnit<WT> A[2], B, C;
        float4 kreg[4], vreg[4];
        // cache rows of the unit, sixteen a wavefront.  K: lane = (row, 16 values), V: lane = (row group, 4 values); rows past the position repeat it
        auto load_kv = [&](int l) __attribute__((always_inline)) {
            const size_t base = (size_t)l * P.kv_layer_stride + soff + ((size_t)ukv * P.seq_len + t0) * 64;
            const unsigned bytes = unit && l < P.L ? (unsigned)un * 256u : 0u;
            const __amdgpu_buffer_rsrc_t rk = ly_rsrc(P.kcache + base, bytes), rv = ly_rsrc(P.vcache + base, bytes);
            const int krow = min(wave * 16 + (lane >> 2), un - 1);
#pragma unroll
            for (int k = 0; k < 4; k++) {
                kreg[k] = __builtin_bit_cast(float4, (u32x4)__builtin_amdgcn_raw_buffer_load_b128(rk, krow * 256 + (lane & 3) * 64 + k * 16, 0, 0));
                vreg[k] = __builtin_bit_cast(float4, (u32x4)__builtin_amdgcn_raw_buffer_load_b128(rv, min(wave * 16 + (lane >> 4) + 4 * k, un - 1) * 256 + (lane & 15) * 16, 0, 0));
            }
        };
        load_kv(0);
        __syncthreads();
        load_q(0, A[0]);
        load_o(0, C);
#pragma unroll 1
        for (int l = 0; l < P.L; l++) {
            const unsigned tag = tag0 | (unsigned)(l + 1);
            // ---- 1: Q | K | V ----
            ly_barrier();
            if (__builtin_amdgcn_readfirstlane(lds_dead)) return;
            if (LY_Q && wave < LY_ND) ly_dot<WT, false>(A[0], xs, wave, P.np_d, red + wave * TR, lane);
            ly_barrier();
            LY_AGAIN();
            load_g(l, wave, A[0]);
            load_g(l, wave + LY_CW, A[1]);
            // ---- 2: attention, sixteen positions a wavefront (nl_block.h's pass) ----
            ly_barrier();
            if (unit) {
                const int kq = lane & 3, vg = lane >> 4, vc = lane & 15, krow = wave * 16 + (lane >> 2);
                const bool kcurrow = t0 + krow == pos;
#pragma unroll 1
                for (int h = 0; h < unh; h++) {
                    const float *q = qs + h * 64;
                    float d0 = 0.f, d1 = 0.f, d2 = 0.f, d3 = 0.f;
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const float4 q4 = *reinterpret_cast<const float4 *>(q + kq * 16 + k * 4);
                        const float4 kc4 = *reinterpret_cast<const float4 *>(kcur + kq * 16 + k * 4);
                        const float4 k4 = kcurrow ? kc4 : kreg[k];
                        d0 = fmaf(q4.x, k4.x, d0); d1 = fmaf(q4.y, k4.y, d1); d2 = fmaf(q4.z, k4.z, d2); d3 = fmaf(q4.w, k4.w, d3);
                    }
                    const float sv = krow < un ? quad_sum((d0 + d1) + (d2 + d3)) * P.scale : -INFINITY;
                    const float mw = wave_max_f32(sv);
                    const float p = krow < un ? exp_f64_as_f32(sv - (mw == -INFINITY ? 0.f : mw)) : 0.f;
                    const float lw = wave_sum_f32(kq == 0 ? p : 0.f);
                    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
                    const float4 vc4 = *reinterpret_cast<const float4 *>(vcur + vc * 4);
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const float pw = __shfl(p, (vg + 4 * k) * 4);
                        const bool vcurrow = t0 + wave * 16 + vg + 4 * k >= pos;        // (its own row and those past it, whose p is 0: what lies there may not be finite)
                        const float4 v4 = vcurrow ? vc4 : vreg[k];
                        o.x = fmaf(pw, v4.x, o.x); o.y = fmaf(pw, v4.y, o.y); o.z = fmaf(pw, v4.z, o.z); o.w = fmaf(pw, v4.w, o.w);
                    }
                    o.x = mf_rows4_sum(o.x); o.y = mf_rows4_sum(o.y); o.z = mf_rows4_sum(o.z); o.w = mf_rows4_sum(o.w);
                    float *wp = wpart + (h * LY_CW + wave) * 68;
                    if (lane < 16) *reinterpret_cast<float4 *>(wp + 4 + vc * 4) = o;
                    if (lane == 0) { wp[0] = mw; wp[1] = lw; }
                }
            }
            ly_barrier();
            // ---- 3: WO ----
            if (LY_D) ly_gather_o(P.go, P.H, tag, Q, xs2, tid);
            ly_barrier();
            if (LY_D && wave < LY_NO) ly_dot<WT, true>(C, xs2, wave, P.np_o, red + wave * 8, lane);
            ly_barrier();
            LY_AGAIN();
            load_d(l, B);
            load_o(l + 1, C);
            // ---- 4: gate and up ----
            ly_barrier();
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int g = wave + i * LY_CW;
                if (LY_I && g < 2 * LY_ND) ly_dot<WT, false>(A[i], xs, g >= LY_ND ? g - LY_ND : g, P.np_d, red + g * TR, lane);
            }
            ly_barrier();
            LY_AGAIN();
            load_q(l + 1, A[0]);
            // ---- 5: down ----
            if (LY_D) ly_gather_h(LY_LOC + LY_NGD, P.t_i, tag, Q, xs2, tid);
            ly_barrier();
            if (LY_D && wave < LY_NI) ly_dot<WT, true>(B, xs2, wave, P.np_i, red + wave * 8, lane);
            ly_barrier();
            LY_AGAIN();
            load_kv(l + 1);
        }
    } else {
        // ================================================ exchange ================================================
        const int gw = wave - LY_CW, gt = tid - LY_CW * 64;
        __syncthreads();
        const int slot = __builtin_amdgcn_readfirstlane(lds_slot);
        // rotation of this workgroup's Q | K | V rows: rows 0-7 of a tile hold elements i, rows 8-15 elements i + 32 (ROWMAP_HEADPERM)
        const int row = lane0 & 15, qhead = min(wg, P.t_qkv - 1) >> 2, qi = (wg & 3) * 8 + (row & 7), qe = qi + (row >> 3) * 32;
        const int qsect = qhead < P.H ? 0 : qhead < P.H + P.KV ? 1 : 2;
        const float ec = P.rope_cos[(long long)pos * 32 + qi], es = P.rope_sin[(long long)pos * 32 + qi];
        LyNorm nw;
#pragma unroll 1
        for (int l = 0; l < P.L; l++) {
            LY_AGAIN();
            const unsigned tag = tag0 | (unsigned)(l + 1);
            // ---- 1 ----
            if (gw == LY_RELAY && l) ly_relay(P.gx, LY_LOC + LY_NGD + LY_NGI, LY_NGD, slot, tag - 1u, Q, lane);
            if (LY_Q || LY_D) {
                double ss = 0.0;
                if (l == 0) {
                    for (int i = gt; i < P.D; i += LY_GT) {
                        const float v = P.x[i];
                        xr[i] = v;
                        xs[ly_at(i)] = v * ly_ptr<float>(tab, l, LY_NORM)[i];
                        ss = fma((double)v, (double)v, ss);
                    }
                } else ss = ly_gather_norm(LY_LOC + LY_NGD + LY_NGI, LY_NGD, tag - 1u, Q, 16u, gt, nw, xr, xs);
                ss = wave_sum_f64(ss);
                if (lane == 0) dred[gw] = ss;
            }
            ly_barrier();
            if (__builtin_amdgcn_readfirstlane(lds_dead)) return;
            float inv = 0.f, bias = 0.f;
            if (gw == 0 && LY_Q) {
                inv = ly_inv_rms(dred, P.D, P.eps);
                if (const float *b = ly_ptr<float>(tab, l, LY_BQ + qsect)) bias = b[(qhead - (qsect == 0 ? 0 : qsect == 1 ? P.H : P.H + P.KV)) * 64 + qe];
            }
            ly_barrier();
            if (gw == 0 && LY_Q) {
                const float v = ly_row_sum(red, LY_ND, lane) * inv + bias, other = dpp_f32<0x128 /* row_ror:8 */>(v);
                const float x0 = row < 8 ? v : other, x1 = row < 8 ? other : v;
                float o = v;
                if (qsect < 2) {
                    if (!P.rope_conj) o = row < 8 ? x0 * ec - x1 * es : x0 * es + x1 * ec;
                    else o = row < 8 ? x0 * ec + x1 * es : -x0 * es + x1 * ec;
                }
                ly_publish<16>(P.gq + (size_t)wg * GPT, tag, o, lane);
            }
            LY_AGAIN();
            // ---- 2: q of the unit's heads, and k, v of the position where the unit sees it: 24 granules each ----
            if (unit) {
                const int nrec = unh + (uown ? 2 : 0), rec = gt / 24, w = gt - rec * 24, ng = nrec * 24;
                if ((gt & ~63) < ng) {
                    const int rc = min(rec, nrec - 1);
                    const int head = rc < unh ? uh0 + rc : rc == unh ? P.H + ukv : P.H + P.KV + ukv;
                    const __amdgpu_buffer_rsrc_t r = ly_rsrc(P.gq, (unsigned)P.t_qkv * (GPT * 16u));
                    u32x4 g;
                    for (int spins = 0;;) {
                        g = ly_granule(r, (unsigned)(head * 24 + w));
                        if (__all(g.x == tag) || !ly_again(Q, spins, 32u, lane)) break;
                    }
                    if (gt < ng) {
                        const int t = w / GPT, r3 = 3 * (w - t * GPT);
                        float *dst = rc < unh ? qs + rc * 64 : rc == unh ? kcur : vcur;
                        const float v[3] = {__uint_as_float(g.y), __uint_as_float(g.z), __uint_as_float(g.w)};
#pragma unroll
                        for (int c = 0; c < 3; c++)
                            if (r3 + c < 16) dst[t * 8 + ((r3 + c) & 7) + ((r3 + c) >> 3) * 32] = v[c];
                    }
                }
            }
            ly_barrier();
            if (uown && uhg == 0 && gt < 128)                            // KV store (go/model.go:552-554)
                (gt < 64 ? P.kcache : P.vcache)[(size_t)l * P.kv_layer_stride + soff + ((size_t)ukv * P.seq_len + pos) * 64 + (gt & 63)] = kcur[gt];
            ly_barrier();
            if (unit)
                for (int h = gw; h < unh; h += LY_GW) {
                    // the eight wavefronts' pieces merged, in order
                    const float *wp = wpart + h * LY_CW * 68;
                    const float mwv = lane < 8 ? wp[min(lane, 7) * 68] : -INFINITY;
                    const float M = wave_max_f32(mwv);
                    const float wgt = lane < 8 && mwv != -INFINITY ? __expf(mwv - M) : 0.f;
                    const float Ls = wave_sum_f32(lane < 8 ? wgt * wp[min(lane, 7) * 68 + 1] : 0.f);
                    float ov = 0.f;
#pragma unroll
                    for (int w = 0; w < LY_CW; w++) ov = fmaf(ly_lane(wgt, w), wp[w * 68 + 4 + lane], ov);
                    // a head's only record is its output
                    const int j = min(lane, LY_REC - 1), hh = uh0 + h;
                    if (nch == 1) ov *= 1.0f / Ls;
                    const float a = __shfl(ov, max(3 * j - 2, 0)), b = __shfl(ov, max(3 * j - 1, 0)), c = __shfl(ov, 3 * j);
                    if (lane < LY_REC)
                        ly_store(nch == 1 ? P.go + (size_t)hh * LY_REC : P.gr + ((size_t)hh * P.rec_max + usplit) * LY_REC, tag, j ? a : M, j ? b : Ls, c, lane);
                }
            if (uown && nch > 1)
                for (int h = gw; h < unh; h += LY_GW) {
                    const u32x4 *rec = P.gr + (size_t)(uh0 + h) * P.rec_max * LY_REC;
                    u32x4 *out = P.go + (size_t)(uh0 + h) * LY_REC;
                    if (nch <= 4) ly_merge_head<2>(rec, out, nch, tag, Q, lane);
                    else ly_merge_head<LY_MAX_REC / 2>(rec, out, nch, tag, Q, lane);
                }
            LY_AGAIN();
            // ---- 3 ----
            if (LY_D) ly_gather_o(P.go, P.H, tag, Q, xs2, tid);
            ly_barrier();
            ly_norm_weights(nw, ly_ptr<float>(tab, l, LY_NORM + 1), LY_NGD, gt);       // (ahead of the polls, which would wait for it)
            float bo = 0.f;
            if (gw == 0 && LY_D)
                if (const float *b = ly_ptr<float>(tab, l, LY_BO)) bo = b[wg * 8 + (lane & 7)];
            ly_barrier();
            if (gw == 0 && LY_D) ly_publish<8>(P.gp + (size_t)wg * LY_HG, tag, xr[wg * 8 + (lane & 7)] + (ly_half_sum(red, LY_NO, lane) + bo), lane);
            LY_AGAIN();
            // ---- 4 ----
            if (gw == LY_RELAY) ly_relay(P.gp, LY_LOC, LY_NGD, slot, tag, Q, lane);
            if (LY_I || LY_D) {
                const double ss = wave_sum_f64(ly_gather_norm(LY_LOC, LY_NGD, tag, Q, 128u, gt, nw, xr, xs));
                if (lane == 0) dred[gw] = ss;
            }
            ly_barrier();
            if (gw == 0 && LY_I) inv = ly_inv_rms(dred, P.D, P.eps);
            ly_barrier();
            if (gw == 0 && LY_I) {
                // lanes 0 - 31: gate, 32 - 63: up; every other share each
                float v = 0.f;
                for (int g = (lane >> 4) & 1; g < LY_ND; g += 2) v += red[(g + (lane >= 32 ? LY_ND : 0)) * TR + row];
                v += __shfl_xor(v, 16);
                const float g = v * inv, u = __shfl_xor(v, 32) * inv;
                ly_publish<16>(P.gh + (size_t)wg * GPT, tag, (g / (1.0f + exp_f64_as_f32(-g))) * u, lane);     // (lanes 0 - 15)
            }
            LY_AGAIN();
            // ---- 5 ----
            if (gw == LY_RELAY) ly_relay(P.gh, LY_LOC + LY_NGD, LY_NGI, slot, tag, Q, lane);
            if (LY_D) ly_gather_h(LY_LOC + LY_NGD, P.t_i, tag, Q, xs2, tid);
            ly_barrier();
            ly_norm_weights(nw, ly_ptr<float>(tab, min(l + 1, P.L - 1), LY_NORM), LY_NGD, gt);
            ly_barrier();
            if (gw == 0 && LY_D) {
                const float v = xr[wg * 8 + (lane & 7)] + ly_half_sum(red, LY_NI, lane);
                if (l + 1 < P.L) ly_publish<8>(P.gx + (size_t)wg * LY_HG, tag, v, lane);
                else if (lane < 8) P.x[wg * 8 + lane] = v;
            }
        }
    }
#undef P
#undef LY_AGAIN
#undef LY_Q
#undef LY_D
#undef LY_I
#undef LY_LOC
#undef LY_NGD
#undef LY_NGI
#undef LY_ND
#undef LY_NO
#undef LY_NI
}

// records of a head
inline int layers_records(int seq_len) { return std::min((seq_len + LY_PASS - 1) / LY_PASS, LY_MAX_REC); }

inline hipError_t launch_layers(int wtype, const LayersParams &P, int grid, hipStream_t st) {
    switch (wtype) {
    case WT_Q8_0: hipLaunchKernelGGL(layers_kernel<WT_Q8_0>, dim3(grid), dim3(LY_THREADS), 0, st, P); break;
    case WT_Q4_0: hipLaunchKernelGGL(layers_kernel<WT_Q4_0>, dim3(grid), dim3(LY_THREADS), 0, st, P); break;
    case WT_Q4_K: hipLaunchKernelGGL(layers_kernel<WT_Q4_K>, dim3(grid), dim3(LY_THREADS), 0, st, P); break;
    case WT_Q6_K: hipLaunchKernelGGL(layers_kernel<WT_Q6_K>, dim3(grid), dim3(LY_THREADS), 0, st, P); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace nl
