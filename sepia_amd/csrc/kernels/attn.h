// attn.h -- the attention half of the GPU ABI (reference src/sepia_gpu.h:
// rel_project :209, banded_attn :226, rel_project_off :253): the dense
// relative-position projection and the banded, GQA, online-softmax
// attention of the reference's attn_forward_chunk (src/sepia.c:1203-1247).
//
// Banded attention runs on the matrix cores. A wave owns 16 rows, each a
// (token, query head) pair whose head uses the workgroup's kv head, and walks
// kv positions in steps of 16 columns:
//   scores  q . k by v_mfma_f32_16x16x4_f32, the wave's q in registers;
//   softmax on the scores' registers: a row's 16 columns are 16 lanes, so
//           its maximum is four DPP steps, and each lane keeps its own part
//           of the row's sum until the end;
//   p . v   by v_mfma_f64_16x16x4_f64.
// Both contractions take their k index in an order that makes every operand
// a 16-byte read: lane group g of four takes k = 16 S + 4 g .. + 3 of each
// sixteen (head dims for the scores, kv rows for p . v) as the k index of
// four matrix ops. The rows of the f64 product are permuted so that register
// r of a lane is the same row in both products (scores: row 4 g + r; f64:
// row g + 4 r), and column j of f64 tile t is head dim 8 j + t, so a lane
// reads 8 consecutive floats of a v row for eight tiles.
//
// Precision follows the reference's CPU loop: scores are f32 dot products
// plus the band bias added in double and rounded once; each weight is
// exp(score - max) rounded to f32; the running sums of weights and of
// weighted v rows are double (f32 sums over 10^5 kv rows drift past the
// reference's 2e-4 relative gate, whose floor is 1e-3 of the largest
// output). The f64 matrix rate (79 TFLOP/s nominal, half the f32 one) is
// what bounds a long chunk of tokens.
//
// Two kernels share that wave:
//   sepia_attn_wave  few rows (a decode token): the waves of a workgroup
//                    take alternate kv steps of the same 16 rows, k and v go
//                    from global memory straight to the operand registers,
//                    and the waves' sums meet in LDS at the end;
//   sepia_attn_tile  many rows (a prefill chunk): four waves of 16 rows each
//                    share the k and v rows of a step through LDS.
// Long kv ranges are split over workgroups too; partials go to scratch and
// sepia_attn_combine folds them.
//
// Measured (64 heads of 128): one token over 20001 kv rows of 8 heads (164
// MB of k and v) 41.9 + 7.8 us, 3.9 TB/s, against 279 + 47 us for scalar
// loops that reduced each score over 16 lanes by shuffles; 500 tokens over
// 1500 + 500 rows 548 us, 105 TFLOP/s over both products, against 6.1 ms.
// Both kernels need two waves a SIMD: with 400 registers and one wave they
// took 68 and 877 us, with spills 98 and 605 us. At 4 tokens over 6004 rows
// (8 heads a kv head: 32 rows) the wave kernel takes 27.8 us, at 8 tokens the
// tile kernel 53 us.
#pragma once
#include "common.h"

#define ATT_RP_ROWS 8       // (t, h) rows per rel-project workgroup
#define ATT_RP_DCH 64       // d_rel columns staged per pass
#define ATT_TB 64           // tokens whose bounds travel in the kernel arguments
#define ATT_BB 256          // tokens per launch of sepia_attn_bounds
#define ATT_KC 32           // kv rows per step of sepia_attn_tile
#define ATT_KS 136          // floats of a staged k row (34 16-byte pieces, 2 mod 4: no bank conflicts)
#define ATT_VS 144          // floats of a staged v row (rows 4 apart differ by 16 banks)
#define ATT_PS 36           // floats of a staged row of weights

// rel_logits[th, r] = sum_d r_vec[th, d] * rel_proj[d, r], an f32 FMA chain
// in d order. Grid (ceil(R / 256), ceil(TH / ATT_RP_ROWS)), 256 threads:
// thread r of the tile computes ATT_RP_ROWS rows, so each rel_proj value is
// read once per workgroup.
extern "C" __global__ __launch_bounds__(256) void sepia_rel_project_f32(
    const float *__restrict__ r_vec, const float *__restrict__ rel_proj, float *__restrict__ rel_logits,
    int64_t TH, int32_t d_rel, int32_t R) {
    __shared__ float rv[ATT_RP_ROWS][ATT_RP_DCH];
    const int64_t th0 = (int64_t)blockIdx.y * ATT_RP_ROWS;
    const int nrow = (int)(TH - th0 < ATT_RP_ROWS ? TH - th0 : ATT_RP_ROWS);
    const int r = (int)blockIdx.x * 256 + (int)threadIdx.x;
    float acc[ATT_RP_ROWS];
#pragma unroll
    for (int i = 0; i < ATT_RP_ROWS; i++) acc[i] = 0.0f;
    for (int d0 = 0; d0 < d_rel; d0 += ATT_RP_DCH) {
        const int nd = d_rel - d0 < ATT_RP_DCH ? d_rel - d0 : ATT_RP_DCH;
        __syncthreads();
        for (int i = threadIdx.x; i < ATT_RP_ROWS * ATT_RP_DCH; i += 256) {
            const int row = i / ATT_RP_DCH, d = i % ATT_RP_DCH;
            rv[row][d] = (row < nrow && d < nd) ? r_vec[(th0 + row) * d_rel + d0 + d] : 0.0f;
        }
        __syncthreads();
        if (r < R) {
            for (int d = 0; d < nd; d++) {
                const float p = rel_proj[(int64_t)(d0 + d) * R + r];
#pragma unroll
                for (int i = 0; i < ATT_RP_ROWS; i++) acc[i] = __builtin_fmaf(rv[i][d], p, acc[i]);
            }
        }
    }
    if (r >= R) return;
#pragma unroll
    for (int i = 0; i < ATT_RP_ROWS; i++)
        if (i < nrow) rel_logits[(th0 + i) * R + r] = acc[i];
}

// Bounds of a batch's tokens: kv positions [lo, hi] (inclusive) and the bias
// scale of each. Up to ATT_TB tokens they are kernel arguments (the caller's
// host arrays need not outlive the call); more are first written to scratch
// as three arrays by sepia_attn_bounds, ATT_BB tokens a launch.
struct AttnTok {
    int32_t lo[ATT_TB], hi[ATT_TB];
    float tau[ATT_TB];
};
struct AttnTokB {
    int32_t lo[ATT_BB], hi[ATT_BB];
    float tau[ATT_BB];
};
extern "C" __global__ __launch_bounds__(ATT_BB) void sepia_attn_bounds(AttnTokB tok, int32_t n, int32_t t0, int32_t T,
                                                                       int32_t *__restrict__ dst) {
    const int i = (int)threadIdx.x;
    if (i >= n) return;
    dst[t0 + i] = tok.lo[i];
    dst[T + t0 + i] = tok.hi[i];
    dst[2 * T + t0 + i] = __builtin_bit_cast(int32_t, tok.tau[i]);
}

typedef float att_f4 __attribute__((ext_vector_type(4)));
typedef double att_d4 __attribute__((ext_vector_type(4)));

// What every attention launch is given. A workgroup's rows are consecutive
// (token, head of the group) pairs: row i of a tile that starts at token tb
// is token tb + i / G, head hk G + i % G.
struct AttnArgs {
    const float *q, *k, *v, *rel;
    const int32_t *gtok;    // bounds in scratch ([3][T]), NULL: in the kernel arguments
    float *out;
    double *part;           // split partials, NULL: one split, straight to out
    int64_t q_pos_base, kv_dim;
    int32_t T, H, Hkv, Dh, R, nsplit, span, TT;   // span: kv rows a split; TT: tokens a tile
    float inv_head_dim;
};

// The largest of a value over the 16 lanes of a DPP row; every lane gets it.
__device__ __forceinline__ float att_max16(float v) {
#define ATT_ROR(n)                                                                                            \
    v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 | n, \
                                                                       0xF, 0xF, false)))
    ATT_ROR(8);
    ATT_ROR(4);
    ATT_ROR(2);
    ATT_ROR(1);
#undef ATT_ROR
    return v;
}

// e^x for x <= 0 (or NaN) in double, within about 2^-51 of it: x = n ln 2 + r,
// |r| <= ln 2 / 2 (ln 2 as the sum of two doubles), e^r as 1 + r q(r) with q
// of degree 9 for the least largest relative error (Remez exchange; 2.3e-16 as
// rounded here) and an exact scaling by 2^n. Below -200 (an f32 zero since
// -104) n stops growing. The rounding to n adds 1.5 * 2^52, which leaves n in
// the sum's low word. Two fused multiply-adds fewer (a Taylor series to degree
// 9 and one ln 2) were 7e-12 off.
__device__ __forceinline__ double att_exp(float x) {
    const double xd = (double)(x < -200.0f ? -200.0f : x);
    const double big = 6755399441055744.0;
    const double t = __builtin_fma(xd, 1.4426950408889634074, big);
    const int n = (int)(uint32_t)__builtin_bit_cast(uint64_t, t);
    const double nd = t - big;
    const double r = __builtin_fma(nd, -2.3190468138462996e-17, __builtin_fma(nd, -0.69314718055994530942, xd));
    double p = 0x1.27315c7a1d3bep-22;
    p = __builtin_fma(p, r, 0x1.72f785aa9806cp-19);
    p = __builtin_fma(p, r, 0x1.a01b59c924b4cp-16);
    p = __builtin_fma(p, r, 0x1.a0197ca67eee6p-13);
    p = __builtin_fma(p, r, 0x1.6c16c0cdd2530p-10);
    p = __builtin_fma(p, r, 0x1.1111112c56a8dp-7);
    p = __builtin_fma(p, r, 0x1.555555558b631p-5);
    p = __builtin_fma(p, r, 0x1.555555554c5bfp-3);
    p = __builtin_fma(p, r, 0x1.ffffffffffe94p-2);
    p = __builtin_fma(p, r, 0x1.0000000000019p+0);
    p = __builtin_fma(p, r, 1.0);
    return __builtin_ldexp(p, n);
}

// A wave's 16 rows, in LDS: a lane reads the four entries of rows 4 g + r
// where it needs them (in registers they would cost 40 of the 256 that two
// workgroups a CU leave a wave).
struct AttnRows {
    int32_t lo[16], hi[16];   // kv bounds (lo > hi: no such row)
    int32_t klim[16];         // the row's band: kv > klim
    float tau[16];
    int64_t rel0[16];         // rel_logits element of kv: rel0 - kv
};
typedef int32_t att_i4 __attribute__((ext_vector_type(4)));
typedef int64_t att_l2 __attribute__((ext_vector_type(2)));

// One wave's state. Lane (j, g) = (lane & 15, lane >> 4) holds rows 4 g + r
// (r = 0..3) of the score columns j.
struct AttnWave {
    const AttnRows *rows;
    float m[4];              // running maximum
    double l[4];             // this lane's part of the running sum
    att_d4 acc[8];           // running weighted v: row 4 g + r, dim 8 j + t
    int32_t lo_min, lo_max, hi_min, hi_max;   // over the wave's rows (lo_min, hi_max: of the rows there are)

    // rows row0 .. row0 + 15 of the tile at token tb
    __device__ __forceinline__ void init(const AttnArgs &a, const AttnTok &tok, int tb, int row0, int hk, AttnRows *rw) {
        const int j = (int)(threadIdx.x & 15), G = a.H / a.Hkv;
        const int nt = a.T - tb < a.TT ? a.T - tb : a.TT;
        const int ti = (row0 + j) / G, h = hk * G + (row0 + j - ti * G), t = tb + ti;
        const bool on = ti < nt;
        // row j's entries (the four lane groups write the same)
        const int tl = on ? t : tb;
        const int32_t lo = on ? (a.gtok ? a.gtok[tl] : tok.lo[tl]) : 1, hi = on ? (a.gtok ? a.gtok[a.T + tl] : tok.hi[tl]) : 0;
        const int64_t qp = a.q_pos_base + tl, kl = qp - a.R;
        rw->lo[j] = lo;
        rw->hi[j] = hi;
        rw->klim[j] = kl < -1 ? -1 : kl > 0x7FFFFFFF ? 0x7FFFFFFF : (int32_t)kl;
        rw->tau[j] = a.gtok ? __builtin_bit_cast(float, a.gtok[2 * a.T + tl]) : tok.tau[tl];
        rw->rel0[j] = ((int64_t)tl * a.H + h) * a.R + qp;
        int lmin = on ? lo : 0x7FFFFFFF, lmax = lo, hmin = hi, hmax = on ? hi : -1;
#pragma unroll
        for (int o = 1; o <= 8; o <<= 1) {
            lmin = min(lmin, __shfl_xor(lmin, o, 16));
            lmax = max(lmax, __shfl_xor(lmax, o, 16));
            hmin = min(hmin, __shfl_xor(hmin, o, 16));
            hmax = max(hmax, __shfl_xor(hmax, o, 16));
        }
        lo_min = __builtin_amdgcn_readfirstlane(lmin);
        lo_max = __builtin_amdgcn_readfirstlane(lmax);
        hi_min = __builtin_amdgcn_readfirstlane(hmin);
        hi_max = __builtin_amdgcn_readfirstlane(hmax);
        rows = rw;
        reset();
        wave_sync();
    }
    __device__ __forceinline__ void reset() {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            m[r] = -INFINITY;
            l[r] = 0.0;
        }
#pragma unroll
        for (int t = 0; t < 8; t++) acc[t] = att_d4{0.0, 0.0, 0.0, 0.0};
    }
    // q of row j, dims 16 S + 4 g .. + 3 (zero past the rows and the head dim)
    template <bool FULL>
    static __device__ __forceinline__ void load_q(const AttnArgs &a, int tb, int row0, int hk, att_f4 *qa) {
        const int lane = (int)(threadIdx.x & 63), j = lane & 15, g = lane >> 4, G = a.H / a.Hkv;
        const int nt = a.T - tb < a.TT ? a.T - tb : a.TT;
        const int ti = (row0 + j) / G, h = hk * G + (row0 + j - ti * G);
        const bool on = ti < nt;
        const float *qr = a.q + ((int64_t)(tb + (on ? ti : 0)) * a.H + h) * a.Dh;
#pragma unroll
        for (int S = 0; S < 8; S++) {
            const int d = 16 * S + 4 * g;
            const att_f4 v = *(const att_f4 *)(qr + (FULL || d < a.Dh ? d : 0));
            qa[S] = on && (FULL || d < a.Dh) ? v : att_f4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
    // LDS written by this wave's lanes before is read by its lanes after
    static __device__ __forceinline__ void wave_sync() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    // the band's logits of kv columns c0 + j (outside the row's band: any)
    __device__ __forceinline__ att_f4 bias(const AttnArgs &a, int32_t c0) const {
        const int g = (int)(threadIdx.x & 63) >> 4;
        const int32_t kv = c0 + (int)(threadIdx.x & 15);
        const att_i4 lo = *(const att_i4 *)(rows->lo + 4 * g), hi = *(const att_i4 *)(rows->hi + 4 * g),
                     kl = *(const att_i4 *)(rows->klim + 4 * g);
        const att_l2 ra = *(const att_l2 *)(rows->rel0 + 4 * g), rb = *(const att_l2 *)(rows->rel0 + 4 * g + 2);
        att_f4 b;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const bool in = kv >= lo[r] && kv <= hi[r] && kv > kl[r];
            b[r] = a.rel[in ? (r < 2 ? ra[r & 1] : rb[r & 1]) - kv : 0];
        }
        return b;
    }
    // scores of a 16-column tile from its dots: (q . k) / head dim + bias
    __device__ __forceinline__ att_f4 score(const AttnArgs &a, att_f4 dot, att_f4 b, int32_t c0) const {
        const int g = (int)(threadIdx.x & 63) >> 4;
        const int32_t kv = c0 + (int)(threadIdx.x & 15);
        const att_i4 kl = *(const att_i4 *)(rows->klim + 4 * g);
        const att_f4 tau = *(const att_f4 *)(rows->tau + 4 * g);
        att_f4 s;
#pragma unroll
        for (int r = 0; r < 4; r++)
            s[r] = (float)((double)(dot[r] * a.inv_head_dim) + (kv > kl[r] ? (double)b[r] * (double)tau[r] : 0.0));
        return s;
    }
    // Running maximum over the NC tiles' scores; sums so far rescaled where
    // it grew; the weights to LDS (ps: 16 rows of ATT_PS floats, the wave's own).
    // A row whose scores so far are all -inf has that as its maximum and takes
    // its weights against 0 (they are 0, and NaN for a NaN): a later score may
    // be finite.
    template <int NC>
    __device__ __forceinline__ void weights(const att_f4 *s, int32_t c0, float *ps) {
        const int lane = (int)(threadIdx.x & 63), j = lane & 15, g = lane >> 4;
        const att_i4 lo = *(const att_i4 *)(rows->lo + 4 * g), hi = *(const att_i4 *)(rows->hi + 4 * g);
        float mn[4];
        bool grew = false;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            float mx = -INFINITY;
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const int32_t kv = c0 + 16 * c + j;
                if (kv >= lo[r] && kv <= hi[r]) mx = fmaxf(mx, s[c][r]);
            }
            mn[r] = fmaxf(m[r], att_max16(mx));
            grew |= mn[r] != m[r];
        }
        if (__ballot(grew)) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const double al = att_exp(mn[r] == m[r] ? 0.0f : m[r] - mn[r]);   // e^0 is 1 exactly
                l[r] *= al;
#pragma unroll
                for (int t = 0; t < 8; t++) acc[t][r] *= al;
                m[r] = mn[r];
            }
        }
        float mb[4];
#pragma unroll
        for (int r = 0; r < 4; r++) mb[r] = m[r] == -INFINITY ? 0.0f : m[r];
#pragma unroll
        for (int c = 0; c < NC; c++) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int32_t kv = c0 + 16 * c + j;
                const uint32_t in = kv >= lo[r] && kv <= hi[r] ? 0xFFFFFFFFu : 0u;
                const float p = __builtin_bit_cast(
                    float, __builtin_bit_cast(uint32_t, (float)att_exp(s[c][r] - mb[r])) & in);
                l[r] += (double)p;
                ps[(4 * g + r) * ATT_PS + 16 * c + j] = p;
            }
        }
        wave_sync();
    }
    // acc += p . v over kv rows 16 S + 4 g + i of a step; vrow(i) gives the 8
    // floats of that row at dims 8 j.
    template <class V>
    __device__ __forceinline__ void pv(const float *ps, int S, V vrow) {
        const int lane = (int)(threadIdx.x & 63), i16 = lane & 15, g = lane >> 4;
        const att_f4 pa = *(const att_f4 *)(ps + (4 * (i16 & 3) + (i16 >> 2)) * ATT_PS + 16 * S + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            att_f4 va, vb;
            vrow(i, va, vb);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 4; t++)
                acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)pa[i], (double)va[t], acc[t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < 4; t++)
                acc[4 + t] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)pa[i], (double)vb[t], acc[4 + t], 0, 0, 0);
        }
    }
    // The same product without the matrix cores, over each row's own kv rows
    // only: 0 * infinity in a matrix op would reach rows that do not see the
    // infinite v.
    __device__ __forceinline__ void pv_masked(const AttnArgs &a, const float *ps, const float *vh, int32_t c0, int n) {
        const int lane = (int)(threadIdx.x & 63), j = lane & 15, g = lane >> 4;
        const int da = 8 * j < a.Dh ? 8 * j : 0, db = 8 * j + 4 < a.Dh ? 8 * j + 4 : 0;
        const att_i4 lo = *(const att_i4 *)(rows->lo + 4 * g), hi = *(const att_i4 *)(rows->hi + 4 * g);
#pragma unroll 1
        for (int c = 0; c < n; c++) {
            const int32_t kv = c0 + c;
            if (kv < lo_min || kv > hi_max) continue;
            const float *vr = vh + (int64_t)kv * a.kv_dim;
            const att_f4 va = *(const att_f4 *)(vr + da), vb = *(const att_f4 *)(vr + db);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t in = kv >= lo[r] && kv <= hi[r] ? 0xFFFFFFFFu : 0u;
                const double p = (double)ps[(4 * g + r) * ATT_PS + c];   // 0 for a row that does not see kv
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    const float v = t < 4 ? va[t & 3] : vb[t & 3];
                    acc[t][r] = __builtin_fma(
                        p, (double)__builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) & in), acc[t][r]);
                }
            }
        }
    }
    // some row of the wave does not see every column of [c, c + n)
    __device__ __forceinline__ bool edge(int64_t c, int n) const { return c < lo_max || c + n - 1 > hi_min; }
    __device__ __forceinline__ void sum_lanes() {
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int o = 1; o <= 8; o <<= 1) l[r] += __shfl_xor(l[r], o, 16);
    }
    // Columns t0 .. t0 + n - 1 of the tiles (dims 8 j + t) of rows 4 g + r to
    // their outputs or to their split's partials: weighted v, then the
    // maximum and the sum. v(t, r), mm, ll: the values.
    template <int N, class V>
    static __device__ __forceinline__ void store(const AttnArgs &a, int tb, int row0, int hk, int x, int t0,
                                                 const float *mm, const double *ll, V v) {
        const int lane = (int)(threadIdx.x & 63), j = lane & 15, g = lane >> 4, G = a.H / a.Hkv;
        const int nt = a.T - tb < a.TT ? a.T - tb : a.TT;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = row0 + 4 * g + r, ti = row / G;
            if (ti >= nt) continue;
            const int64_t th = (int64_t)(tb + ti) * a.H + hk * G + (row - ti * G);
            if (a.part) {
                double *p = a.part + (th * a.nsplit + x) * (a.Dh + 2);
#pragma unroll
                for (int t = 0; t < N; t++)
                    if (8 * j + t0 + t < a.Dh) p[8 * j + t0 + t] = v(t, r);
                if (j == 0 && t0 == 0) {
                    p[a.Dh] = (double)mm[r];
                    p[a.Dh + 1] = ll[r];
                }
            } else {
                const double inv = 1.0 / ll[r];
                float *o = a.out + th * a.Dh;
#pragma unroll
                for (int t = 0; t < N; t++)
                    if (8 * j + t0 + t < a.Dh) o[8 * j + t0 + t] = (float)(v(t, r) * inv);
            }
        }
    }
};

// Scores' dots of NC column tiles, each as two chains of 64 products: qa(S)
// and kb(c, S) give q of row j and k of column j of tile c, dims 16 S + 4 g
// .. + 3. The scheduling barriers keep the reads a few at a time (all at
// once cost 32 registers a tile).
template <int NC, class Q, class K>
__device__ __forceinline__ void att_dots(Q qa, K kb, att_f4 *dot) {
    att_f4 s0[NC], s1[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) s0[c] = s1[c] = att_f4{0.0f, 0.0f, 0.0f, 0.0f};
    att_f4 kv[2][NC], qv[2];
    qv[0] = qa(0);
#pragma unroll
    for (int c = 0; c < NC; c++) kv[0][c] = kb(c, 0);
#pragma unroll
    for (int S = 0; S < 8; S++) {
        if (S + 1 < 8) {
            qv[(S + 1) & 1] = qa(S + 1);
#pragma unroll
            for (int c = 0; c < NC; c++) kv[(S + 1) & 1][c] = kb(c, S + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; i += 2)
#pragma unroll
            for (int c = 0; c < NC; c++) {
                s0[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[S & 1][i], kv[S & 1][c][i], s0[c], 0, 0, 0);
                s1[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[S & 1][i + 1], kv[S & 1][c][i + 1], s1[c], 0, 0, 0);
            }
    }
#pragma unroll
    for (int c = 0; c < NC; c++) dot[c] = s0[c] + s1[c];
}
// a NaN or an infinity among the four (each times zero is then a NaN)
__device__ __forceinline__ bool att_nonfinite(att_f4 v) {
    return !((v[0] * 0.0f + v[1] * 0.0f) + (v[2] * 0.0f + v[3] * 0.0f) == 0.0f);
}

template <bool B> struct AttBool { static constexpr bool value = B; };

// Few rows: workgroup (kv head x, tile y of TT tokens (TT G <= 16), split z),
// ATT_WV waves. Wave w walks the split's 16-column steps w, w + ATT_WV, ...;
// the next step's k loads are issued once this step's scores are formed and
// its v loads once its product is. q is read back from LDS for every step:
// in registers it does not fit beside the sums and the k and v in flight.
// The waves' sums meet in LDS, where each wave adds two of the eight tiles,
// in wave order. A wave that met a NaN or an infinity in the v rows of a step
// that not all its rows see walks its steps again with the masked product
// (here and not inside the loop, whose registers it would take). FULL: the
// head dim is 128.
#define ATT_WV 4
template <bool FULL>
__device__ __forceinline__ void attn_wave(const AttnArgs &a, const AttnTok &tok) {
    __shared__ __attribute__((aligned(16))) double xacc[ATT_WV][8][4][64];
    __shared__ double xl[ATT_WV][4][64];
    __shared__ float xm[ATT_WV][4][64];
    __shared__ __attribute__((aligned(16))) AttnRows rw[ATT_WV];
    static_assert(sizeof(float) * (16 * ATT_KS + ATT_WV * 16 * ATT_PS) <= sizeof xacc, "q and the weights share xacc");
    const int lane = (int)(threadIdx.x & 63), j = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int hk = (int)blockIdx.x, tb = (int)blockIdx.y * a.TT, x = (int)blockIdx.z;
    float *qs = (float *)xacc, *ps = qs + 16 * ATT_KS + w * 16 * ATT_PS;
    AttnWave W;
    W.init(a, tok, tb, 0, hk, &rw[w]);
    if (w == 0) {
        att_f4 qa[8];
        AttnWave::load_q<FULL>(a, tb, 0, hk, qa);
#pragma unroll
        for (int S = 0; S < 8; S++) *(att_f4 *)(qs + j * ATT_KS + 16 * S + 4 * g) = qa[S];
    }
    const int64_t s0 = (int64_t)W.lo_min + (int64_t)x * a.span;
    const int32_t last = (int32_t)(W.hi_max < s0 + a.span - 1 ? W.hi_max : s0 + a.span - 1);
    const float *kh = a.k + (int64_t)hk * a.Dh, *vh = a.v + (int64_t)hk * a.Dh;
    att_f4 kb[8], vb[4][2];
    const att_f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    auto load_k = [&](int64_t c0) {
        const int64_t kv = c0 + j < last ? c0 + j : last;
        const float *kr = kh + kv * a.kv_dim + 4 * g;
#pragma unroll
        for (int S = 0; S < 8; S++) kb[S] = *(const att_f4 *)(kr + (FULL || 16 * S + 4 * g < a.Dh ? 16 * S : -4 * g));
    };
    auto load_v = [&](int64_t c0) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int64_t kv = c0 + 4 * g + i < last ? c0 + 4 * g + i : last;
            const float *vr = vh + kv * a.kv_dim + (FULL || 8 * j < a.Dh ? 8 * j : 0);
            vb[i][0] = *(const att_f4 *)vr;
            vb[i][1] = *(const att_f4 *)(vr + (FULL || 8 * j + 4 < a.Dh ? 4 : 0));
        }
    };
    auto walk = [&](auto masked) {
        bool bad = false;
        int64_t c = s0 + 16 * w;
        if (c <= last) {
            load_k(c);
            load_v(c);
        }
        for (; c <= last; c += 16 * ATT_WV) {
            const int32_t c0 = (int32_t)c;
            const att_f4 b = W.bias(a, c0);
            att_f4 dot;
            att_dots<1>([&](int S) { return *(const att_f4 *)(qs + j * ATT_KS + 16 * S + 4 * g); },
                        [&](int, int S) { return FULL || 16 * S + 4 * g < a.Dh ? kb[S] : zero; }, &dot);
            const int64_t cn = c + 16 * ATT_WV;
            if (cn <= last) load_k(cn);
            const att_f4 s = W.score(a, dot, b, c0);
            W.weights<1>(&s, c0, ps);
            if constexpr (decltype(masked)::value) {
                W.pv_masked(a, ps, vh, c0, 16);
            } else {
                if (W.edge(c, 16)) {
#pragma unroll
                    for (int i = 0; i < 4; i++) bad = bad || att_nonfinite(vb[i][0]) || att_nonfinite(vb[i][1]);
                }
                W.pv(ps, 0, [&](int i, att_f4 &va, att_f4 &vc) {
                    va = vb[i][0];
                    vc = vb[i][1];
                });
                if (cn <= last) load_v(cn);
            }
        }
        return __ballot(bad) != 0;
    };
    __syncthreads();   // q is staged
    if (walk(AttBool<false>{})) {
        W.reset();
        walk(AttBool<true>{});
    }
    W.sum_lanes();
    float M[4];
#pragma unroll
    for (int r = 0; r < 4; r++) xm[w][r][lane] = W.m[r];
    __syncthreads();   // and every wave is done with q and its weights
#pragma unroll
    for (int r = 0; r < 4; r++) {
        M[r] = xm[0][r][lane];
#pragma unroll
        for (int o = 1; o < ATT_WV; o++) M[r] = fmaxf(M[r], xm[o][r][lane]);
        const double e = att_exp(W.m[r] == M[r] ? 0.0f : W.m[r] - M[r]);
        xl[w][r][lane] = W.l[r] * e;
#pragma unroll
        for (int t = 0; t < 8; t++) xacc[w][t][r][lane] = W.acc[t][r] * e;
    }
    __syncthreads();
    double L[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        L[r] = xl[0][r][lane];
#pragma unroll
        for (int o = 1; o < ATT_WV; o++) L[r] += xl[o][r][lane];
    }
    AttnWave::store<2>(a, tb, 0, hk, x, 2 * w, M, L, [&](int t, int r) {
        double v = xacc[0][2 * w + t][r][lane];
#pragma unroll
        for (int o = 1; o < ATT_WV; o++) v += xacc[o][2 * w + t][r][lane];
        return v;
    });
}
extern "C" __global__ __launch_bounds__(64 * ATT_WV, 2) void sepia_attn_wave(AttnArgs a, AttnTok tok) {
    attn_wave<true>(a, tok);
}
extern "C" __global__ __launch_bounds__(64 * ATT_WV, 2) void sepia_attn_wave_d(AttnArgs a, AttnTok tok) {
    attn_wave<false>(a, tok);
}

// Many rows: workgroup (kv head x, tile y of TT tokens (TT G <= 64), split
// z), 4 waves of 16 rows. A step's ATT_KC k and v rows are staged in LDS for
// all four waves (each thread 4 16-byte pieces of either, the next step's in
// its registers while this one computes). kv heads are the fastest grid
// dimension: workgroup ids go to the 8 XCDs in turn, so an XCD's L2 keeps the
// k and v of its own heads. The last tiles, whose causal ranges are longest,
// start first.
template <bool FULL>
__device__ __forceinline__ void attn_tile(const AttnArgs &a, const AttnTok &tok) {
    __shared__ __attribute__((aligned(16))) float ks[ATT_KC * ATT_KS];
    __shared__ __attribute__((aligned(16))) float vs[ATT_KC * ATT_VS];
    __shared__ __attribute__((aligned(16))) float ps_all[4][16 * ATT_PS];
    __shared__ int32_t rng[2][4];
    const int tid = (int)threadIdx.x, lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hk = (int)blockIdx.x, tb = ((int)gridDim.y - 1 - (int)blockIdx.y) * a.TT, x = (int)blockIdx.z;
    float *ps = ps_all[w];
    __shared__ __attribute__((aligned(16))) AttnRows rw[4];
    AttnWave W;
    W.init(a, tok, tb, 16 * w, hk, &rw[w]);
    att_f4 qa[8];
    AttnWave::load_q<FULL>(a, tb, 16 * w, hk, qa);
    if (lane == 0) {
        rng[0][w] = W.lo_min;
        rng[1][w] = W.hi_max;
    }
    __syncthreads();
    const int32_t t_lo = min(min(rng[0][0], rng[0][1]), min(rng[0][2], rng[0][3]));
    const int32_t t_hi = max(max(rng[1][0], rng[1][1]), max(rng[1][2], rng[1][3]));
    const int64_t s0 = (int64_t)t_lo + (int64_t)x * a.span;
    const int32_t last = (int32_t)(t_hi < s0 + a.span - 1 ? t_hi : s0 + a.span - 1);
    const float *kh = a.k + (int64_t)hk * a.Dh, *vh = a.v + (int64_t)hk * a.Dh;
    const att_f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    att_f4 kn[4], vn[4];
    auto load = [&](int64_t c0) {   // piece p = tid + 256 i: row p / 32, floats 4 (p % 32) ..
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int p = tid + 256 * i, d = 4 * (p & 31);
            const int64_t kv = c0 + (p >> 5) < last ? c0 + (p >> 5) : last;
            const int64_t at = kv * a.kv_dim + (FULL || d < a.Dh ? d : 0);
            kn[i] = *(const att_f4 *)(kh + at);
            vn[i] = *(const att_f4 *)(vh + at);
        }
    };
    auto walk = [&](auto masked) {
        bool bad = false;
        if (s0 <= last) load(s0);
        for (int64_t c = s0; c <= last; c += ATT_KC) {
            const int32_t c0 = (int32_t)c;
            __syncthreads();   // the waves are done with the step before
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int p = tid + 256 * i;
                *(att_f4 *)(ks + (p >> 5) * ATT_KS + 4 * (p & 31)) = FULL || 4 * (p & 31) < a.Dh ? kn[i] : zero;
                *(att_f4 *)(vs + (p >> 5) * ATT_VS + 4 * (p & 31)) = vn[i];
            }
            __syncthreads();
            if (c + ATT_KC <= last) load(c + ATT_KC);
            if (c > W.hi_max || c + ATT_KC - 1 < W.lo_min) continue;   // nothing for this wave's rows
            att_f4 s[2], dot[2];
#pragma unroll
            for (int cc = 0; cc < 2; cc++) s[cc] = W.bias(a, c0 + 16 * cc);
            att_dots<2>([&](int S) { return qa[S]; },
                        [&](int cc, int S) { return *(const att_f4 *)(ks + (16 * cc + j) * ATT_KS + 16 * S + 4 * g); },
                        dot);
#pragma unroll
            for (int cc = 0; cc < 2; cc++) s[cc] = W.score(a, dot[cc], s[cc], c0 + 16 * cc);
            W.weights<2>(s, c0, ps);
            if constexpr (decltype(masked)::value) {
                W.pv_masked(a, ps, vh, c0, ATT_KC);
            } else {
                if (W.edge(c, ATT_KC)) {
                    for (int i = lane; i < ATT_KC * 32; i += 64)
                        bad = bad || att_nonfinite(*(const att_f4 *)(vs + (i >> 5) * ATT_VS + 4 * (i & 31)));
                }
#pragma unroll
                for (int S = 0; S < ATT_KC / 16; S++)
                    W.pv(ps, S, [&](int i, att_f4 &va, att_f4 &vb) {
                        const float *vr = vs + (16 * S + 4 * g + i) * ATT_VS + 8 * j;
                        va = *(const att_f4 *)vr;
                        vb = *(const att_f4 *)(vr + 4);
                    });
            }
        }
        return __syncthreads_or(bad) != 0;
    };
    if (walk(AttBool<false>{})) {   // as in attn_wave, for the four waves together
        W.reset();
        walk(AttBool<true>{});
    }
    W.sum_lanes();
    AttnWave::store<8>(a, tb, 16 * w, hk, x, 0, W.m, W.l, [&](int t, int r) { return W.acc[t][r]; });
}

extern "C" __global__ __launch_bounds__(256, 2) void sepia_attn_tile(AttnArgs a, AttnTok tok) { attn_tile<true>(a, tok); }
extern "C" __global__ __launch_bounds__(256, 2) void sepia_attn_tile_d(AttnArgs a, AttnTok tok) {
    attn_tile<false>(a, tok);
}

// Fold of token blockIdx.y, head blockIdx.x: its nsplit partials in split
// order, in double: out[t, h, d] = sum_x acc_x[d] e^(m_x - M) / sum_x l_x
// e^(m_x - M), rounded to f32. The threads first share the splits' factors
// (a split that had none of the token's rows has maximum -infinity and sum
// zero: factor 0), then each sums its dim, eight loads at a time.
#define ATT_FOLD 1024   // splits at most
extern "C" __global__ __launch_bounds__(128) void sepia_attn_combine(const double *__restrict__ part, int32_t H,
                                                                     int32_t Dh, int32_t nsplit,
                                                                     float *__restrict__ out) {
    __shared__ double f[ATT_FOLD], lx[ATT_FOLD];
    __shared__ float red[2];
    const int d = (int)threadIdx.x;
    const int64_t th = (int64_t)blockIdx.y * H + blockIdx.x;
    const double *pb = part + th * nsplit * (Dh + 2);
    float M = -INFINITY;
    for (int x = d; x < nsplit; x += 128) {
        const double *px = pb + (int64_t)x * (Dh + 2) + Dh;
        f[x] = px[0];
        lx[x] = px[1];
        M = fmaxf(M, (float)f[x]);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
    if ((d & 63) == 0) red[d >> 6] = M;
    __syncthreads();
    M = fmaxf(red[0], red[1]);
    for (int x = d; x < nsplit; x += 128) f[x] = f[x] == -INFINITY && lx[x] == 0.0 ? 0.0 : exp(f[x] - (double)M);
    __syncthreads();
    double L = 0.0, o = 0.0;
    int x = 0;
    for (; x + 8 <= nsplit; x += 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = d < Dh ? pb[(int64_t)(x + u) * (Dh + 2) + d] : 0.0;
#pragma unroll
        for (int u = 0; u < 8; u++) {
            L = __builtin_fma(lx[x + u], f[x + u], L);
            o = __builtin_fma(v[u], f[x + u], o);
        }
    }
    for (; x < nsplit; x++) {
        L = __builtin_fma(lx[x], f[x], L);
        o = __builtin_fma(d < Dh ? pb[(int64_t)x * (Dh + 2) + d] : 0.0, f[x], o);
    }
    if (d < Dh) out[th * Dh + d] = (float)(o / L);
}
