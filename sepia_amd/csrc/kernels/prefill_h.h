// prefill_h.h -- the prefill MoE projections on the f16 matrix cores: the
// batched layer of prefill.h with the same grouping and combine, for layers
// in the real checkpoint's formats (IQ2_XS, IQ3_XXS, IQ4_XS routed; Q5_K,
// Q6_K, Q8_0 shared) and for mixes of those with Q2_K, Q3_K and Q4_K.
//
// Activations (x per token for gate/up, h per pair for down) travel as "PH"
// rows: per row a power-of-two scale s with 2^15 s > max|v| (+inf when the
// row holds a NaN or an infinity, which then makes every output of the row
// non-finite), and per column v' = v / s (|v'| < 2^15, exact) as two f16
// planes, hi = f16(v') and lo = f16(v' - hi): together within 2^-23 |v'| (two
// roundings) or 2^-25 (lo's, among the f16 subnormals), which is at most
// 2^-39 of the row's largest: beside an outlier 10^4 times the rest, the rest
// keep their 22 bits (with |v'| < 1 the floor was 2^-24 of the outlier, and
// outputs that it does not reach were 2.6e-3 off).
// 128 columns of a row are a 576-byte record: hi (128 f16, column order),
// lo (128 f16), then four 16-byte groups, one per 32 columns, for the min
// terms of Q2_K, Q4_K and Q5_K: the two 16-column sums of v', each / 16 (so
// that it fits f16) as three f16 (together exact, or within 2^-25), and two
// zeros.
//
// Weights enter v_mfma_f32_16x16x32_f16 as exact f16 integer codes, decoded
// from the raw blocks in registers (the products hi * code and lo * code are
// exact in f32; the matrix cores add them in f32). Per weight row n and
// 256-column block, with C the f32 dot of the codes with v' (x is the
// v' the record holds, w the weights of src/quants.c's dequant):
//   IQ2_XS   code = +-grid * (2 s + 1) * 2^-14, s the 4-bit scale of its
//            16 weights (|code| <= 43 * 31 * 2^-14),
//            sum w x = d C 2^14 / 8                     (quants.c:179-201)
//   IQ3_XXS  code = +-grid * (2 s + 1) * 2^-14, 4-bit s per 32 weights
//            (|code| <= 62 * 31 * 2^-14), sum w x = d C 2^14 / 4
//            (quants.c:203-226)
//   Q4_K     code = q * sc, 6-bit sc per 32 (<= 15 * 63); sum w x = d C -
//   Q5_K     dmin sum_j m_j S_j (Q5_K: code <= 31 * 63), the min terms as one
//            more matrix op: the records' sums against the mins, times 16
//            (quants.c:104-151)
//   Q2_K     the same with 4-bit sc and m per 16 weights (<= 3 * 15)
//   Q3_K     code = (q - 4) * (sc - 32), sc per 16; sum w x = d C
//   Q6_K     int8 sc per 16 weights split as 16 a + b (b in 0..15):
//            codes (q - 32) b and (q - 32) a, sum w x = d (C_b + 16 C_a)
//            (quants.c:153-177)
//   IQ4_XS   code = level (int8 table), per 32 columns
//            sum w x = sum_32 d (ls - 32) C_32          (quants.c:228-248)
//   Q8_0     code = q, per 32 columns sum w x = sum_32 d_32 C_32
//            (quants.c:85-94)
// Every code is an integer of magnitude < 2048 (the IQ codes times 2^-14),
// so exact in f16. The K-quant codes come from the byte b by a permute that
// makes the half 0x64bb (1024 + b, exact) and a packed f16 add or
// multiply-add that removes the 1024 and applies the scale. The IQ codes
// come from the grid byte b and a sign byte (0x80 or 0x00, a table per sign
// index) by one permute per two codes that makes the half +-b 2^-24 (the
// f16 subnormal with mantissa b), then one packed f16 multiply by
// (2 s + 1) 2^10: every intermediate exact. (The multiply reads the
// subnormal as such: f16 denormals are on in the kernels' default FP mode,
// and a flush would zero every IQ code, which every IQ parity case shows.)
//
// Workgroup: one unit (<= 64 pairs of one expert, MT = 1..4 M tiles of 16) x
// 8 waves; a wave computes two N tiles of 16 weight rows (gate/up: the same
// rows of gate and of up, so silu(gate) * up needs no exchange) x the unit's
// M tiles. A wave's weights come G blocks (256 columns) of its rows at a time,
// as whole 16-byte pieces along the rows, to registers a group ahead and from
// there to its own part of LDS, where its lanes read what they decode. The
// unit's records, half a block at a time, go through registers to a double
// buffer in LDS that all waves read, one barrier a half.
//
// What bounds it: the LDS pipe (activation reads, codebook gathers at 2-3
// times their conflict-free cost) and the latency between its results and
// the matrix ops, at two waves a SIMD. Measured, gate/up + down at hidden 6144,
// inter 3072, 256 experts, IQ2_XS / IQ3_XXS with Q5_K / Q6_K shared: 1999
// tokens 3.30 + 1.87 ms (units of 64 pairs; 4.36 + 2.94 ms with units of 32
// whose 16 waves staged single blocks by LDS DMA), 512 tokens 1.30 + 0.77 ms
// (1.57 + 1.09), 9 tokens 328 + 203 us (363 + 238). Loads alone take 125 us
// of the 328: a wave instruction that reads whole pieces along a row touches
// each line once; lanes loading just what they decode took 369 us for the
// same bytes. Four N tiles a wave for the larger units (half the activation
// reads, groups of one block) took 3.35 + 1.97 ms; all of a half's table
// reads at once 397 us for 9 tokens; units of up to 16 pairs in a launch of
// their own with two workgroups a CU 334 + 203 us there, but 538 + 1044 us
// for the two gate/up launches of 512 tokens.
#pragma once
#include "prefill_q.h"

#define PH_UM 64                       // pairs per unit
#define PH_REC 576                     // bytes of a 128-column PH record
#define PH_LREC 608                    // a staged record (38 16-byte pieces, 2 mod 4: no LDS bank conflicts)
#define PH_WAVES 8                     // waves of a workgroup

typedef _Float16 ph_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 ph_h8 __attribute__((ext_vector_type(8)));
typedef uint32_t ph_u4 __attribute__((ext_vector_type(4)));

// BB: block bytes (256 columns); QN: dwords of a lane's half block, HN: of
// what it needs of the block besides; G, GL: blocks of a weight group for
// units of up to two M tiles and of more (what the LDS holds); STEP: scale
// per 32-column step applied in f32 (else once per block); MIN: min terms.
template <int T> struct PhFmt;
template <> struct PhFmt<ST_Q2_K> { static constexpr int BB = 84, QN = 4, HN = 1, G = 4, GL = 2; static constexpr bool STEP = false, MIN = true; };
template <> struct PhFmt<ST_Q3_K> { static constexpr int BB = 110, QN = 2, HN = 6, G = 4, GL = 2; static constexpr bool STEP = false, MIN = false; };
template <> struct PhFmt<ST_Q4_K> { static constexpr int BB = 144, QN = 4, HN = 4, G = 2, GL = 2; static constexpr bool STEP = false, MIN = true; };
template <> struct PhFmt<ST_Q5_K> { static constexpr int BB = 176, QN = 4, HN = 6, G = 2, GL = 1; static constexpr bool STEP = false, MIN = true; };
template <> struct PhFmt<ST_Q6_K> { static constexpr int BB = 210, QN = 8, HN = 1, G = 2, GL = 1; static constexpr bool STEP = false, MIN = false; };
template <> struct PhFmt<ST_IQ2_XS> { static constexpr int BB = 74, QN = 3, HN = 1, G = 4, GL = 2; static constexpr bool STEP = false, MIN = false; };
template <> struct PhFmt<ST_IQ3_XXS> { static constexpr int BB = 98, QN = 3, HN = 1, G = 4, GL = 2; static constexpr bool STEP = false, MIN = false; };
template <> struct PhFmt<ST_IQ4_XS> { static constexpr int BB = 136, QN = 8, HN = 2, G = 2, GL = 2; static constexpr bool STEP = true, MIN = false; };
template <> struct PhFmt<ST_Q8_0> { static constexpr int BB = 272, QN = 12, HN = 1, G = 1, GL = 1; static constexpr bool STEP = true, MIN = false; };

// LDS: [record stages 2 x 16 MT x PH_LREC][weight groups: 8 waves x 2 tiles
// x 16 rows x PW pieces] ... [IQ2_XS grid 4 KB / IQ3_XXS grid 1 KB][128 x 8
// sign bytes][row tables]
#define PH_LDS_BYTES 163840
#define PH_O_ROWS (PH_LDS_BYTES - 16 * PH_UM)
#define PH_O_SIGNS (PH_O_ROWS - 1024)
#define PH_O_TAB (PH_O_SIGNS - 4096)

// --------------------------------------------------------- rows -> PH ----
// One workgroup per row: src row r (K floats at src + r * ld) into its
// records at rec + r * ldr and its scale at scale[r]. Thread i converts the
// 16-column groups i, i + 256, ...
extern "C" __global__ __launch_bounds__(256) void sepia_ph_quant(const float *__restrict__ src, int64_t ld,
                                                                 int64_t K, uint8_t *__restrict__ rec, int64_t ldr,
                                                                 float *__restrict__ scale) {
    __shared__ float red[4];
    const int64_t r = blockIdx.x;
    const float *row = src + r * ld;
    // (each times zero: 0, or NaN for a NaN or an infinity; a plain sum of
    // large finite values could overflow into one)
    float m = 0.0f;
    for (int64_t c = 4 * (int64_t)threadIdx.x; c < K; c += 1024) {
        const float4 v = *(const float4 *)(row + c);
        m = mq_nonfinite_max(fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)))),
                             (v.x * 0.0f + v.y * 0.0f) + (v.z * 0.0f + v.w * 0.0f));
    }
    m = pq_wave_max(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    // s = 2^e, 2^15 s > m (exact scaling): e = the exponent of m's leading
    // bit + 1 - 15, held to where s is a normal float (1 / s is one then too).
    // Where that holds it, m < 2^-111; rows below 2^-126 are multiples of
    // 2^-149, whose v' are multiples of 2^-23, exact.
    const bool fin = m < INFINITY;
    int e = 0;
    if (fin && m > 0.0f) (void)frexpf(m, &e);
    e = e - 15 < -126 ? -126 : e - 15;
    const float s = !fin ? INFINITY : ldexpf(1.0f, e), inv = fin ? ldexpf(1.0f, -e) : 0.0f;
    if (threadIdx.x == 0) scale[r] = s;
    uint8_t *out = rec + r * ldr;
    for (int64_t gi = threadIdx.x; gi < K / 16; gi += 256) {
        const float4 *x4 = (const float4 *)(row + 16 * gi);
        uint8_t *blk = out + (gi >> 3) * PH_REC;
        const int j = (int)(gi & 7);
        float sum = 0.0f;
        _Float16 h[16], l[16];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const float4 t = x4[c];
            const float a[4] = {t.x * inv, t.y * inv, t.z * inv, t.w * inv};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                sum += a[i];
                h[4 * c + i] = (_Float16)a[i];
                l[4 * c + i] = (_Float16)(a[i] - (float)h[4 * c + i]);
            }
        }
#pragma unroll
        for (int i = 0; i < 2; i++) {
            *(uint4 *)(blk + 32 * j + 16 * i) = *(const uint4 *)(h + 8 * i);
            *(uint4 *)(blk + 256 + 32 * j + 16 * i) = *(const uint4 *)(l + 8 * i);
        }
        sum = fin ? sum * 0.0625f : 0.0f;
        const _Float16 s0 = (_Float16)sum, s1 = (_Float16)(sum - (float)s0),
                       s2 = (_Float16)(sum - (float)s0 - (float)s1);
        _Float16 *sp = (_Float16 *)(blk + 512 + 16 * (j >> 1)) + 3 * (j & 1);
        sp[0] = s0;
        sp[1] = s1;
        sp[2] = s2;
        if (j & 1) sp[3] = sp[4] = (_Float16)0.0f;
    }
}

// ------------------------------------------------------------- decoders --
// Bytes 0, 1 (sel 0x04010400) or 2, 3 (sel 0x04030402) of v as the halves
// 0x64bb: 1024 + b, exact.
__device__ __forceinline__ ph_h2 ph_bias2(uint32_t v, uint32_t sel) {
    return __builtin_bit_cast(ph_h2, __builtin_amdgcn_perm(0x64646464u, v, sel));
}
#define PH_SEL_LO 0x04010400u
#define PH_SEL_HI 0x04030402u
// 8 codes b - off from the 8 bytes of g (exact f16 integers)
__device__ __forceinline__ ph_h8 ph_codes_sub(uint2 g, ph_h2 off) {
    ph_h2 c[4] = {ph_bias2(g.x, PH_SEL_LO) - off, ph_bias2(g.x, PH_SEL_HI) - off, ph_bias2(g.y, PH_SEL_LO) - off,
                  ph_bias2(g.y, PH_SEL_HI) - off};
    return __builtin_bit_cast(ph_h8, c);
}
__device__ __forceinline__ ph_h2 ph_splat(float v) {
    const _Float16 h = (_Float16)v;
    return ph_h2{h, h};
}
// A small integer's exact f16 in both halves (a direct 16-bit integer to f16
// convert, no f32 step): |v| <= 2048.
__device__ __forceinline__ ph_h2 ph_splat_u(uint32_t v) {
    const _Float16 h = (_Float16)(uint16_t)v;
    return ph_h2{h, h};
}
// The sign bytes of the 128 IQ sign indices, 8 bytes each: byte j 0x80
// where bit j of iq_signs(index) is set (code j negative), else 0x00.
__device__ __forceinline__ void ph_fill_signs(uint8_t *st) {
    for (int i = threadIdx.x; i < 128; i += blockDim.x) {
        const uint32_t s = iq_signs((uint32_t)i);
        uint2 m = make_uint2(0u, 0u);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            m.x |= ((s >> j) & 1u) << (8 * j + 7);
            m.y |= ((s >> (j + 4)) & 1u) << (8 * j + 7);
        }
        *(uint2 *)(st + 8 * i) = m;
    }
}
// 8 IQ codes from the grid bytes g and the sign bytes sg (codes 0..3 in .x,
// 4..7 in .y): the halves +-b 2^-24 (low byte the grid byte, high byte the
// sign byte) times s2 = (2 s + 1) 2^10
__device__ __forceinline__ ph_h8 ph_codes_iq(uint2 g, uint2 sg, ph_h2 s2) {
    const ph_h2 c[4] = {__builtin_bit_cast(ph_h2, __builtin_amdgcn_perm(sg.x, g.x, 0x05010400u)) * s2,
                        __builtin_bit_cast(ph_h2, __builtin_amdgcn_perm(sg.x, g.x, 0x07030602u)) * s2,
                        __builtin_bit_cast(ph_h2, __builtin_amdgcn_perm(sg.y, g.y, 0x05010400u)) * s2,
                        __builtin_bit_cast(ph_h2, __builtin_amdgcn_perm(sg.y, g.y, 0x07030602u)) * s2};
    return __builtin_bit_cast(ph_h8, c);
}
template <int T>
__device__ __forceinline__ void ph_fill_tables(uint8_t *smem) {
    if constexpr (T == ST_IQ2_XS) {
        for (int i = threadIdx.x; i < 512; i += blockDim.x) ((uint64_t *)(smem + PH_O_TAB))[i] = c_iq2xs_grid[i];
        ph_fill_signs(smem + PH_O_SIGNS);
    } else if constexpr (T == ST_IQ3_XXS) {
        for (int i = threadIdx.x; i < 256; i += blockDim.x) ((uint32_t *)(smem + PH_O_TAB))[i] = c_iq3xxs_grid[i];
        ph_fill_signs(smem + PH_O_SIGNS);
    }
}

// The IQ4 levels + 128 as bytes (0..241), for the biased conversion.
__device__ __forceinline__ constexpr uint32_t ph_iq4_word(int k) {
    constexpr int8_t v[16] = SEPIA_IQ4NL_VALUES_INIT;
    return (uint32_t)(uint8_t)(v[4 * k] + 128) | ((uint32_t)(uint8_t)(v[4 * k + 1] + 128) << 8) |
           ((uint32_t)(uint8_t)(v[4 * k + 2] + 128) << 16) | ((uint32_t)(uint8_t)(v[4 * k + 3] + 128) << 24);
}
// levels + 128 of the four codes in the low nibbles of the bytes of c
__device__ __forceinline__ uint32_t ph_iq4_levels(uint32_t c) {
    constexpr uint32_t T0 = ph_iq4_word(0), T1 = ph_iq4_word(1), T2 = ph_iq4_word(2), T3 = ph_iq4_word(3);
    const uint32_t sel = c & 0x07070707u;
    const uint32_t lo = __builtin_amdgcn_perm(T1, T0, sel), hi = __builtin_amdgcn_perm(T3, T2, sel);
    return __builtin_amdgcn_perm(hi, lo, ((c >> 1) & 0x04040404u) | 0x03020100u);
}

// N dwords of a staged row at byte p. M: whether p is 2 bytes past a dword
// (else at one): two aligned dwords around each, funnel-shifted.
template <int N, bool M>
__device__ __forceinline__ void ph_gld(const uint8_t *p, uint32_t *q) {
    const uint32_t at = pf_lds(p) - (M ? 2u : 0u);
    uint32_t d[N + 1];
#pragma unroll
    for (int i = 0; i < N + (M ? 1 : 0); i++)
        d[i] = *(const __attribute__((address_space(3))) uint32_t *)(size_t)(at + 4u * (uint32_t)i);
#pragma unroll
    for (int i = 0; i < N; i++) q[i] = M ? __builtin_amdgcn_alignbit(d[i + 1], d[i], 16) : d[i];
}

// What lane group g needs of the block at p besides the half's codes. M: the
// block starts 2 bytes past a dword.
template <int T, bool M>
__device__ __forceinline__ void ph_load_head(const uint8_t *p, int g, uint32_t *h) {
    if constexpr (T == ST_Q2_K) {
        ph_gld<1, M>(p + 80, h);   // d, dmin
    } else if constexpr (T == ST_Q3_K) {
        ph_gld<2, M>(p + 8 * g, h);       // hmask bytes 8 g ..
        ph_gld<3, M>(p + 96, h + 2);      // scales: low nibbles, then the high bits
        ph_gld<1, !M>(p + 106, h + 5);    // d in the high half
    } else if constexpr (T == ST_Q4_K) {
        ph_gld<4, M>(p, h);   // d, dmin, 12 scale bytes
    } else if constexpr (T == ST_Q5_K) {
        ph_gld<4, M>(p, h);
        ph_gld<2, M>(p + 16 + 8 * g, h + 4);   // qh bytes 8 g ..
    } else if constexpr (T == ST_Q6_K) {
        ph_gld<1, !M>(p + 206, h);   // d in the high half
    } else if constexpr (T == ST_IQ2_XS || T == ST_IQ3_XXS) {
        ph_gld<1, M>(p, h);   // d in the low half
    } else if constexpr (T == ST_IQ4_XS) {
        ph_gld<2, M>(p, h);   // d, scales_h; scales_l
    }
}
// What it decodes of half hb (columns 128 hb .. + 127). K step s (0..3) of
// the half takes columns 32 s + 8 g .. + 7 of it, except IQ2_XS and
// IQ3_XXS, whose lane group takes 32 g + 8 s .. + 7 (a lane's codes are then
// adjacent bytes, ph_chunked).
template <int T, bool M>
__device__ __forceinline__ void ph_load_half(const uint8_t *p, int hb, int g, uint32_t *q) {
    if constexpr (T == ST_Q2_K) {
        ph_gld<2, M>(p + 16 + 32 * hb + 8 * g, q);
        ph_gld<2, M>(p + 8 * hb, q + 2);   // its scale bytes
    } else if constexpr (T == ST_Q3_K) {
        ph_gld<2, M>(p + 32 + 32 * hb + 8 * g, q);
    } else if constexpr (T == ST_Q4_K || T == ST_Q5_K) {
        const int o = (T == ST_Q4_K ? 16 : 48) + 64 * hb + 8 * g;
        ph_gld<2, M>(p + o, q);
        ph_gld<2, M>(p + o + 32, q + 2);
    } else if constexpr (T == ST_Q6_K) {
        ph_gld<2, M>(p + 64 * hb + 8 * g, q);
        ph_gld<2, M>(p + 64 * hb + 32 + 8 * g, q + 2);
        ph_gld<2, M>(p + 128 + 32 * hb + 8 * g, q + 4);   // qh
        ph_gld<2, M>(p + 192 + 8 * hb, q + 6);            // its scales
    } else if constexpr (T == ST_IQ2_XS) {
        ph_gld<2, !M>(p + 2 + 32 * hb + 8 * g, q);
        ph_gld<1, !M>(p + 66 + 4 * hb, q + 2);   // the half's scales, byte g the lane group's
    } else if constexpr (T == ST_IQ3_XXS) {
        ph_gld<2, !M>(p + 2 + 32 * hb + 8 * g, q);
        ph_gld<1, !M>(p + 66 + 16 * hb + 4 * g, q + 2);
    } else if constexpr (T == ST_IQ4_XS) {
#pragma unroll
        for (int s = 0; s < 4; s++) ph_gld<2, M>(p + 8 + 16 * (4 * hb + s) + 8 * (g & 1), q + 2 * s);
    } else {   // Q8_0: step 4 hb + s at 34 (4 hb + s), a dword for even s
        ph_gld<2, !M>(p + 136 * hb + 2 + 8 * g, q);
        ph_gld<1, M>(p + 136 * hb, q + 2);   // d in the low half
        ph_gld<2, M>(p + 136 * hb + 36 + 8 * g, q + 3);
        ph_gld<1, !M>(p + 136 * hb + 34, q + 5);
        ph_gld<2, !M>(p + 136 * hb + 70 + 8 * g, q + 6);
        ph_gld<1, M>(p + 136 * hb + 68, q + 8);
        ph_gld<2, M>(p + 136 * hb + 104 + 8 * g, q + 9);
        ph_gld<1, !M>(p + 136 * hb + 102, q + 11);
    }
}
template <int T>
__device__ __forceinline__ constexpr bool ph_chunked() { return T == ST_IQ2_XS || T == ST_IQ3_XXS; }

__device__ __forceinline__ float ph_hlo(uint32_t v) { return f16_bits_to_f32(v & 0xFFFFu); }
__device__ __forceinline__ float ph_hhi(uint32_t v) { return f16_bits_to_f32(v >> 16); }
// Byte i of the dwords at h.
__device__ __forceinline__ uint32_t ph_byte(const uint32_t *h, int i) { return (h[i >> 2] >> (8 * (i & 3))) & 255u; }
// The 6-bit scale of sub-block j of Q4_K and Q5_K from the block's first 16
// bytes (the packing of get_scale_min_k4, src/quants.c:96-102; scale byte i
// is byte 4 + i).
__device__ __forceinline__ uint32_t ph_scale_6(const uint32_t *h, int j) {
    return j < 4 ? ph_byte(h, 4 + j) & 63u : (ph_byte(h, 8 + j) & 15u) | ((ph_byte(h, j) >> 6) << 4);
}

// What a lane decodes for a K step: the 8 codes (two operands for Q6_K) and,
// for the STEP formats, the step's scale.
struct PhB {
    ph_h8 b, b2;
    float sc;
};
// The IQ formats' table entries of K step s: grid and sign bytes, read a step
// ahead of ph_decode.
struct PhG {
    uint2 gr, sg;
};
template <int T>
__device__ __forceinline__ PhG ph_gather(const uint32_t *q, const uint8_t *tab, const uint8_t *signs, int s) {
    PhG r;
    if constexpr (T == ST_IQ2_XS) {   // u16 s: grid index (9 bits), sign index (7 bits)
        const uint32_t v = q[s >> 1] >> (16 * (s & 1));
        r.gr = *(const __attribute__((address_space(3))) uint2 *)(size_t)pf_lds(tab + 8 * (v & 511u));
        r.sg = *(const __attribute__((address_space(3))) uint2 *)(size_t)pf_lds(signs + 8 * ((v >> 9) & 127u));
    } else if constexpr (T == ST_IQ3_XXS) {   // bytes 2 s, 2 s + 1: grid indices (4 codes each); sign index s at bit 7 s
        const uint32_t ix = q[s >> 1] >> (16 * (s & 1));
        r.gr.x = *(const __attribute__((address_space(3))) uint32_t *)(size_t)pf_lds(tab + 4 * (ix & 255u));
        r.gr.y = *(const __attribute__((address_space(3))) uint32_t *)(size_t)pf_lds(tab + 4 * ((ix >> 8) & 255u));
        r.sg = *(const __attribute__((address_space(3))) uint2 *)(size_t)pf_lds(signs + 8 * ((q[2] >> (7 * s)) & 127u));
    }
    return r;
}
template <int T>
__device__ __forceinline__ PhB ph_decode(const uint32_t *h, const uint32_t *q, const PhG &G, int hb, int s, int g) {
    PhB r;
    if constexpr (T == ST_IQ2_XS) {   // 4-bit scale: nibble s >> 1 of the lane group's byte
        r.b = ph_codes_iq(G.gr, G.sg, ph_splat_u((2u * ((q[2] >> (8 * g + 4 * (s >> 1))) & 15u) + 1u) << 10));
    } else if constexpr (T == ST_IQ3_XXS) {   // 4-bit scale at bit 28
        r.b = ph_codes_iq(G.gr, G.sg, ph_splat_u((2u * (q[2] >> 28) + 1u) << 10));
    } else if constexpr (T == ST_IQ4_XS) {
        // 8 bytes of the step's 16, nibble g >> 1; 6-bit scale ls of group 4 hb + s
        const int j = 4 * hb + s;
        const uint32_t sh = 4u * (uint32_t)(g >> 1);
        const uint2 lv = make_uint2(ph_iq4_levels(q[2 * s] >> sh), ph_iq4_levels(q[2 * s + 1] >> sh));
        r.b = ph_codes_sub(lv, ph_splat(1152.0f));
        const uint32_t ls = ((h[1] >> (4 * j)) & 15u) | (((h[0] >> (16 + 2 * j)) & 3u) << 4);
        r.sc = ph_hlo(h[0]) * (float)((int32_t)ls - 32);
    } else if constexpr (T == ST_Q4_K || T == ST_Q5_K) {
        // nibble s & 1 of bytes 32 (s >> 1) + 8 g .. (q[2 (s >> 1)], + 1); Q5_K: bit 4 hb + s of qh
        const int j = 4 * hb + s, k = 2 * (s >> 1);
        const uint32_t nsh = 4u * (uint32_t)(s & 1);
        uint32_t c0 = (q[k] >> nsh) & 0x0F0F0F0Fu, c1 = (q[k + 1] >> nsh) & 0x0F0F0F0Fu;
        if constexpr (T == ST_Q5_K) {
            c0 |= ((h[4] >> j) & 0x01010101u) << 4;
            c1 |= ((h[5] >> j) & 0x01010101u) << 4;
        }
        r.b = ph_codes_sub(make_uint2(c0, c1), ph_splat(1024.0f)) * (_Float16)(uint16_t)ph_scale_6(h, j);
    } else if constexpr (T == ST_Q2_K) {
        // bit pair s of the bytes; scale byte 2 s + (g >> 1) of the half, low nibble
        const uint32_t c0 = (q[0] >> (2 * s)) & 0x03030303u, c1 = (q[1] >> (2 * s)) & 0x03030303u;
        const uint32_t sc = (q[2 + (s >> 1)] >> (16 * (s & 1) + 8 * (g >> 1))) & 15u;
        r.b = ph_codes_sub(make_uint2(c0, c1), ph_splat(1024.0f)) * (_Float16)(uint16_t)sc;
    } else if constexpr (T == ST_Q3_K) {
        // bit pair s of the bytes, high bit 4 hb + s of hmask; scale j = 8 hb + 2 s + (g >> 1): nibble hb of
        // byte 2 s + (g >> 1), its high bits 2 (j >> 2) of byte 8 + (j & 3)
        const int b = 4 * hb + s;
        const uint32_t c0 = ((q[0] >> (2 * s)) & 0x03030303u) | (((h[0] >> b) & 0x01010101u) << 2);
        const uint32_t c1 = ((q[1] >> (2 * s)) & 0x03030303u) | (((h[1] >> b) & 0x01010101u) << 2);
        const uint32_t gs = 8u * (uint32_t)(g >> 1);
        const uint32_t lo = (h[2 + (s >> 1)] >> (16 * (s & 1) + 4 * hb + gs)) & 15u;
        const uint32_t hi = (h[4] >> (16 * (s & 1) + 2 * (2 * hb + (s >> 1)) + gs)) & 3u;
        r.b = ph_codes_sub(make_uint2(c0, c1), ph_splat(1028.0f)) * (_Float16)(int16_t)((int32_t)(lo | (hi << 4)) - 32);
    } else if constexpr (T == ST_Q6_K) {
        // quarter s: low 4 bits from ql[32 (s & 1) + 8 g ..] (nibble s >> 1), high 2 from qh bits 2 s; int8 scale
        // 2 s + (g >> 1) of the half, split as 16 a + b
        const int k = 2 * (s & 1);
        const uint32_t nsh = 4u * (uint32_t)(s >> 1), hsh = 2u * (uint32_t)s;
        const uint32_t c0 = ((q[k] >> nsh) & 0x0F0F0F0Fu) | (((q[4] >> hsh) & 0x03030303u) << 4);
        const uint32_t c1 = ((q[k + 1] >> nsh) & 0x0F0F0F0Fu) | (((q[5] >> hsh) & 0x03030303u) << 4);
        const int32_t sc = (int32_t)(int8_t)((q[6 + (s >> 1)] >> (16 * (s & 1) + 8 * (g >> 1))) & 255u);
        const ph_h8 q32 = ph_codes_sub(make_uint2(c0, c1), ph_splat(1056.0f));   // q - 32
        r.b = q32 * (_Float16)(int16_t)(sc & 15);                               // (q - 32) b
        r.b2 = q32 * (_Float16)(int16_t)(sc >> 4);                              // (q - 32) a
    } else {   // Q8_0
        r.b = ph_codes_sub(make_uint2(q[3 * s] ^ 0x80808080u, q[3 * s + 1] ^ 0x80808080u), ph_splat(1152.0f));
        r.sc = ph_hlo(q[3 * s + 2]);
    }
    return r;
}
// The mins of a half as a matrix operand against the record's sum groups:
// lane group g has columns 32 g .. + 31, three terms of each 16-column sum.
template <int T>
__device__ __forceinline__ ph_h8 ph_mins(const uint32_t *h, const uint32_t *q, int hb, int g) {
    _Float16 a, b;
    const uint32_t gs = 8u * (uint32_t)g;
    if constexpr (T == ST_Q2_K) {
        const uint32_t v = q[2 + (g >> 1)] >> (16 * (g & 1));   // scale bytes 2 g, 2 g + 1 of the half: high nibbles
        a = (_Float16)(uint16_t)((v >> 4) & 15u);
        b = (_Float16)(uint16_t)((v >> 12) & 15u);
    } else {
        const uint32_t m = hb == 0 ? (h[2] >> gs) & 63u : ((h[3] >> (gs + 4)) & 15u) | (((h[2] >> (gs + 6)) & 3u) << 4);
        a = b = (_Float16)(uint16_t)m;
    }
    return ph_h8{a, a, a, b, b, b, (_Float16)0.0f, (_Float16)0.0f};
}

// ----------------------------------------------------------- projection --
template <bool B> struct PhBool { static constexpr bool value = B; };

// One projection workgroup (see the top of the file). GU: wave w computes
// rows r0 + 16 w .. of gate (W0, tile 0) and up (W1, tile 1), h[pair][row] =
// silu(gate) * up in f32; down: rows r0 + 32 w .. of W0, out[pair][row] in
// f32. rows: those of the matrix, a multiple of 256 as the host checks.
template <int T, bool GU, int MT>
__device__ __forceinline__ void ph_proj(uint8_t *smem, const uint8_t *W0, const uint8_t *W1, uint64_t row_bytes,
                                        int64_t nb, const uint8_t *rec, const int64_t *roff, const int32_t *pair,
                                        const float *srow, int nv, int64_t r0, int64_t rows, float *__restrict__ out,
                                        int64_t ld_out) {
    typedef PhFmt<T> F;
    constexpr int NT = 2, G = MT <= 2 ? F::G : F::GL, QN = F::QN, HN = F::HN, HT = GU ? 1 : 2;
    // a group's bytes of a row, from the dword at or below its start (odd
    // blocks of a format of 4 k + 2 bytes start 2 bytes past one; only G = 1
    // groups do), as PW pieces; KW wave instructions a tile
    constexpr int PW = (G * F::BB + (G == 1 && F::BB % 4 ? 2 : 0) + 15) / 16, KW = (16 * PW + 63) / 64;
    constexpr uint32_t O_W = 2u * 16u * MT * PH_LREC;
    static_assert(O_W + PH_WAVES * NT * 16 * 16 * PW <= (T == ST_IQ2_XS || T == ST_IQ3_XXS ? PH_O_TAB : PH_O_ROWS), "LDS");
    const int tid = (int)threadIdx.x, l = tid & 63, n = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t grow = r0 + 16 * HT * w;   // the wave's first row
    // Always true, which the compiler does not know: a branch on it ends the
    // basic block at every half of the unrolled loop below. As straight-line
    // code the kernels spilled 889 registers (9 tokens 539 -> 556 us, 300
    // tokens of a mixed layer 557 -> 592).
    const bool whole = grow < rows;
    const int nbi = (int)nb, nst = 2 * nbi;
    const uint8_t *tab = smem + PH_O_TAB, *signs = smem + PH_O_SIGNS;
    ph_fill_tables<T>(smem);   // published by the first barrier
    // records: piece tid + 512 i of a half is row m = piece / 32 of the unit,
    // 16-byte column group piece % 32 (hi, then lo); a K step's four lane
    // groups read adjacent pieces
    const uint8_t *asrc[MT];
    uint32_t adst[MT];
    const uint8_t *ssrc = nullptr;
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int p = tid + 512 * i, m = p >> 5, c = p & 31, cg = c & 15;
        asrc[i] = rec + roff[m] + 16 * c;
        adst[i] = (uint32_t)(m * PH_LREC + 256 * (c >> 4) + 16 * (ph_chunked<T>() ? 4 * (cg & 3) + (cg >> 2) : cg));
    }
    if (F::MIN) ssrc = rec + roff[tid < 64 * MT ? tid >> 2 : 0] + 512 + 16 * (tid & 3);
    // Loads return in order, so the records of units of up to two M tiles are
    // fetched AD halves ahead: a wait for records issued after a weight group
    // is one for that group too.
    constexpr int AD = MT <= 2 ? 4 : 1;   // divides a turn's halves
    ph_u4 ar[AD][MT], sr[AD];
    auto a_load = [&](int t, int slot) {
        t = t < nst ? t : nst - 1;
#pragma unroll
        for (int i = 0; i < MT; i++) ar[slot][i] = *(const ph_u4 *)(asrc[i] + (uint32_t)t * PH_REC);
        if (F::MIN) sr[slot] = *(const ph_u4 *)(ssrc + (uint32_t)t * PH_REC);
    };
    auto a_store = [&](int t, int slot) {
        uint8_t *st = smem + (uint32_t)(t & 1) * (16 * MT * PH_LREC);
#pragma unroll
        for (int i = 0; i < MT; i++) *(ph_u4 *)(st + adst[i]) = ar[slot][i];
        if (F::MIN && tid < 64 * MT) *(ph_u4 *)(st + (tid >> 2) * PH_LREC + 512 + 16 * (tid & 3)) = sr[slot];
    };
    // weights: piece q = 64 k + lane of a tile's group is row q / PW, bytes
    // 16 (q % PW) .. of it; pieces past the row's last block take the group's
    // first (the last one that holds block bytes may run up to 12 bytes past
    // the matrix, into the 256 that every device buffer of the library
    // carries past its data, dev_bytes in sepia_hip.c)
    uint32_t wrow[KW], wcol[KW];
#pragma unroll
    for (int k = 0; k < KW; k++) {
        const int q = 64 * k + l < 16 * PW ? 64 * k + l : 0, m = q / PW;
        wrow[k] = (uint32_t)((uint64_t)m * row_bytes);
        wcol[k] = 16u * (uint32_t)(q - m * PW);
    }
    // (from the wave's first row: 32-bit offsets then reach its rows in a matrix of any size)
    const uint64_t wfirst = (uint64_t)grow * row_bytes;
    const uint8_t *Wt[NT] = {W0 + wfirst, GU ? W1 + wfirst : W0 + wfirst + 16 * row_bytes};
    uint8_t *wl = smem + O_W + (uint32_t)w * (NT * 16 * 16 * PW);
    ph_u4 wr[NT][KW];
    auto w_load = [&](int b) {   // the group of blocks b ..
        const uint32_t at = ((uint32_t)b * F::BB) & ~3u, left = (uint32_t)nbi * F::BB - at;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int k = 0; k < KW; k++) {
                typedef ph_u4 U4 __attribute__((aligned(4)));
                wr[t][k] = *(const U4 *)(Wt[t] + at + (uint64_t)(wrow[k] + (wcol[k] < left ? wcol[k] : 0u)));
            }
    };
    auto w_store = [&]() {
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int k = 0; k < KW; k++)
                if (64 * (k + 1) <= 16 * PW || 64 * k + l < 16 * PW)
                    *(ph_u4 *)(wl + t * (16 * 16 * PW) + 1024 * k + 16 * l) = wr[t][k];
    };
    pf_f32x4 acc[NT][MT], cb[NT][MT], cb2[T == ST_Q6_K ? NT : 1][T == ST_Q6_K ? MT : 1],
        cm[F::MIN ? NT : 1][F::MIN ? MT : 1];
    const pf_f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
        for (int mt = 0; mt < MT; mt++) acc[t][mt] = zero;
    // half hb of block b (o: where it starts in the staged group)
    auto half = [&](auto mis, int o, int hb) {
        constexpr bool M = decltype(mis)::value;
        const uint8_t *As = smem + (uint32_t)hb * (16 * MT * PH_LREC) + n * PH_LREC + 16 * g;
        uint32_t q[NT][QN], h[NT][HN];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const uint8_t *blk = wl + (16 * t + n) * (16 * PW) + o;
            ph_load_half<T, M>(blk, hb, g, q[t]);
            ph_load_head<T, M>(blk, g, h[t]);
        }
        if (hb == 0) {
#pragma unroll
            for (int t = 0; t < NT; t++)
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    cb[t][mt] = zero;
                    if constexpr (T == ST_Q6_K) cb2[t][mt] = zero;
                    if constexpr (F::MIN) cm[t][mt] = zero;
                }
        }
        // Pipelined by one K step: step s + 1's table entries and activations
        // are on their way from LDS while step s's matrix ops run; its codes
        // are made of them after.
        PhB B[NT];
        PhG Gt[NT];
        ph_h8 a1[2];
#pragma unroll
        for (int t = 0; t < NT; t++) Gt[t] = ph_gather<T>(q[t], tab, signs, 0);
        auto a_read = [&](int s, int mt, int pl) {
            return *(const __attribute__((address_space(3))) ph_h8 *)(size_t)pf_lds(As + 16 * mt * PH_LREC + 256 * pl + 64 * s);
        };
#pragma unroll
        for (int pl = 0; pl < 2; pl++) a1[pl] = a_read(0, 0, pl);
#pragma unroll
        for (int t = 0; t < NT; t++) B[t] = ph_decode<T>(h[t], q[t], Gt[t], hb, 0, g);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            ph_h8 a2[2][2];
            a2[0][0] = a1[0];
            a2[0][1] = a1[1];
            if (s + 1 < 4) {
#pragma unroll
                for (int t = 0; t < NT; t++) Gt[t] = ph_gather<T>(q[t], tab, signs, s + 1);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) {
                if (mt + 1 < MT) {
#pragma unroll
                    for (int pl = 0; pl < 2; pl++) a2[(mt + 1) & 1][pl] = a_read(s, mt + 1, pl);
                } else if (s + 1 < 4) {
#pragma unroll
                    for (int pl = 0; pl < 2; pl++) a1[pl] = a_read(s + 1, 0, pl);
                }
                const ph_h8 ah = a2[mt & 1][0], al = a2[mt & 1][1];
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    if constexpr (F::STEP) {
                        pf_f32x4 c = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, B[t].b, zero, 0, 0, 0);
                        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, B[t].b, c, 0, 0, 0);
#pragma unroll
                        for (int k = 0; k < 4; k++) acc[t][mt][k] = __builtin_fmaf(B[t].sc, c[k], acc[t][mt][k]);
                    } else {
                        cb[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, B[t].b, cb[t][mt], 0, 0, 0);
                        cb[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, B[t].b, cb[t][mt], 0, 0, 0);
                        if constexpr (T == ST_Q6_K) {
                            cb2[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, B[t].b2, cb2[t][mt], 0, 0, 0);
                            cb2[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, B[t].b2, cb2[t][mt], 0, 0, 0);
                        }
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (s + 1 < 4) {
#pragma unroll
                for (int t = 0; t < NT; t++) B[t] = ph_decode<T>(h[t], q[t], Gt[t], hb, s + 1, g);
            }
        }
        if constexpr (F::MIN) {   // mins . sums
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const ph_h8 mb = ph_mins<T>(h[t], q[t], hb, g);
#pragma unroll
                for (int mt = 0; mt < MT; mt++) {
                    const ph_h8 sa =
                        *(const __attribute__((address_space(3))) ph_h8 *)(size_t)pf_lds(As + 16 * mt * PH_LREC + 512);
                    cm[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(sa, mb, cm[t][mt], 0, 0, 0);
                }
            }
        }
        if (!F::STEP && hb == 1) {
#pragma unroll
            for (int t = 0; t < NT; t++) {
                // IQ: 2^14 / 8, 2^14 / 4
                const float d = T == ST_IQ2_XS    ? ph_hlo(h[t][0]) * 2048.0f
                                : T == ST_IQ3_XXS ? ph_hlo(h[t][0]) * 4096.0f
                                : T == ST_Q3_K    ? ph_hhi(h[t][HN - 1])
                                : T == ST_Q6_K    ? ph_hhi(h[t][0])
                                                  : ph_hlo(h[t][0]);
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        float c = cb[t][mt][k];
                        if constexpr (T == ST_Q6_K) c = __builtin_fmaf(16.0f, cb2[t][mt][k], c);
                        acc[t][mt][k] = __builtin_fmaf(d, c, acc[t][mt][k]);
                        if constexpr (F::MIN)
                            acc[t][mt][k] = __builtin_fmaf(-16.0f * ph_hhi(h[t][0]), cm[t][mt][k], acc[t][mt][k]);
                    }
            }
        }
    };
    // Every load is unconditional (past the last block, the last one again): a
    // wait after a branch around loads would be for all of them.
#pragma unroll
    for (int i = 0; i < AD; i++) a_load(i, i);
    w_load(0);
    a_store(0, 0);
    if constexpr (AD > 1) a_load(AD, 0);
    __syncthreads();
    // a group, or two blocks, a turn: a block's alignment, a record slot's
    // registers and where a group starts are then known at compile time
    constexpr int U = G < 2 ? 2 : G;
    for (int b0 = 0; b0 < nbi; b0 += U) {
#pragma unroll
        for (int i = 0; i < 2 * U; i++) {
            const int b = b0 + i / 2, hb = i % 2, t_st = 2 * b + hb;
            if (b >= nbi) break;
            if constexpr (AD == 1) a_load(t_st + 1, 0);
            if (i % (2 * G) == 0) {   // a new group
                w_store();
                w_load(b + G < nbi ? b + G : b);
                asm volatile("" ::: "memory");
            }
            const int o = (i / 2 % G) * F::BB + (G == 1 && F::BB % 4 ? i / 2 * 2 : 0);
            if (whole) {
                if (F::BB % 4 && (i / 2) % 2) half(PhBool<true>{}, o, hb);
                else half(PhBool<false>{}, o, hb);
            }
            // the next half's records to LDS (the buffer the half before used)
            if constexpr (AD == 1) {
                a_store(t_st + 1, 0);
            } else {
                a_store(t_st + 1, (i + 1) % AD);
                a_load(t_st + 1 + AD, (i + 1) % AD);
            }
            __syncthreads();
        }
    }
    // y = s_pair * acc; lane: pairs 16 mt + 4 g + k, rows grow + 16 t + n
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int m = 16 * mt + 4 * g + k;
            if (m >= nv) continue;
            const float sp = srow[m];
            float *o = out + (int64_t)pair[m] * ld_out + grow + n;
            if constexpr (GU) {
                o[0] = silu_f32(acc[0][mt][k] * sp) * (acc[1][mt][k] * sp);
            } else {
                o[0] = acc[0][mt][k] * sp;
                o[16] = acc[1][mt][k] * sp;
            }
        }
}

// The unit's row tables: record offset, pair and scale of its rows (those
// past its pairs repeat the first; their outputs are discarded).
__device__ __forceinline__ void ph_unit_rows(const int32_t *pairs, int nv, bool by_token, int32_t n_sel, int64_t ldr,
                                             const float *scale, uint8_t *smem, int64_t *&roff, int32_t *&pair,
                                             float *&srow) {
    roff = (int64_t *)(smem + PH_O_ROWS);
    pair = (int32_t *)(roff + PH_UM);
    srow = (float *)(pair + PH_UM);
    if (threadIdx.x < PH_UM) {
        const int32_t p = pairs[threadIdx.x < (unsigned)nv ? (int)threadIdx.x : 0];
        const int64_t row = by_token ? (int64_t)(p / n_sel) : (int64_t)p;
        pair[threadIdx.x] = p;
        roff[threadIdx.x] = row * ldr;
        srow[threadIdx.x] = scale[row];
    }
    __syncthreads();
}

// The launch has one workgroup per row slice (gate/up: 128 rows of each
// matrix; down: 256 rows) and unit.
#define PH_CASE(T, GU)                                                                                         \
    case T:                                                                                                    \
        if (nv > 48) ph_proj<T, GU, 4>(smem, W0, W1, row_bytes, nb, rec, roff, pair, srow, nv, r0, rows, out, ld_out); \
        else if (nv > 32) ph_proj<T, GU, 3>(smem, W0, W1, row_bytes, nb, rec, roff, pair, srow, nv, r0, rows, out, ld_out); \
        else if (nv > 16) ph_proj<T, GU, 2>(smem, W0, W1, row_bytes, nb, rec, roff, pair, srow, nv, r0, rows, out, ld_out); \
        else ph_proj<T, GU, 1>(smem, W0, W1, row_bytes, nb, rec, roff, pair, srow, nv, r0, rows, out, ld_out); \
        break;
template <bool GU>
__device__ __forceinline__ void ph_run(int32_t type, uint8_t *smem, const uint8_t *W0, const uint8_t *W1,
                                       uint64_t row_bytes, int64_t nb, const uint8_t *rec, const int64_t *roff,
                                       const int32_t *pair, const float *srow, int nv, int64_t r0, int64_t rows,
                                       float *out, int64_t ld_out) {
    switch (type) {
        PH_CASE(ST_IQ2_XS, GU)
        PH_CASE(ST_IQ3_XXS, GU)
        PH_CASE(ST_IQ4_XS, GU)
        PH_CASE(ST_Q2_K, GU)
        PH_CASE(ST_Q3_K, GU)
        PH_CASE(ST_Q4_K, GU)
        PH_CASE(ST_Q5_K, GU)
        PH_CASE(ST_Q6_K, GU)
        PH_CASE(ST_Q8_0, GU)
    default: break;
    }
}
// 256-column blocks of a row (a projection's n_blocks counts Q8_0's
// 32-column blocks; its 256-column block is eight of them, 272 bytes).
__device__ __forceinline__ int64_t ph_nb(int32_t t, int64_t n_blocks) { return t == ST_Q8_0 ? n_blocks / 8 : n_blocks; }

// Gate/up: workgroup (128-row slice bx of I, unit by); hf[p][row] = silu(gate
// . x_t) * (up . x_t) in f32 for the unit's pairs p (token t = p / n_sel).
// The host launches it only when every projection of the layer has one of
// the formats above, with 4-byte-aligned rows, and H and I are multiples of
// 256.
extern "C" __global__ __launch_bounds__(64 * PH_WAVES) void sepia_ph_gateup(
    PfProj gate, PfProj up, PfProj s_gate, PfProj s_up, int32_t n_routed, int32_t n_sel, int64_t I, int64_t H,
    const uint8_t *__restrict__ phx, const float *__restrict__ phxs, const int32_t *__restrict__ list,
    const int32_t *__restrict__ units, const int32_t *__restrict__ n_units, float *__restrict__ hf) {
    const PfSlot slot = pf_slot(n_units[0]);
    if (slot.y >= n_units[0]) return;
    extern __shared__ __attribute__((aligned(16))) uint8_t pf_smem[];
    const int32_t *un = units + 3 * slot.y;
    const int32_t e = un[0], nv = un[2];
    const bool routed = e < n_routed;
    const PfProj &G = routed ? gate : s_gate, &U = routed ? up : s_up;
    const int64_t ei = routed ? e : e - n_routed;
    int64_t *roff;
    int32_t *pair;
    float *srow;
    ph_unit_rows(list + un[1], nv, true, n_sel, (H / 128) * PH_REC, phxs, pf_smem, roff, pair, srow);
    ph_run<true>(G.type, pf_smem, G.base + ei * G.stride, U.base + ei * U.stride, G.row_bytes, ph_nb(G.type, G.n_blocks),
                 phx, roff, pair, srow, nv, slot.x * 128, I, hf, I);
}

// Down: workgroup (256-row slice bx of H, unit by); yp[p][row] = down_e .
// h_p in f32 (h_p the PH row p). Same launch conditions.
extern "C" __global__ __launch_bounds__(64 * PH_WAVES) void sepia_ph_down(
    PfProj down, PfProj s_down, int32_t n_routed, int64_t I, int64_t H, const uint8_t *__restrict__ phh,
    const float *__restrict__ phhs, const int32_t *__restrict__ list, const int32_t *__restrict__ units,
    const int32_t *__restrict__ n_units, float *__restrict__ yp) {
    const PfSlot slot = pf_slot(n_units[0]);
    if (slot.y >= n_units[0]) return;
    extern __shared__ __attribute__((aligned(16))) uint8_t pf_smem[];
    const int32_t *un = units + 3 * slot.y;
    const int32_t e = un[0], nv = un[2];
    const bool routed = e < n_routed;
    const PfProj &D = routed ? down : s_down;
    const int64_t ei = routed ? e : e - n_routed;
    const uint8_t *wd = D.base + ei * D.stride;
    int64_t *roff;
    int32_t *pair;
    float *srow;
    ph_unit_rows(list + un[1], nv, false, 1, (I / 128) * PH_REC, phhs, pf_smem, roff, pair, srow);
    ph_run<false>(D.type, pf_smem, wd, wd, D.row_bytes, ph_nb(D.type, D.n_blocks), phh, roff, pair, srow, nv, slot.x * 256,
                  H, yp, H);
}
