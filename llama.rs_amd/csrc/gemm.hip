// gemm.hip — dequantize x GEMM for batched prefill on the gfx950 matrix cores.
//
// Y[m][n] = sum_k A[m][k] * W[n][k]: A = M tokens x K activations (f32, packed
// by the producing kernel or launch_gemm_pack, gemm_pack.h), W = a resident
// N x K GGUF weight (Q4_K, Q5_K, Q6_K or Q8_0).  Replaces the reference's
// prefill GEMM (shaders/mul_mm.comp, dispatched by matmul::dispatch_mul_mm_q4k,
// crates/llama-vulkan/src/matmul.rs:433-465), which quantizes A to int8.
//   precision 1  A and dequant(W) rounded to bf16 once, f32 accumulation
//   precision 3  f32-grade, for prefill whose logits must match the f32
//                forward: the weights go to the matrix cores as exact whole
//                numbers in f16 (sub-block scale times quant: at most 1953 for
//                Q4_K / Q5_K; Q6_K products above 2048 and Q8_0's f16 scale
//                times quant as f16 hi + lo), the activations as f16 hi + lo
//                (22 bits under their super-block's own power of two).  Two
//                products a weight (three for Q6_K / Q8_0) accumulate in f32
//                over a super-block of 256; its f16 scale and the activations'
//                power of two multiply the sum once (fold).  The K-quant
//                minima are one more K-step: minima x sub-block sums.
// With both operands split into bf16 hi + lo and three products this took 1.7
// times as long (32B gate / up at 512 tokens 978 -> 575 us; bf16 hi + lo is
// 4e-6 from the 64-bit result, this 2e-7 to 3e-7).
//
// Tiling.  A 256-thread workgroup owns 32 MT tokens x 256 weight rows, each of
// its four wavefronts MT x 2 tiles of 32 x 32.  A wavefront unpacks its own 64
// rows' weights from registers straight into matrix operands, so weights never
// go through LDS and no wavefront waits for another's dequant; the activations
// are copied to LDS by global_load_lds in the order in which they are read (no
// padding, no address arithmetic, no bank conflicts).  A stage is half a
// super-block: the next stage's copies and weight loads are issued, then the
// current one computes, then one barrier.  Two independent workgroups per CU
// fill each other's waits (one workgroup of eight wavefronts in lockstep took
// 98 against 63 us at 512 x 5120 x 5120).
//
// What bounds it.  Where a CU has two workgroups at precision 3, the matrix and the
// vector pipe together (132 matrix operations of 32 clocks and about 610 vector
// operations of 4.8 clocks per wavefront and super-block; up to four vector
// operations hide behind a matrix one) and the card's power: 32B gate / up of 512
// tokens has the one busy for 60 % of the time and the other for 43 %, at 1.8 to
// 1.9 GHz, and its 1.1 PFLOP/s of products compare with 1.27 (bf16) and 1.37 (f16)
// of a large library product; down 57 and 52 %.  Fewer workgroups leave waits that
// no pipe fills: the bf16 512 x 13824 x 5120 is 216 workgroups of four row tiles
// on 256 CUs, 31 and 31 % busy at 2.2 GHz; the same at precision 3 48 and 35 %.
#include "gemm_pack.h"
#include "gemm_plan.h"
#include "quant_dev.h"

namespace lrs {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((address_space(3))) void lds_void;

constexpr int PG_MAX_SEG = 3;
struct PgSeg {
    const uint8_t *q;  // weight, tiled layout (tiled.h)
    float *y;          // [M][ldy]
    uint32_t N, ldy, nt0, noff;
};
struct PgArgs {
    // what a workgroup needs to find its tile, in one 64-byte line (spread over
    // two, a short launch starts 0.3 us later)
    const uint8_t *a;  // planes (gemm_pack.h)
    float *part;
    uint32_t nm, nn, ks, kz0, kn;  // kz0, kn: the launch's slices of the ks
    uint32_t nseg, nseg0, nsb, M, ntot;
    uint32_t accum, cont;  // cont: k_reduce_ks: y holds the sum of the slices before kz0
    PgSeg seg[PG_MAX_SEG];
};

__device__ __forceinline__ f16x2 as_h2(uint32_t v) { return __builtin_bit_cast(f16x2, v); }
// Raw bytes of one lane for 128 elements (half a super-block) of its weight
// row: lane group hf holds the pieces of 16 elements whose index is odd / even.
// A stage loads only the words it uses: a register that a load in flight will
// write and nobody reads would be handed out again, and its next use would wait
// for that load.  Q4_K / Q5_K: h0 = f16 d and dmin, sc and mn the packed scales
// and minima of the half (raw words); Q6_K: sc the half's two scale words.
template <uint32_t T> struct WHalf;
template <> struct WHalf<T_Q4_K> { uint32_t h0, h1, h2, h3; u32x4 q[2]; };
template <> struct WHalf<T_Q5_K> { uint32_t h0, h1, h2, h3; u32x4 qh, q[2]; };
template <> struct WHalf<T_Q6_K> { u32x2 sc; u32x4 la, lb, qh; uint32_t d; };
template <> struct WHalf<T_Q8_0> { u32x4 q[4]; uint32_t d[4]; };  // d: the f16 scales of the whole super-block

// Addresses: c is uniform (the chunk of the wavefront's first row tile, in
// scalar registers), o the lane's 32-bit offset to its own row tile, so that a
// load needs no 64-bit address arithmetic per lane.
__device__ __forceinline__ u32x4 ldo(const uint8_t *c, uint32_t o) { return *reinterpret_cast<const u32x4 *>(c + o); }

// Q8_0: 16-byte piece k (K-steps 2 k, 2 k + 1 of the half) of the lane's row
__device__ __forceinline__ u32x4 q8_piece(const uint8_t *c, uint32_t o, uint32_t r, uint32_t hf, int half, int k) {
    return ldo(c + (2 * half + (k >> 1)) * 1088 + 512 * (k & 1), o + 256 * hf + 16 * r);
}

// c + o = the super-block's chunk (Q8_0: its first 64-element unit's chunk) of the row's tile
template <uint32_t T, int PREC>
__device__ __forceinline__ void wload(const uint8_t *c, uint32_t o, uint32_t r, uint32_t hf, int half, WHalf<T> &w) {
    const uint32_t o0 = o + 16 * r, o1 = o0 + 256 * hf;
    if constexpr (T == T_Q4_K || T == T_Q5_K) {
        // precision 3 takes d, dmin and the minima once, with the second half
        if (half == 1) {
            const u32x4 h = ldo(c, o0);
            w.h0 = h.x, w.h1 = h.y, w.h2 = h.z, w.h3 = h.w;
        } else if (PREC == 3) {
            w.h1 = *reinterpret_cast<const uint32_t *>(c + 4 + o0);
        } else {
            w.h0 = *reinterpret_cast<const uint32_t *>(c + o0);
            const u32x2 h = *reinterpret_cast<const u32x2 *>(c + 4 + o0);
            w.h1 = h.x, w.h2 = h.y;
        }
    }
    if constexpr (T == T_Q4_K) {
        w.q[0] = ldo(c + 256 + 1024 * half, o1);
        w.q[1] = ldo(c + 768 + 1024 * half, o1);
    } else if constexpr (T == T_Q5_K) {
        w.qh = ldo(c + 256, o1);
        w.q[0] = ldo(c + 768 + 1024 * half, o1);
        w.q[1] = ldo(c + 1280 + 1024 * half, o1);
    } else if constexpr (T == T_Q6_K) {
        w.sc = *reinterpret_cast<const u32x2 *>(c + 8 * half + o0);
        w.la = ldo(c + 256 + 512 * half, o1);
        w.lb = ldo(c + 1280 + 512 * half, o1);
        w.qh = ldo(c + 2304 + 512 * half, o1);
        if (PREC == 1 || half == 1) w.d = *reinterpret_cast<const uint16_t *>(c + 3328 + (o + 2 * r));
    } else {
#pragma unroll
        for (int k = 0; k < 4; k++) w.q[k] = q8_piece(c, o, r, hf, half, k);
#pragma unroll
        for (int u = 0; u < 4; u++) w.d[u] = *reinterpret_cast<const uint32_t *>(c + u * 1088 + 1024 + (o + 4 * r));
    }
}

// the 6-bit scales (minima) of sub-blocks 4 half .. 4 half + 3 as bytes of a
// word, from header words h1 (h2) and h3
template <class W>
__device__ __forceinline__ uint32_t k4_scales(const W &w, int half) {
    return half == 0 ? w.h1 & 0x3F3F3F3Fu : (w.h3 & 0x0F0F0F0Fu) | ((w.h1 >> 2) & 0x30303030u);
}
template <class W>
__device__ __forceinline__ uint32_t k4_mins(const W &w, int half) {
    return half == 0 ? w.h2 & 0x3F3F3F3Fu : ((w.h3 >> 4) & 0x0F0F0F0Fu) | ((w.h2 >> 2) & 0x30303030u);
}

// words 2 pair, 2 pair + 1 of a piece
__device__ __forceinline__ uint32_t pw(const u32x4 &v, int pair, int i) { return v[2 * pair + i]; }

// Q8_0: the f16 scales of a super-block share a power of two 2^ex > max |d|
// (an f16 scale over it is a fraction, exact in f16 but for scales 2^14 below
// the largest, whose last bits fall under 2^-24 of it)
__device__ __forceinline__ int q8_exp(const uint32_t (&d)[4]) {
    uint32_t m = 0;
#pragma unroll
    for (int u = 0; u < 4; u++) m = max(m, max(d[u] & 0x7FFFu, (d[u] >> 16) & 0x7FFFu));
    int ex;
    (void)frexpf(h2f((uint16_t)m), &ex);
    return m ? ex : 0;
}

// (v & M) | 0x64006400 (two f16 of 1024 + the masked bits) as one instruction:
// the constants are hidden from the compiler, which would fold them into two
// instructions with a literal each
template <uint32_t M>
__device__ __forceinline__ uint32_t and_1024(uint32_t v) {
    uint32_t m = M, k = 0x64006400u;
    asm("" : "+s"(m));
    asm("" : "+v"(k));
    return (v & m) | k;
}
// the bytes (b0, b2) or (b1, b3) of a word as a pair of f16 whole numbers + 1024
__device__ __forceinline__ f16x2 pair02(uint32_t v) { return as_h2((v & 0x00FF00FFu) | 0x64006400u); }
__device__ __forceinline__ f16x2 pair13(uint32_t v) { return pair02(v >> 8); }
__device__ __forceinline__ f16x2 both(_Float16 v) { return f16x2{v, v}; }
__device__ __forceinline__ f16x2 both(float v) { return both((_Float16)v); }

// the f16 scales of half a super-block's K-steps 2 s, 2 s + 1 (s = 0..3)
template <uint32_t T> struct SHalf { f16x2 a, b; };  // (s = 0, 2), (s = 1, 3); Q6_K: (0, 1), (2, 3)
template <uint32_t T>
__device__ __forceinline__ SHalf<T> scales(const WHalf<T> &w, int half, uint32_t hf, int ex) {
    SHalf<T> s;
    if constexpr (T == T_Q4_K || T == T_Q5_K) {
        // the odd sub-blocks are the high nibbles, unpacked times 16
        const uint32_t v = k4_scales(w, half);
        s.a = pair02(v) - both(1024.0f);
        s.b = (pair13(v) - both(1024.0f)) * both(0.0625f);
    } else if constexpr (T == T_Q6_K) {
        // int8 scales 8 half + 2 quarter + hf
        s.a = pair02((w.sc.x >> (8 * hf)) ^ 0x00800080u) - both(1152.0f);
        s.b = pair02((w.sc.y >> (8 * hf)) ^ 0x00800080u) - both(1152.0f);
    } else {
        float d[4];
#pragma unroll
        for (int i = 0; i < 4; i++) d[i] = ldexpf(h2f((uint16_t)(w.d[2 * half + (i >> 1)] >> (16 * (i & 1)))), -ex);
        s.a = f16x2{(_Float16)d[0], (_Float16)d[2]};
        s.b = f16x2{(_Float16)d[1], (_Float16)d[3]};
    }
    return s;
}

// B operand of K-step t (0..7 of the half) for precision 3: bh + bl is the
// weight without the super-block's factor (fold), exact
template <uint32_t T>
__device__ __forceinline__ void bfrag_int(const WHalf<T> &w, const SHalf<T> &sc, int half, int t, f16x8 &bh, f16x8 &bl) {
    const int s = t >> 1, pair = t & 1;
    const f16x2 sv = T == T_Q6_K ? both(s < 2 ? sc.a[s & 1] : sc.b[s & 1]) : both(s & 1 ? sc.b[s >> 1] : sc.a[s >> 1]);
    // the constants that take the unpacking offset off: -1024 sc (K-quants)
    const f16x2 cv = sv * both(-1024.0f);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        f16x2 f[2];
        if constexpr (T == T_Q4_K || T == T_Q5_K) {
            // (1024 + q) sc - 1024 sc, or with the nibble in bits 4..7
            // (1024 + 16 q) sc / 16 - 64 sc: whole numbers up to 1953, exact
            const int hi = s & 1;
            const uint32_t v = pw(w.q[s >> 1], pair, i);
            uint32_t e0 = hi ? and_1024<0x00F000F0u>(v) : and_1024<0x000F000Fu>(v);
            uint32_t e1 = hi ? and_1024<0x00F000F0u>(v >> 8) : and_1024<0x000F000Fu>(v >> 8);
            if constexpr (T == T_Q5_K) {
                const uint32_t h = pw(w.qh, pair, i) >> (4 * half + s);
                e0 |= (h & 0x00010001u) << (hi ? 8 : 4);
                e1 |= ((h >> 8) & 0x00010001u) << (hi ? 8 : 4);
            }
            f[0] = __builtin_elementwise_fma(as_h2(e0), sv, cv);
            f[1] = __builtin_elementwise_fma(as_h2(e1), sv, cv);
        } else {
            // whole numbers q times the scale, rounded to f16, and the exact
            // remainder of that rounding (Q6_K: of products above 2048)
            f16x2 q0, q1;
            if constexpr (T == T_Q6_K) {
                const uint32_t l = pw((s & 1) ? w.lb : w.la, pair, i) >> (4 * (s >> 1));
                const uint32_t hb = pw(w.qh, pair, i);
                const uint32_t h = s == 0 ? hb << 4 : s == 1 ? hb << 2 : s == 2 ? hb : hb >> 2;
                q0 = as_h2(and_1024<0x000F000Fu>(l) | (h & 0x00300030u)) - both(1056.0f);
                q1 = as_h2(and_1024<0x000F000Fu>(l >> 8) | ((h >> 8) & 0x00300030u)) - both(1056.0f);
            } else {
                const uint32_t v = pw(w.q[s], pair, i) ^ 0x80808080u;
                q0 = pair02(v) - both(1152.0f);
                q1 = pair13(v) - both(1152.0f);
            }
            f[0] = q0 * sv;
            f[1] = q1 * sv;
            const f16x2 g0 = __builtin_elementwise_fma(q0, sv, -f[0]), g1 = __builtin_elementwise_fma(q1, sv, -f[1]);
            bl[4 * i] = g0[0];
            bl[4 * i + 1] = g0[1];
            bl[4 * i + 2] = g1[0];
            bl[4 * i + 3] = g1[1];
        }
        bh[4 * i] = f[0][0];
        bh[4 * i + 1] = f[0][1];
        bh[4 * i + 2] = f[1][0];
        bh[4 * i + 3] = f[1][1];
    }
}

// precision 1: the f32 scale and offset of K-steps 2 s, 2 s + 1 of a half
template <uint32_t T> struct AHalf { float a[4], o[4]; };
template <uint32_t T>
__device__ __forceinline__ AHalf<T> affine(const WHalf<T> &w, int half, uint32_t hf) {
    AHalf<T> r;
#pragma unroll
    for (int s = 0; s < 4; s++) {
        if constexpr (T == T_Q4_K || T == T_Q5_K) {
            const uint32_t sc = (k4_scales(w, half) >> (8 * s)) & 0xFF, m = (k4_mins(w, half) >> (8 * s)) & 0xFF;
            r.a[s] = __fmul_rn(h2f((uint16_t)(w.h0 & 0xFFFF)), (float)sc);
            r.o[s] = -__fmul_rn(h2f((uint16_t)(w.h0 >> 16)), (float)m);
        } else if constexpr (T == T_Q6_K) {
            const uint32_t sw = w.sc[s >> 1] >> (16 * (s & 1));
            r.a[s] = __fmul_rn(h2f((uint16_t)w.d), (float)(int8_t)((sw >> (8 * hf)) & 0xFF));
        } else {
            r.a[s] = h2f((uint16_t)(w.d[2 * half + (s >> 1)] >> (16 * (s & 1))));
        }
    }
    return r;
}

// B operand of K-step t, precision 1: the weights in f32 (one fused
// multiply-add each: dequant.rs's value for Q6_K and Q8_0; Q4_K / Q5_K without
// the rounding of d sc q), rounded to bf16
template <uint32_t T>
__device__ __forceinline__ bf16x8 bfrag_bf16(const WHalf<T> &w, const AHalf<T> &af, int half, int t) {
    const int s = t >> 1, pair = t & 1;
    const float o = T == T_Q6_K ? -32.0f * af.a[s] : T == T_Q8_0 ? -128.0f * af.a[s] : af.o[s];  // exact products
    u32x4 b;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        uint32_t q;
        if constexpr (T == T_Q8_0) {
            q = pw(w.q[s], pair, i) ^ 0x80808080u;
        } else if constexpr (T == T_Q6_K) {
            const uint32_t hb = pw(w.qh, pair, i);
            q = ((pw((s & 1) ? w.lb : w.la, pair, i) >> (4 * (s >> 1))) & 0x0F0F0F0Fu) |
                ((s == 0 ? hb << 4 : s == 1 ? hb << 2 : s == 2 ? hb : hb >> 2) & 0x30303030u);
        } else {
            q = (pw(w.q[s >> 1], pair, i) >> (4 * (s & 1))) & 0x0F0F0F0Fu;
            if constexpr (T == T_Q5_K) q |= ((pw(w.qh, pair, i) >> (4 * half + s)) & 0x01010101u) << 4;
        }
        // hidden: the compiler would turn the byte conversions into shifts,
        // knowing which bits of the bytes are set
        asm("" : "+v"(q));
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = fmaf(af.a[s], (float)((q >> (8 * k)) & 0xFF), o);
        typedef __attribute__((ext_vector_type(2))) float f32x2;
        b[2 * i] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{v[0], v[2]}), bf16x2));
        b[2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{v[1], v[3]}), bf16x2));
    }
    return __builtin_bit_cast(bf16x8, b);
}

// the eight minima as f16, in the order of the sub-block sums
template <class W>
__device__ __forceinline__ f16x8 min_frag(const W &w) {
    f16x8 m;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t v = k4_mins(w, i);
        const f16x2 f0 = pair02(v) - both(1024.0f), f1 = pair13(v) - both(1024.0f);
        m[4 * i] = f0[0];
        m[4 * i + 1] = f0[1];
        m[4 * i + 2] = f1[0];
        m[4 * i + 3] = f1[1];
    }
    return m;
}

template <int PREC, int MT> struct PgLds {
    static constexpr int STEP = PREC == 3 ? 2048 : 1024;  // bytes of a K-step of a row tile
    static constexpr int STAGE = MT * 8 * STEP;
    static constexpr int SUMS = PREC == 3 ? MT * 2048 : 16;
};

template <uint32_t T, int PREC, int MT, int NT> struct PgTile {
static __device__ __forceinline__ void run(const PgArgs &g, const PgSeg &sg, uint32_t kz, uint32_t mb, uint32_t n0,
                                           uint8_t *As0, uint8_t *As1, uint8_t *Ss) {
    using L = PgLds<PREC, MT>;
    constexpr uint32_t BB = gemm_block_bytes(PREC);
    constexpr bool MINS = T == T_Q4_K || T == T_Q5_K;
    const uint32_t tid = threadIdx.x, lane = tid & 63, hf = lane >> 5;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t s0 = kz * g.nsb / g.ks, s1 = (kz + 1) * g.nsb / g.ks;  // super-blocks of the K slice
    const uint32_t nw0 = n0 + 32 * NT * wave;  // this wavefront's rows
    const uint32_t nmt = (g.M + 31) / 32;

    constexpr uint32_t CH = T == T_Q8_0 ? 4 * tchunk_bytes(T) : tchunk_bytes(T);  // bytes per super-block
    const uint32_t r = lane & 15, last = (sg.N + 15) / 16 - 1;
    const uint32_t tile0 = min(nw0 / 16, last);
    const uint8_t *const wp = sg.q + (size_t)tile0 * g.nsb * CH;
    uint32_t wo[NT];
#pragma unroll
    for (int i = 0; i < NT; i++) wo[i] = (min(nw0 / 16 + 2 * i + ((lane >> 4) & 1), last) - tile0) * g.nsb * CH;
    // activation blocks of the row tiles (past the last one: a copy of it)
    const uint8_t *ap[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) ap[i] = g.a + (size_t)min(mb * MT + i, nmt - 1) * g.nsb * BB;

    auto dma = [&](uint32_t sb, int half, uint8_t *dst) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int u = 0; u < 8 * L::STEP / 1024 / PG_WAVES; u++) {
                const uint32_t un = wave + PG_WAVES * u;
                __builtin_amdgcn_global_load_lds(ap[i] + ((size_t)sb * BB + half * 8 * L::STEP + 1024 * un) + 16 * lane,
                                                 (lds_void *)(dst + i * 8 * L::STEP + 1024 * un), 16, 0, 0);
            }
    };
    auto dma_sums = [&](uint32_t sb) __attribute__((always_inline)) {
        if constexpr (PREC == 3) {
            if (wave < 2)
#pragma unroll
                for (int i = 0; i < MT; i++)
                    __builtin_amdgcn_global_load_lds(ap[i] + (size_t)sb * BB + GP_SUMS + 1024 * wave + 16 * lane,
                                                     (lds_void *)(Ss + (sb & 1) * L::SUMS + i * 2048 + 1024 * wave),
                                                     16, 0, 0);
        }
    };

    f32x16 tot[MT][NT], acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) tot[i][j][e] = 0.f;

    auto scale4 = [&](uint32_t sb, int i, int q) __attribute__((always_inline)) {
        return *reinterpret_cast<const float4 *>(Ss + (sb & 1) * L::SUMS + i * 2048 + 1024 + 4 * (8 * q + 4 * hf));
    };
    // one half of a super-block from its LDS stage
    // operands of a K-step: the activations' hi (and lo) parts, the weights'
    // hi (and for Q6_K and Q8_0 lo) parts; precision 1 uses the hi members
    constexpr bool LO = PREC == 3 && (T == T_Q6_K || T == T_Q8_0);
    struct FragA { u32x4 h[MT], l[PREC == 3 ? MT : 1]; };
    struct FragB { u32x4 h[NT], l[LO ? NT : 1]; };
    // Half a super-block from its LDS stage.  The operands of K-step t + 1 are
    // read and unpacked while step t's matrix operations run: the scheduling
    // groups put about as many vector operations behind each matrix operation
    // as there are.
    auto compute = [&](int half, const uint8_t *As, WHalf<T> (&w)[NT], const uint8_t *nxt, int nhalf)
                       __attribute__((always_inline)) {
        SHalf<T> sc[NT];
        AHalf<T> af[NT];
#pragma unroll
        for (int j = 0; j < NT; j++) {
            if constexpr (PREC == 3) {
                int ex = 0;
                if constexpr (T == T_Q8_0) ex = q8_exp(w[j].d);
                sc[j] = scales<T>(w[j], half, hf, ex);
            } else {
                af[j] = affine<T>(w[j], half, hf);
            }
        }
        FragA fa[2];
        FragB fb[2];
        auto lfrag = [&](int t, FragA &A, FragB &B) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < MT; i++) {
                A.h[i] = *reinterpret_cast<const u32x4 *>(As + (i * 8 + t) * L::STEP + 16 * lane);
                if constexpr (PREC == 3)
                    A.l[i] = *reinterpret_cast<const u32x4 *>(As + (i * 8 + t) * L::STEP + 1024 + 16 * lane);
            }
#pragma unroll
            for (int j = 0; j < NT; j++) {
                if constexpr (PREC == 3) {
                    f16x8 bh, bl;
                    bfrag_int<T>(w[j], sc[j], half, t, bh, bl);
                    B.h[j] = __builtin_bit_cast(u32x4, bh);
                    if constexpr (LO) B.l[j] = __builtin_bit_cast(u32x4, bl);
                } else {
                    B.h[j] = __builtin_bit_cast(u32x4, bfrag_bf16<T>(w[j], af[j], half, t));
                }
            }
        };
        auto mma = [&](const u32x4 &a, const u32x4 &b, f32x16 &c) __attribute__((always_inline)) {
            if constexpr (PREC == 3)
                c = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b),
                                                           c, 0, 0, 0);
            else
                c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                            __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
        };
        if (PREC == 3 && half == 0) {
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;
        }
        lfrag(0, fa[0], fb[0]);
#pragma unroll
        for (int t = 0; t < 8; t++) {
            if (t < 7) lfrag(t + 1, fa[(t + 1) & 1], fb[(t + 1) & 1]);
            const FragA &A = fa[t & 1];
            const FragB &B = fb[t & 1];
            if constexpr (LO) {
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int i = 0; i < MT; i++) mma(A.h[i], B.l[j], acc[i][j]);
            }
            if constexpr (PREC == 3) {
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int i = 0; i < MT; i++) mma(A.l[i], B.h[j], acc[i][j]);
            }
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int i = 0; i < MT; i++) mma(A.h[i], B.h[j], PREC == 3 ? acc[i][j] : tot[i][j]);
            constexpr int NM = MT * NT * (LO ? 3 : PREC == 3 ? 2 : 1);  // matrix operations of a step
            constexpr int NV = PREC == 1 ? (NT * 25 + NM - 1) / NM : LO ? 6 : 5;
#pragma unroll
            for (int z = 0; z < NM; z++) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);   // a matrix operation
                __builtin_amdgcn_sched_group_barrier(0x2, NV, 0);  // vector operations
                if (z < (PREC == 3 ? 2 : 1) * MT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // an LDS read
            }
            if constexpr (T == T_Q8_0) {
                if (t & 1)
#pragma unroll
                    for (int j = 0; j < NT; j++) w[j].q[t >> 1] = q8_piece(nxt, wo[j], r, hf, nhalf, t >> 1);
            }
        }
    };
    // the super-block's whole-number sums times its scales, into the totals
    auto fold = [&](uint32_t sb, const WHalf<T> (&w)[NT]) __attribute__((always_inline)) {
        if constexpr (PREC == 3) {
#pragma unroll
            for (int j = 0; j < NT; j++) {
                float d, dm = 0.f;
                f16x8 mf;
                if constexpr (T == T_Q6_K) {
                    d = h2f((uint16_t)w[j].d);
                } else if constexpr (T == T_Q8_0) {
                    d = ldexpf(1.0f, q8_exp(w[j].d));
                } else {
                    d = h2f((uint16_t)(w[j].h0 & 0xFFFF));
                    dm = h2f((uint16_t)(w[j].h0 >> 16));
                    mf = min_frag(w[j]);
                }
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    f32x16 q;
                    if constexpr (MINS) {
                        const f16x8 sf =
                            *reinterpret_cast<const f16x8 *>(Ss + (sb & 1) * L::SUMS + i * 2048 + 16 * lane);
#pragma unroll
                        for (int e = 0; e < 16; e++) q[e] = 0.f;
                        q = __builtin_amdgcn_mfma_f32_32x32x16_f16(sf, mf, q, 0, 0, 0);
                    }
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float4 s = scale4(sb, i, e);
                        const float sv[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            const int x = 4 * e + k;
                            const float v = MINS ? fmaf(acc[i][j][x], d, -(q[x] * dm)) : acc[i][j][x] * d;
                            tot[i][j][x] = fmaf(v, sv[k], tot[i][j][x]);
                        }
                    }
                }
            }
        }
    };
    auto sync = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wavefront's copies and loads have arrived
        __syncthreads();
    };

    // Stages of half a super-block: the next stage's copy and weight loads are
    // issued first, then the current one computes from the other LDS array.
    // Q8_0 holds one set of weight registers (its pieces are the widest) and
    // refills each piece once its K-steps are done.
    WHalf<T> w0[NT], w1[NT];
    const uint8_t *cw = wp + (size_t)s0 * CH;
    dma(s0, 0, As0);
    dma_sums(s0);
#pragma unroll
    for (int j = 0; j < NT; j++) wload<T, PREC>(cw, wo[j], r, hf, 0, w0[j]);
    sync();
    for (uint32_t sb = s0; sb < s1; sb++) {
        const uint32_t nx = min(sb + 1, s1 - 1);  // past the end: the last block again, unused
        const uint8_t *nw = wp + (size_t)nx * CH;
        dma(sb, 1, As1);
        if constexpr (T != T_Q8_0)
#pragma unroll
            for (int j = 0; j < NT; j++) wload<T, PREC>(cw, wo[j], r, hf, 1, w1[j]);
        __builtin_amdgcn_sched_barrier(0);
        compute(0, As0, w0, cw, 1);
        sync();
        dma(nx, 0, As0);
        if (sb + 1 < s1) dma_sums(nx);
        if constexpr (T != T_Q8_0)
#pragma unroll
            for (int j = 0; j < NT; j++) wload<T, PREC>(nw, wo[j], r, hf, 0, w0[j]);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (T == T_Q8_0) {
            compute(1, As1, w0, nw, 0);
            fold(sb, w0);
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int u = 0; u < 4; u++)
                    w0[j].d[u] = *reinterpret_cast<const uint32_t *>(nw + u * 1088 + 1024 + (wo[j] + 4 * r));
        } else {
            compute(1, As1, w1, nw, 0);
            fold(sb, w1);
        }
        cw = nw;
        sync();
    }
    // D layout: lane l, register e -> row 8(e/4) + 4(l/32) + e%4, column l%32
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const uint32_t n = nw0 + 32 * j + (lane & 31);
        if (n >= sg.N) continue;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const uint32_t m = 32 * (mb * MT + i) + 8 * (e >> 2) + 4 * hf + (e & 3);
                if (m < g.M) {
                    if (g.kn > 1) {
                        g.part[((size_t)(kz - g.kz0) * g.M + m) * g.ntot + sg.noff + n] = tot[i][j][e];
                    } else {
                        float *o = sg.y + (size_t)m * sg.ldy + n;
                        *o = g.accum ? *o + tot[i][j][e] : tot[i][j][e];
                    }
                }
            }
    }
}
};

template <uint32_t T0, uint32_t T1, int PREC, int MT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_pgemm(PgArgs g) {
    using L = PgLds<PREC, MT>;
    constexpr int NT = 2;  // weight-row tiles of 32 per wavefront
    __shared__ __attribute__((aligned(16))) uint8_t As0[L::STAGE];
    __shared__ __attribute__((aligned(16))) uint8_t As1[L::STAGE];
    __shared__ __attribute__((aligned(16))) uint8_t Ss[2 * L::SUMS];
    const uint32_t ntile = g.nm * g.nn * g.kn, per = (ntile + 7) / 8;
    const uint32_t t0 = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per || t0 >= ntile) return;
    // row tiles of one weight tile run next to each other (they share its bytes
    // in an XCD's L2); the last segment, of the slower type, starts first
    const uint32_t mb = t0 % g.nm, t = t0 / g.nm, nt = g.nn - 1 - t % g.nn, kz = g.kz0 + t / g.nn;
    uint32_t si = 0;
#pragma unroll
    for (int i = 1; i < PG_MAX_SEG; i++)
        if ((uint32_t)i < g.nseg && nt >= g.seg[i].nt0) si = i;
    const PgSeg sg = g.seg[si];
    const uint32_t n0 = (nt - sg.nt0) * 32 * NT * PG_WAVES;
    if (T0 == T1 || si < g.nseg0)
        PgTile<T0, PREC, MT, NT>::run(g, sg, kz, mb, n0, As0, As1, Ss);
    else
        PgTile<T1, PREC, MT, NT>::run(g, sg, kz, mb, n0, As0, As1, Ss);
}



// y[m][n] (+)= sum over the K slices of part[z][m][noff + n], slices in order,
// four outputs per thread (N % 4 == 0, else one)
template <int V>
__global__ __launch_bounds__(256) void k_reduce_ks(PgArgs g) {
    const PgSeg sg = g.seg[blockIdx.z];
    const uint32_t n = V * (blockIdx.x * 256 + threadIdx.x), m = blockIdx.y;
    if (n >= sg.N) return;
    typedef __attribute__((ext_vector_type(V))) float fv;
    const float *p = g.part + (size_t)m * g.ntot + sg.noff + n;
    const size_t st = (size_t)g.M * g.ntot;
    fv *o = reinterpret_cast<fv *>(sg.y + (size_t)m * sg.ldy + n);
    fv v = *reinterpret_cast<const fv *>(p);
    if (g.cont) v = *o + v;
    for (uint32_t z = 1; z < g.kn; z++) v += *reinterpret_cast<const fv *>(p + z * st);
    *o = g.accum ? *o + v : v;
}

// rows of f32 into the GEMM's input layout: workgroup = 32 rows x one super-block
template <int PREC>
__global__ __launch_bounds__(256) void k_gemm_pack(const float *__restrict__ a, uint32_t M, uint32_t nsb,
                                                   uint8_t *__restrict__ p) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const uint32_t row = 32 * (blockIdx.x / nsb) + 8 * i + (threadIdx.x >> 5);
        const uint32_t c = 32 * (blockIdx.x % nsb) + (threadIdx.x & 31);
        if (row >= M) return;
        const float *x = a + ((size_t)row * nsb) * 256 + 8 * c;
        const float4 u = *reinterpret_cast<const float4 *>(x), w = *reinterpret_cast<const float4 *>(x + 4);
        const float v[8] = {u.x, u.y, u.z, u.w, w.x, w.y, w.z, w.w};
        gp_store8<PREC>(v, row, c, nsb, p);
    }
}

hipError_t launch_gemm_pack(const float *a, uint32_t M, uint32_t K, int prec, uint8_t *planes, hipStream_t s) {
    if (M == 0 || K == 0 || K % 256) return hipErrorInvalidValue;
    const dim3 grid((M + 31) / 32 * (K / 256));
    if (prec == 3)
        hipLaunchKernelGGL((k_gemm_pack<3>), grid, dim3(256), 0, s, a, M, K / 256, planes);
    else
        hipLaunchKernelGGL((k_gemm_pack<1>), grid, dim3(256), 0, s, a, M, K / 256, planes);
    return hipGetLastError();
}

size_t gemm_planes_bytes(uint32_t M, uint32_t K, int prec) {
    return (size_t)((M + 31) / 32) * (K / 256) * gemm_block_bytes(prec);
}

using GemmFn = void (*)(PgArgs);

template <uint32_t T0, uint32_t T1>
static GemmFn pick_gemm_shape(int prec, uint32_t mt) {
    if (prec == 3) return mt == 1 ? k_pgemm<T0, T1, 3, 1> : k_pgemm<T0, T1, 3, 2>;
    return mt == 1 ? k_pgemm<T0, T1, 1, 1> : mt == 2 ? k_pgemm<T0, T1, 1, 2> : k_pgemm<T0, T1, 1, 4>;
}

// the kernel for weight types t0 (the first segments) and t1 (the rest)
static GemmFn pick_gemm(uint32_t t0, uint32_t t1, int prec, uint32_t mt) {
    if (t0 == T_Q4_K && t1 == T_Q4_K) return pick_gemm_shape<T_Q4_K, T_Q4_K>(prec, mt);
    if (t0 == T_Q5_K && t1 == T_Q5_K) return pick_gemm_shape<T_Q5_K, T_Q5_K>(prec, mt);
    if (t0 == T_Q6_K && t1 == T_Q6_K) return pick_gemm_shape<T_Q6_K, T_Q6_K>(prec, mt);
    if (t0 == T_Q8_0 && t1 == T_Q8_0) return pick_gemm_shape<T_Q8_0, T_Q8_0>(prec, mt);
    // a prompt block's q / k with a Q6_K v (the K-quant mixes)
    if (t0 == T_Q4_K && t1 == T_Q6_K) return pick_gemm_shape<T_Q4_K, T_Q6_K>(prec, mt);
    if (t0 == T_Q5_K && t1 == T_Q6_K) return pick_gemm_shape<T_Q5_K, T_Q6_K>(prec, mt);
    return nullptr;
}

bool gemm_segs_supported(const WeightView *w, uint32_t nseg) {
    if (nseg == 0 || nseg > (uint32_t)PG_MAX_SEG) return false;
    uint32_t nseg0 = 1;
    while (nseg0 < nseg && w[nseg0].type == w[0].type) nseg0++;
    for (uint32_t i = 0; i < nseg; i++) {
        if (w[i].n_in != w[0].n_in || !is_tiled(w[i].type)) return false;
        if (i >= nseg0 && w[i].type != w[nseg0].type) return false;  // at most two types, in two runs
    }
    return pick_gemm(w[0].type, w[nseg - 1].type, 3, 1) != nullptr;
}

hipError_t launch_gemm_segs(const WeightView *w, float *const *y, const uint32_t *ldy, uint32_t nseg,
                            const uint8_t *planes, uint32_t M, int prec, hipStream_t s, bool accum, float *work,
                            size_t work_bytes, uint32_t *ks_out) {
    if (M == 0 || !planes || !gemm_segs_supported(w, nseg) || w[0].n_in == 0 || w[0].n_in % 256)
        return hipErrorInvalidValue;
    uint32_t Ns[PG_MAX_SEG], ts[PG_MAX_SEG];
    for (uint32_t i = 0; i < nseg; i++) Ns[i] = w[i].n_out, ts[i] = w[i].type;
    const PgPlan p = pg_plan(M, Ns, ts, nseg, w[0].n_in / 256, prec);
    PgArgs g = {};
    g.a = planes;
    g.nseg = nseg;
    g.nseg0 = 1;
    while (g.nseg0 < nseg && w[g.nseg0].type == w[0].type) g.nseg0++;
    uint32_t nt = 0, ntot = 0, nmax = 0;
    bool v4 = true;
    for (uint32_t i = 0; i < nseg; i++) {
        const uint32_t N = w[i].n_out;
        g.seg[i] = {w[i].q, y[i], N, ldy[i], nt, ntot};
        nt += (N + PG_ROWS - 1) / PG_ROWS;
        ntot += N;
        nmax = std::max(nmax, N);
        v4 = v4 && N % 4 == 0 && ldy[i] % 4 == 0 && ((uintptr_t)y[i] & 15) == 0;
    }
    g.M = M;
    g.nsb = w[0].n_in / 256;
    // Where the scratch holds fewer partial sums than there are slices, the
    // slices go by in rounds of as many as it holds (one: straight to y), added
    // in the same order: a call's bits depend on its sizes and types alone.  A
    // sum that starts from y, or that the caller reduces, has its scratch.
    uint32_t fit = p.ks;
    if (pg_bytes(p, M, Ns, nseg) > work_bytes) {
        if (accum || ks_out) return hipErrorInvalidValue;
        fit = (uint32_t)std::max<size_t>(1, work_bytes / ((size_t)M * ntot * sizeof(float)));
    }
    g.nm = (M + 32 * p.mt - 1) / (32 * p.mt);
    g.nn = nt;
    g.ntot = ntot;
    g.ks = p.ks;
    g.part = work;
    const GemmFn fn = pick_gemm(w[0].type, w[nseg - 1].type, prec, p.mt);
    for (; g.kz0 < g.ks; g.kz0 += g.kn) {
        g.kn = std::min(fit, g.ks - g.kz0);
        g.cont = g.kz0 ? 1u : 0u;
        g.accum = accum || (g.kn == 1 && g.cont) ? 1u : 0u;
        const uint32_t grid = 8 * ((g.nm * g.nn * g.kn + 7) / 8);
        hipLaunchKernelGGL(fn, dim3(grid), dim3(64 * PG_WAVES), 0, s, g);
        if (ks_out) {
            *ks_out = g.ks;  // the caller reduces the slices (launch_norm_rows)
        } else if (g.kn > 1) {
            if (v4)
                hipLaunchKernelGGL((k_reduce_ks<4>), dim3((nmax + 1023) / 1024, M, nseg), dim3(256), 0, s, g);
            else
                hipLaunchKernelGGL((k_reduce_ks<1>), dim3((nmax + 255) / 256, M, nseg), dim3(256), 0, s, g);
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace lrs
