// quant.hip — device-layout repack, seeded synthetic blocks and bit-exact
// dequant for the GGUF block types on the decode path (gfx950).
//
// Dequant follows ggml_cpu::dequant_to_f32 (crates/ggml-cpu/src/dequant.rs:
// 58-258) element by element with the same f32 operation order; the library
// is compiled with -ffp-contract=off, so d1*q - m1 rounds twice as in Rust.
#include "lrs_internal.h"
#include "quant_dev.h"

namespace lrs {

static unsigned grid_for(uint64_t n, unsigned bs) {
    uint64_t g = (n + bs - 1) / bs;
    if (g > 65536u * 4u) g = 65536u * 4u;
    if (g == 0) g = 1;
    return (unsigned)g;
}

// ---------------------------------------------------------------------------
// GGUF row-major blocks <-> device layout (tiled.h for the matvec types, the
// GGUF bytes as they are for the others).  One thread per device word; every
// padding byte is written as zero.
// ---------------------------------------------------------------------------
__global__ void k_repack_from_gguf(const uint8_t *__restrict__ g, WeightView w, size_t dev_bytes,
                                   uint8_t *__restrict__ q) {
    const uint32_t bb = (uint32_t)block_bytes(w.type);
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < dev_bytes / 4;
         i += (size_t)gridDim.x * blockDim.x) {
        uint32_t v = 0;
        for (int k = 0; k < 4; k++) {
            uint32_t row, blk, o;
            if (tinv(w.type, w.n_in, w.n_out, 4 * i + k, row, blk, o))
                v |= (uint32_t)g[((size_t)row * w.nb + blk) * bb + o] << (8 * k);
        }
        reinterpret_cast<uint32_t *>(q)[i] = v;
    }
}

__global__ void k_repack_to_gguf(WeightView w, size_t dev_bytes, uint8_t *__restrict__ g) {
    const uint32_t bb = (uint32_t)block_bytes(w.type);
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < dev_bytes;
         i += (size_t)gridDim.x * blockDim.x) {
        uint32_t row, blk, o;
        if (tinv(w.type, w.n_in, w.n_out, i, row, blk, o)) g[((size_t)row * w.nb + blk) * bb + o] = w.q[i];
    }
}

hipError_t launch_repack_from_gguf(const uint8_t *gguf_dev, WeightView w, uint8_t *q, hipStream_t s) {
    const size_t db = weight_dev_bytes(w.type, w.n_in, w.n_out);
    if (!is_tiled(w.type)) return hipMemcpyAsync(q, gguf_dev, db, hipMemcpyDeviceToDevice, s);
    hipLaunchKernelGGL(k_repack_from_gguf, dim3(grid_for(db / 4, 256)), dim3(256), 0, s, gguf_dev, w, db, q);
    return hipGetLastError();
}

hipError_t launch_repack_to_gguf(WeightView w, uint8_t *gguf_dev, hipStream_t s) {
    const size_t db = weight_dev_bytes(w.type, w.n_in, w.n_out);
    if (!is_tiled(w.type)) return hipMemcpyAsync(gguf_dev, w.q, db, hipMemcpyDeviceToDevice, s);
    hipLaunchKernelGGL(k_repack_to_gguf, dim3(grid_for(db, 256)), dim3(256), 0, s, w, db, gguf_dev);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// seeded synthetic blocks: the same counter-based hash and field rules as the
// host generator, so any block can be regenerated bit-identically on the CPU
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}
__device__ __forceinline__ uint64_t hsh(uint64_t seed, uint64_t blk, uint32_t j) {
    return mix64(seed * 0x9E3779B97F4A7C15ULL + blk * 0xD1B54A32D192ED03ULL +
                 (uint64_t)j * 0x8CB92BA72F3D8DD7ULL + 0x2545F4914F6CDD1DULL);
}
__device__ __forceinline__ float h_unif(uint64_t h, float lo, float hi) {
    float u = __fmul_rn((float)(uint32_t)(h >> 40), 1.0f / 16777216.0f);
    float span = __fsub_rn(hi, lo);
    return __fadd_rn(lo, __fmul_rn(span, u));
}
// binary16 round-to-nearest-even narrowing, integer-only
__device__ __forceinline__ uint16_t f2h_rne(float f) {
    uint32_t x = __float_as_uint(f);
    uint32_t sign = (x >> 16) & 0x8000u, exp = (x >> 23) & 0xFFu, man = x & 0x7FFFFFu;
    if (exp == 0xFF) return (uint16_t)(sign | (man ? (0x7E00u | (man >> 13)) : 0x7C00u));
    int32_t e = (int32_t)exp - 127 + 15;
    if (e >= 31) return (uint16_t)(sign | 0x7C00u);
    if (e <= 0) {
        if (e < -10) return (uint16_t)sign;
        uint32_t m = man | 0x800000u, sh = (uint32_t)(14 - e);
        uint32_t q = m >> sh, rem = m & ((1u << sh) - 1u), half = 1u << (sh - 1u);
        if (rem > half || (rem == half && (q & 1u))) q++;
        return (uint16_t)(sign | q);
    }
    uint32_t h = ((uint32_t)e << 10) | (man >> 13), rem = man & 0x1FFFu;
    if (rem > 0x1000u || (rem == 0x1000u && (h & 1u))) h++;
    return (uint16_t)(sign | h);
}
__device__ __forceinline__ uint8_t hbyte(uint64_t h) { return (uint8_t)(h >> 56); }

__device__ uint16_t gen_d16(uint32_t t, uint64_t seed, uint64_t blk, int mode, float lo, float hi,
                            bool is_min) {
    if (t == T_Q6_K) return f2h_rne(h_unif(hsh(seed, blk, 208), lo, hi));
    if (!is_min) return f2h_rne(h_unif(hsh(seed, blk, 0), lo, hi));
    if (mode == 1) {
        float d = h2f(f2h_rne(h_unif(hsh(seed, blk, 0), lo, hi)));
        return f2h_rne(__fmul_rn(d, t == T_Q4_K ? 7.5f : 15.5f));
    }
    return f2h_rne(h_unif(hsh(seed, blk, 1), lo, hi));
}

// GGUF byte `o` of synthetic block `blk`
__device__ uint8_t gen_byte(uint32_t t, uint64_t seed, uint64_t blk, uint32_t o, int mode,
                            float lo, float hi) {
    switch (t) {
    case T_Q8_0: {
        if (o < 2) {
            uint16_t v = gen_d16(t, seed, blk, mode, lo, hi, false);
            return (uint8_t)(o == 0 ? (v & 0xFF) : (v >> 8));
        }
        uint64_t h = hsh(seed, blk, o - 1);
        int q = (int)(((h >> 32) * 255ULL) >> 32) - 127;
        return (uint8_t)(int8_t)q;
    }
    case T_Q4_K:
    case T_Q5_K: {
        if (o < 4) {
            uint16_t v = gen_d16(t, seed, blk, mode, lo, hi, o >= 2);
            return (uint8_t)((o & 1) ? (v >> 8) : (v & 0xFF));
        }
        if (o < 16 && mode == 1) {
            // packed 6-bit scales with mins equal to scales
            uint32_t k = o - 4;  // 0..11
            auto sc = [&](uint32_t j) { return (uint32_t)(hbyte(hsh(seed, blk, 4 + j)) & 63); };
            if (k < 4) return (uint8_t)((sc(k) & 63) | ((sc(k + 4) >> 4) << 6));
            if (k < 8) return (uint8_t)((sc(k - 4) & 63) | ((sc(k) >> 4) << 6));
            uint32_t j = k - 8;
            return (uint8_t)((sc(j + 4) & 15) | ((sc(j + 4) & 15) << 4));
        }
        return hbyte(hsh(seed, blk, o));
    }
    case T_Q6_K: {
        if (o < 192) return hbyte(hsh(seed, blk, o));
        if (o < 208) return (uint8_t)(int8_t)((int)(hsh(seed, blk, o) >> 57) - 64);
        uint16_t v = gen_d16(t, seed, blk, mode, lo, hi, false);
        return (uint8_t)(o == 208 ? (v & 0xFF) : (v >> 8));
    }
    default:
        return 0;
    }
}

// synthetic weight straight into the device layout: one thread per device
// word, each byte the generator byte of its GGUF (block, offset); the block
// index is the GGUF row-major one (row * nb + block), as on the host
__global__ void k_generate(WeightView w, size_t dev_bytes, uint64_t seed, int mode, float lo, float hi,
                           uint8_t *__restrict__ q) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < dev_bytes / 4;
         i += (size_t)gridDim.x * blockDim.x) {
        uint32_t v = 0;
        for (int k = 0; k < 4; k++) {
            uint32_t row, blk, o;
            if (tinv(w.type, w.n_in, w.n_out, 4 * i + k, row, blk, o))
                v |= (uint32_t)gen_byte(w.type, seed, (uint64_t)row * w.nb + blk, o, mode, lo, hi) << (8 * k);
        }
        reinterpret_cast<uint32_t *>(q)[i] = v;
    }
}

hipError_t launch_generate(WeightView w, uint8_t *q, uint64_t seed, int mode, float d_lo, float d_hi,
                           hipStream_t s) {
    if (!is_tiled(w.type)) return hipErrorInvalidValue;
    const size_t db = weight_dev_bytes(w.type, w.n_in, w.n_out);
    hipLaunchKernelGGL(k_generate, dim3(grid_for(db / 4, 256)), dim3(256), 0, s, w, db, seed, mode,
                       d_lo, d_hi, q);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// dequant (bit-exact with dequant.rs)
// ---------------------------------------------------------------------------
// One wavefront turns 256 consecutive elements of a row (a super-block, or four
// Q8_0 units) into one contiguous KB of f32: lane l makes elements 4 l .. 4 l + 3
// from one word of quants (two for Q5_K / Q6_K) and the run's scale bytes, which
// the lanes of a run share.  Bound by the f32 written; a thread per element that
// looked every byte up through toff took 640 us for a 5120 x 5120 Q5_K weight,
// this 29.4 us (123 MB moved, 4.2 TB/s; a
// large copy reaches 4.9 TB/s).
typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ uint32_t ld32(const uint8_t *p) { return *reinterpret_cast<const uint32_t *>(p); }
__device__ __forceinline__ uint32_t ld16(const uint8_t *p) { return *reinterpret_cast<const uint16_t *>(p); }

// elements 4 l .. 4 l + 3 of super-block u (Q8_0: of the 256 elements from 256 u) of row `row`
template <uint32_t T>
__device__ __forceinline__ f32x4 deq4(const WeightView &w, uint32_t row, uint32_t u, uint32_t l) {
    const uint32_t r = row % TILE_ROWS, e = 4 * l;
    const uint8_t *tile = w.q + (size_t)(row / TILE_ROWS) * tunits(T, w.n_in) * tchunk_bytes(T);
    f32x4 v;
    if constexpr (T == T_Q8_0) {
        const uint8_t *c = tile + (size_t)(4 * u + (e >> 6)) * tchunk_bytes(T);
        const uint32_t b = (e >> 5) & 1, q = ld32(c + 16 * (16 * (2 * b + ((e >> 4) & 1)) + r) + (e & 15));
        const float d = h2f((uint16_t)ld16(c + 1024 + 4 * r + 2 * b));
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = __fmul_rn((float)(int8_t)((q >> (8 * i)) & 0xFF), d);
    } else if constexpr (T == T_Q4_K || T == T_Q5_K) {
        constexpr uint32_t QS = T == T_Q4_K ? 256 : 768;
        const uint8_t *c = tile + (size_t)u * tchunk_bytes(T);
        const uint32_t j = e >> 6, hi = (e >> 5) & 1, sub = 2 * j + hi, x = e & 31;
        uint32_t q = (ld32(c + QS + 1024 * (j >> 1) + 16 * (16 * (2 * (j & 1) + (x >> 4)) + r) + (x & 15)) >> (4 * hi)) &
                     0x0F0F0F0Fu;
        if constexpr (T == T_Q5_K)
            q |= ((ld32(c + 256 + 16 * (16 * (x >> 4) + r) + (x & 15)) >> sub) & 0x01010101u) << 4;
        const uint32_t h = ld32(c + 16 * r), s0 = ld32(c + 16 * r + 4), s1 = ld32(c + 16 * r + 8),
                       s2 = ld32(c + 16 * r + 12), sh = 8 * (sub & 3);
        const uint32_t a = (s0 >> sh) & 0xFF, m = (s1 >> sh) & 0xFF, x2 = (s2 >> sh) & 0xFF;
        const uint32_t sc = sub < 4 ? a & 63 : (x2 & 0xF) | ((a >> 6) << 4);
        const uint32_t mn = sub < 4 ? m & 63 : (x2 >> 4) | ((m >> 6) << 4);
        const float d1 = __fmul_rn(h2f((uint16_t)(h & 0xFFFF)), (float)sc);
        const float m1 = __fmul_rn(h2f((uint16_t)(h >> 16)), (float)mn);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = __fsub_rn(__fmul_rn(d1, (float)((q >> (8 * i)) & 0xFF)), m1);
    } else {  // T_Q6_K
        const uint8_t *c = tile + (size_t)u * tchunk_bytes(T);
        const uint32_t half = e >> 7, quarter = (e >> 5) & 3, x = e & 31, pc = 16 * (16 * (2 * half + (x >> 4)) + r) + (x & 15);
        const uint32_t lo = (ld32(c + 256 + 1024 * (quarter & 1) + pc) >> (4 * (quarter >> 1))) & 0x0F0F0F0Fu;
        const uint32_t q = lo | (((ld32(c + 2304 + pc) >> (2 * quarter)) & 0x03030303u) << 4);
        const float s = (float)(int8_t)c[16 * r + 8 * half + (x >> 4) + 2 * quarter];
        const float ds = __fmul_rn(h2f((uint16_t)ld16(c + 3328 + 2 * r)), s);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = __fmul_rn(ds, (float)((int)((q >> (8 * i)) & 0xFF) - 32));
    }
    return v;
}

// VEC: `out` is 16-byte aligned (rows are whole blocks, so every store is)
template <bool VEC>
__device__ __forceinline__ void put4(float *__restrict__ o, f32x4 v) {
    if constexpr (VEC)
        *reinterpret_cast<f32x4 *>(o) = v;
    else
        for (int i = 0; i < 4; i++) o[i] = v[i];
}

// workgroup = 256 elements of the 16 rows of a tile, a wavefront every fourth row
template <uint32_t T, bool VEC>
__global__ __launch_bounds__(256) void k_dequant(WeightView w, uint32_t nu, float *__restrict__ out) {
    const uint32_t u = blockIdx.x % nu, row0 = blockIdx.x / nu * TILE_ROWS, l = threadIdx.x & 63;
    if (256 * u + 4 * l >= w.n_in) return;  // Q8_0: the row's last, partial 256 elements
#pragma unroll
    for (uint32_t i = 0; i < TILE_ROWS / 4; i++) {
        const uint32_t row = row0 + 4 * i + (threadIdx.x >> 6);
        if (row < w.n_out) put4<VEC>(out + (size_t)row * w.n_in + 256 * u + 4 * l, deq4<T>(w, row, u, l));
    }
}

// rows[r] selects a row; out is [n_rows][n_in] (embedding lookup, ops.rs:11-26
// on the dequantized table); workgroup = 1024 elements of one row
template <uint32_t T, bool VEC>
__global__ __launch_bounds__(256) void k_dequant_rows(WeightView w, const uint32_t *__restrict__ rows, uint32_t n_rows,
                                                      uint32_t nq, float *__restrict__ out) {
    const uint32_t r = blockIdx.x / nq, u = 4 * (blockIdx.x % nq) + (threadIdx.x >> 6), l = threadIdx.x & 63;
    const uint32_t row = min(rows[r], w.n_out - 1);  // ids are validated on the host
    if (256 * u + 4 * l < w.n_in) put4<VEC>(out + (size_t)r * w.n_in + 256 * u + 4 * l, deq4<T>(w, row, u, l));
}

// the types that are kept as GGUF bytes (F32, F16, Q4_0): one element per thread
__global__ void k_dequant_raw(WeightView w, const uint32_t *__restrict__ rows, uint32_t n_rows,
                              float *__restrict__ out) {
    const uint32_t be = (uint32_t)block_elems(w.type);
    const uint64_t n = (uint64_t)n_rows * w.n_in;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x) {
        uint64_t e = i;
        if (rows) e = (uint64_t)min(rows[i / w.n_in], w.n_out - 1) * w.n_in + i % w.n_in;
        out[i] = deq_elem(w, e / be, (uint32_t)(e % be));
    }
}

// rows null: every row of w
template <uint32_t T, bool VEC>
static void start_dequant(const WeightView &w, const uint32_t *rows, uint32_t n_rows, float *out, hipStream_t s) {
    const uint32_t nu = (w.n_in + 255) / 256;
    if (rows)
        hipLaunchKernelGGL((k_dequant_rows<T, VEC>), dim3(n_rows * ((nu + 3) / 4)), dim3(256), 0, s, w, rows, n_rows,
                           (nu + 3) / 4, out);
    else
        hipLaunchKernelGGL((k_dequant<T, VEC>), dim3(ttiles(w.n_out) * nu), dim3(256), 0, s, w, nu, out);
}

static hipError_t dequant(const WeightView &w, const uint32_t *rows, uint32_t n_rows, float *out, hipStream_t s) {
    const bool vec = ((uintptr_t)out & 15) == 0;
#define LRS_DEQ(T)                                                 \
    case T:                                                        \
        if (vec) start_dequant<T, true>(w, rows, n_rows, out, s);  \
        else start_dequant<T, false>(w, rows, n_rows, out, s);     \
        break;
    switch (w.type) {
        LRS_DEQ(T_Q8_0)
        LRS_DEQ(T_Q4_K)
        LRS_DEQ(T_Q5_K)
        LRS_DEQ(T_Q6_K)
    default:
        hipLaunchKernelGGL(k_dequant_raw, dim3(grid_for((uint64_t)n_rows * w.n_in, 256)), dim3(256), 0, s, w, rows,
                           n_rows, out);
    }
#undef LRS_DEQ
    return hipGetLastError();
}

hipError_t launch_dequant(WeightView w, float *out, hipStream_t s) { return dequant(w, nullptr, w.n_out, out, s); }

hipError_t launch_dequant_rows(WeightView w, const uint32_t *rows_dev, uint32_t n_rows, float *out,
                               hipStream_t s) {
    return dequant(w, rows_dev, n_rows, out, s);
}

}  // namespace lrs
