// prefill.hip — the per-token ops of a batched prompt block (n tokens at
// positions pos0 .. pos0+n-1) around the matrix-core GEMMs of gemm.hip:
// RMSNorm per row and SwiGLU (both written straight as the next GEMM's input,
// gemm_pack.h), bias + RoPE + f16 KV append after the q/k/v
// GEMMs, causal GQA attention over the cache.  The formulas of the decode
// kernels (Model::forward, crates/llama-model/src/model.rs:99-266; ops.rs:
// 56-66, 952-988; attention.rs:76-166), which is what the reference's
// prefill_residente (gpu.rs:673-697) drives in blocks of batch_size() tokens;
// the attention runs on the matrix cores (f16 hi/lo operands, f32
// accumulation), so its summation order differs from the per-token kernel.
#include "gemm_pack.h"

namespace lrs {

// X += the ks K-slice partials part[z][row][E] of a split o / down GEMM (summed
// in slice order, then added to X, as k_reduce_ks does; ks 0: none), then the
// row X[r] * scale_r * w, scale_r = 1 / sqrt(mean(X[r]^2) + eps), as a GEMM
// input (gemm_pack.h) and, with Y, in f32.  Workgroup = a row.  Load latency
// bounds it, so a thread has all of its eight elements' loads in flight (a
// wider row takes more passes, whose elements are read back for the second
// half).  us at E = 5120, 256 threads that went over the row four elements at a
// time and read it back -> this: 512 rows norm alone 15.9 -> 11.0, with the
// slices of o and down 20.3 -> 17.5; 19 rows of 11 to 22 slices 11.6 (a reduce
// launch of its own and a norm) -> 7.6.
__global__ __launch_bounds__(1024) void k_norm_rows(const float *__restrict__ part, uint32_t ks, float *X,
                                                    const float *__restrict__ w, float eps, uint32_t E,
                                                    float *__restrict__ Y, uint8_t *__restrict__ planes) {
    __shared__ float red[16];
    const size_t plane = (size_t)gridDim.x * E, r0 = (size_t)blockIdx.x * E;
    float *const x = X + r0;
    const uint32_t i0 = 8 * threadIdx.x, step = 8 * blockDim.x;
    float v0[8], g0[8];  // the first pass's elements and weights
    auto load8 = [](const float *p, float (&v)[8]) __attribute__((always_inline)) {
        const float4 a = *reinterpret_cast<const float4 *>(p), b = *reinterpret_cast<const float4 *>(p + 4);
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
    };
    auto store8 = [](float *p, const float (&v)[8]) __attribute__((always_inline)) {
        *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
        *reinterpret_cast<float4 *>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
    };
    if (i0 < E) load8(w + i0, g0);
    float ss = 0.f;
    for (uint32_t i = i0; i < E; i += step) {
        float v[8];
        load8(x + i, v);
        if (ks) {
            float p[8];
            load8(part + r0 + i, p);
#pragma unroll 4
            for (uint32_t z = 1; z < ks; z++) {
                float q[8];
                load8(part + z * plane + r0 + i, q);
#pragma unroll
                for (int k = 0; k < 8; k++) p[k] += q[k];
            }
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] += p[k];
            store8(x + i, v);
        }
#pragma unroll
        for (int k = 0; k < 8; k++) {
            ss = fmaf(v[k], v[k], ss);
            if (i == i0) v0[k] = v[k];
        }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) ss += __shfl_xor(ss, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    float tot = 0.f;
    for (uint32_t i = 0; i < blockDim.x / 64; i++) tot += red[i];
    const float scale = 1.0f / sqrtf(tot / (float)E + eps);
    for (uint32_t i = i0; i < E; i += step) {
        float v[8], g[8];
        if (i == i0) {
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = v0[k], g[k] = g0[k];
        } else {
            load8(x + i, v);
            load8(w + i, g);
        }
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = (v[k] * scale) * g[k];
        if (Y) store8(Y + r0 + i, v);
        gp_store8<3>(v, blockIdx.x, i >> 3, E >> 8, planes);
    }
}

// q/k/v GEMM outputs -> bias, adjacent-pair RoPE on q and k at position
// pos0 + token, q to f32, k and v to the f16 cache.  One thread per pair.
struct QkvPost {
    const float *qt, *kt, *vt;     // [n][qd], [n][kvd], [n][kvd]
    const float *bq, *bk, *bv;     // biases or null
    const float *freq;             // [rope_dim / 2]
    float *q;                      // [n][qd]
    _Float16 *kc, *vc;             // this layer's caches [n_kv][ctx][hd]
    uint32_t n, pos0, qd, kvd, hd, rope_dim, ctx;
};

__global__ void k_qkv_post(QkvPost a) {
    const uint32_t b = blockIdx.y;
    const uint32_t np = (a.qd + 2 * a.kvd) / 2;  // pairs per token
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np || b >= a.n) return;
    const uint32_t e = 2 * i, pos = a.pos0 + b;
    const float *src;
    const float *bias;
    uint32_t off;
    int kind;  // 0 q, 1 k, 2 v
    if (e < a.qd) {
        kind = 0, off = e, src = a.qt + (size_t)b * a.qd, bias = a.bq;
    } else if (e < a.qd + a.kvd) {
        kind = 1, off = e - a.qd, src = a.kt + (size_t)b * a.kvd, bias = a.bk;
    } else {
        kind = 2, off = e - a.qd - a.kvd, src = a.vt + (size_t)b * a.kvd, bias = a.bv;
    }
    float x0 = src[off], x1 = src[off + 1];
    if (bias) {
        x0 = x0 + bias[off];
        x1 = x1 + bias[off + 1];
    }
    const uint32_t dd = off % a.hd;
    if (kind < 2 && dd < a.rope_dim) {
        // ops.rs:952-975: theta = pos * freq[dd / 2]
        const float th = (float)pos * a.freq[dd >> 1];
        float sn, cs;
        sincosf(th, &sn, &cs);
        const float r0 = x0 * cs - x1 * sn, r1 = x0 * sn + x1 * cs;
        x0 = r0;
        x1 = r1;
    }
    if (kind == 0) {
        a.q[(size_t)b * a.qd + off] = x0;
        a.q[(size_t)b * a.qd + off + 1] = x1;
    } else {
        _Float16 *c = kind == 1 ? a.kc : a.vc;
        const uint32_t hh = off / a.hd;
        const size_t o = ((size_t)hh * a.ctx + pos) * a.hd + dd;
        c[o] = (_Float16)x0;
        c[o + 1] = (_Float16)x1;
    }
}

// Causal GQA attention of the block: token b (position pos0 + b) attends to
// cache positions 0..pos0+b (attention.rs:76-166 per token).
struct AttnPre {
    const float *q;                 // [n][n_head * hd]
    const _Float16 *kc, *vc;        // [n_kv][ctx][hd]
    float *out;                     // [S][n][n_head * hd]: each split's sum of e^(s - m) v
    float2 *ml;                     // [S][n][n_head]: its {m, sum of e^(s - m)}
    uint32_t n, pos0, n_head, n_kv, ctx, S;
    float scale;
};

// On the matrix cores: workgroup (32-token query block,
// KV head, group of NW query heads of the GQA group), one wavefront per query
// head: NW = the whole group for head_dim <= 128; at head_dim 256 at most 4
// wavefronts (the query and output registers of a wavefront exceed half the
// register file, so one wavefront per SIMD).  Per chunk of 32 cache positions each wavefront forms the transposed
// score tile S^T = K Q^T (32 positions x 32 queries) with
// v_mfma_f32_32x32x16_f16: K is the f16 cache (exact), Q is split into f16
// hi + lo after scaling each query by a power of two (2^-e >= 1 / max |q|),
// so the products carry 22 bits of q.  In that layout a lane owns one query
// and 16 of the chunk's positions, so the online softmax (running max m,
// sum l) needs one cross-lane step per reduction.  The probabilities, split
// into f16 hi + lo, are the B operand of O^T += V^T P^T straight from the
// score registers: the K index of that product is the position order in
// which the score layout holds them (4 positions of the lane's half, then the
// 4 positions 8 further), and V^T is read from LDS in the same order.
// K is staged with global_load_lds into an XOR-swizzled row layout
// (conflict-free 16-byte reads), V into a transposed, padded layout: through
// registers, or at head_dim 256 (no registers to spare) through a row-major
// LDS copy transposed after each chunk.  The next chunk's loads are in flight
// during the current chunk's matrix work.
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void_t;

template <int HD, int NW>
__global__ __launch_bounds__(64 * NW) void k_attn_pf_mma(AttnPre a) {
    constexpr int NT = 64 * NW;
    constexpr int KS = HD / 16;           // K-steps of S^T (16 dims each)
    constexpr int OT = HD / 32;           // O^T tiles of 32 dims
    constexpr int NPR = HD / 8;           // 16-byte pieces per K / V row
    constexpr int NPC = 32 * NPR;         // pieces per chunk
    constexpr int VLD = 36;               // V^T row (f16): 72 B, conflict-free 8-byte reads
    constexpr int NVP = (NPC + NT - 1) / NT;
    constexpr bool VLDS = HD > 128;       // V staged through LDS instead of registers
    __shared__ __attribute__((aligned(16))) _Float16 Ks[2][32 * HD];
    __shared__ __attribute__((aligned(16))) _Float16 Vt[2][HD * VLD];
    __shared__ __attribute__((aligned(16))) _Float16 Vraw[VLDS ? 32 * HD : 8];
    const uint32_t rep = a.n_head / a.n_kv, ng = (rep + NW - 1) / NW;
    // the last query blocks have the most positions: they start first
    const uint32_t qb = gridDim.x / a.S - 1 - blockIdx.x / a.S, sp = blockIdx.x % a.S, kh = blockIdx.y / ng;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, hf = lane >> 5;
    const uint32_t hl = (blockIdx.y % ng) * NW + wave;  // query head within the group
    const bool hact = hl < rep;                         // an idle wavefront stages and stores nothing
    const uint32_t h = kh * rep + (hact ? hl : rep - 1);
    const uint32_t q0 = qb * 32, qi = q0 + (lane & 31);
    const uint32_t qr = qi < a.n ? qi : a.n - 1;  // lanes past the block compute a copy, store nothing
    const uint32_t qpos = a.pos0 + qr;
    const uint32_t kend = a.pos0 + min(q0 + 32, a.n);  // positions 0..kend-1 are attended
    const uint32_t nall = (kend + 31) / 32, share = (nall + a.S - 1) / a.S;
    const uint32_t c0 = sp * share, nch = min(c0 + share, nall);  // this split's chunks
    const size_t row = (size_t)sp * a.n + qi;
    if (c0 >= nall) {  // more splits than chunks: an empty share
        if (hf == 0 && qi < a.n && hact) a.ml[row * a.n_head + h] = make_float2(-INFINITY, 0.f);
        return;
    }
    const _Float16 *kb = a.kc + (size_t)kh * a.ctx * HD;
    const _Float16 *vb = a.vc + (size_t)kh * a.ctx * HD;

    // K chunk c -> Ks[buf]: LDS slot s (16 B) holds row s / NPR, piece
    // (s % NPR) ^ (row % NPR); wavefront instruction i fills slots 64i..64i+63
    auto stage_k = [&](uint32_t c, uint32_t buf) {
        for (uint32_t i = wave; i < NPC / 64; i += NW) {
            const uint32_t sl = 64 * i + lane, row = sl / NPR, pc = (sl % NPR) ^ (row % NPR);
            const uint32_t kp = min(32 * c + row, kend - 1);  // past the end: any finite row (masked)
            __builtin_amdgcn_global_load_lds(kb + (size_t)kp * HD + 8 * pc,
                                             (lds_void_t *)(Ks[buf] + 64 * 8 * i), 16, 0, 0);
        }
    };
    // V chunk c: piece p = (row p % 32, dims 8 (p / 32)..), through registers
    // (load_v, store_v) or, at head_dim 256, global_load_lds into Vraw slot p
    // and an LDS transpose (vraw_to_vt)
    uint4 vr[VLDS ? 1 : NVP];
    auto stage_vraw = [&](uint32_t c) {
        for (uint32_t i = wave; i < NPC / 64; i += NW) {
            const uint32_t p = 64 * i + lane, row = p % 32, kp = min(32 * c + row, kend - 1);
            __builtin_amdgcn_global_load_lds(vb + (size_t)kp * HD + 8 * (p / 32),
                                             (lds_void_t *)(Vraw + 64 * 8 * i), 16, 0, 0);
        }
    };
    auto vraw_to_vt = [&](uint32_t buf) {
        for (uint32_t p = tid; p < (uint32_t)NPC; p += NT) {
            const uint4 v = *reinterpret_cast<const uint4 *>(Vraw + 8 * p);
            const _Float16 *hv = reinterpret_cast<const _Float16 *>(&v);
            const uint32_t row = p % 32, d0 = 8 * (p / 32);
#pragma unroll
            for (int e = 0; e < 8; e++) Vt[buf][(d0 + e) * VLD + row] = hv[e];
        }
    };
    auto load_v = [&](uint32_t c) {
#pragma unroll
        for (int j = 0; j < (VLDS ? 1 : NVP); j++) {
            const uint32_t p = tid + NT * j;
            if (p < (uint32_t)NPC) {
                const uint32_t row = p % 32, kp = min(32 * c + row, kend - 1);
                vr[j] = *reinterpret_cast<const uint4 *>(vb + (size_t)kp * HD + 8 * (p / 32));
            }
        }
    };
    auto store_v = [&](uint32_t buf) {
#pragma unroll
        for (int j = 0; j < (VLDS ? 1 : NVP); j++) {
            const uint32_t p = tid + NT * j;
            if (p < (uint32_t)NPC) {
                const uint32_t row = p % 32, d0 = 8 * (p / 32);
                const _Float16 *hv = reinterpret_cast<const _Float16 *>(&vr[j]);
#pragma unroll
                for (int e = 0; e < 8; e++) Vt[buf][(d0 + e) * VLD + row] = hv[e];
            }
        }
    };

    // this lane's query: dims 16 k + 8 hf .. + 7 of every K-step, scaled by
    // 2^-e (e from the head's max |q|, both halves), split into f16 hi + lo
    f16x8_t qh[KS], ql[KS];
    float qsc;
    {
        const float *qp = a.q + ((size_t)qr * a.n_head + h) * HD + 8 * hf;
        float qv[KS][8];
        float qm = 0.f;
#pragma unroll
        for (int k = 0; k < KS; k++) {
            const float4 x0 = *reinterpret_cast<const float4 *>(qp + 16 * k);
            const float4 x1 = *reinterpret_cast<const float4 *>(qp + 16 * k + 4);
            qv[k][0] = x0.x; qv[k][1] = x0.y; qv[k][2] = x0.z; qv[k][3] = x0.w;
            qv[k][4] = x1.x; qv[k][5] = x1.y; qv[k][6] = x1.z; qv[k][7] = x1.w;
#pragma unroll
            for (int e = 0; e < 8; e++) qm = fmaxf(qm, fabsf(qv[k][e]));
        }
        qm = fmaxf(qm, __shfl_xor(qm, 32, 64));
        int ex;
        frexpf(qm, &ex);
        ex = ex < -60 ? -60 : ex;
        qsc = ldexpf(1.0f, ex) * a.scale;
#pragma unroll
        for (int k = 0; k < KS; k++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float x = ldexpf(qv[k][e], -ex);
                const _Float16 xh = (_Float16)x;
                qh[k][e] = xh;
                ql[k][e] = (_Float16)(x - (float)xh);
            }
    }

    f32x16_t o[OT];
#pragma unroll
    for (int t = 0; t < OT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[t][r] = 0.f;
    float m = -INFINITY, l = 0.f;

    stage_k(c0, 0);
    if constexpr (VLDS) {
        stage_vraw(c0);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        vraw_to_vt(0);
    } else {
        load_v(c0);
        store_v(0);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    for (uint32_t c = c0; c < nch; c++) {
        const uint32_t cur = (c - c0) & 1;
        const bool more = c + 1 < nch;
        if (more) {
            stage_k(c + 1, cur ^ 1);
            if constexpr (VLDS)
                stage_vraw(c + 1);
            else
                load_v(c + 1);
        }
        // S^T = K Q^T: lane (query l%32) gets positions 8(r/4) + 4 hf + r%4
        f32x16_t sc;
#pragma unroll
        for (int r = 0; r < 16; r++) sc[r] = 0.f;
        const uint32_t krow = lane & 31;
#pragma unroll
        for (int k = 0; k < KS; k++) {
            const uint32_t sl = krow * NPR + ((2 * k + hf) ^ (krow % NPR));
            const f16x8_t kf = *reinterpret_cast<const f16x8_t *>(Ks[cur] + 8 * sl);
            sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, ql[k], sc, 0, 0, 0);
            sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qh[k], sc, 0, 0, 0);
        }
        // online softmax of this query over the chunk (causal mask)
        float cmax = -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const uint32_t kp = 32 * c + 8 * (r >> 2) + 4 * hf + (r & 3);
            sc[r] = kp <= qpos ? sc[r] * qsc : -INFINITY;
            cmax = fmaxf(cmax, sc[r]);
        }
        cmax = fmaxf(cmax, __shfl_xor(cmax, 32, 64));
        // a query before all of the share's positions so far has only -inf:
        // any finite maximum then gives zeros
        const float mn = fmaxf(m, cmax) == -INFINITY ? -1e30f : fmaxf(m, cmax);
        const float alpha = expf(m - mn);
        float ps = 0.f;
        f16x8_t ph[2], pl[2];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const float p = expf(sc[r] - mn);
            ps += p;
            const _Float16 x = (_Float16)p;
            ph[r >> 3][r & 7] = x;
            pl[r >> 3][r & 7] = (_Float16)(p - (float)x);
        }
        ps += __shfl_xor(ps, 32, 64);
        l = l * alpha + ps;
        m = mn;
        // O^T (dims x queries) = alpha O^T + V^T P^T; K slot j of step s is
        // position 16 s + 4 hf + j (j < 4) or 16 s + 8 + 4 hf + j - 4
#pragma unroll
        for (int t = 0; t < OT; t++) {
#pragma unroll
            for (int r = 0; r < 16; r++) o[t][r] *= alpha;
            const _Float16 *vrow = Vt[cur] + (32 * t + (lane & 31)) * VLD + 4 * hf;
#pragma unroll
            for (int st = 0; st < 2; st++) {
                const f16x4_t v0 = *reinterpret_cast<const f16x4_t *>(vrow + 16 * st);
                const f16x4_t v1 = *reinterpret_cast<const f16x4_t *>(vrow + 16 * st + 8);
                const f16x8_t va = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, pl[st], o[t], 0, 0, 0);
                o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va, ph[st], o[t], 0, 0, 0);
            }
        }
        if constexpr (!VLDS) {
            if (more) store_v(cur ^ 1);
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if constexpr (VLDS) {
            if (more) {
                vraw_to_vt(cur ^ 1);
                __syncthreads();
            }
        }
    }
    // out[token][head][dim]: lane holds dims 32 t + 8 (r/4) + 4 hf + r%4
    if (qi < a.n && hact) {
        if (hf == 0) a.ml[row * a.n_head + h] = make_float2(m, l);
        float *op = a.out + (row * a.n_head + h) * HD;
#pragma unroll
        for (int t = 0; t < OT; t++)
#pragma unroll
            for (int g = 0; g < 4; g++)
                *reinterpret_cast<float4 *>(op + 32 * t + 8 * g + 4 * hf) =
                    make_float4(o[t][4 * g], o[t][4 * g + 1], o[t][4 * g + 2], o[t][4 * g + 3]);
    }
}

// The splits of k_attn_pf_mma merged (softmax over the union of their
// positions), times sigmoid(gate) for the hybrid (gate_quant.comp; qg holds a
// head's query, then its gate), as the o projection's GEMM input.  Workgroup =
// 8 rows x one super-block, eight elements per thread; the splits go by in
// fours whose loads are in flight together (one at a time the 11 splits of a
// 19-token turn took 34 us).
__global__ __launch_bounds__(256) void k_attn_merge(const float *__restrict__ part, const float2 *__restrict__ ml,
                                                    const float *__restrict__ qg, uint32_t S, uint32_t n,
                                                    uint32_t n_head, uint32_t hd, uint8_t *__restrict__ planes) {
    const uint32_t qd = n_head * hd, row = 8 * blockIdx.y + (threadIdx.x >> 5);
    if (row >= n) return;
    const uint32_t c = 32 * blockIdx.x + (threadIdx.x & 31), e = 8 * c, h = e / hd;
    float m = -INFINITY, l = 0.f, v[8] = {};
    for (uint32_t s0 = 0; s0 < S; s0 += 4) {
        float2 p[4];
        float4 a[4], b[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const size_t r = (size_t)min(s0 + i, S - 1) * n + row;
            p[i] = ml[r * n_head + h];
            if (s0 + i >= S) p[i] = make_float2(-INFINITY, 0.f);
            a[i] = *reinterpret_cast<const float4 *>(part + r * qd + e);
            b[i] = *reinterpret_cast<const float4 *>(part + r * qd + e + 4);
        }
        const float mn = fmaxf(fmaxf(fmaxf(p[0].x, p[1].x), fmaxf(p[2].x, p[3].x)), m);
        const float old = m == -INFINITY ? 0.f : expf(m - mn);
        l *= old;
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] *= old;
        m = mn;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (p[i].y == 0.f) continue;  // an empty share: its sums were not written
            const float w = expf(p[i].x - m);
            l = fmaf(p[i].y, w, l);
            const float x[8] = {a[i].x, a[i].y, a[i].z, a[i].w, b[i].x, b[i].y, b[i].z, b[i].w};
#pragma unroll
            for (int k = 0; k < 8; k++) v[k] = fmaf(w, x[k], v[k]);
        }
    }
    const float inv = 1.0f / l;
    const float *g = qg ? qg + (size_t)row * 2 * qd + (size_t)h * 2 * hd + hd + e % hd : nullptr;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        v[i] *= inv;
        if (g) v[i] = v[i] * (1.0f / (1.0f + expf(-g[i])));
    }
    gp_store8<3>(v, row, c, qd >> 8, planes);
}

hipError_t launch_norm_rows(const float *part, uint32_t ks, float *X, const float *w, float eps, uint32_t E,
                            uint32_t n, float *Y, uint8_t *planes, hipStream_t s) {
    if (E == 0 || E % 256 || !planes) return hipErrorInvalidValue;
    const uint32_t threads = min(1024u, (E / 8 + 63) / 64 * 64);
    hipLaunchKernelGGL(k_norm_rows, dim3(n), dim3(threads), 0, s, part, ks, X, w, eps, E, Y, planes);
    return hipGetLastError();
}

hipError_t launch_qkv_post(const float *qt, const float *kt, const float *vt, const float *bq,
                           const float *bk, const float *bv, const float *freq, float *q,
                           _Float16 *kc, _Float16 *vc, uint32_t n, uint32_t pos0, uint32_t qd,
                           uint32_t kvd, uint32_t hd, uint32_t rope_dim, uint32_t ctx,
                           hipStream_t s) {
    QkvPost a = {qt, kt, vt, bq, bk, bv, freq, q, kc, vc, n, pos0, qd, kvd, hd, rope_dim, ctx};
    const uint32_t np = (qd + 2 * kvd) / 2;
    hipLaunchKernelGGL(k_qkv_post, dim3((np + 255) / 256, n), dim3(256), 0, s, a);
    return hipGetLastError();
}

// Splits of the cache positions of a block of n tokens: about one workgroup
// per CU (the five wavefronts of the 32B shape's head groups leave no room for
// a second), at most one split per chunk of the last query block.  With the
// merge, 32B shape, us per layer: 512 tokens from position 0 64 -> 47 (four
// splits a block: 70), 19 tokens behind 333 positions 42 -> 18.
uint32_t attn_prefill_splits(uint32_t n, uint32_t pos0, uint32_t n_head, uint32_t n_kv, uint32_t hd) {
    const uint32_t rep = n_head / n_kv, ng = hd == 256 ? (rep + 3) / 4 : 1;
    const uint32_t wgs = (n + 31) / 32 * n_kv * ng, chunks = (pos0 + n + 31) / 32;
    const uint32_t want = (256 + wgs - 1) / wgs;
    return want < chunks ? want : chunks;
}

hipError_t launch_attn_prefill(const float *q, const _Float16 *kc, const _Float16 *vc, const float *qg, float *part,
                               float2 *ml, uint32_t n, uint32_t pos0, uint32_t n_head, uint32_t n_kv,
                               uint32_t hd, uint32_t ctx, uint8_t *planes, hipStream_t s) {
    if (n == 0 || n_kv == 0 || n_head % n_kv || n_head / n_kv > 8 || (n_head * hd) % 256)
        return hipErrorInvalidValue;
    const uint32_t S = attn_prefill_splits(n, pos0, n_head, n_kv, hd);
    AttnPre a = {q, kc, vc, part, ml, n, pos0, n_head, n_kv, ctx, S, 1.0f / sqrtf((float)hd)};
    const uint32_t rep = n_head / n_kv;
    // wavefronts per workgroup: the whole group, or at head_dim 256 an even
    // share of it in groups of at most 4
    const uint32_t nw = hd == 256 ? (rep + (rep + 3) / 4 - 1) / ((rep + 3) / 4) : rep;
    void (*fn)(AttnPre) = nullptr;
#define LRS_PF_NW(W)                                                                     \
    case W:                                                                              \
        fn = hd == 64 ? k_attn_pf_mma<64, W> : hd == 128 ? k_attn_pf_mma<128, W> : nullptr; \
        break;
    if (hd == 64 || hd == 128) {
        switch (nw) {
            LRS_PF_NW(1) LRS_PF_NW(2) LRS_PF_NW(3) LRS_PF_NW(4)
            LRS_PF_NW(5) LRS_PF_NW(6) LRS_PF_NW(7) LRS_PF_NW(8)
        }
    } else if (hd == 256) {
        switch (nw) {
        case 1: fn = k_attn_pf_mma<256, 1>; break;
        case 2: fn = k_attn_pf_mma<256, 2>; break;
        case 3: fn = k_attn_pf_mma<256, 3>; break;
        case 4: fn = k_attn_pf_mma<256, 4>; break;
        }
    }
#undef LRS_PF_NW
    if (!fn) return hipErrorInvalidValue;
    const uint32_t ng = (rep + nw - 1) / nw;
    hipLaunchKernelGGL(fn, dim3((n + 31) / 32 * S, n_kv * ng), dim3(64 * nw), 0, s, a);
    hipLaunchKernelGGL(k_attn_merge, dim3(n_head * hd / 256, (n + 7) / 8), dim3(256), 0, s, part, ml, qg, S, n,
                       n_head, hd, planes);
    return hipGetLastError();
}

// silu(G) * U (ops.rs:978-988: g / (1 + e^-g) * u) as the down projection's
// GEMM input; workgroup = 32 rows x one super-block
__global__ __launch_bounds__(256) void k_swiglu_pack(const float *__restrict__ G,
                                                     const float *__restrict__ U, uint32_t F, uint32_t n,
                                                     uint8_t *__restrict__ planes) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint32_t row = 32 * blockIdx.y + 8 * k + (threadIdx.x >> 5);
        if (row >= n) return;
        const uint32_t c = 32 * blockIdx.x + (threadIdx.x & 31);
        const size_t i = (size_t)row * F + 8 * c;
        float v[8];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const float4 g = *reinterpret_cast<const float4 *>(G + i + 4 * h);
            const float4 u = *reinterpret_cast<const float4 *>(U + i + 4 * h);
            v[4 * h] = (g.x / (1.0f + expf(-g.x))) * u.x;
            v[4 * h + 1] = (g.y / (1.0f + expf(-g.y))) * u.y;
            v[4 * h + 2] = (g.z / (1.0f + expf(-g.z))) * u.z;
            v[4 * h + 3] = (g.w / (1.0f + expf(-g.w))) * u.w;
        }
        gp_store8<3>(v, row, c, F >> 8, planes);
    }
}

hipError_t launch_swiglu_pack(const float *G, const float *U, uint32_t F, uint32_t n, uint8_t *planes,
                              hipStream_t s) {
    if (F % 256 || n == 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_swiglu_pack, dim3(F / 256, (n + 31) / 32), dim3(256), 0, s, G, U, F, n, planes);
    return hipGetLastError();
}

}  // namespace lrs
