// Launch shape of the prompt GEMM (gemm.hip): arithmetic on sizes and types
// only, so that a host program compiles it alone.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

#include "../../include/lrs.h"

namespace lrs {

constexpr int PG_WAVES = 4;  // wavefronts of a workgroup
constexpr uint32_t PG_ROWS = 64 * PG_WAVES;  // weight rows of a workgroup

// Launch shape of a GEMM: row tiles of 32 tokens per workgroup, K slices.
struct PgPlan {
    uint32_t mt, ks;
};

inline uint32_t pg_tiles(uint32_t M, const uint32_t *N, uint32_t nseg, uint32_t mt) {
    uint32_t nn = 0;
    for (uint32_t i = 0; i < nseg; i++) nn += (N[i] + PG_ROWS - 1) / PG_ROWS;
    return (M + 32 * mt - 1) / (32 * mt) * nn;
}

// us per super-block of n workgroups that share a CU, measured with Q4_K
// weights at K = 5120: the first workgroups of a CU hide each other's waits.
// `fit`: workgroups that fit a CU at once (by registers)
inline double pg_unit(int prec, uint32_t mt, uint32_t fit, uint32_t n) {
    static const double p3m1[3] = {2.5, 4.4, 6.6}, p3m2[2] = {3.6, 6.4};
    static const double p1m1[3] = {2.0, 3.0, 4.2}, p1m2[3] = {2.7, 4.8, 6.4}, p1m4[2] = {4.4, 7.8};
    const double *c = prec == 3 ? (mt == 1 ? p3m1 : p3m2) : mt == 1 ? p1m1 : mt == 2 ? p1m2 : p1m4;
    return n / fit * c[fit - 1] + (n % fit ? c[n % fit - 1] : 0.0);
}

// The shape with the least expected time: the workgroups that a CU gets, and
// for K slices the partial sums written and read back (at about 7 TB/s, most
// of them in the memory-side cache) and the launch that adds them.
inline PgPlan pg_plan(uint32_t M, const uint32_t *N, const uint32_t *type, uint32_t nseg, uint32_t nsb, int prec) {
    // precision 3: Q6_K and Q8_0 take a third product, Q5_K more unpacking;
    // precision 1: their unpacking shows where a workgroup has few row tiles.
    // While every workgroup runs at once the slowest counts, else the average
    uint32_t ntot = 0;
    bool wide = false;  // a type whose operands take more registers
    for (uint32_t i = 0; i < nseg; i++) {
        ntot += N[i];
        wide = wide || type[i] == LRS_TYPE_Q6_K || type[i] == LRS_TYPE_Q5_K;
    }
    PgPlan best = {1, 1};
    double best_cost = 1e30;
    for (uint32_t mt = 1; mt <= (prec == 3 ? 2u : 4u); mt *= 2) {
        if (mt > 1 && M <= 16 * mt) break;
        double slow = 1.0, mean = 0.0;
        for (uint32_t i = 0; i < nseg; i++) {
            const double rel = type[i] == LRS_TYPE_Q4_K ? 1.0
                               : prec == 1       ? (mt == 4 ? 1.05 : 1.25)
                                                 : type[i] == LRS_TYPE_Q5_K ? 1.2 : 1.5;
            slow = std::max(slow, rel);
            mean += rel * N[i] / ntot;
        }
        const uint32_t tiles = pg_tiles(M, N, nseg, mt);
        const uint32_t fit = mt == (prec == 3 ? 2u : 4u) || (wide && !(prec == 1 && mt == 1)) ? 2 : 3;
        for (uint32_t ks = 1; ks <= nsb && ks <= 32; ks++) {
            if (ks > 1 && (tiles >= 2048 || M > 65535)) break;  // the reduce's grid has a y row per token
            const uint32_t len = (nsb + ks - 1) / ks, per = (tiles * ks + 255) / 256;
            const double rel = per < fit ? slow : per == fit ? 0.5 * (slow + mean) : mean;
            double cost = (len + 0.5) * rel * pg_unit(prec, mt, fit, per);
            if (ks > 1) cost += 5.0 + (2.0 * ks + 1) * M * ntot * 4.0 / 7e6;
            if (cost < best_cost * 0.98) {
                best_cost = cost;
                best = {mt, ks};
            }
        }
    }
    return best;
}

// bytes of the partial sums of a plan
inline size_t pg_bytes(const PgPlan &p, uint32_t M, const uint32_t *N, uint32_t nseg) {
    size_t ntot = 0;
    for (uint32_t i = 0; i < nseg; i++) ntot += N[i];
    return p.ks > 1 ? p.ks * ntot * M * sizeof(float) : 0;
}

// scratch of the K-sliced form of one call
inline size_t gemm_work_bytes(uint32_t M, const uint32_t *N, const uint32_t *type, uint32_t nseg, uint32_t K,
                              int prec) {
    return pg_bytes(pg_plan(M, N, type, nseg, K / 256, prec), M, N, nseg);
}

// ... of any call of up to M rows.  Fewer rows can take so many more slices
// that they need more (13824 x 4096 Q4_K, precision 3: 290 rows 64.1 MB, 512
// rows 42.5), at no particular row counts, so each is looked at: 0.2 ms for 512.
inline size_t gemm_work_most(uint32_t M, const uint32_t *N, const uint32_t *type, uint32_t nseg, uint32_t K,
                             int prec) {
    size_t most = 0;
    for (uint32_t m = 1; m <= M; m++) most = std::max(most, gemm_work_bytes(m, N, type, nseg, K, prec));
    return most;
}

}  // namespace lrs
