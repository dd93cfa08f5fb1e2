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

// us per super-block of 1, 2, ... workgroups that share a CU (the first ones hide
// each other's waits), as many as fit it by registers.  The bf16 form's, and
// Q8_0's, are fitted to launches of every shape forced in turn on random weights:
// matrices and groups from 2048 x 2048 to 2 x 27648 x 5120, 2 to 2048 rows, up to
// 32 slices, weights from memory and from the cache, 38 000 launches.  Over them
// the shape chosen in bf16 takes 1.0 % longer than the best (geometric mean; at
// most 22 %), and with Q8_0 at precision 3 1.2 % (12 %).  Costs of Q4_K times a
// factor per type took 3.7 % (51 %: Q4_K in bf16, 384 x 13824 x 5120 as one row
// tile 116 us, as four 79) and 3.1 % (32 %).  The K-quants' at precision 3 (2 %)
// are those factors: fitted costs took 0.5 % over these calls, but a prompt block
// of 12 to 32 tokens, where the launch that adds the slices costs 5 us, was up to
// 6 % slower.
struct PgCost {
    uint32_t fit;
    double us[4];
};
inline PgCost pg_cost(int prec, uint32_t mt, uint32_t type) {
    const int t = type == LRS_TYPE_Q4_K ? 0 : type == LRS_TYPE_Q5_K ? 1 : type == LRS_TYPE_Q6_K ? 2 : 3;
    static const PgCost p3[2][4] = {
        {{3, {2.5, 4.4, 6.6}}, {2, {3.0, 5.28}}, {2, {3.75, 6.6}}, {3, {3.8, 5.6, 9.4}}},
        {{2, {3.6, 6.4}}, {2, {4.32, 7.68}}, {2, {5.4, 9.6}}, {2, {5.4, 8.8}}}};
    static const PgCost p1[3][4] = {
        {{4, {2.0, 3.3, 4.6, 6.5}}, {3, {2.4, 3.7, 5.3}}, {3, {2.4, 4.1, 6.0}}, {4, {2.8, 3.6, 5.2, 7.0}}},
        {{3, {2.7, 4.5, 6.4}}, {2, {3.5, 5.0}}, {2, {3.4, 5.6}}, {3, {3.4, 4.8, 6.4}}},
        {{2, {4.3, 6.5}}, {2, {4.6, 8.0}}, {2, {4.6, 8.1}}, {2, {4.7, 6.8}}}};
    return prec == 3 ? p3[mt / 2][t] : p1[mt / 2][t];
}

// The shape with the least expected time: the super-blocks of a workgroup (and
// part of one to start it), times what they cost with the workgroups that a CU
// gets; for K slices the partial sums written and read back (most of them in the
// memory-side cache) and the launch that adds them.
inline PgPlan pg_plan(uint32_t M, const uint32_t *N, const uint32_t *type, uint32_t nseg, uint32_t nsb, int prec) {
    double ntot = 0;
    for (uint32_t i = 0; i < nseg; i++) ntot += N[i];
    PgPlan best = {1, 1};
    double best_cost = 1e30;
    for (uint32_t mt = 1; mt <= (prec == 3 ? 2u : 4u); mt *= 2) {
        if (mt > 1 && M <= 16 * mt) break;
        const uint32_t tiles = pg_tiles(M, N, nseg, mt);
        // a launch of two types is compiled for the larger's registers
        uint32_t fit = 4;
        for (uint32_t i = 0; i < nseg; i++) fit = std::min(fit, pg_cost(prec, mt, type[i]).fit);
        for (uint32_t ks = 1; ks <= nsb && ks <= 32; ks++) {
            if (ks > 1 && (tiles >= 2048 || M > 65535)) break;  // the reduce's grid has a y row per token
            const uint32_t len = (nsb + ks - 1) / ks, per = (tiles * ks + 255) / 256;
            // while every workgroup runs at once the slowest type counts, else the average
            double slow = 0.0, mean = 0.0;
            for (uint32_t i = 0; i < nseg; i++) {
                const PgCost c = pg_cost(prec, mt, type[i]);
                const double u = per / fit * c.us[fit - 1] + (per % fit ? c.us[per % fit - 1] : 0.0);
                slow = std::max(slow, u);
                mean += u * N[i] / ntot;
            }
            const double u = per < fit ? slow : per == fit ? 0.5 * (slow + mean) : mean;
            const double moved = (2.0 * ks + 1) * M * ntot * 4.0;
            double cost = (len + (prec == 3 ? 0.5 : 0.3)) * u;
            if (ks > 1) cost += prec == 3 ? 5.0 + moved / 7e6 : 1.0 + 0.2 * ks + moved / 8e6;
            if (cost < best_cost * 0.98) {  // fewer row tiles and slices where it is close
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
// rows none), at no particular row counts, so each is looked at: 0.2 ms for 512.
inline size_t gemm_work_most(uint32_t M, const uint32_t *N, const uint32_t *type, uint32_t nseg, uint32_t K,
                             int prec) {
    size_t most = 0;
    for (uint32_t m = 1; m <= M; m++) most = std::max(most, gemm_work_bytes(m, N, type, nseg, K, prec));
    return most;
}

}  // namespace lrs
