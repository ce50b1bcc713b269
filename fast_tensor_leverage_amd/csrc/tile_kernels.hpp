// tile_kernels.hpp -- descents of 16 samples per wave on the FP64 matrix cores.
//
// The group kernels (sampler_kernels.hpp) read every node of every sample's
// path into registers: 24 nodes of 4.2 KB per sample and mode at R = 32,
// I = 2^23, and that read (64 B per clock and CU from the L1, at about half of
// its rate) is what bounds them once the samples are taken in order.  Here a
// wave holds the x vectors of 16 samples that are neighbours in the order and
// evaluates x^T G x of one node for all of them: G in the A operand, read once
// per 16 samples, the x vectors in the B operand,
//   v_mfma_f64_16x16x4f64: A[i][k] in lane 16k + i, B[k][j] in lane 16k + j,
//   D[4v + l/16][l%16] in item v of lane l.
// Lane l keeps x_{4t + l/16} of sample l%16 for t = 0, 1, ..., which is the B
// operand of every step and also the factor that item v of a result tile is
// multiplied by, so nothing moves between lanes but the final sum over l/16.
// Samples of the tile that stand at different nodes are served one node after
// the other.  Deep in the tree each sample stands alone and the group kernel is
// the better one: a descent stops when a level took more than kTileStop nodes
// and is resumed there.  With J samples in the order of their uniforms that is
// about two levels past log2(J / 16): level 13.8 on average for J = 50,000, of 18
// at I = 2^23, R = 32.
#pragma once

#include "sampler_kernels.hpp"

namespace ftl {

// Loads of a node in flight per wave, and waves per SIMD (782 blocks at J =
// 50,000 are just over three per CU, so a fourth is worth more than longer
// chunks; above R = 80 its 128 registers spill).
template <int NB>
struct TileCfg {
    static constexpr int kChunk = NB <= 6 ? 16 : 4 * NB;
    static constexpr int kWaves = NB <= 6 ? 4 : 3;
};

// x^T G x of the tile's samples for one node (a wave-uniform address), in every
// lane of the sample.  Only the stored triangle is used: 16 x 16 block (p, q),
// p <= q, adds G_pq^T x_p to y_q, a diagonal block as its strict upper part plus
// half of its diagonal, and the result is twice the sum of x_q^T y_q.  A load
// then takes four row segments of up to 16 entries (mirroring the diagonal
// blocks instead spread each of their loads over some 35 cache lines, and the
// address unit bounded the kernel).  Lanes outside the triangle or past R read
// an entry of their row segment and use zero.
template <int NB, typename TN>
__device__ __forceinline__ double tile_form(const TN* __restrict__ node, const double (&x)[4 * NB], uint32_t R,
                                            uint32_t lane) {
    uint32_t kr = lane >> 4;
    const uint32_t ci = lane & 15;
    // load offsets are formed per call, above R = 96 per block column: hoisted,
    // or shared between the columns, they take the registers of a wave per SIMD
    if constexpr (NB > 2 && NB <= 6) asm volatile("" : "+v"(kr));
    const char* base = reinterpret_cast<const char*>(node);
    auto entry = [&](uint32_t e) { return *reinterpret_cast<const TN*>(base + e * (uint32_t)sizeof(TN)); };
    double total = 0.0;
#pragma unroll
    for (int q = 0; q < NB; q++) {
        lg_f64x4 acc = {0.0, 0.0, 0.0, 0.0};
        if constexpr (NB > 6) asm volatile("" : "+v"(kr));
        const uint32_t b = min(16 * q + ci, R - 1);
        // entry (r, c) sits at rb(r) + c, rb(r) = r R - r (r + 1) / 2; the rows
        // of a lane are kr, kr + 4, ...
        uint32_t rb = kr * R - kr * (kr + 1) / 2, step = 4 * R - 4 * kr - 10;
#pragma unroll
        for (int t0 = 0; t0 < 4 * (q + 1); t0 += TileCfg<NB>::kChunk) {
            TN g[TileCfg<NB>::kChunk];
#pragma unroll
            for (int u = 0; u < TileCfg<NB>::kChunk; u++) {
                const int t = t0 + u;
                if (t < 4 * q) {
                    g[u] = entry(rb + b);
                } else if (t < 4 * (q + 1)) {
                    const uint32_t r = 4 * t + kr;
                    g[u] = entry(r < R ? rb + max(r, b) : R * (R + 1) / 2 - 1);
                }
                rb += step;
                step -= 16;
            }
#pragma unroll
            for (int u = 0; u < TileCfg<NB>::kChunk; u++) {
                const int t = t0 + u;
                double v = t < 4 * (q + 1) ? (double)g[u] : 0.0;
                if (t >= 4 * q) {
                    const uint32_t e = 4 * (t - 4 * q) + kr;
                    v = e < ci ? v : e == ci ? 0.5 * v : 0.0;
                }
                if (t < 4 * (q + 1)) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(v, x[t], acc, 0, 0, 0);
            }
            if constexpr (NB > 2) __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int v = 0; v < 4; v++) total += acc[v] * x[4 * q + v];
    }
    return 2.0 * pair_sum32(pair_sum16(total));
}

// The descent of descend (partition_tree.hpp:251-332) for the tile's samples,
// from the root to the leaves or to the level at which more than `stop` nodes
// were needed; depth: the sample's level on return.
template <int NB, bool USE32>
__device__ __forceinline__ void tile_descend(const ModeDev& md, const Shape& sh, uint32_t ts64, uint32_t ts32,
                                             const double* tree64, const double (&x)[4 * NB], uint32_t R, double u,
                                             bool active, uint32_t stop, uint32_t lane, uint32_t& c, double& low,
                                             double& high, double& m, uint32_t& depth) {
    m = tile_form<NB, double>(tree64, x, R, lane);
    c = 0;
    low = 0.0;
    high = 1.0;
    const uint32_t lfill = (uint32_t)sh.lfill_level, nodes = (uint32_t)sh.node_count;
    uint32_t d = 0;
    while (d <= lfill) {
        const uint32_t child = 2 * c + 1;
        // the guarded tail level: a leaf on the lfill level stops here
        const bool go = active && child < nodes;
        uint64_t rem = __ballot(go);
        uint32_t n = 0;
        while (rem) {
            const uint32_t node = (uint32_t)__builtin_amdgcn_readlane((int)child, __builtin_ctzll(rem));
            double mL;
            if (!USE32 || d + 1 < md.d64)
                mL = tile_form<NB, double>(tree64 + (uint64_t)node * ts64, x, R, lane);
            else
                mL = tile_form<NB, float>(md.tree32 + ((uint64_t)node - md.n64) * ts32, x, R, lane);
            const bool mine = go && child == node;
            if (mine) {
                const double cutoff = low + mL / m;
                if (u <= cutoff) {
                    c = child;
                    high = cutoff;
                } else {
                    c = child + 1;
                    low = cutoff;
                }
            }
            rem &= ~__ballot(mine);
            n++;
        }
        d++;
        if (n > stop) break;
    }
    depth = d;
}

// Nodes that one level may take for a tile before the group kernel goes on.
constexpr uint32_t kTileStop = 2;

// Eigen stage of sampled mode a.mi_begin: the eigen row of every sample to
// a.st_r.  Samples in the order of their eigen uniforms.
template <int NB>
__global__ void __launch_bounds__(256, TileCfg<NB>::kWaves) k_tile_eigen(DrawArgs a) {
    const uint32_t lane = threadIdx.x & 63, kr = lane >> 4;
    const uint64_t tile = (uint64_t)ordered_block(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6);
    if (tile * 16 >= a.J) return;
    const uint64_t slot = tile * 16 + (lane & 15);
    const bool active = slot < a.J;
    const uint64_t i = a.perm[active ? slot : a.J - 1];
    const uint32_t R = (uint32_t)a.R;
    const int k = a.order[a.mi_begin];
    const ModeDev& md = a.mode[k];
    double x[4 * NB];
#pragma unroll
    for (int t = 0; t < 4 * NB; t++) {
        const uint32_t e = 4 * t + kr;
        x[t] = e < R ? (a.mi_begin > 0 ? a.h_state[i * R + e] : 1.0) : 0.0;
    }
    const double u = a.draws ? a.draws[(uint64_t)k * a.J + i] : philox_uniform(a.seed, a.call, i, 2 * k);
    uint32_t c, depth;
    double low, high, m;
    tile_descend<NB, false>(md, a.esh, a.ts64, a.ts32, md.etree, x, R, u, active, ~0u, lane, c, low, high, m, depth);
    if (active && kr == 0) a.st_r[i] = (uint32_t)leaf_index(a.esh, c);
}

// Upper levels of the Gram descent of sampled mode a.mi_begin: {low, high, m,
// node and level} of every sample to a.st_s.  Samples in the order of their
// Gram uniforms.
template <int NB, bool USE32>
__global__ void __launch_bounds__(256, TileCfg<NB>::kWaves) k_tile_gram(DrawArgs a) {
    const uint32_t lane = threadIdx.x & 63, kr = lane >> 4;
    const uint64_t tile = (uint64_t)ordered_block(blockIdx.x, gridDim.x) * 4 + (threadIdx.x >> 6);
    if (tile * 16 >= a.J) return;
    const uint64_t slot = tile * 16 + (lane & 15);
    const bool active = slot < a.J;
    const uint64_t i = a.perm[active ? slot : a.J - 1];
    const uint32_t R = (uint32_t)a.R;
    const int k = a.order[a.mi_begin];
    const ModeDev& md = a.mode[k];
    const double* er = md.E + (uint64_t)a.st_r[i] * R;
    double x[4 * NB];
#pragma unroll
    for (int t = 0; t < 4 * NB; t++) {
        const uint32_t e = 4 * t + kr;
        x[t] = e < R ? (a.mi_begin > 0 ? a.h_state[i * R + e] * er[e] : er[e]) : 0.0;
    }
    const double u = a.draws ? a.draws[(uint64_t)a.N * a.J + (uint64_t)k * a.J + i]
                             : philox_uniform(a.seed, a.call, i, 2 * k + 1);
    uint32_t c, depth;
    double low, high, m;
    tile_descend<NB, USE32>(md, md.sh, a.ts64, a.ts32, md.tree64, x, R, u, active, kTileStop, lane, c, low, high, m,
                            depth);
    if (active && kr == 0) {
        double* st = a.st_s + i * 4;
        st[0] = low;
        st[1] = high;
        st[2] = m;
        st[3] = __longlong_as_double((long long)((uint64_t)depth << 32 | c));
    }
}

}  // namespace ftl
