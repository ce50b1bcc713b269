// jacobi.hpp -- block-level cyclic Jacobi eigensolver for small symmetric
// matrices (R <= 128), used by computeM and by the sampled-Gram pseudo-inverse
// of the ALS step.
#pragma once

#include "ftl_common.hpp"
#include "wave_ops.hpp"

namespace ftl {

// ---------------------------------------------------------------------------
// Cyclic Jacobi eigensolver for one symmetric R x R matrix held by a block.
// Round-robin pair order (circle method); a round rotates its R/2 disjoint
// pairs (p, q): J^T A J applied to the 2x2 blocks where a row pair meets a
// column pair, the row rotation before the column rotation, and V J, V stored
// transposed (row v holds eigenvector column v).  Rotation annihilating
// A[p][q], p < q (Golub & Van Loan Alg. 8.5.2), skipped when
// |A[p][q]| <= eps*sqrt(|A[p][p] A[q][q]|).  Products and sums are rounded
// individually (no contraction).  On return lam is ascending and Vout column
// v holds the eigenvector of lam[v].
// ---------------------------------------------------------------------------
constexpr int kJacobiSmallR = 64;

// Rotations of a round, pair by pair: {c, s} with top' = c top - s bottom,
// bottom' = s top + c bottom, s = 0 for a skipped pair.
struct JacobiShared {
    double2 rot[2][64];
    int p[64], q[64], act[64];
    double c[64], s[64];
};

// 1/x and 1/sqrt(x): v_rcp_f64 / v_rsq_f64 estimates plus one Newton step.
__device__ inline double fast_rcp(double x) {
    double r = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, r, 1.0);
    return fma(r, e, r);
}

__device__ inline double fast_rsq(double x) {
    double r = __builtin_amdgcn_rsq(x);
    const double h = 0.5 * x * r;
    const double e = fma(-h, r, 0.5);
    return fma(r, e, r);
}

// The rotation of tangent t != 0.
__device__ inline void jacobi_cs(double t, double& c, double& s) {
#pragma clang fp contract(off)
    c = fast_rsq(1.0 + t * t);
    s = t * c;
}

// Rotation (c, s) of tangent t annihilating apq = A[p][q]; false (c = 1, s = t = 0)
// when it is negligible.
__device__ inline bool jacobi_rotation(double app, double aqq, double apq, double& c, double& s, double& t) {
#pragma clang fp contract(off)
    c = 1.0;
    s = t = 0.0;
    const double eps = 2.220446049250313e-16;
    // |apq| <= eps sqrt(|app aqq|), compared in squares (no square root on
    // the round's critical path)
    if (apq * apq <= (eps * eps) * fabs(app * aqq) || apq == 0.0) return false;
    // hardware reciprocal / reciprocal square root, each refined by one
    // Newton step (error ~1 ulp; the rotation stays orthogonal to working
    // precision)
    const double tau = (aqq - app) * fast_rcp(2.0 * apq);
    if (fabs(tau) > 1e150) {
        t = 0.5 * fast_rcp(tau);
    } else {
        const double x = 1.0 + tau * tau;
        const double sq = x * fast_rsq(x);
        t = (tau >= 0 ? 1.0 : -1.0) * fast_rcp(fabs(tau) + sq);
    }
    jacobi_cs(t, c, s);
    return true;
}

// The same from A; false also when q is the padding index of an odd size.
__device__ inline bool jacobi_rotation(const double* A, int LD, int R, int p, int q, double& c, double& s) {
    c = 1.0;
    s = 0.0;
    if (q >= R) return false;
    double t;
    return jacobi_rotation(A[p * LD + p], A[q * LD + q], A[p * LD + q], c, s, t);
}

// Sweep cap of the cyclic Jacobi iteration (quadratic convergence takes
// 6-10 sweeps for R <= 128 in FP64).
constexpr int kJacobiMaxSweeps = 40;

// Eigensolves of this translation unit's kernels that stopped at the sweep
// cap (one device counter per source file and device; read on the host with
// jacobi_capped_read).
static __device__ uint32_t g_jacobi_capped = 0;

static inline uint64_t jacobi_capped_read() {
    uint32_t v = 0;
    FTL_HIP_CHECK(hipDeviceSynchronize());
    FTL_HIP_CHECK(hipMemcpyFromSymbol(&v, HIP_SYMBOL(g_jacobi_capped), sizeof(v), 0, hipMemcpyDeviceToHost));
    return v;
}

// Stable ascending sort of A's diagonal; Vout (R x R, dense) column v is the
// eigenvector of lam[v].  Vout may be A.
template <int BS>
__device__ __forceinline__ void jacobi_sorted(const double* A, int LD, const double* V, int LV, int R, double* lam,
                                              double* Vout, double* diag_tmp) {
    for (int v = threadIdx.x; v < R; v += BS) diag_tmp[v] = A[v * LD + v];
    __syncthreads();
    for (int w = threadIdx.x; w < R * R; w += BS) {
        const int v = w / R, i = w - v * R;
        const double d = diag_tmp[v];
        int rank = 0;
        for (int u = 0; u < R; u++) {
            const double du = diag_tmp[u];
            rank += (du < d) || (du == d && u < v);
        }
        if (i == 0) lam[rank] = d;
        Vout[i * R + rank] = V[v * LV + i];
    }
}

// The order the matrix is padded to (a zero row and column when odd) and the
// row length of A: odd, so rows start in different LDS banks.  Above
// kJacobiSmallR the general solver's A is not padded.
__host__ __device__ constexpr int jacobi_n2(int R) { return R + (R & 1); }
__host__ __device__ inline int jacobi_ld(int R) { return R <= kJacobiSmallR ? jacobi_n2(R) + 1 : R + 1; }

// Element of pair k's top / bottom in round `round`, m = n2 - 1 rounds a sweep:
// position 0 fixed, the others moving by one a round.
__device__ inline int jacobi_top(uint32_t k, uint32_t round, uint32_t m) {
    const uint32_t a = k - 1 + round;
    return k == 0 ? 0 : (int)(1 + min(a, a - m));
}
__device__ inline int jacobi_bottom(uint32_t k, uint32_t round, uint32_t m) {
    const uint32_t a = m - 1 - k + round;
    return (int)(1 + min(a, a - m));
}

// Entry (slot sr of row pair kr, slot sc of column pair kc) of J^T A J for the
// rotations `rot` of round `round` (slot 0 top, 1 bottom).
__device__ inline double jacobi_entry_after(const double* A, int LD, const double2* rot, uint32_t round, uint32_t m,
                                            uint32_t kr, uint32_t sr, uint32_t kc, uint32_t sc) {
#pragma clang fp contract(off)
    const double* At = A + jacobi_top(kr, round, m) * LD;
    const double* Ab = A + jacobi_bottom(kr, round, m) * LD;
    const int t2 = jacobi_top(kc, round, m), b2 = jacobi_bottom(kc, round, m);
    const double2 g = rot[kr], g2 = rot[kc];
    const double att = At[t2], atb = At[b2], abt = Ab[t2], abb = Ab[b2];
    double xt = sr ? abt : att, xb = sr ? abb : atb;
    if (g.y != 0.0) {
        const double u = sr ? g.y : g.x, v = sr ? g.x : -g.y;
        xt = u * att + v * abt;
        xb = u * atb + v * abb;
    }
    double x = sc ? xb : xt;
    if (g2.y != 0.0) {
        const double u = sc ? g2.y : g2.x, v = sc ? g2.x : -g2.y;
        x = u * xt + v * xb;
    }
    return x;
}

// Rotation of pair k, whose elements in its round are P (top) and Q, to rot[k]
// (and its tangent, of the same sign, to log[k]); whether it is applied.
__device__ __forceinline__ bool jacobi_put(double2* rot, double* log, uint32_t k, int R, int P, int Q, double app,
                                           double aqq, double apq) {
    double c = 1.0, s = 0.0, t = 0.0;
    const bool act = max(P, Q) < R && jacobi_rotation(app, aqq, apq, c, s, t);
    rot[k] = make_double2(c, P < Q ? s : -s);
    if (log) log[k] = P < Q ? t : -t;
    return act;
}

// Rotation of pair k in the round after `round`, from A and the rotations of
// `round`: its top is the top of pair k + 1 (the last pair's its own bottom),
// its bottom the bottom of pair k - 1 (the first pair's the top of pair 1).
__device__ __forceinline__ bool jacobi_next_rotation(const double* A, int LD, int R, const double2* rot,
                                                     uint32_t round, uint32_t m, uint32_t np, uint32_t k, double2* out,
                                                     double* log) {
    const uint32_t rn = round + 1 == m ? 0 : round + 1;
    const int P = jacobi_top(k, rn, m), Q = jacobi_bottom(k, rn, m);
    uint32_t kp, sp, kq, sq;
    if (k == 0) {
        kp = 0, sp = 0;
        kq = np > 1 ? 1 : 0, sq = np > 1 ? 0 : 1;
    } else {
        const bool last = k + 1 == np;
        kp = last ? k : k + 1, sp = last ? 1 : 0;
        kq = k - 1, sq = 1;
    }
    if (P > Q) {
        const uint32_t t = kp, u = sp;
        kp = kq, sp = sq;
        kq = t, sq = u;
    }
    const double app = jacobi_entry_after(A, LD, rot, round, m, kp, sp, kp, sp);
    const double aqq = jacobi_entry_after(A, LD, rot, round, m, kq, sq, kq, sq);
    const double apq = jacobi_entry_after(A, LD, rot, round, m, kp, sp, kq, sq);
    return jacobi_put(out, log, k, R, P, Q, app, aqq, apq);
}

// Items first, first + step, ... of J^T A J of a round: item it is the 2x2
// block of row pair it / np and column pair it % np.  BATCH items are loaded
// before any is written.  An may be A.
template <int BATCH>
__device__ __forceinline__ void jacobi_apply(const double* A, double* An, int LD, const double2* rot, uint32_t round,
                                             uint32_t m, uint32_t np, uint32_t first, uint32_t step) {
#pragma clang fp contract(off)
    uint32_t k = first / np, k2 = first - k * np;
    const uint32_t dk = step / np, dk2 = step - dk * np;
    for (uint32_t it = first; it < np * np; it += BATCH * step) {
        double2 g[BATCH], g2[BATCH];
        int t[BATCH], b[BATCH], t2[BATCH], b2[BATCH];
        double att[BATCH], atb[BATCH], abt[BATCH], abb[BATCH];
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
            // items past the end are those of pair 0 again, not written
            const bool in = u == 0 || it + u * step < np * np;
            const uint32_t kr = in ? k : 0, kc = in ? k2 : 0;
            g[u] = rot[kr];
            g2[u] = rot[kc];
            t[u] = jacobi_top(kr, round, m) * LD;
            b[u] = jacobi_bottom(kr, round, m) * LD;
            t2[u] = jacobi_top(kc, round, m);
            b2[u] = jacobi_bottom(kc, round, m);
            att[u] = A[t[u] + t2[u]];
            atb[u] = A[t[u] + b2[u]];
            abt[u] = A[b[u] + t2[u]];
            abb[u] = A[b[u] + b2[u]];
            k += dk;
            k2 += dk2;
            if (k2 >= np) {
                k2 -= np;
                k++;
            }
        }
#pragma unroll
        for (int u = 0; u < BATCH; u++) {
            if (u > 0 && it + u * step >= np * np) break;
            double rtt = att[u], rtb = atb[u], rbt = abt[u], rbb = abb[u];
            if (g[u].y != 0.0) {
                rtt = g[u].x * att[u] - g[u].y * abt[u];
                rbt = g[u].y * att[u] + g[u].x * abt[u];
                rtb = g[u].x * atb[u] - g[u].y * abb[u];
                rbb = g[u].y * atb[u] + g[u].x * abb[u];
            }
            double ntt = rtt, ntb = rtb, nbt = rbt, nbb = rbb;
            if (g2[u].y != 0.0) {
                ntt = g2[u].x * rtt - g2[u].y * rtb;
                ntb = g2[u].y * rtt + g2[u].x * rtb;
                nbt = g2[u].x * rbt - g2[u].y * rbb;
                nbb = g2[u].y * rbt + g2[u].x * rbb;
            }
            An[t[u] + t2[u]] = ntt;
            An[t[u] + b2[u]] = ntb;
            An[b[u] + t2[u]] = nbt;
            An[b[u] + b2[u]] = nbb;
        }
    }
}

// Whether a pair p < q of A does not meet the skip test (in the thread's share).
template <int BS>
__device__ __forceinline__ int jacobi_open(const double* A, int LD, int R) {
    int open = 0;
    for (int w = threadIdx.x; w < R * R; w += BS) {
        const int p = w / R, q = w - (w / R) * R;
        if (p < q) {
            const double apq = A[p * LD + q];
            const double thr = (2.220446049250313e-16 * 2.220446049250313e-16) * fabs(A[p * LD + p] * A[q * LD + q]);
            open |= !(apq * apq <= thr || apq == 0.0);
        }
    }
    return open;
}

// R <= kJacobiSmallR: one barrier per round.  A is double-buffered (A0 holds the
// matrix, n2 x LD with the padding zero), and while the other waves apply round
// r to A (current to next buffer) and V, wave 0 forms the rotations of round
// r + 1 from the few entries of the next A that they need, so the chain of a
// round is one rotation, not a rotation and an update.  The waves of A and of V
// are separate, and a thread derives the elements of its pairs from the round
// number, so that an item costs its entries and one {c, s} pair per rotation in
// LDS traffic, which bounds a round from R = 48 on.  The operations on every
// entry and their order are those of the two-barrier form: a pair whose top is
// its larger index only has the sign of its s turned.  k_gram_pinv over 700- and
// 300-row Gaussian / ill-conditioned factors, two barriers a round -> this (us):
// R = 32 156 / 296 -> 113 / 203, R = 16 59 / 123 -> 45 / 91.  Vout may be A1; A0 is
// overwritten.  Returns false (in every thread) when the sweep cap ended the
// iteration before every pair met the skip test.
template <int BS>
__device__ __forceinline__ bool jacobi_small(double* A0, double* A1, double* V, int R, double* lam, double* Vout,
                                             JacobiShared& js, double* diag_tmp) {
#pragma clang fp contract(off)
    constexpr int NWV = BS / 64, NA = NWV / 2, NV = NWV - 1 - NA;
    static_assert(NV >= 1, "a wave for the rotations, for A and for V");
    const int tid = threadIdx.x, wave = tid >> 6;
    const int n2 = jacobi_n2(R), LD = n2 + 1, LV = R + 1;
    const uint32_t m = n2 - 1, np = n2 / 2;
    for (int e = tid; e < R * R; e += BS) V[(e / R) * LV + e % R] = (e / R == e % R) ? 1.0 : 0.0;
    __syncthreads();
    // items of V: (k, i), i fastest; a thread's next item is a fixed step on
    const uint32_t ta = tid - 64, tv = tid - 64 * (1 + NA);
    const uint32_t nv = np * (uint32_t)R;
    const uint32_t kv = tv / R, iv = tv - kv * R, dv = (64 * NV) / R, div = 64 * NV - dv * R;
    int cur = 0;
    bool carry = false;
    if (tid < (int)np) {
        const int P = jacobi_top(tid, 0, m), Q = jacobi_bottom(tid, 0, m);
        const int p = min(P, Q), q = max(P, Q);
        carry = jacobi_put(js.rot[0], nullptr, tid, R, P, Q, A0[p * LD + p], A0[q * LD + q], A0[p * LD + q]);
    }
    __syncthreads();
    bool converged = false;
    for (int sweep = 0; sweep < kJacobiMaxSweeps; sweep++) {
        int any = carry;
        for (uint32_t r = 0; r < m; r++) {
            const double* A = cur ? A1 : A0;
            double* An = cur ? A0 : A1;
            const double2* rot = js.rot[cur];
            if (wave == 0) {
                if (tid < (int)np) {
                    carry = jacobi_next_rotation(A, LD, R, rot, r, m, np, tid, js.rot[cur ^ 1], nullptr);
                    if (r + 1 < m) any |= carry;
                }
            } else if (wave <= NA) {
                jacobi_apply<1>(A, An, LD, rot, r, m, np, ta, 64 * NA);
            } else {
                uint32_t k = kv, i = iv;
                for (uint32_t it = tv; it < nv; it += 64 * NV) {
                    const double2 g = rot[k];
                    if (g.y != 0.0) {
                        double* vt = V + jacobi_top(k, r, m) * LV + i;
                        double* vb = V + jacobi_bottom(k, r, m) * LV + i;
                        const double x = *vt, y = *vb;
                        *vt = g.x * x - g.y * y;
                        *vb = g.y * x + g.x * y;
                    }
                    k += dv;
                    i += div;
                    if (i >= (uint32_t)R) {
                        i -= R;
                        k++;
                    }
                }
            }
            __syncthreads();
            cur ^= 1;
        }
        if (!__syncthreads_or(any)) {
            converged = true;
            break;
        }
        // converged when every pair meets the skip test: the next sweep would
        // rotate nothing, so stopping here gives the same result
        if (!__syncthreads_or(jacobi_open<BS>(cur ? A1 : A0, LD, R))) {
            converged = true;
            break;
        }
    }
    jacobi_sorted<BS>(cur ? A1 : A0, LD, V, LV, R, lam, Vout, diag_tmp);
    if (!converged && tid == 0) atomicAdd(&g_jacobi_capped, 1u);
    __syncthreads();
    return converged;
}

// Ranks from which computeM's eigensolves are split over launches: one block
// diagonalises A and logs its rotations, then a wave per row of V applies them
// (k_cm_vectors).  V's updates are a third of a round's FP64 operations and half of
// its entries, and inside the block they share its one CU's LDS and FP64 issue
// with A's (above R = 64 V did not fit the LDS at all).  G's part of computeM,
// Gaussian / ill-conditioned: R = 64 0.31 / 0.59 ms (one block 0.53 / 0.94), R = 128
// 1.49 / 2.90 (4.46 / 7.63).  At R = 32 the extra launches cost what V does.
constexpr int kJacobiSplitR = 33;

// Two buffers of A up to this rank (149 KB at 96).
constexpr int kJacobiDoubleR = 96;

__host__ __device__ inline uint64_t jacobi_solve_lds_doubles(uint64_t R) {
    const uint64_t n2 = (uint64_t)jacobi_n2((int)R);
    return (R <= (uint64_t)kJacobiDoubleR ? 2 : 1) * n2 * (n2 + 1);
}
// Doubles of a matrix's log of rotations: their tangents, from which (c, s)
// follow bit for bit, for every sweep up to the cap.
__host__ __device__ constexpr uint64_t jacobi_log_doubles(uint64_t R) {
    const uint64_t n2 = (uint64_t)jacobi_n2((int)R);
    return kJacobiMaxSweeps * (n2 - 1) * (n2 / 2);
}

// A (n2 x (n2 + 1), padding zero) diagonalised: lam ascending, rank[v] the place
// of diagonal entry v, *rounds the rounds done and their tangents in log (n2 / 2
// per round).  TWO: A1 is the second buffer; else two barriers a round, in place.
template <int BS, bool TWO>
__device__ __forceinline__ void jacobi_solve(double* A0, double* A1, int R, double* log, double* lam, int* rank,
                                             int* rounds, JacobiShared& js, double* diag_tmp) {
    const int tid = threadIdx.x, wave = tid >> 6;
    const int n2 = jacobi_n2(R), LD = n2 + 1;
    const uint32_t m = n2 - 1, np = n2 / 2;
    int cur = 0;
    bool carry = false;
    auto first = [&](const double* A, int buf, uint32_t round, double* to) {
        const int P = jacobi_top(tid, round, m), Q = jacobi_bottom(tid, round, m);
        const int p = min(P, Q), q = max(P, Q);
        return jacobi_put(js.rot[buf], to, tid, R, P, Q, A[p * LD + p], A[q * LD + q], A[p * LD + q]);
    };
    double* lg = log;  // the log of the round
    if constexpr (TWO) {
        if (tid < (int)np) carry = first(A0, 0, 0, lg);
        __syncthreads();
    }
    bool converged = false;
    for (int sweep = 0; sweep < kJacobiMaxSweeps; sweep++) {
        int any = carry;
        for (uint32_t r = 0; r < m; r++, lg += np) {
            if constexpr (TWO) {
                const double* A = cur ? A1 : A0;
                if (wave == 0) {
                    if (tid < (int)np) {
                        // the log of the round after the last sweep's last one
                        // is not part of it
                        const bool in = sweep + 1 < kJacobiMaxSweeps || r + 1 < m;
                        carry = jacobi_next_rotation(A, LD, R, js.rot[cur], r, m, np, tid, js.rot[cur ^ 1],
                                                     in ? lg + np : nullptr);
                        if (r + 1 < m) any |= carry;
                    }
                } else {
                    jacobi_apply<1>(A, cur ? A0 : A1, LD, js.rot[cur], r, m, np, tid - 64, BS - 64);
                }
                __syncthreads();
                cur ^= 1;
            } else {
                if (tid < (int)np) any |= first(A0, 0, r, lg);
                __syncthreads();
                // four items in flight, unless most of a thread's four are past
                // the end (R = 100: 1.58 against 1.94 ms)
                if (np * np > 3 * BS) jacobi_apply<4>(A0, A0, LD, js.rot[0], r, m, np, tid, BS);
                else jacobi_apply<1>(A0, A0, LD, js.rot[0], r, m, np, tid, BS);
                __syncthreads();
            }
        }
        if (!__syncthreads_or(any)) {
            converged = true;
            break;
        }
        if (!__syncthreads_or(jacobi_open<BS>(TWO && cur ? A1 : A0, LD, R))) {
            converged = true;
            break;
        }
    }
    const double* A = TWO && cur ? A1 : A0;
    for (int v = tid; v < R; v += BS) diag_tmp[v] = A[v * LD + v];
    __syncthreads();
    for (int v = tid; v < R; v += BS) {
        const double d = diag_tmp[v];
        int at = 0;
        for (int u = 0; u < R; u++) {
            const double du = diag_tmp[u];
            at += (du < d) || (du == d && u < v);
        }
        lam[at] = d;
        rank[v] = at;
    }
    if (tid == 0) *rounds = (int)((lg - log) / np);
    if (!converged && tid == 0) atomicAdd(&g_jacobi_capped, 1u);
}

// DPP shifts of a wave by one lane: lane i takes lane i + 1's / i - 1's value.
__device__ inline double wave_from_next(double v) { return dpp_f64<0x130>(v); }
__device__ inline double wave_from_prev(double v) { return dpp_f64<0x138>(v); }

// Row i of V after the logged rotations, in registers: lane k (of the row's LPR
// lanes, one per pair) holds the entries of pair k's top and bottom in place of
// the round, and hands them on to the neighbouring lanes.  put(v, x): entry x of
// eigenvector column v.  V starts as the identity.
template <int LPR, class Put>
__device__ __forceinline__ void jacobi_row(const double* log, int rounds, int R, int i, int lane, Put put) {
#pragma clang fp contract(off)
    const uint32_t m = jacobi_n2(R) - 1, np = jacobi_n2(R) / 2;
    const uint32_t k = lane & (LPR - 1), kc = k < np ? k : np - 1;
    double x = jacobi_top(k, 0, m) == i ? 1.0 : 0.0, y = jacobi_bottom(k, 0, m) == i ? 1.0 : 0.0;
    if (k >= np) x = y = 0.0;
    constexpr int AH = 8;  // tangents loaded ahead
    double g[AH];
    const double* src = log + kc;
#pragma unroll
    for (int u = 0; u < AH; u++) g[u] = src[(uint64_t)min(u, rounds - 1) * np];
    for (int r0 = 0; r0 < rounds; r0 += AH) {
        // off the chain of the rounds: a launch at R = 128 122 us, inside it 168
        double c[AH], s[AH];
#pragma unroll
        for (int u = 0; u < AH; u++) {
            jacobi_cs(g[u], c[u], s[u]);
            g[u] = src[(uint64_t)min(r0 + AH + u, rounds - 1) * np];
        }
#pragma unroll
        for (int u = 0; u < AH; u++) {
            if (r0 + u < rounds) {
                double xn = x, yn = y;
                if (s[u] != 0.0) {
                    xn = c[u] * x - s[u] * y;
                    yn = s[u] * x + c[u] * y;
                }
                if (np > 1) {
                    const double up = wave_from_next(xn), down = wave_from_prev(yn);
                    x = k == 0 ? xn : k + 1 == np ? yn : up;
                    y = k == 0 ? up : down;
                } else {
                    x = xn;
                    y = yn;
                }
            }
        }
    }
    if (k < np) {
        const int t = jacobi_top(k, 0, m), b = jacobi_bottom(k, 0, m);
        if (t < R) put(t, x);
        if (b < R) put(b, y);
    }
}

template <int BS>
__device__ __forceinline__ bool jacobi_large(double* A, double* V, int R, double* lam, double* Vout, JacobiShared& js,
                                             double* diag_tmp) {
#pragma clang fp contract(off)
    const int tid = threadIdx.x;
    const int LD = R + 1;  // odd leading dimension: rows start in different LDS banks
    const int n2 = R + (R & 1);
    const int npairs = n2 / 2;
    for (int e = tid; e < R * R; e += BS) V[(e / R) * LD + e % R] = (e / R == e % R) ? 1.0 : 0.0;
    __syncthreads();
    bool converged = false;
    for (int sweep = 0; sweep < kJacobiMaxSweeps; sweep++) {
        int any = 0;
        // circle-method positions of pair tid's elements, advanced by one (mod
        // n2 - 1) per round instead of recomputed by division
        int pa = tid - 1, pb = n2 - 2 - tid;
        for (int round = 0; round + 1 < n2; round++) {
            // rotations of this round, each computed once from the current A
            if (tid < npairs) {
                int p = tid == 0 ? 0 : 1 + pa, q = 1 + pb;  // tid < n2/2: q's position is never the fixed one
                if (p > q) {
                    const int t = p;
                    p = q;
                    q = t;
                }
                double c, s;
                const bool act = jacobi_rotation(A, LD, R, p, q, c, s);
                js.p[tid] = p;
                js.q[tid] = q;
                js.c[tid] = c;
                js.s[tid] = s;
                js.act[tid] = act;
                any |= act;
            }
            pa = pa + 1 == n2 - 1 ? 0 : pa + 1;
            pb = pb + 1 == n2 - 1 ? 0 : pb + 1;
            __syncthreads();
            // J^T A J in place: the 2x2 block where row pair k meets column
            // pair k2 belongs to one thread, which applies the row rotation
            // and then the column rotation (the operation order of applying
            // all row rotations, then all column rotations)
            for (int it = tid; it < npairs * npairs; it += BS) {
                const int k = it / npairs, k2 = it - (it / npairs) * npairs;
                const bool act1 = js.act[k], act2 = js.act[k2];
                if (!act1 && !act2) continue;
                const int p = js.p[k], q = js.q[k], p2 = js.p[k2], q2 = js.q[k2];
                const double c = js.c[k], s = js.s[k], c2 = js.c[k2], s2 = js.s[k2];
                // an index of value R (padding of an odd size) only occurs in
                // inactive pairs; its entries are treated as absent
                const bool qv = q < R, q2v = q2 < R;
                const double app2 = A[p * LD + p2];
                const double apq2 = q2v ? A[p * LD + q2] : 0.0;
                const double aqp2 = qv ? A[q * LD + p2] : 0.0;
                const double aqq2 = qv && q2v ? A[q * LD + q2] : 0.0;
                double rpp2 = app2, rpq2 = apq2, rqp2 = aqp2, rqq2 = aqq2;
                if (act1) {
                    rpp2 = c * app2 - s * aqp2;
                    rqp2 = s * app2 + c * aqp2;
                    rpq2 = c * apq2 - s * aqq2;
                    rqq2 = s * apq2 + c * aqq2;
                }
                double npp2 = rpp2, npq2 = rpq2, nqp2 = rqp2, nqq2 = rqq2;
                if (act2) {
                    npp2 = c2 * rpp2 - s2 * rpq2;
                    npq2 = s2 * rpp2 + c2 * rpq2;
                    nqp2 = c2 * rqp2 - s2 * rqq2;
                    nqq2 = s2 * rqp2 + c2 * rqq2;
                }
                A[p * LD + p2] = npp2;
                if (q2v) A[p * LD + q2] = npq2;
                if (qv) A[q * LD + p2] = nqp2;
                if (qv && q2v) A[q * LD + q2] = nqq2;
            }
            // V J, on the transposed store: entry (i, pair k2), i fastest
            for (int it = tid; it < R * npairs; it += BS) {
                const int k2 = it / R, i = it - (it / R) * R;
                if (!js.act[k2]) continue;
                const int p = js.p[k2], q = js.q[k2];
                const double c = js.c[k2], s = js.s[k2];
                const double vp = V[p * LD + i], vq = V[q * LD + i];
                V[p * LD + i] = c * vp - s * vq;
                V[q * LD + i] = s * vp + c * vq;
            }
            __syncthreads();
        }
        if (!__syncthreads_or(any)) {
            converged = true;
            break;
        }
        // converged when every pair meets the skip test: the next sweep would
        // rotate nothing, so stopping here gives the same result
        int open = 0;
        for (int w = tid; w < R * R; w += BS) {
            const int p = w / R, q = w - (w / R) * R;
            if (p < q) {
                const double apq = A[p * LD + q];
                const double thr = (2.220446049250313e-16 * 2.220446049250313e-16) * fabs(A[p * LD + p] * A[q * LD + q]);
                open |= !(apq * apq <= thr || apq == 0.0);
            }
        }
        if (!__syncthreads_or(open)) {
            converged = true;
            break;
        }
    }
    jacobi_sorted<BS>(A, LD, V, LD, R, lam, Vout, diag_tmp);
    if (!converged && tid == 0) atomicAdd(&g_jacobi_capped, 1u);
    __syncthreads();
    return converged;
}

// Storage of a block.  R <= kJacobiSmallR: both buffers of A, the second also
// the eigenvectors, and V, all in LDS.  Above: A in LDS, V ((R+1) R) and the
// eigenvectors (R^2) in the block's global scratch.
__host__ __device__ inline uint64_t jacobi_lds_doubles(uint64_t R) {
    if (R > (uint64_t)kJacobiSmallR) return (R + 1) * R;
    const uint64_t n2 = (uint64_t)jacobi_n2((int)R);
    return 2 * n2 * (n2 + 1) + R * (R + 1);
}

// Block size of the one-block Jacobi kernels.  Measured on computeM at R=32
// (N=3, I=2^23): 1024 threads 80 + 72 us, 256 threads 98 + 127 us -- the
// element-wise phases around the rotations (P_k, V, E, eigen tree) gain
// more from the extra waves than the barriers cost.
inline uint32_t jacobi_threads_for(uint64_t R) { (void)R; return 1024u; }

struct JacobiStore {
    double *A, *A1, *V, *vecs;
};

__device__ inline JacobiStore jacobi_store_small(double* smem, int R) {
    const int n2 = jacobi_n2(R), n = n2 * (n2 + 1);
    JacobiStore st;
    st.A = smem;
    st.A1 = st.vecs = smem + n;
    st.V = smem + 2 * n;
    return st;
}

__device__ inline JacobiStore jacobi_store(double* smem, double* work, int R) {
    if (R <= kJacobiSmallR) return jacobi_store_small(smem, R);
    JacobiStore st;
    st.A = st.A1 = smem;
    st.V = work;
    st.vecs = work + (R + 1) * R;
    return st;
}

// A (rows and columns [0, n), row length LD) from f(r, c), zero past R.
template <int BS, class F>
__device__ __forceinline__ void jacobi_fill(double* A, int R, int n, int LD, F f) {
    for (int e = threadIdx.x; e < n * n; e += BS) {
        const int r = e / n, c = e - (e / n) * n;
        A[r * LD + c] = r < R && c < R ? f(r, c) : 0.0;
    }
}
template <int BS, class F>
__device__ __forceinline__ void jacobi_fill(double* A, int R, F f) {
    jacobi_fill<BS>(A, R, R <= kJacobiSmallR ? jacobi_n2(R) : R, jacobi_ld(R), f);
}

// Eigendecomposition of st.A (jacobi_fill, then a barrier).
template <int BS>
__device__ __forceinline__ bool jacobi_block(const JacobiStore& st, int R, double* lam, JacobiShared& js,
                                             double* diag_tmp) {
    if (R <= kJacobiSmallR) return jacobi_small<BS>(st.A, st.A1, st.V, R, lam, st.vecs, js, diag_tmp);
    return jacobi_large<BS>(st.A, st.V, R, lam, st.vecs, js, diag_tmp);
}

}  // namespace ftl
