// hbem_solve.hip -- lu.solve / lu.adjoint().solve of randomized_svd::sv
// (randsvd.cpp:99-146) on thin right-hand sides (n x nc), batched over
// matrices, reading the factors of hbem_dense.hip in place.
#include <algorithm>

#include "hbem_complex.hpp"

namespace hbem {

// ---------------------------------------------------------------------------
// Thin triangular solves
// ---------------------------------------------------------------------------
// A = P^T L U with L (unit lower) and U in one column-major array LU.  All four
// substitutions read LU in place, always down its columns:
//   A x = b:    L y = P b forward, U x = y backward -- right-looking: once the
//               block's unknowns are known, columns of L (below) / U (above)
//               update the other rows;
//   A^H x = b:  U^H y = b forward, L^H z = y backward, x = P^T z -- left-
//               looking: (U^H y)_i = sum_j conj(U(j, i)) y_j runs down column
//               i of U above the diagonal (of L below it for L^H), so each
//               block first gathers its rows' sums from the finished unknowns.
//
// A pass goes block by block of 64 rows, and its length is the chain of the
// blocks: wavefront 0 solves block s while the other seven do what does not
// need it -- the coupling of block s - 1 and older to the rows beyond block s
// (right-looking) or to block s + 1 (left-looking) -- and load into registers what
// comes next, the coupling of blocks s and s + 1 and the diagonal block s + 1;
// after the barrier they apply block s's coupling to block s + 1 from those
// registers and lay the next diagonal block into LDS.  The right-hand sides stay
// in LDS.  With everything after a block's solve in sequence, a sweep's pass with
// q = 20 at order 602 (12 matrices) took 15.8 ms and a Newton pass at order 1000 (32
// matrices) 73.3 ms; with this form and panels of 512 rows from order 513 on (below)
// 12.0 and 62.6 ms.
//
// Panels (below) of 512 rows: one workgroup streams a triangle at 26 GB/s, the many of
// a coupling at 5 TB/s, but each panel costs two launches.  128 rows were 4% slower
// (12.5 and 64.9 ms), 256 rows faster for few matrices (11.7 ms) but slower for many (256
// of order 800, whose solves read the factors at 4 TB/s: 25.2 against 24.3 ms; the
// mixed sweep of order 4000 184 against 181 ms).
constexpr int kSolvePanel = 512;
constexpr int kSolveThreads = 512;
constexpr int kSolveWork = kSolveThreads / 64 - 1;   // wavefronts beside the block solve
constexpr int kTS = 65;   // padded row stride of the 64 x 64 LDS diagonal block

template <int NC>
struct SolveLds {
    cdbl tile[64 * kTS];      // the current diagonal block (see stage_column)
    cdbl dinv[64];            // its reciprocal pivots
    cdbl xb[2][64 * NC];      // solutions of the last two blocks, [row][right-hand side]
};

// The diagonal block [r0, r0 + bs)^2 of a pass is solved as a strictly lower one in
// LDS: tile(i, j), i > j, op(i, j) of the pass with rows and columns reversed for
// backward passes, zero elsewhere.  op(i, j) = LU(i, j), or conj(LU(j, i)) for adj.
// With a non-unit diagonal the block is (M D^-1) y = w, x = D^-1 y: the entries are
// scaled by the reciprocal pivots as they are staged, so that a step's dependence
// chain is one broadcast and one complex multiply-add.  Every complex product is
// explicit FMAs, so the bits do not depend on how the compiler contracts the code.
//
// A wavefront stages column q of LU (lane p: row p; v its entry, d LU(p, p)).
__device__ __forceinline__ void stage_column(cdbl v, cdbl d, int q, int bs, bool adj, bool lower, cdbl* tile, cdbl* dinv) {
    const int p = threadIdx.x & 63;
    const bool unit = lower != adj;           // L forward, L^H backward
    const int i = adj ? q : p, j = adj ? p : q;
    const bool in = p < bs && q < bs && (lower ? i > j : i < j);
    if (adj) v = cconj(v);
    if (!unit) {
        if (adj) d = cconj(d);
        else d = bcast_lane(d, q);            // column q's pivot
        const cdbl r = crecip(d);
        v = cmulx(v, r);
        if (p == q && q < bs) dinv[lower ? q : bs - 1 - q] = r;
    }
    const int ti = lower ? i : bs - 1 - i, tj = lower ? j : bs - 1 - j;
    const bool rev = !lower && (i >= bs || j >= bs);   // outside the block: zero at its own place
    tile[(rev ? i : ti) * kTS + (rev ? j : tj)] = in ? v : mk(0, 0);
}

// Element at byte offset 16 or 8 (c n + i) of a column block, c < 64: a uniform base and
// a 32-bit offset, one register an address where 64-bit ones spilled.
template <class F>
__device__ __forceinline__ F at(const F* block, int i, int c, int n) {
    return *reinterpret_cast<const F*>(reinterpret_cast<const char*>(block) + (unsigned)(sizeof(F) * ((unsigned)c * (unsigned)n + (unsigned)i)));
}

template <int J>
__device__ __forceinline__ double row_bcast(double x) {
    const unsigned long long b = __double_as_longlong(x);
    const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x150 + J, 0xf, 0xf, true);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x150 + J, 0xf, 0xf, true);
    return __longlong_as_double(((unsigned long long)hi << 32) | lo);
}

// Wavefront 0: solves the staged block for the rows r0 .. r0 + bs - 1 of w
// ([row][NC]) in place and leaves the solution in xb (zero beyond bs).  Lane l
// holds rows 16 s + l % 16, s < 4, of right-hand sides l / 16 (+ 4): step j
// broadcasts its unknown within each row of sixteen lanes by DPP (row_newbcast) and
// updates the sub-blocks of sixteen rows from its own on, the tile entries two steps
// ahead: 14 instructions a step with two right-hand sides, where a lane per row and
// readlane broadcasts took 45.
template <int NC>
__device__ __forceinline__ void diag_solve(int r0, int bs, bool lower, bool unit, cdbl* w, const cdbl* tile,
                                           const cdbl* dinv, cdbl* xb) {
    constexpr int G = (NC + 3) / 4;
    const int lane = threadIdx.x & 63, l16 = lane & 15, rh = lane >> 4;
    cdbl x[4][G];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int i = 16 * s + l16, c = rh + 4 * g;
            x[s][g] = i < bs && c < NC ? w[(r0 + (lower ? i : bs - 1 - i)) * NC + c] : mk(0, 0);
        }
    const cdbl* t0 = tile + l16 * kTS;
    cdbl lv[2][2][4];                         // [buffer][step][sub-block]
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int s = 0; s < 4; ++s) lv[0][u][s] = t0[16 * s * kTS + u];
    static_for<32>([&](auto pair) {
        constexpr int k = decltype(pair)::value, cur = k & 1, j0 = 2 * k, jn = j0 + 2;
        if constexpr (k + 1 < 32) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int s = jn / 16; s < 4; ++s) lv[cur ^ 1][u][s] = t0[16 * s * kTS + jn + u];
        }
        static_for<2>([&](auto step) {
            constexpr int u = decltype(step)::value, j = j0 + u, sb = j / 16;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const cdbl xj = mk(row_bcast<j % 16>(x[sb][g].x), row_bcast<j % 16>(x[sb][g].y));
#pragma unroll
                for (int s = sb; s < 4; ++s) cfms(x[s][g], lv[cur][u][s], xj);
            }
        });
        __builtin_amdgcn_sched_barrier(0);    // no further ahead: the registers
    });
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const int i = 16 * s + l16, o = lower ? i : bs - 1 - i;
        const bool in = i < bs;
        cdbl d = mk(1, 0);
        if (!unit) d = dinv[in ? i : 0];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int c = rh + 4 * g;
            cdbl v = x[s][g];
            if (!unit) v = cmulx(v, d);
            if (c < NC) {
                if (in) w[(r0 + o) * NC + c] = v;
                xb[(in ? o : i) * NC + c] = in ? v : mk(0, 0);
            }
        }
    }
}

// Sums of the N doubles v over a wavefront: value k is left in the lanes l with l / (64
// / N) = k.  Pairs of values are exchanged and added half by half (v_permlane32_swap,
// v_permlane16_swap), the rest by DPP and shuffles.
__device__ __forceinline__ void swap_add(double& a, double b, bool half) {
    const unsigned long long x = __double_as_longlong(a), y = __double_as_longlong(b);
    unsigned long long p, q;
    if (half) {
        const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
        p = ((unsigned long long)hi[0] << 32) | lo[0];
        q = ((unsigned long long)hi[1] << 32) | lo[1];
    } else {
        const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
        p = ((unsigned long long)hi[0] << 32) | lo[0];
        q = ((unsigned long long)hi[1] << 32) | lo[1];
    }
    a = __longlong_as_double(p) + __longlong_as_double(q);
}
template <int M, int O, int N>
__device__ __forceinline__ void sum_step(double (&v)[N]) {
    if constexpr (M >= 1) {
        const bool up = threadIdx.x & O;
#pragma unroll
        for (int i = 0; i < M; ++i) {
            const double keep = up ? v[i + M] : v[i], give = up ? v[i] : v[i + M];
            v[i] = keep + __shfl_xor(give, O, 64);
        }
    } else {
        v[0] += __shfl_xor(v[0], O, 64);
    }
    if constexpr (O > 1) sum_step<M / 2, O / 2>(v);
}
template <int N>
__device__ __forceinline__ double wave_sums(double (&v)[N]) {
    static_assert(N == 8 || N == 16 || N == 32, "");
#pragma unroll
    for (int i = 0; i < N / 2; ++i) swap_add(v[i], v[i + N / 2], true);
#pragma unroll
    for (int i = 0; i < N / 4; ++i) swap_add(v[i], v[i + N / 4], false);
    sum_step<N / 8, 8>(v);
    return v[0];
}

// Columns and right-hand sides whose lane sums fit 32 values at a time.
template <int NC>
constexpr int kSumCols = NC <= 2 ? 8 : (NC <= 4 ? 4 : 2);
template <int V>
constexpr int kPow2 = V <= 8 ? 8 : (V <= 16 ? 16 : 32);

// w rows i0 .. i0 + cols - 1 minus the sums over the wavefront of acc
template <int NC, int CP>
__device__ __forceinline__ void subtract_sums(cdbl (&acc)[CP][NC], int i0, int cols, cdbl* w) {
    constexpr int V = kPow2<CP * NC * 2>, L = 64 / V;
    const int lane = threadIdx.x & 63;
    double v[V];
#pragma unroll
    for (int k = 0; k < V; ++k) v[k] = 0.0;
#pragma unroll
    for (int q = 0; q < CP; ++q)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            v[(q * NC + c) * 2] = acc[q][c].x;
            v[(q * NC + c) * 2 + 1] = acc[q][c].y;
        }
    const double t = wave_sums<V>(v);
    const int k = lane / L;
    if (lane % L == 0 && k < cols * NC * 2) reinterpret_cast<double*>(w)[(size_t)i0 * NC * 2 + k] -= t;
}

// Right-looking pass with the column-major factor: L (lower, unit) forward or U
// backward, over the rows [pb, pe) (the whole matrix, or one panel of the panelled
// form); w: row pb's right-hand sides.  A wavefront covers 16 rows x 4 groups of 16
// columns of a block's coupling (lane = row + 16 group), the groups' sums added by
// shuffles.
template <int NC, class F>
__device__ __forceinline__ void subst_right(const F* M, int n, bool lower, cdbl* w, SolveLds<NC>& S, int pb, int pe) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int l16 = lane & 15, grp = lane >> 4;
    const int nblk = (pe - pb + 63) / 64;
    auto rb = [&](int s) { return pb + 64 * (lower ? s : nblk - 1 - s); };   // first row of the s-th block solved
    auto bsz = [&](int s) { return min(64, pe - rb(s)); };
    // sixteen columns of the block [r0, r0 + bs) at row i (clamped addresses)
    auto load16 = [&](auto& t, int i, int r0, int bs) {
        const F* B = M + (size_t)r0 * n;
#pragma unroll
        for (int u = 0; u < 16; ++u) t[u] = at(B, i, min(16 * grp + u, bs - 1), n);
    };
    // rows i of a wavefront minus the block's columns times its unknowns
    auto apply16 = [&](const auto& t, int i, bool live, int bs, const cdbl* xb) {
        cdbl acc[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] = mk(0, 0);
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int j = 16 * grp + u;
            const cdbl tv = j < bs ? to_cdbl(t[u]) : mk(0, 0);
#pragma unroll
            for (int c = 0; c < NC; ++c) cfma(acc[c], tv, xb[j * NC + c]);
            if (u % 2 == 1) __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int o = 16; o < 64; o <<= 1) {
                acc[c].x += __shfl_xor(acc[c].x, o, 64);
                acc[c].y += __shfl_xor(acc[c].y, o, 64);
            }
        if (grp == 0 && live) {
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                cdbl& y = w[(i - pb) * NC + c];
                y = y - acc[c];
            }
        }
    };
    // the first diagonal block, by all wavefronts
    for (int q = wv; q < 64; q += kSolveWork + 1) {
        const int r0 = rb(0), bs = bsz(0), p = min(lane, bs - 1), qc = min(q, bs - 1);
        stage_column(to_cdbl(M[(r0 + p) + (size_t)(r0 + qc) * n]), to_cdbl(M[(r0 + p) + (size_t)(r0 + p) * n]), q, bs, false,
                     lower, S.tile, S.dinv);
    }
    __syncthreads();
    for (int s = 0; s < nblk; ++s) {
        const int r0 = rb(s), bs = bsz(s);
        const bool next = s + 1 < nblk;
        const int rn = next ? rb(s + 1) : r0, bn = next ? bsz(s + 1) : bs;
        F pre[22];                               // wavefronts 1-4: the coupling of s + 1 and s; 5-7: columns of block s + 1
        F dg{};
        if (wv == 0) {
            diag_solve<NC>(r0 - pb, bs, lower, lower, w, S.tile, S.dinv, S.xb[s & 1]);
        } else {
            // the coupling of block s - 1 to the rows beyond block s
            if (s > 0) {
                const int rp = rb(s - 1), bp = bsz(s - 1);
                const int ia = lower ? r0 + bs : pb, ib = lower ? pe : r0;
                for (int i0 = ia + 16 * (wv - 1); i0 < ib; i0 += 16 * kSolveWork) {
                    F t[16];
                    load16(t, min(i0 + l16, ib - 1), rp, bp);
                    apply16(t, i0 + l16, i0 + l16 < ib, bp, S.xb[(s - 1) & 1]);
                }
            }
            if (next) {
                if (wv <= 4) {
                    load16(pre, rn + min(16 * (wv - 1) + l16, bn - 1), r0, bs);
                } else {
                    const int p = min(lane, bn - 1);
                    const F* B = M + (size_t)rn * n;
                    if (!lower) dg = at(B, rn + p, p, n);
#pragma unroll
                    for (int u = 0; u < 22; ++u) pre[u] = at(B, rn + p, min(wv - 5 + 3 * u, bn - 1), n);
                }
            }
        }
        __syncthreads();                          // block s solved, the older couplings in
        if (next && wv > 0) {
            if (wv <= 4) {
                const int i = 16 * (wv - 1) + l16;
                apply16(pre, rn + i, i < bn, bs, S.xb[s & 1]);
            } else {
#pragma unroll
                for (int u = 0; u < 22; ++u) {
                    if (wv - 5 + 3 * u < 64)
                        stage_column(to_cdbl(pre[u]), to_cdbl(dg), wv - 5 + 3 * u, bn, false, lower, S.tile, S.dinv);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        __syncthreads();
    }
}

// Left-looking pass with the conjugate transpose of the factor: U^H (lower) forward
// or L^H (unit) backward, over the rows [pb, pe).  A wavefront sums columns of the
// factor over finished unknowns, its lanes down the columns: block s + 1's sums over
// the blocks before s beside block s's solve, those over block s after it.  (The
// unknowns outside [pb, pe) are gathered beforehand.)
template <int NC, class F>
__device__ __forceinline__ void subst_left(const F* M, int n, bool lower, cdbl* w, SolveLds<NC>& S, int pb, int pe) {
    constexpr int CB = NC <= 3 ? 5 : (NC == 4 ? 4 : (NC == 5 ? 3 : 2));   // columns at a time beside the solve: two rounds
    constexpr int CU = kSumCols<NC>;                                      // ... and after it
    constexpr int TW = NC <= 2 ? 2 : 1;                                   // 64-row sweeps' loads in flight
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int nblk = (pe - pb + 63) / 64;
    auto rb = [&](int s) { return pb + 64 * (lower ? s : nblk - 1 - s); };
    auto bsz = [&](int s) { return min(64, pe - rb(s)); };
    for (int q = wv; q < 64; q += kSolveWork + 1) {
        const int r0 = rb(0), bs = bsz(0), p = min(lane, bs - 1), qc = min(q, bs - 1);
        stage_column(to_cdbl(M[(r0 + p) + (size_t)(r0 + qc) * n]), to_cdbl(M[(r0 + p) + (size_t)(r0 + p) * n]), q, bs, true,
                     lower, S.tile, S.dinv);
    }
    __syncthreads();
    for (int s = 0; s < nblk; ++s) {
        const int r0 = rb(s), bs = bsz(s);
        const bool next = s + 1 < nblk;
        const int rn = next ? rb(s + 1) : r0, bn = next ? bsz(s + 1) : bs;
        F pre[22];                               // wavefronts 1-4: columns of the coupling; 5-7: of block s + 1
        F dg{};
        if (wv == 0) {
            diag_solve<NC>(r0 - pb, bs, lower, !lower, w, S.tile, S.dinv, S.xb[s & 1]);
        } else if (next) {
            const F* B = M + (size_t)rn * n;
            if (s > 0) {
                const int ja = lower ? pb : r0 + bs, jb = lower ? r0 : pe;   // finished before block s
                const int T = (jb - ja + 63) >> 6;
                for (int q0 = CB * (wv - 1); q0 < bn; q0 += CB * kSolveWork) {
                    cdbl acc[CB][NC];
#pragma unroll
                    for (int q = 0; q < CB; ++q)
#pragma unroll
                        for (int c = 0; c < NC; ++c) acc[q][c] = mk(0, 0);
                    for (int tt = 0; tt < T; tt += TW) {
                        F mv[TW][CB];
#pragma unroll
                        for (int h = 0; h < TW; ++h) {
                            const int jc = min(ja + lane + 64 * (tt + h), jb - 1);
#pragma unroll
                            for (int q = 0; q < CB; ++q) mv[h][q] = at(B, jc, min(q0 + q, bn - 1), n);
                        }
#pragma unroll
                        for (int h = 0; h < TW; ++h) {
                            const int j = ja + lane + 64 * (tt + h);
                            cdbl xj[NC];
#pragma unroll
                            for (int c = 0; c < NC; ++c) xj[c] = j < jb ? w[(min(j, jb - 1) - pb) * NC + c] : mk(0, 0);
#pragma unroll
                            for (int q = 0; q < CB; ++q) {
                                const cdbl t = cconj(to_cdbl(mv[h][q]));
#pragma unroll
                                for (int c = 0; c < NC; ++c) cfma(acc[q][c], t, xj[c]);
                            }
                        }
                    }
                    subtract_sums<NC, CB>(acc, rn - pb + q0, min(CB, bn - q0), w);
                }
            }
            if (wv <= 4) {
#pragma unroll
                for (int u = 0; u < 16; ++u) pre[u] = at(B, r0 + min(lane, bs - 1), min(16 * (wv - 1) + u, bn - 1), n);
            } else {
                const int p = min(lane, bn - 1);
                if (lower) dg = at(B, rn + p, p, n);
#pragma unroll
                for (int u = 0; u < 22; ++u) pre[u] = at(B, rn + p, min(wv - 5 + 3 * u, bn - 1), n);
            }
        }
        __syncthreads();                          // block s solved, the older sums in
        if (next && wv > 0) {
            if (wv <= 4) {
                cdbl xj[NC];
#pragma unroll
                for (int c = 0; c < NC; ++c) xj[c] = S.xb[s & 1][lane * NC + c];   // zero beyond the block
#pragma unroll
                for (int u0 = 0; u0 < 16; u0 += CU) {
                    cdbl acc[CU][NC];
#pragma unroll
                    for (int q = 0; q < CU; ++q) {
                        const cdbl t = cconj(to_cdbl(pre[u0 + q]));
#pragma unroll
                        for (int c = 0; c < NC; ++c) {
                            acc[q][c] = mk(0, 0);
                            cfma(acc[q][c], t, xj[c]);
                        }
                    }
                    const int q0 = 16 * (wv - 1) + u0;
                    subtract_sums<NC, CU>(acc, rn - pb + q0, min(CU, bn - q0), w);
                }
            } else {
#pragma unroll
                for (int u = 0; u < 22; ++u) {
                    if (wv - 5 + 3 * u < 64)
                        stage_column(to_cdbl(pre[u]), to_cdbl(dg), wv - 5 + 3 * u, bn, true, lower, S.tile, S.dinv);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        __syncthreads();
    }
}

// one workgroup of kSolveThreads threads per matrix
template <class F, int NC>
__global__ __launch_bounds__(kSolveThreads) void k_solve_thin(const F* __restrict__ LU, long long ms,
                                                              const int* __restrict__ perm, int n,
                                                              cdbl* __restrict__ X, int adj) {
    __shared__ SolveLds<NC> S;
    __shared__ cdbl w[kSolvePanel * NC];
    const int b = blockIdx.x;
    const int* p = perm + (size_t)b * n;
    cdbl* x = X + (size_t)b * n * NC;
    const F* lu = LU + (size_t)b * ms;
    const int tid = threadIdx.x;
    // A = P^T L U:  w = P x, L y = w, U z = y;  A^H = U^H L^H P:  U^H y = x, L^H z = y, x = P^T z
    for (int e = tid; e < n * NC; e += blockDim.x) {
        const int i = e % n, c = e / n;
        w[i * NC + c] = x[(adj ? i : p[i]) + (size_t)c * n];
    }
    __syncthreads();
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
        if (!adj) subst_right<NC>(lu, n, pass == 0, w, S, 0, n);
        else subst_left<NC>(lu, n, pass == 0, w, S, 0, n);
    }
    for (int e = tid; e < n * NC; e += blockDim.x) {
        const int i = e % n, c = e / n;
        x[(adj ? p[i] : i) + (size_t)c * n] = w[i * NC + c];
    }
}

// Panelled form of the thin solves for orders above kSolvePanel: the
// passes run panel by panel of kSolvePanel rows.  A panel's triangle is solved
// by one workgroup per matrix (k_solve_panel: the blocked substitution above,
// restricted to the panel); the panel's coupling to the other rows runs on
// many workgroups per matrix: a right-looking pass then updates every row
// after the panel with the panel's columns (k_panel_update), a left-looking
// pass first gathers into the panel's rows the sums over the unknowns finished
// before it (k_panel_gather).  Each entry of the factors is still read once,
// but the bulk of the reads no longer waits on one workgroup per matrix.

// w = P x (A x = b) or w = x (A^H x = b)
static __global__ void k_thin_in(const int* __restrict__ perm, int n, int nc, const cdbl* __restrict__ X, int adj,
                          cdbl* __restrict__ work) {
    const int b = blockIdx.y;
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (long long)n * nc) return;
    const int i = (int)(e % n), c = (int)(e / n);
    const cdbl* x = X + (size_t)b * n * nc;
    work[(size_t)b * n * nc + e] = adj ? x[e] : x[perm[(size_t)b * n + i] + (size_t)c * n];
}

// x = w (A x = b) or x = P^T w (A^H x = b)
static __global__ void k_thin_out(const int* __restrict__ perm, int n, int nc, cdbl* __restrict__ X, int adj,
                           const cdbl* __restrict__ work) {
    const int b = blockIdx.y;
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (long long)n * nc) return;
    const int i = (int)(e % n), c = (int)(e / n);
    cdbl* x = X + (size_t)b * n * nc;
    const cdbl v = work[(size_t)b * n * nc + e];
    if (adj) x[perm[(size_t)b * n + i] + (size_t)c * n] = v;
    else x[e] = v;
}

// Right-looking coupling of the unknowns [cb, ce) (one panel, staged in xs)
// onto row i: w_i -= sum_j M(i, j) w_j, the sum in column order.  A thread per
// row (consecutive rows: the loads run down the columns), LR column loads in
// flight.
template <int NC>
__device__ __forceinline__ void stage_unknowns(const cdbl* w, int n, int cb, int ce, cdbl* xs) {
    const int pw = ce - cb;
    for (int e = threadIdx.x; e < pw * NC; e += blockDim.x) {
        const int j = e % pw, c = e / pw;
        xs[j * NC + c] = w[cb + j + (size_t)c * n];
    }
}
template <class F, int NC>
__device__ __forceinline__ void couple_right_row(const F* M, int n, cdbl* w, int cb, int ce, int i, const cdbl* xs) {
    constexpr int LR = sizeof(F) == sizeof(cflt) ? 16 : 8;
    const int pw = ce - cb;
    cdbl acc[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = mk(0, 0);
    const F* mr = M + i + (size_t)cb * n;
    for (int j0 = 0; j0 < pw; j0 += LR) {
        F t[LR];
#pragma unroll
        for (int u = 0; u < LR; ++u) t[u] = mr[(size_t)min(j0 + u, pw - 1) * n];
#pragma unroll
        for (int u = 0; u < LR; ++u) {
            if (j0 + u < pw) {
                const cdbl tv = to_cdbl(t[u]);
#pragma unroll
                for (int c = 0; c < NC; ++c) cfma(acc[c], tv, xs[(j0 + u) * NC + c]);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        cdbl& y = w[i + (size_t)c * n];
        y = y - acc[c];
    }
}

// Left-looking coupling of the unknowns [ja, jb) onto rows i0 .. i0 + 3 (those
// below re): w_i -= sum_j conj(M(j, i)) w_j.  One wavefront, lanes down the
// columns (lane j mod 64: ja is a multiple of 64), two sweeps' loads in
// flight; the lane sums are reduced by shuffles in a fixed order.
template <class F, int NC>
__device__ __forceinline__ void couple_left_quad(const F* M, int n, cdbl* w, int ja, int jb, int i0, int re) {
    const int lane = threadIdx.x & 63;
    const int qmax = min(4, re - i0) - 1;
    cdbl acc[4][NC];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[q][c] = mk(0, 0);
    const int T = (jb - ja + 63) >> 6;
    for (int tt = 0; tt < T; tt += 2) {
        cdbl xj[2][NC];
        F mv[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int jc = min(ja + lane + 64 * (tt + h), jb - 1);
#pragma unroll
            for (int c = 0; c < NC; ++c) xj[h][c] = w[jc + (size_t)c * n];
#pragma unroll
            for (int q = 0; q < 4; ++q) mv[h][q] = M[jc + (size_t)(i0 + min(q, qmax)) * n];
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool in = ja + lane + 64 * (tt + h) < jb;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const cdbl t = (in && q <= qmax) ? cconj(to_cdbl(mv[h][q])) : mk(0, 0);
#pragma unroll
                for (int c = 0; c < NC; ++c) cfma(acc[q][c], t, xj[h][c]);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                acc[q][c].x += __shfl_xor(acc[q][c].x, o, 64);
                acc[q][c].y += __shfl_xor(acc[q][c].y, o, 64);
            }
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (lane == q && q <= qmax) {
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                cdbl& y = w[i0 + q + (size_t)c * n];
                y = y - acc[q][c];
            }
        }
}

// One panel [pb, pe) of a pass (0: L, or U^H; 1: U, or L^H), blocks 0 .. batch - 1
// (one of kSolveThreads threads per matrix), and beside it, in blocks batch + cwg b + k, a coupling that does not touch the
// panel: the unknowns [cb, ce) onto the rows [rb, re) of matrix b,
// right-looking (a thread per row, 512 rows a block) or, for adj, left-looking
// (a wavefront per four rows, 32 rows a block).  The coupling blocks take the
// CUs the batch's panel solves leave idle.  Up to kFuseNc right-hand sides:
// with more, the left-looking sums do not fit beside the panel solve's registers,
// and the couplings run as launches of their own.
constexpr int kFuseNc = 3;
template <class F, int NC>
__global__ __launch_bounds__(kSolveThreads) void k_solve_panel(const F* __restrict__ LU, long long ms, int n, int pass,
                                                               int adj, cdbl* __restrict__ work, int pb, int pe,
                                                               int batch, int cwg, int cb, int ce, int rb, int re) {
    __shared__ SolveLds<NC> S;
    __shared__ cdbl wl[kSolvePanel * NC];
    if ((int)blockIdx.x < batch) {
        const int b = blockIdx.x, pw = pe - pb;
        cdbl* w = work + (size_t)b * n * NC;
        const F* lu = LU + (size_t)b * ms;
        for (int e = threadIdx.x; e < pw * NC; e += blockDim.x) wl[(e % pw) * NC + e / pw] = w[pb + e % pw + (size_t)(e / pw) * n];
        __syncthreads();
        if (!adj) subst_right<NC>(lu, n, pass == 0, wl, S, pb, pe);
        else subst_left<NC>(lu, n, pass == 0, wl, S, pb, pe);
        for (int e = threadIdx.x; e < pw * NC; e += blockDim.x) w[pb + e % pw + (size_t)(e / pw) * n] = wl[(e % pw) * NC + e / pw];
        return;
    }
    if constexpr (NC <= kFuseNc) {
        const int q = blockIdx.x - batch, b = q / cwg, k = q - b * cwg;
        cdbl* w = work + (size_t)b * n * NC;
        const F* M = LU + (size_t)b * ms;
        if (!adj) {
            cdbl* xs = wl;                            // the panel solve's LDS is not used by this block
            stage_unknowns<NC>(w, n, cb, ce, xs);
            __syncthreads();
            const int i = rb + k * blockDim.x + threadIdx.x;
            if (i < re) couple_right_row<F, NC>(M, n, w, cb, ce, i, xs);
        } else {
            const int i0 = rb + (k * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 4;
            if (i0 < re) couple_left_quad<F, NC>(M, n, w, cb, ce, i0, re);
        }
    }
}

// The same couplings on their own.  Right-looking, 64 rows a block: wavefront
// v sums the unknowns cb + 128 v .. + 127 for the block's rows (lane = row,
// so the loads still run down the columns in 64-row segments), and the four
// partial sums are added in a fixed order, ((0 + 1) + (2 + 3)), by wavefront 0:
// each thread's chain of dependent load rounds is a quarter as long as with
// one thread per row over the whole panel.  The quarters are fixed column
// ranges from the panel's start, so a panel padded with zero columns gives the
// same sums.
template <class F, int NC>
__global__ __launch_bounds__(256) void k_panel_update(const F* __restrict__ LU, long long ms, int n,
                                                      cdbl* __restrict__ work, int cb, int ce, int rb, int re) {
    constexpr int LR = sizeof(F) == sizeof(cflt) ? 16 : 8;
    constexpr int QW = kSolvePanel / 4;
    __shared__ cdbl xs[kSolvePanel * NC];
    __shared__ cdbl part[4][64][NC];
    const int b = blockIdx.y, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    cdbl* w = work + (size_t)b * n * NC;
    stage_unknowns<NC>(w, n, cb, ce, xs);
    __syncthreads();
    const int i = rb + blockIdx.x * 64 + lane;
    const int q0 = wv * QW, q1 = min(ce - cb, q0 + QW);
    cdbl acc[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = mk(0, 0);
    if (i < re) {
        const F* mr = LU + (size_t)b * ms + i + (size_t)cb * n;
        for (int j0 = q0; j0 < q1; j0 += LR) {
            F t[LR];
#pragma unroll
            for (int u = 0; u < LR; ++u) t[u] = mr[(size_t)min(j0 + u, q1 - 1) * n];
#pragma unroll
            for (int u = 0; u < LR; ++u) {
                if (j0 + u < q1) {
                    const cdbl tv = to_cdbl(t[u]);
#pragma unroll
                    for (int c = 0; c < NC; ++c) cfma(acc[c], tv, xs[(j0 + u) * NC + c]);
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) part[wv][lane][c] = acc[c];
    __syncthreads();
    if (wv == 0 && i < re) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            cdbl& y = w[i + (size_t)c * n];
            y = y - ((part[0][lane][c] + part[1][lane][c]) + (part[2][lane][c] + part[3][lane][c]));
        }
    }
}

// Left-looking, 16 rows a block.
template <class F, int NC>
__global__ __launch_bounds__(256) void k_panel_gather(const F* __restrict__ LU, long long ms, int n,
                                                      cdbl* __restrict__ work, int ja, int jb, int rb, int re) {
    const int b = blockIdx.y;
    const int i0 = rb + (blockIdx.x * 4 + (threadIdx.x >> 6)) * 4;
    if (i0 >= re) return;                     // whole wavefront; no barrier in this kernel
    couple_left_quad<F, NC>(LU + (size_t)b * ms, n, work + (size_t)b * n * NC, ja, jb, i0, re);
}

// Panelled substitution (n > kSolvePanel).  A pass solves its panels in
// order; every row must have taken the couplings of all panels solved before
// its own, in that order.  After panel p's solve, the next panel's rows take
// p's coupling (a small launch); the rows beyond the next panel take it in
// the launch that solves the next panel, beside that solve.  Left-looking
// passes (adj) gather instead: the next panel's rows take the unknowns solved
// before p beside p's solve, then p's own unknowns.  A row's sums are split
// only at panel boundaries and at fixed offsets inside a panel, and which
// launch serves a row depends only on its panel, so a matrix padded at the
// end gives the same bits (a panel of zeros and the identity adds zeros to the others,
// so the one-kernel form of an order below kSolvePanel gives them too).  Above
// kFuseNc right-hand sides: each panel's coupling as a launch of its own,
// all rows at once, after its solve (right-looking) or before it (left).
template <class F, int NC>
static void solve_thin_nc(const F* LU, long long ms, const int* perm, int n, int batch, cdbl* X, bool adj, cdbl* work,
                          hipStream_t st) {
    const int a = adj ? 1 : 0;
    if (n <= kSolvePanel) {
        hipLaunchKernelGGL((k_solve_thin<F, NC>), dim3(batch), dim3(kSolveThreads), 0, st, LU, ms, perm, n, X, a);
        return;
    }
    const dim3 gio((unsigned)(((long long)n * NC + 255) / 256), (unsigned)batch);
    hipLaunchKernelGGL(k_thin_in, gio, dim3(256), 0, st, perm, n, NC, X, a, work);
    const int np = (n + kSolvePanel - 1) / kSolvePanel;
    auto first = [&](int p) { return p * kSolvePanel; };
    auto last = [&](int p) { return min(n, (p + 1) * kSolvePanel); };
    if constexpr (NC > kFuseNc) {
        for (int pass = 0; pass < 2; ++pass) {
            const bool lower = pass == 0;
            for (int t = 0; t < np; ++t) {
                const int p = lower ? t : np - 1 - t;
                const int pb = first(p), pe = last(p);
                if (adj && (lower ? pb > 0 : pe < n))
                    hipLaunchKernelGGL((k_panel_gather<F, NC>), dim3((unsigned)((pe - pb + 15) / 16), (unsigned)batch),
                                       dim3(256), 0, st, LU, ms, n, work, lower ? 0 : pe, lower ? pb : n, pb, pe);
                hipLaunchKernelGGL((k_solve_panel<F, NC>), dim3((unsigned)batch), dim3(kSolveThreads), 0, st, LU, ms, n,
                                   pass, a, work, pb, pe, batch, 1, 0, 0, 0, 0);
                const int rb = lower ? pe : 0, re = lower ? n : pb;
                if (!adj && re > rb)
                    hipLaunchKernelGGL((k_panel_update<F, NC>), dim3((unsigned)((re - rb + 63) / 64), (unsigned)batch),
                                       dim3(256), 0, st, LU, ms, n, work, pb, pe, rb, re);
            }
        }
        hipLaunchKernelGGL(k_thin_out, gio, dim3(256), 0, st, perm, n, NC, X, a, work);
        return;
    }
    for (int pass = 0; pass < 2; ++pass) {
        const bool lower = pass == 0;
        for (int t = 0; t < np; ++t) {
            const int p = lower ? t : np - 1 - t;
            const int pb = first(p), pe = last(p);
            const bool next = t + 1 < np;
            const int np_ = lower ? p + 1 : p - 1;             // the next panel of the pass
            const int nb = next ? first(np_) : 0, ne = next ? last(np_) : 0;
            int cb = 0, ce = 0, rb = 0, re = 0;                 // the coupling beside this solve
            if (!adj && t > 0) {
                const int pp = lower ? p - 1 : p + 1;          // the panel solved before
                cb = first(pp);
                ce = last(pp);
                rb = lower ? pe : 0;                           // the rows beyond this panel
                re = lower ? n : pb;
            } else if (adj && next) {
                cb = lower ? 0 : pe;
                ce = lower ? pb : n;
                rb = nb;
                re = ne;
            }
            const bool cpl = ce > cb && re > rb;
            const int cwg = !cpl ? 0 : (adj ? (re - rb + kSolveThreads / 16 - 1) / (kSolveThreads / 16) : (re - rb + kSolveThreads - 1) / kSolveThreads);
            hipLaunchKernelGGL((k_solve_panel<F, NC>), dim3((unsigned)(batch + batch * cwg)), dim3(kSolveThreads), 0, st,
                               LU, ms, n, pass, a, work, pb, pe, batch, cwg > 0 ? cwg : 1, cb, ce, rb, re);
            if (!next) continue;
            if (!adj)
                hipLaunchKernelGGL((k_panel_update<F, NC>), dim3((unsigned)((ne - nb + 63) / 64), (unsigned)batch),
                                   dim3(256), 0, st, LU, ms, n, work, pb, pe, nb, ne);
            else
                hipLaunchKernelGGL((k_panel_gather<F, NC>), dim3((unsigned)((ne - nb + 15) / 16), (unsigned)batch),
                                   dim3(256), 0, st, LU, ms, n, work, pb, pe, nb, ne);
        }
    }
    hipLaunchKernelGGL(k_thin_out, gio, dim3(256), 0, st, perm, n, NC, X, a, work);
}

template <class F>
static void solve_thin_impl(const F* LU, long long ms, const int* perm, int n, int batch, cdbl* X, int nc, bool adj,
                            cdbl* work, hipStream_t st) {
    switch (nc) {
    case 1: solve_thin_nc<F, 1>(LU, ms, perm, n, batch, X, adj, work, st); break;
    case 2: solve_thin_nc<F, 2>(LU, ms, perm, n, batch, X, adj, work, st); break;
    case 3: solve_thin_nc<F, 3>(LU, ms, perm, n, batch, X, adj, work, st); break;
    case 4: solve_thin_nc<F, 4>(LU, ms, perm, n, batch, X, adj, work, st); break;
    case 5: solve_thin_nc<F, 5>(LU, ms, perm, n, batch, X, adj, work, st); break;
    case 6: solve_thin_nc<F, 6>(LU, ms, perm, n, batch, X, adj, work, st); break;
    case 7: solve_thin_nc<F, 7>(LU, ms, perm, n, batch, X, adj, work, st); break;
    default: solve_thin_nc<F, 8>(LU, ms, perm, n, batch, X, adj, work, st); break;
    }
}

// (the instances for FP32 factors are compiled by hbem_solve_f32.hip)
#ifndef HBEM_SOLVE_F32
void lu_solve_thin_batched(const cdbl* LU, long long ms, const int* perm, int n, int batch, cdbl* X, int nc, bool adj,
                           cdbl* work, hipStream_t st) {
    solve_thin_impl(LU, ms, perm, n, batch, X, nc, adj, work, st);
}
#else
void lu_solve_thin_batched_f32(const cflt* LU, long long ms, const int* perm, int n, int batch, cdbl* X, int nc,
                               bool adj, cdbl* work, hipStream_t st) {
    solve_thin_impl(LU, ms, perm, n, batch, X, nc, adj, work, st);
}
#endif

}  // namespace hbem
