// hbem_radial.hip -- assembly of T's entries from radial functionals.
//
// Every operator entry (m, n) -- P1 hat m on panels m-1, m against hat n on
// panels n-1, n -- is a sum over the quadrature nodes of its four panel pairs
// of a geometric factor times a function of the node distance r alone: H0 or
// H1 of kappa r times a power of r (galerkin_builder.cpp:346-832).  For fixed
// kappa it is a linear functional of that function.  An unordered pair (m, n)
// has five that do not depend on kappa: of the hats the double layer test m /
// trial n and test n / trial m, the weak part of the hypersingular layer and the
// single layer; of the panels m, n the curl part of the hypersingular layer,
// which enters the four entries over a panel pair with the signs of the hats'
// slopes -- kept per panel pair, its rounding cancels in the layer's action on
// smooth traces as the quadrature loops' does (compressed per pair of hats it
// cost a digit of the transmission solution).  The functionals are compressed
// once per geometry onto a few radial points shared by all pairs of a distance
// band:
//
//   far bands   the function is analytic on the band's interval, so its
//               polynomial interpolant at p Chebyshev points is exact to
//               rounding for a small p (band_order: 16-24 on well-resolved
//               meshes), and sum_n c_n g(r_n) = sum_j C_j g(r_j) with C the
//               transposed interpolation of the quadrature coefficients c
//               (k_radial_far);
//   near band   (band 0, all pairs inside radius R, touching panels among them)
//               J0, J1 / x and the entire parts of Y0, Y1 -- what is left
//               without ln x and 1/x -- are entire in r^2, so the transposition
//               on [0, R^2] of the coefficients and of the coefficients times
//               ln(r / R), plus the sums of c / r^2 and of c, reproduces the
//               (singular) quadrature sums (k_radial_near).  The functions span
//               orders of magnitude over [0, R], so every coefficient has to be
//               right to its own last digits: the nodes' Lagrange weights are
//               formed from the differences r^2 - r_j^2 (near_weight).
//
// The points being the band's, one Hankel pair per point and kappa serves every
// pair of the band (k_band_basis), and the evaluation is a real x complex
// matrix product [functionals of the pairs x points] [points x kappa] on the
// FP64 matrix cores (k_band_eval) -- where the node loops evaluate Ns^2 Hankel
// pairs and 17 sums per panel pair and kappa.
//
// The interpolation degrees are chosen for a tier of kappa d_max (d_max the
// largest panel diameter).  A wavenumber's tier depends on its own kappa only
// and a column of the product on its own column of the basis, so a
// wavenumber's bits do not depend on the others of its call or on the batch.
//
// Records: [pair m >= n][nv values per derivative order][column], index m (m + 1) / 2
// + n: K(m, n), K(n, m), W without its curl part, V, the curl part of panels m, n,
// and V(n, m) where nv = 6 (the quirk of the coinciding single layer's
// k-derivatives, HBEM_FLAG_QUIRK_SLP_COINC_DER, is not symmetric); without the
// factor i/4 (galerkin_builder.cpp:1014-1017).
#include <algorithm>
#include <cmath>

#include "hbem_internal.hpp"

namespace hbem {

__device__ __forceinline__ long long tri_ll(int i, int j) { return (long long)i * (i + 1) / 2 + j; }
__device__ __forceinline__ void tri_mn(int rec, int& m, int& n) {
    int i = (int)((sqrt(8.0 * (double)rec + 1.0) - 1.0) * 0.5);
    while (tri_ll(i, 0) > rec) --i;
    while (tri_ll(i + 1, 0) <= rec) ++i;
    m = i;
    n = rec - (int)tri_ll(i, 0);
}

// ---------------------------------------------------------------------------
// Setup
// ---------------------------------------------------------------------------
// Band of every pair of hats from the interval [lo, hi] of the Gauss-node
// distances of its four panel pairs: 0 (near) when hi <= R or the pair touches a
// singular panel pair (band[rec] != 0 on entry), else 1 + floor((lo - first) /
// step); band b covers [first + (b - 1) step, first + b step + W], W the largest
// width an interval can have where a hat's two panels meet, so it holds the whole
// interval.  Consecutive panels of a mesh need not meet (several curves in one
// mesh, an open arc): a pair over such a seam may leave its band, where the
// polynomials grow without bound, and is marked kBandOutside.
// Four lanes a pair, one panel pair each.
__global__ __launch_bounds__(256) void k_radial_band(const double* __restrict__ gtab, int N, int ns, int npairs, double R,
                                                     double first, double step, double width,
                                                     unsigned short* __restrict__ band) {
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int rec = (int)(id >> 2) < npairs ? (int)(id >> 2) : npairs - 1, ab = (int)id & 3;
    const bool touch = band[rec] != 0;
    int m, n;
    tri_mn(rec, m, n);
    double lo = 1e300, hi = 0.0;
    const int P = (ab & 1) ? m : (m == 0 ? N - 1 : m - 1);
    const int Q = (ab >> 1) ? n : (n == 0 ? N - 1 : n - 1);
    for (int i = 0; i < ns; ++i) {
        const double* gi = gtab + ((size_t)P * ns + i) * 5;
        const double x = gi[0], y = gi[1];
        for (int j = 0; j < ns; ++j) {
            const double* gj = gtab + ((size_t)Q * ns + j) * 5;
            const double vx = x - gj[0], vy = y - gj[1];
            const double r2 = vx * vx + vy * vy;
            lo = fmin(lo, r2);
            hi = fmax(hi, r2);
        }
    }
#pragma unroll
    for (int o = 1; o < 4; o <<= 1) {
        lo = fmin(lo, __shfl_xor(lo, o, 64));
        hi = fmax(hi, __shfl_xor(hi, o, 64));
    }
    lo = sqrt(lo);
    hi = sqrt(hi);
    if (ab == 0 && (id >> 2) < npairs) {
        unsigned short b = 0;
        bool in = hi <= R;
        if (!touch && !in) {
            b = (unsigned short)(1 + (int)fmin(fmax(floor((lo - first) / step), 0.0), kBandOutside - 2.0));
            const double end = first + b * step;
            in = lo >= end - step && hi <= end + width;
        }
        band[rec] = in ? b : (unsigned short)kBandOutside;
    }
}

// Skip flags of the general panel pairs (the reference's isArrayZero tests,
// galerkin_builder.cpp:470-495, 852-870) at the pair's triangular index: bit 0
// all |v.N_j| < eps (double layer, test i), bit 1 test j, bit 2 all
// |tau_i.tau_j| < eps.
__global__ __launch_bounds__(256) void k_radial_flags(const double* __restrict__ gtab, int ns, int npairs,
                                                      unsigned char* __restrict__ flags) {
    const int rec = blockIdx.x * blockDim.x + threadIdx.x;
    if (rec >= npairs) return;
    int i, j;
    tri_mn(rec, i, j);
    unsigned f = 7;
    for (int a = 0; a < ns && f; ++a) {
        const double* gi = gtab + ((size_t)i * ns + a) * 5;
        for (int b = 0; b < ns && f; ++b) {
            const double* gj = gtab + ((size_t)j * ns + b) * 5;
            const double vx = gi[0] - gj[0], vy = gi[1] - gj[1];
            if (!(fabs(vx * gj[3] - vy * gj[2]) < kDblEps)) f &= ~1u;
            if (!(fabs(vy * gi[2] - vx * gi[3]) < kDblEps)) f &= ~2u;
            if (!(fabs(gi[3] * gj[3] + gi[2] * gj[2]) < kDblEps)) f &= ~4u;
        }
    }
    flags[rec] = (unsigned char)f;
}

// Where a coefficient lies: pairs go in tiles of 16, and a tile's table is
// [p / 4 steps][nf functionals][64] with element (point & 3) * 16 + pair & 15 --
// the first operand of v_mfma_f64_16x16x4f64 as one coalesced load per step and
// functional.
__device__ __forceinline__ size_t tile_elem(int j, int nf, int f, int row) {
    return ((size_t)(j >> 2) * nf + f) * 64 + (j & 3) * 16 + row;
}

// Sums of 64 values over groups of G lanes: lane l of a group is left with the
// totals of values (64 / G) l .. (64 / G) l + 64 / G - 1 in v[0 ..].  Each step
// exchanges and halves the values a lane carries (63 exchanges for G = 64,
// against 384 for 64 separate butterflies).
template <int O, int N>
__device__ __forceinline__ void exchange_halves(double (&v)[64]) {
    const bool up = threadIdx.x & O;
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
        const double keep = up ? v[i + N / 2] : v[i], give = up ? v[i] : v[i + N / 2];
        v[i] = keep + __shfl_xor(give, O, 64);
    }
    if constexpr (O > 1) exchange_halves<O / 2, N / 2>(v);
}

// The five quadrature coefficients of a Gauss node of panel pair (P, Q) for the
// hats (m, n): double layer test P / trial Q and test Q / trial P, curl part (of
// panels m, n only), weak part, single layer; returns r^2.
struct PairNode {
    int P, Q, sa, sb;
    double fk, ft, fb, cu;
};
__device__ __forceinline__ PairNode pair_node(int m, int n, int ab, int N, const unsigned char* __restrict__ flags) {
    PairNode x;
    x.sa = ab & 1;
    x.sb = ab >> 1;
    x.P = x.sa ? m : (m == 0 ? N - 1 : m - 1);
    x.Q = x.sb ? n : (n == 0 ? N - 1 : n - 1);
    const unsigned f = flags[x.P > x.Q ? tri_ll(x.P, x.Q) : tri_ll(x.Q, x.P)];
    const bool rev = x.P < x.Q;               // bit 0 belongs to the larger panel index as test panel
    x.fk = (f & (rev ? 2u : 1u)) ? 0.0 : 1.0;
    x.ft = (f & (rev ? 1u : 2u)) ? 0.0 : 1.0;
    x.fb = (f & 4u) ? 0.0 : 2.0;
    x.cu = ab == 3 ? 1.0 : 0.0;
    return x;
}
__device__ __forceinline__ double gauss_node(const PairNode& x, int i, int j, const double* __restrict__ gtab, int ns,
                                             const double* __restrict__ xg, const double* __restrict__ wg, double (&c)[5]) {
    const double* gi = gtab + ((size_t)x.P * ns + i) * 5;
    const double* gj = gtab + ((size_t)x.Q * ns + j) * 5;
    const double vx = gi[0] - gj[0], vy = gi[1] - gj[1];
    const double xs = xg[i], xt = xg[j];
    const double w = wg[i] * wg[j];
    const double wb = w * (x.sa ? 1.0 - xs : xs) * (x.sb ? 1.0 - xt : xt);
    c[0] = x.fk * wb * (vx * gj[3] - vy * gj[2]) * gi[4];
    c[1] = x.ft * wb * (vy * gi[2] - vx * gi[3]) * gj[4];
    c[2] = x.cu * w;
    c[3] = x.fb * wb * (gi[3] * gj[3] + gi[2] * gj[2]);
    c[4] = wb * (gi[4] * gj[4]);
    return vx * vx + vy * vy;
}

// Coefficients of the far bands.  L = 16 lanes per pair, two workgroups per tile (64,
// eight, where there are few pairs: see launch_radial_far): lanes over the Gauss nodes
// of the four panel pairs; per node the five
// quadrature coefficients and the Chebyshev polynomials T_q of its position in
// the band are formed, twelve q at a time (60 register sums a lane, totalled over
// the pair's lanes together), and the moments mu_q are carried to the points by
// C_j = sum_q (2 - delta_q0) / p T_q(s_j) mu_q (costab, built on the host).  The
// T_q recurrence runs for the nodes only, where its errors meet the decaying
// coefficients of the smooth function; a recurrence over the points would not be
// damped.  The two double-layer coefficients are stored divided by r_j (they
// multiply H1 / r).
template <int L>
__global__ __launch_bounds__(128) void k_radial_far(const int* __restrict__ recs, const BandTile* __restrict__ tiles,
                                                    int tile0, const Band* __restrict__ bands,
                                                    const double* __restrict__ gtab, const double* __restrict__ xg,
                                                    const double* __restrict__ wg, int N, int ns,
                                                    const unsigned char* __restrict__ flags,
                                                    const double* __restrict__ costab, double* __restrict__ tab, int pmax) {
    constexpr int QC = 12, PB = 128 / L, BT = 16 / PB;   // pairs of a workgroup, workgroups of a tile
    extern __shared__ double mu_s[];          // [PB][pmax][5]
    const int row = (blockIdx.x % BT) * PB + threadIdx.x / L, l = threadIdx.x % L;
    const int tile = tile0 + blockIdx.x / BT;
    double* mu = mu_s + (size_t)(threadIdx.x / L) * pmax * 5;
    const BandTile bt = tiles[tile];
    const Band bd = bands[bt.band];
    const int rec = recs[(size_t)tile * 16 + row];
    const int p = bd.p, nn = ns * ns;
    int m = 0, n = 0;
    if (rec >= 0) tri_mn(rec, m, n);
    const double ia = 1.0 / bd.a;
    for (int q0 = 0; q0 < p; q0 += QC) {
        double s[64];
#pragma unroll
        for (int f = 0; f < 64; ++f) s[f] = 0.0;
        for (int ab = 0; ab < 4 && rec >= 0; ++ab) {
            const PairNode pn = pair_node(m, n, ab, N, flags);
            for (int nd = l; nd < nn; nd += L) {
                const int i = nd / ns, j = nd - i * ns;
                double c[5];
                const double r = sqrt(gauss_node(pn, i, j, gtab, ns, xg, wg, c));
                const double u = (r - bd.c) * ia, u2 = u + u;
                double tp = u, tc = 1.0;      // T_{q-1}, T_q (T_{-1} = T_1)
                for (int q = 0; q < q0; ++q) {
                    const double tn = fma(u2, tc, -tp);
                    tp = tc;
                    tc = tn;
                }
#pragma unroll
                for (int q = 0; q < QC; ++q) {
#pragma unroll
                    for (int g = 0; g < 5; ++g) s[q * 5 + g] = fma(tc, c[g], s[q * 5 + g]);
                    const double tn = fma(u2, tc, -tp);
                    tp = tc;
                    tc = tn;
                }
            }
        }
        exchange_halves<L / 2, 64>(s);
#pragma unroll
        for (int k = 0; k < 64 / L; ++k) {
            const int f = 64 / L * l + k;
            if (f < QC * 5 && q0 * 5 + f < p * 5) mu[q0 * 5 + f] = s[k];
        }
    }
    __syncthreads();
    const double* ct = costab + bd.cos;       // [j][q], weighted
    const double* rj = costab + bd.rad;
    double* out = tab + bt.off;
    for (int it = l; it < p * 5; it += L) {
        const int j = it / 5, g = it - 5 * j;
        double v = 0.0;
        for (int q = 0; q < p; ++q) v = fma(ct[j * p + q], mu[q * 5 + g], v);
        out[tile_elem(j, 5, g, row)] = g < 2 ? v / rj[j] : v;
    }
}

// Lagrange weights of the near band's points at a node: l_j = prod_{k != j} (u -
// u_k) / (u_j - u_k) with u = r^2 times a power of two (iS, near 1 / R^2), u_j doubles
// (the points are defined by them) and lam[j] = prod_{k != j} 1 / (u_j - u_k); pts:
// [u_j][lam], near_stride(p) each (-1 and 0 beyond p).  Products of differences, each
// good to a few rounding errors of itself: the weights are too, also those a thousand
// times smaller than the largest.  (Sums of Chebyshev polynomials, which the far bands
// take, leave every weight with the rounding of the largest: at kappa d = 20, where
// J1 / r falls by 10^4 over the band, K of a 64-panel polygon was off by 2.0e-13 and V
// by 5.7e-14; these leave 3.8e-14 and 8.1e-15, the node loops 4.5e-14 and 2.2e-14.)
// u's last bit is made one, up or down, and the points' are zero: no node names a point.
__device__ __forceinline__ double near_node(double r2, double iS) {
    const long long b = __double_as_longlong(r2 * iS);
    return __longlong_as_double(b & 1 ? b : (b & 2 ? b - 1 : b + 1));
}
__device__ __forceinline__ double near_product(const double* __restrict__ pts, int p, double u) {
    double w = 1.0;
    for (int k = 0; k < p; ++k) w *= u - pts[k];
    return w;
}
// 1 / d by two Newton steps
__device__ __forceinline__ double fast_recip(double d) {
    double y = __builtin_amdgcn_rcp(d);
    y = fma(fma(-d, y, 1.0), y, y);
    return fma(fma(-d, y, 1.0), y, y);
}

typedef double dbl4 __attribute__((ext_vector_type(4)));
// s + x, what rounding takes from it added to e (Knuth's TwoSum)
__device__ __forceinline__ void two_sum(dbl4& s, dbl4 x, dbl4& e) {
#pragma clang fp contract(off)
    const dbl4 t = s + x, b = t - s;
    e += (s - (t - b)) + (x - b);
    s = t;
}

// Moments of the singular panel pairs for the near band (composite rules,
// galerkin_builder.cpp:17-306, 553-832): local functionals of a pair (i, j), entry
// q = a + 2 b: double layer test i (local a) / trial j (b) [0..3] and test j (a) /
// trial i (b) [4..7], curl weight [8], weak part [9..12] and single layer [13..16]
// test i (a) / trial j (b); times the Lagrange weight of point q, and that times
// (2/pi) ln(r / R) [17..33].  A pair's table serves the four pairs of hats over it;
// adjacent pairs have one table per node half.  ext[25]: sums of c / r^2 of the
// double-layer functionals, then the sums of c of the seventeen (0 for the curl
// weight, see k_radial_near).
//
// Sixteen of the seventeen functionals and the weights are the operands of a
// matrix product over the nodes, [16 x nodes] [nodes x 32 q] and the same with the
// logarithm, so a wavefront evaluates 64 nodes (a lane each), hands them through
// LDS to the lanes that v_mfma_f64_16x16x4f64 wants them in, and multiplies; the
// curl weight and ext ride along as multiply-adds.  The product bounds it: one
// workgroup (pair, half) reads nothing but its two panels.  Node tables in memory
// read by one workgroup per two q took 0.55 ms for a 200-panel polygon's pairs
// (order 11) and 5.2 ms for the 400-panel star's (order 16); this form 0.29 and
// 2.53 ms.
constexpr int kMomLocal = kRadialMoments;
constexpr int kMomQ = 32;                     // q per workgroup
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
template <int CLS>
__global__ __launch_bounds__(256) void k_radial_moments(const int* __restrict__ ent, const double* __restrict__ panels,
                                                        const double* __restrict__ coefs,
                                                        const double* __restrict__ xc, const double* __restrict__ wc, int nc,
                                                        double R, double iS, const double* __restrict__ pts, int p,
                                                        double* __restrict__ mom, double* __restrict__ ext) {
    constexpr int LD = 17, WAVE = 64 * LD + 3 * 64;   // doubles of a wavefront
    __shared__ double sh[4 * WAVE];
    __shared__ int nz[3];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, l16 = lane & 15, lk = lane >> 4;
    const int e = blockIdx.x, h = blockIdx.y, q0 = blockIdx.z * kMomQ;
    const int nn = nc * nc;
    const int pi = ent[3 * (size_t)e], pj = ent[3 * (size_t)e + 1];
    const bool swap = ent[3 * (size_t)e + 2] != 0;
    const double* gi = panels + 8 * (size_t)pi;
    const double* gj = panels + 8 * (size_t)pj;
    const double iR2 = 1.0 / (R * R);
    const int P = near_stride(p);
    double* buf = sh + wv * WAVE;
    double *sln = buf + 64 * LD, *scu = sln + 64, *sir = scu + 64;
    if (tid < 3) nz[tid] = 0;
    __syncthreads();
    dbl4 tot[2][2] = {}, err[2][2] = {};      // [16 q][without, with the logarithm]: sums and their rounding errors
    double curl[2][2] = {}, ex = 0.0, ec = 0.0;
    bool any[3] = {false, false, false};
    for (int n0 = 64 * wv; n0 < nn; n0 += 256) {
        const int nd = n0 + lane < nn ? n0 + lane : nn - 1, a = nd / nc, b = nd - a * nc;
        const bool in = n0 + lane < nn;
        cdbl zi, zj, ti, tj;
        double w, bi[2], bj[2];
        if (CLS == 1) {
            const double t = xc[a], sx = t * xc[b];
            w = t * wc[a] * wc[b];
            const double si = h == 0 ? sx : t, sj = h == 0 ? t : sx;
            panel_eval(gi, coefs, si, !swap, zi, ti);
            panel_eval(gj, coefs, sj, swap, zj, tj);
            bi[0] = swap ? si : 1.0 - si;
            bi[1] = swap ? 1.0 - si : si;
            bj[0] = swap ? 1.0 - sj : sj;
            bj[1] = swap ? sj : 1.0 - sj;
        } else {
            const double t = xc[b], sx = t * (1.0 - xc[a]);
            w = t * wc[a] * wc[b];
            panel_eval(gi, coefs, sx, false, zi, ti);
            panel_eval(gi, coefs, t, false, zj, tj);
            bi[0] = sx; bi[1] = 1.0 - sx; bj[0] = t; bj[1] = 1.0 - t;
        }
        if (!in) w = 0.0;
        const cdbl v = zi - zj;
        const double r2 = v.x * v.x + v.y * v.y, ni = hypot(ti.x, ti.y), nj = hypot(tj.x, tj.y);
        const double vd = (v.x * tj.y - v.y * tj.x) * ni, vt = (v.y * ti.x - v.x * ti.y) * nj;
        const double td = ti.y * tj.y + ti.x * tj.x;
        any[0] = any[0] || (in && !(fabs(vd) < kDblEps));
        any[1] = any[1] || (in && !(fabs(vt) < kDblEps));
        any[2] = any[2] || (in && !(fabs(td) < kDblEps));
        const double u = near_node(r2, iS);
        double* o = buf + lane * LD;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double pbb = bi[q & 1] * bj[q >> 1], pbt = bj[q & 1] * bi[q >> 1];
            const double pw = CLS == 1 ? pbb : pbb + pbt;
            o[q] = w * vd * pbb;
            o[4 + q] = w * vt * pbt;
            o[8 + q] = w * (2.0 * td) * pw;
            o[12 + q] = w * (ni * nj) * pw;
        }
        sln[lane] = r2 > 0.0 ? 0.5 * kTwoOverPi * log(r2 * iR2) : 0.0;
        scu[lane] = CLS == 1 ? w : 2.0 * w;
        sir[lane] = r2 > 0.0 ? 1.0 / r2 : 0.0;
        wave_lds_fence();
        double fa[16];
#pragma unroll
        for (int s = 0; s < 16; ++s) fa[s] = buf[(4 * s + lk) * LD + l16];
        wave_lds_fence();
        const double wp = near_product(pts, p, u);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int j = q0 + 16 * c + q;
                o[q] = (wp * pts[P + j]) * fast_recip(u - pts[j]);
            }
            wave_lds_fence();
            dbl4 acc[2] = {};                 // this chunk's 64 nodes
#pragma unroll
            for (int s = 0; s < 16; ++s) {
                const double t = buf[(4 * s + lk) * LD + l16], tl = t * sln[4 * s + lk], cu = scu[4 * s + lk];
                acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[s], t, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[s], tl, acc[1], 0, 0, 0);
                curl[c][0] = fma(cu, t, curl[c][0]);
                curl[c][1] = fma(cu, tl, curl[c][1]);
                if (c == 0) {
                    ex = fma(fa[s], sir[4 * s + lk], ex);
                    ec += fa[s];
                }
            }
            // a singular pair's nodes fill many chunks, whose running sum would leave
            // the coefficients with three times the rounding error of one
#pragma unroll
            for (int g = 0; g < 2; ++g) two_sum(tot[c][g], acc[g], err[c][g]);
            wave_lds_fence();
        }
    }
    for (int k = 0; k < 3; ++k)
        if (any[k]) nz[k] = 1;
    // the four wavefronts' sums through LDS, added in order: [c][log][16][16],
    // then curl [c][log][16], then the sums of c / r^2 [16] and of c [16]
    __syncthreads();
    for (int c = 0; c < 2; ++c)
        for (int g = 0; g < 2; ++g) {
            for (int v = 0; v < 4; ++v) buf[((c * 2 + g) * 16 + 4 * v + lk) * 16 + l16] = tot[c][g][v] + err[c][g][v];
            double t = curl[c][g];
            t += __shfl_xor(t, 16, 64);
            t += __shfl_xor(t, 32, 64);
            if (lk == 0) buf[1024 + (c * 2 + g) * 16 + l16] = t;
        }
    ex += __shfl_xor(ex, 16, 64);
    ex += __shfl_xor(ex, 32, 64);
    ec += __shfl_xor(ec, 16, 64);
    ec += __shfl_xor(ec, 32, 64);
    if (lk == 0) {
        buf[1088 + l16] = ex;
        buf[1104 + l16] = ec;
    }
    __syncthreads();
    auto total = [&](int k) { return (sh[k] + sh[WAVE + k]) + (sh[2 * WAVE + k] + sh[3 * WAVE + k]); };
    const bool f0 = nz[0] != 0, f1 = nz[1] != 0, f2 = nz[2] != 0;   // isArrayZero (galerkin_builder.cpp:470-495, 852-870)
    const size_t eh = (size_t)e * gridDim.y + h;
    // functional kk of a table whose sixteen products lie at base, stride st
    auto value = [&](int kk, int base, int st, double curl_sum) {
        if (kk == 8) return curl_sum;
        if (kk > 8) return kk > 12 || f2 ? total(base + st * (kk - 1)) : 0.0;
        if (CLS == 1) return (kk < 4 ? f0 : f1) ? total(base + st * kk) : 0.0;
        return kk < 4 ? (f0 ? total(base + st * kk) : 0.0) + (f1 ? total(base + st * (4 + kk)) : 0.0) : 0.0;
    };
    for (int it = tid; it < kMomQ * kMomLocal; it += 256) {
        const int q = it / kMomLocal, k = it - q * kMomLocal, g = (q >> 4) * 2 + (k >= 17 ? 1 : 0);
        if (q0 + q >= p) break;
        mom[(eh * p + q0 + q) * kMomLocal + k] = value(k % 17, g * 256 + (q & 15), 16, total(1024 + g * 16 + (q & 15)));
    }
    if (q0 == 0 && tid < kRadialSums)
        ext[eh * kRadialSums + tid] = tid < 8 ? value(tid, 1088, 1, 0.0) : value(tid - 8, 1104, 1, 0.0);
}

// Coefficients of the near band.  One wavefront per pair of hats: the Gauss nodes
// of its general panel pairs over the lanes, six points at a time (60 register sums a
// lane, totalled over the lanes together), and the moments of its singular panel
// pairs from their tables.  Table per point: the five coefficients, then those of
// (2/pi) ln(r / R); ext [tile][7][16]: sum c / r^2 of the two double-layer
// functionals, the five sums of c, for the curl part less one: the constant that its
// first k-derivative takes from the 1 / x of H1, -2i / (pi kappa) of every panel pair,
// cancels in the hats (record_W), but for the quadrature rules' own defect of the
// integral of 1 (curl_s of the singular pairs', curl_g of the general ones), and its
// rounding errors would not, 1 / (kappa h)^2 times the entry's.  The far bands drop it
// too (k_band_eval).
__global__ __launch_bounds__(128) void k_radial_near(const RadialNear* __restrict__ ent, int nent,
                                                     const BandTile* __restrict__ tiles, const Band* __restrict__ bands,
                                                     const double* __restrict__ gtab, const double* __restrict__ xg,
                                                     const double* __restrict__ wg, int N, int ns,
                                                     const unsigned char* __restrict__ flags,
                                                     const double* __restrict__ mom_c, const double* __restrict__ ext_c,
                                                     const double* __restrict__ mom_a, const double* __restrict__ ext_a,
                                                     const double* __restrict__ costab, double iS, double curl_s,
                                                     double curl_g, double* __restrict__ tab, double* __restrict__ ext, int pmax, int cache) {
    constexpr int QC = 6;
    extern __shared__ double mu_s[];          // [2 wavefronts]([pmax][10], [cache]{product, log} of the nodes)
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int x = blockIdx.x * 2 + wv;        // the grid covers the tiles' 16 pairs each, two a workgroup
    const int tile = x >> 4, row = x & 15;
    double* mu = mu_s + (size_t)wv * (pmax * 10 + 2 * cache);
    double* nodes = mu + pmax * 10;           // (a lane reads what it wrote)
    const BandTile bt = tiles[tile];
    const Band bd = bands[bt.band];
    const int p = bd.p, nn = ns * ns;
    const bool live = x < nent;               // else the padding of the last tile
    const RadialNear en = ent[live ? x : 0];
    const double iR2 = 1.0 / (bd.a * bd.a);   // near band: a = R
    const double* pts = costab + bd.cos;
    const int P = near_stride(p);
    double ex[7] = {};                        // sums of c / r^2 (double layer), of c (not curl)
    for (int q0 = 0; q0 < p; q0 += QC) {
        double s[64];
#pragma unroll
        for (int f = 0; f < 64; ++f) s[f] = 0.0;
        for (int ab = 0; ab < 4 && live; ++ab) {
            if ((en.type[ab] & 3) != 3) continue;
            const PairNode pn = pair_node(en.m, en.n, ab, N, flags);
            for (int nd = lane; nd < nn; nd += 64) {
                const int i = nd / ns, j = nd - i * ns;
                double c[5];
                const double r2 = gauss_node(pn, i, j, gtab, ns, xg, wg, c);
                const double u = near_node(r2, iS);
                double wp, lr;
                const int at = ab * nn + nd;
                if (q0 == 0 || !cache) {
                    lr = r2 > 0.0 ? 0.5 * kTwoOverPi * log(r2 * iR2) : 0.0;
                    wp = near_product(pts, p, u);
                    if (cache) {
                        nodes[2 * at] = wp;
                        nodes[2 * at + 1] = lr;
                    }
                } else {
                    wp = nodes[2 * at];
                    lr = nodes[2 * at + 1];
                }
                if (q0 == 0) {
                    if (r2 > 0.0) {
                        ex[0] += c[0] / r2;
                        ex[1] += c[1] / r2;
                    }
#pragma unroll
                    for (int g = 0; g < 5; ++g)
                        if (g != 2) ex[2 + g] += c[g];
                }
#pragma unroll
                for (int q = 0; q < QC; ++q) {
                    const int k = q0 + q;     // < P, lam 0 beyond p
                    const double t = (wp * pts[P + k]) * fast_recip(u - pts[k]), tl = t * lr;
#pragma unroll
                    for (int g = 0; g < 5; ++g) {
                        s[q * 10 + g] = fma(t, c[g], s[q * 10 + g]);
                        s[q * 10 + 5 + g] = fma(tl, c[g], s[q * 10 + 5 + g]);
                    }
                }
            }
        }
        exchange_halves<32, 64>(s);
        if (lane < QC * 10 && q0 * 10 + lane < p * 10) mu[q0 * 10 + lane] = s[0];
    }
#pragma unroll
    for (int g = 0; g < 7; ++g)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ex[g] += __shfl_xor(ex[g], o, 64);
    __syncthreads();
    // the singular panel pairs' local moments: functional g of panel pair ab
    auto local = [&](int ab, int g) {
        const int sa = ab & 1, sb = ab >> 1;
        const int P = sa ? en.m : (en.m == 0 ? N - 1 : en.m - 1), Q = sb ? en.n : (en.n == 0 ? N - 1 : en.n - 1);
        const int q = sa + 2 * sb, qt = sb + 2 * sa;
        const bool coi = (en.type[ab] & 3) == 0, rev = P < Q;   // rev: Q is the pair's first panel
        if (g == 0) return coi || !rev ? q : 4 + q;
        if (g == 1) return coi || rev ? qt : 4 + qt;
        if (g == 2) return 8;
        // one panel: entry (0, 1) = entry (1, 0) (galerkin_builder.cpp:571-573, 744-746)
        return (g == 3 ? 9 : 13) + (coi ? (q == 2 ? 1 : q) : (rev ? qt : q));
    };
    double* out = tab + bt.off;
    for (int it = lane; it < p * 10; it += 64) {
        const int j = it / 10, g = it - 10 * j, g5 = g % 5;
        double v = mu[it];
        for (int ab = 0; ab < 4 && live; ++ab) {
            const int cls = en.type[ab] & 3, e = en.type[ab] >> 2;
            if (cls == 3 || (g5 == 2 && ab != 3)) continue;
            const int k = j * kMomLocal + (g >= 5 ? 17 : 0) + local(ab, g5);
            const size_t st = (size_t)p * kMomLocal;
            v += cls == 0 ? mom_c[e * st + k] : mom_a[2 * e * st + k] + mom_a[(2 * e + 1) * st + k];
        }
        out[tile_elem(j, 10, g, row)] = v;
    }
    if (lane < 7) {
        double v = 0.0;
#pragma unroll
        for (int g = 0; g < 7; ++g)
            if (lane == g) v = ex[g];
        for (int ab = 0; ab < 4 && live; ++ab) {
            const int cls = en.type[ab] & 3, e = en.type[ab] >> 2;
            if (lane == 4) {
                if (ab == 3) v = cls == 3 ? curl_g : curl_s;
                continue;
            }
            if (cls == 3) continue;
            const int k = lane < 2 ? local(ab, lane) : 8 + local(ab, lane - 2);
            const size_t st = kRadialSums;
            v += cls == 0 ? ext_c[e * st + k] : ext_a[2 * e * st + k] + ext_a[(2 * e + 1) * st + k];
        }
        ext[((size_t)tile * 7 + lane) * 16 + row] = v;
    }
}

// ---------------------------------------------------------------------------
// Evaluation
// ---------------------------------------------------------------------------
// The radial functions at every band's points for the group's slots s (its
// columns' inner slots, then the outer ones): basis[(off + 2 j + i) nslots + s].
// Far bands: i = 0 H0, i = 1 H1 at kappa r_j.  Near band: (J0, entire part of
// Y0 plus (2/pi) ln(kappa R / 2) J0) and the same of J1 / r, Y1 / r; complex
// kappa: the sums J + iY of these, and at offset nbasis i J0, i J1 / r.
// The points are those of the transposition, s_j in extended precision: what the
// doubles r_j and kappa r_j leave out of the argument enters by the derivatives
// (A&S 9.1.27-28), as a phase kappa r of 100 rounded to 64 bits would put 1e-14 on
// every pair of the band.
// Up to x = 8 the entire parts A = J0, B = J1 / x, C, D of Y0 and Y1 by their power
// series in y = x^2 / 64 (A&S 9.1.10-9.1.13), whose terms grow to 100 and cancel: by the
// compensated Horner scheme (Graillat, Langlois and Louvet: each step's rounding errors,
// by fma and TwoSum, in a second Horner recurrence), the coefficients in two doubles.
// ser: [kSeriesDeg + 1][A, B, C, D], then the residuals.
__device__ __forceinline__ void series_comp(const double* __restrict__ ser, double z, double (&v)[4]) {
#pragma clang fp contract(off)
    const double* lo = ser + 4 * (kSeriesDeg + 1);
    double e[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        v[f] = ser[4 * kSeriesDeg + f];
        e[f] = lo[4 * kSeriesDeg + f];
    }
    for (int i = kSeriesDeg - 1; i >= 0; --i) {
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            const double a = ser[4 * i + f], p = v[f] * z, pe = fma(v[f], z, -p);
            const double s = p + a, t = s - p, se = (p - (s - t)) + (a - t);
            e[f] = fma(e[f], z, (pe + se) + lo[4 * i + f]);
            v[f] = s;
        }
    }
#pragma unroll
    for (int f = 0; f < 4; ++f) v[f] += e[f];
}

__global__ __launch_bounds__(256) void k_band_basis(RadialParams P, const Band* __restrict__ bands,
                                                    const double* __restrict__ costab, int nslots) {
    const int b = blockIdx.y;
    const Band bd = bands[b];
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= bd.p * nslots) return;
    const int j = id / nslots, s = id - j * nslots;
    const int q = P.cols[s % P.ncolg] + (s >= P.ncolg ? P.nslot2 : 0);
    const double r = costab[bd.rad + j], dr = costab[bd.rad + bd.p + j];
    cdbl* o = P.basis + ((size_t)bd.basis + 2 * j) * nslots + s;
    if (P.kapi) {
        const cdbl kap = mk(P.kap[q], P.kapi[q]), z = r * kap;
        const cdbl d = mk(fma(r, kap.x, -z.x) + dr * kap.x, fma(r, kap.y, -z.y) + dr * kap.y);
        if (b > 0) {
            cdbl h0, h1;
            if (cabsd(z) < 8.0) {
                // (the continued fraction is slow next to |z| = 2 and leaves 2e-15)
                cdbl c0, c1;
                bessel_entire_cplx(z, h0, c0, h1, c1);
                const cdbl L2 = kTwoOverPi * clogd(0.5 * z), y0 = c0 + L2 * h0;
                const cdbl y1 = z * (c1 + L2 * h1) - kTwoOverPi * recip(z), J1 = z * h1;
                h0 = mk(h0.x - y0.y, h0.y + y0.x);
                h1 = mk(J1.x - y1.y, J1.y + y1.x);
            } else {
                hankel01_cplx(z, h0, h1);
            }
            o[0] = h0 - d * h1;
            o[nslots] = h1 + d * (h0 - cdiv(h1, z));
            return;
        }
        // J0 (1 + (2i/pi) ln(kappa R / 2)) + i C and the same of J1 / r, then the
        // factors i J0, i J1 / r of the coefficients with (2/pi) ln(r / R)
        cdbl j0, c0, j1, c1;
        bessel_entire_cplx(z, j0, c0, j1, c1);
        const cdbl t = cdiv(d, z), zd = z * d, e0 = j0, e1 = j1, f0 = c0;
        j0 = j0 - zd * e1;
        j1 = j1 + t * (e0 - 2.0 * e1);
        c0 = c0 - zd * c1 + (kTwoOverPi * t) * (mk(1.0, 0.0) - e0);
        c1 = c1 + t * (f0 - 2.0 * c1 - kTwoOverPi * e1);
        const cdbl lR = mk(1.0, 0.0) + mk(0.0, kTwoOverPi) * clogd(0.5 * bd.a * kap);
        const cdbl b1 = kap * j1, d1 = kap * c1;
        o[0] = j0 * lR + mk(-c0.y, c0.x);
        o[nslots] = b1 * lR + mk(-d1.y, d1.x);
        cdbl* ol = P.basis + ((size_t)P.nbasis + 2 * j) * nslots + s;
        ol[0] = mk(-j0.y, j0.x);
        ol[nslots] = mk(-b1.y, b1.x);
        return;
    }
    const double kap = P.kap[q], x = kap * r, d = fma(kap, r, -x) + kap * dr, xi = 1.0 / x;
    double A, B, C, Dd;                        // J0 = A, J1 = x B, entire parts C of Y0 and x Dd of Y1
    if (x < 8.0) {
        // polynomials in y = x^2 / 64, whose rounding is one more residual of the
        // argument: (x^2 - fl(x^2)) / (2 x)
        const double x2 = x * x, t = (d + 0.5 * fma(x, x, -x2) * xi) * xi;
        double v[4];
        series_comp(costab, x2 * (1.0 / 64.0), v);
        A = fma(-x2 * t, v[1], v[0]);
        B = fma(t, fma(-2.0, v[1], v[0]), v[1]);
        C = fma(kTwoOverPi * t, 1.0 - v[0], fma(-x2 * t, v[3], v[2]));
        Dd = fma(t, v[2] - 2.0 * v[3] - kTwoOverPi * v[1], v[3]);
        if (b > 0) {
            const double L2 = kTwoOverPi * fma(d, xi, log(0.5 * x)), xd = x + d, J1 = xd * B;
            o[0] = mk(A, fma(L2, A, C));
            o[nslots] = mk(J1, fma(L2, J1, fma(xd, Dd, -kTwoOverPi * fma(-d * xi, xi, xi))));
            return;
        }
    } else {
        double j0, y0, j1, y1;
        bessel_jy01_f<0>(x, 0.0, 0.0, xi, 1.0 / sqrt(kPi * x), j0, y0, j1, y1);
        const double J0 = fma(-d, j1, j0), Y0 = fma(-d, y1, y0);
        const double J1 = fma(d, fma(-j1, xi, j0), j1), Y1 = fma(d, fma(-y1, xi, y0), y1);
        if (b > 0) {
            o[0] = mk(J0, Y0);
            o[nslots] = mk(J1, Y1);
            return;
        }
        const double L2 = kTwoOverPi * fma(d, xi, log(0.5 * x)), xr = fma(-d * xi, xi, xi);
        A = J0;
        C = fma(-L2, J0, Y0);
        B = J1 * xr;
        Dd = (fma(-L2, J1, Y1) + kTwoOverPi * xr) * xr;
    }
    const double lR = kTwoOverPi * log(0.5 * (kap * bd.a));
    o[0] = mk(A, fma(lR, A, C));
    o[nslots] = mk(kap * B, kap * fma(lR, B, Dd));
}

// One complex sum of four pairs (the accumulator rows of a lane).
struct Sum4 {
    dbl4 re, im;
};

// The scalings at the end of double_layer_*, hypersingular_*, single_layer_* for
// one slot: sums per order -> value of order t.
template <class K>
struct SlotScale {
    K kap, kr, k2h, kinv, nk2h, nkap2;        // kappa, k, kappa^2 / 2, 1 / kappa, -kappa^2 / 2, -2 kappa
    double c, sqc;
};
// Real scalings with every operation fixed by the source (no contraction left
// to the compiler): an order's value is the same in every instantiation.
__device__ __forceinline__ cdbl scaled(double k, cdbl b) {
#pragma clang fp contract(off)
    return mk(k * b.x, k * b.y);
}
__device__ __forceinline__ cdbl scaled(cdbl k, cdbl b) { return k * b; }
__device__ __forceinline__ cdbl minus(cdbl a, cdbl b) {
#pragma clang fp contract(off)
    return mk(a.x - b.x, a.y - b.y);
}
__device__ __forceinline__ cdbl nmadd(double k, cdbl b, cdbl a) { return mk(fma(-k, b.x, a.x), fma(-k, b.y, a.y)); }   // a - k b
__device__ __forceinline__ cdbl nmadd(cdbl k, cdbl b, cdbl a) { return a - k * b; }
template <class K>
__device__ __forceinline__ cdbl value_K(const SlotScale<K>& s, int t, cdbl s0, cdbl s1, cdbl s2) {
    if (t == 0) return scaled(s.kap, s0);
    if (t == 1) return scaled(s.kr * s.c, s1);
    return scaled(s.c, nmadd(s.kap, s2, s1));
}
template <class K>
__device__ __forceinline__ cdbl value_V(const SlotScale<K>& s, int t, cdbl v0, cdbl v1, cdbl v2) {
    if (t == 0) return v0;
    if (t == 1) return scaled(-s.sqc, v1);
    return scaled(-s.c, nmadd(s.kinv, v1, v2));
}
// curl part of a panel pair
template <class K>
__device__ __forceinline__ cdbl value_A(const SlotScale<K>& s, int t, cdbl a0, cdbl a1, cdbl a2) {
    if (t == 0) return a0;
    if (t == 1) return scaled(-s.sqc, a1);
    return scaled(-s.c, nmadd(s.kinv, a1, a2));
}
// the rest of W
template <class K>
__device__ __forceinline__ cdbl value_W(const SlotScale<K>& s, int t, cdbl b0, cdbl b1, cdbl b2) {
    if (t == 0) return scaled(s.nk2h, b0);
    if (t == 1) return scaled(s.sqc, nmadd(s.kap, b0, scaled(s.k2h, b1)));
    return scaled(s.c, minus(nmadd(s.nkap2, b1, scaled(s.k2h, nmadd(s.kinv, b1, b2))), b0));
}

__device__ __forceinline__ void load_slot(const RadialParams& P, int q, SlotScale<double>& s) {
    s.kap = P.kap[q];
    s.kr = P.kr[q];
    s.c = P.cv[q];
    s.k2h = 0.5 * s.kap * s.kap;
    s.kinv = 1.0 / s.kap;
    s.nk2h = -s.k2h;
    s.nkap2 = -2.0 * s.kap;
    s.sqc = sqrt(s.c);
}
__device__ __forceinline__ void load_slot(const RadialParams& P, int q, SlotScale<cdbl>& s) {
    s.kap = mk(P.kap[q], P.kapi[q]);
    s.kr = mk(P.kr[q], P.kri[q]);
    s.c = P.cv[q];
    s.k2h = 0.5 * s.kap * s.kap;
    s.kinv = recip(s.kap);
    s.nk2h = (-1.0) * s.k2h;
    s.nkap2 = -2.0 * s.kap;
    s.sqc = sqrt(s.c);
}

// sum v of s plus i k e
__device__ __forceinline__ void add_i(Sum4& s, int v, double k, double e) { s.im[v] = fma(k, e, s.im[v]); }
__device__ __forceinline__ void add_i(Sum4& s, int v, cdbl k, double e) {
    s.re[v] = fma(-k.y, e, s.re[v]);
    s.im[v] = fma(k.x, e, s.im[v]);
}

// Sums of NF functionals starting at f0 (all of one kind: KIND 0 double layer,
// 1 the others) for orders 0..D and the lane's one (two: DIFF) slots.
template <int D, bool DIFF, bool NEAR, class K, int KIND, int NF>
__device__ __forceinline__ void band_sums(const double* __restrict__ a, int f0, const cdbl* __restrict__ bs, int nslots,
                                          int s0, int s1, const double* __restrict__ rj, int p, const double* __restrict__ ex,
                                          const K* ikap, const cdbl* __restrict__ bl, Sum4 (&S)[D + 1][NF][DIFF ? 2 : 1]) {
    constexpr int H = DIFF ? 2 : 1, NA = NEAR ? 10 : 5;
    constexpr bool CN = NEAR && sizeof(K) == sizeof(cdbl);   // near band, complex kappa
    const int lane = threadIdx.x & 63, lk = lane >> 4;
#pragma unroll
    for (int t = 0; t <= D; ++t)
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int h = 0; h < H; ++h) S[t][f][h].re = S[t][f][h].im = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 2
    for (int st = 0; st < (p >> 2); ++st) {
        const int j = 4 * st + lk;
        double c[NF], cl[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            c[f] = a[((size_t)st * NA + f0 + f) * 64 + lane];
            if (NEAR) cl[f] = a[((size_t)st * NA + 5 + f0 + f) * 64 + lane];
        }
        cdbl g[2][H], l[2][H];                 // the two radial functions, inner and outer slot (l: see k_band_basis)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            // order 0 of KIND 0 takes function 1, of KIND 1 function 0; order 1 the other
            if (D == 0 && i == (KIND == 0 ? 0 : 1)) continue;
#pragma unroll
            for (int h = 0; h < H; ++h) {
                g[i][h] = bs[(size_t)(2 * j + i) * nslots + (h ? s1 : s0)];
                if (CN) l[i][h] = bl[(size_t)(2 * j + i) * nslots + (h ? s1 : s0)];
            }
        }
        const double r = D > 0 ? rj[j] : 1.0, r2 = r * r;
#pragma unroll
        for (int t = 0; t <= D; ++t) {
            const int i = ((KIND == 0) == ((t & 1) == 0)) ? 1 : 0;
            // far: r^t; near (functions of H1 / r): orders 0, 1, 2 of K 1, 1, r^2, of the others 1, r^2, r^2
            const double sc = NEAR ? (t == 2 || (t == 1 && KIND == 1) ? r2 : 1.0) : (t == 0 ? 1.0 : (t == 1 ? r : r2));
            const bool one = t == 0 || (NEAR && t == 1 && KIND == 0);
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const double cf = one ? c[f] : c[f] * sc;
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    S[t][f][h].re = __builtin_amdgcn_mfma_f64_16x16x4f64(cf, g[i][h].x, S[t][f][h].re, 0, 0, 0);
                    S[t][f][h].im = __builtin_amdgcn_mfma_f64_16x16x4f64(cf, g[i][h].y, S[t][f][h].im, 0, 0, 0);
                }
                if (NEAR) {
                    const double lf = one ? cl[f] : cl[f] * sc;
#pragma unroll
                    for (int h = 0; h < H; ++h) {
                        if (CN) S[t][f][h].re = __builtin_amdgcn_mfma_f64_16x16x4f64(lf, l[i][h].x, S[t][f][h].re, 0, 0, 0);
                        S[t][f][h].im = __builtin_amdgcn_mfma_f64_16x16x4f64(lf, CN ? l[i][h].y : g[i][h].x, S[t][f][h].im, 0, 0, 0);
                    }
                }
            }
        }
    }
    if (NEAR) {
        // the -2 / (pi x) of Y1: Y1 / r takes the sums of c / r^2, Y1 r those of c
#pragma unroll
        for (int t = 0; t <= D; ++t) {
            const bool y1 = (KIND == 0) == ((t & 1) == 0);
            if (!y1) continue;
#pragma unroll
            for (int f = 0; f < NF; ++f)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const double e = ex[(size_t)(KIND == 0 && t == 0 ? f0 + f : 2 + f0 + f) * 16 + 4 * v + lk];
#pragma unroll
                    for (int h = 0; h < H; ++h) add_i(S[t][f][h], v, ikap[h], e);
                }
        }
    }
}

// Records of one tile of 16 pairs for 16 columns: a wavefront forms the sums of
// the double layer, the hypersingular layer (curl and weak parts) and the single layer in turn on the
// matrix cores (lane l: column l & 15, pairs 4 v + (l >> 4) in accumulator
// element v, see hbem_dense.hip for the instruction's layout), scales them and
// writes the slot's values, or (DIFF) the differences T is formed from, K
// inner - outer, W and V outer - inner (gen_sol_op.cpp:59-74), of the column's
// two slots.
template <int D, bool DIFF, bool NEAR, class K>
__global__ __launch_bounds__(256) void k_band_eval(RadialParams P, const int* __restrict__ recs,
                                                   const BandTile* __restrict__ tiles, int tile0, int ntile,
                                                   const Band* __restrict__ bands, const double* __restrict__ costab,
                                                   const double* __restrict__ tab, const double* __restrict__ ext) {
    constexpr int H = DIFF ? 2 : 1;
    const int lane = threadIdx.x & 63, l16 = lane & 15, lk = lane >> 4;
    const int nkt = (P.ncolg + 15) >> 4;
    const long long w = (long long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (w >= (long long)ntile * nkt) return;  // whole wavefront; the kernel has no barrier
    const int tile = tile0 + (int)(w / nkt), kt = (int)(w % nkt);
    const int ci = kt * 16 + l16, cc = ci < P.ncolg ? ci : P.ncolg - 1;
    const bool act = ci < P.ncolg;
    const BandTile bt = tiles[tile];
    const Band bd = bands[bt.band];
    const int nslots = P.ncolg * H;
    const double* a = tab + bt.off;
    const cdbl* bs = P.basis + (size_t)bd.basis * nslots;
    const cdbl* bl = P.basis + (size_t)P.nbasis * nslots;   // near band, complex kappa
    const double* rj = costab + bd.rad;
    const double* ex = NEAR ? ext + (size_t)tile * 7 * 16 : nullptr;
    const int col = P.cols[cc];
    SlotScale<K> sl[H];
    K ikap[H];                                 // -(2/pi) / kappa
#pragma unroll
    for (int h = 0; h < H; ++h) {
        load_slot(P, col + h * P.nslot2, sl[h]);
        ikap[h] = (-kTwoOverPi) * sl[h].kinv;
    }
    int rec[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) rec[v] = act ? recs[(size_t)tile * 16 + 4 * v + lk] : -1;
    const size_t ncol = P.ncol;
    auto put = [&](int v, int t, int q, const cdbl (&x)[H]) {
        if (rec[v] < 0) return;
        const cdbl y = !DIFF ? x[0] : (q < 2 ? minus(x[0], x[H - 1]) : minus(x[H - 1], x[0]));
        cdbl* o = P.out + ((size_t)rec[v] * (P.nv * (D + 1)) + P.nv * t + q) * ncol + col;
        o[0] = y;
    };
    auto at = [](const Sum4& s, int v) { return mk(s.re[v], s.im[v]); };
    {
        Sum4 S[D + 1][2][H];
        band_sums<D, DIFF, NEAR, K, 0, 2>(a, 0, bs, nslots, cc, P.ncolg + cc, rj, bd.p, ex, ikap, bl, S);
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int f = 0; f < 2; ++f)
#pragma unroll
                for (int t = 0; t <= D; ++t) {
                    cdbl x[H];
#pragma unroll
                    for (int h = 0; h < H; ++h)
                        x[h] = value_K(sl[h], t, at(S[0][f][h], v), at(S[D >= 1 ? 1 : 0][f][h], v), at(S[D][f][h], v));
                    put(v, t, f, x);
                }
    }
    {
        Sum4 S[D + 1][2][H];
        band_sums<D, DIFF, NEAR, K, 1, 2>(a, 2, bs, nslots, cc, P.ncolg + cc, rj, bd.p, ex, ikap, bl, S);
        if (D >= 1 && !NEAR) {
            // the curl part's constant (see k_radial_near)
#pragma unroll
            for (int h = 0; h < H; ++h)
#pragma unroll
                for (int v = 0; v < 4; ++v) add_i(S[D >= 1 ? 1 : 0][0][h], v, ikap[h], -1.0);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int t = 0; t <= D; ++t) {
                cdbl x[H], y[H];
#pragma unroll
                for (int h = 0; h < H; ++h) {
                    y[h] = value_A(sl[h], t, at(S[0][0][h], v), at(S[D >= 1 ? 1 : 0][0][h], v), at(S[D][0][h], v));
                    x[h] = value_W(sl[h], t, at(S[0][1][h], v), at(S[D >= 1 ? 1 : 0][1][h], v), at(S[D][1][h], v));
                }
                put(v, t, 4, y);
                put(v, t, 2, x);
            }
    }
    {
        Sum4 S[D + 1][1][H];
        band_sums<D, DIFF, NEAR, K, 1, 1>(a, 4, bs, nslots, cc, P.ncolg + cc, rj, bd.p, ex, ikap, bl, S);
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int t = 0; t <= D; ++t) {
                cdbl x[H];
#pragma unroll
                for (int h = 0; h < H; ++h)
                    x[h] = value_V(sl[h], t, at(S[0][0][h], v), at(S[D >= 1 ? 1 : 0][0][h], v), at(S[D][0][h], v));
                put(v, t, 3, x);
            }
    }
}

// ---------------------------------------------------------------------------
// Records from local matrices (the node-loop kernels): the local matrices L
// [panel pair][16 (D+1)][lcols].  Group column i: L column i, or (lout > 0) the
// difference of columns i and lout + i.  W is written whole, its curl part zero.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_records_from_locals(const cdbl* __restrict__ L, int lcols, int D, int lout,
                                                             int npairs, const int* __restrict__ cols, int ncolg, int N,
                                                             cdbl* __restrict__ out, int ncol, int nv) {
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= (long long)npairs * ncolg) return;
    const int rec = (int)(id / ncolg), ci = (int)(id - (long long)rec * ncolg);
    int m, n;
    tri_mn(rec, m, n);
    const int nslot = 16 * (D + 1);
    cdbl* o = out + (size_t)rec * (nv * (D + 1)) * ncol + cols[ci];
    for (int t = 0; t <= D; ++t) {
        cdbl e[5][2][2];                       // K(m, n), K(n, m), W, V, V(n, m)
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            const int P = a == 0 ? (m == 0 ? N - 1 : m - 1) : m;
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const int Q = b == 0 ? (n == 0 ? N - 1 : n - 1) : n;
                const bool fwd = P >= Q;
                const cdbl* l = L + ((size_t)(fwd ? tri_ll(P, Q) : tri_ll(Q, P)) * nslot + 16 * t) * lcols + ci;
                // K(n, m) takes the transposed block, or (one panel) entry (b, a)
                const int q = a + 2 * b, qt = b + 2 * a;
                const int sk = fwd ? q : 4 + q, st = P == Q ? qt : (fwd ? 4 + qt : qt);
                const int sw = 8 + (fwd ? q : qt), sv = 12 + (fwd ? q : qt);
                const int slot[5] = {sk, st, sw, sv, P == Q ? 12 + qt : sv};
#pragma unroll
                for (int y = 0; y < 5; ++y) {
                    cdbl v = l[(size_t)slot[y] * lcols];
                    if (lout > 0) {
                        const cdbl w = l[(size_t)slot[y] * lcols + lout];
                        v = y < 2 ? v - w : w - v;
                    }
                    e[y][a][b] = v;
                }
            }
        }
        // (e00 + e11) + (e01 + e10): under (m, n) -> (n, m) the symmetric layers
        // exchange e01 and e10 only
#pragma unroll
        for (int y = 0; y < 5; ++y) {
            const int at = y < 4 ? y : 5;
            if (at < nv) o[(size_t)(nv * t + at) * ncol] = (e[y][0][0] + e[y][1][1]) + (e[y][0][1] + e[y][1][0]);
        }
        o[(size_t)(nv * t + 4) * ncol] = mk(0, 0);
    }
}

// ---------------------------------------------------------------------------
// Consumers of the records
// ---------------------------------------------------------------------------
__device__ __forceinline__ cdbl quarter_i(cdbl v) { return mk(-0.25 * v.y, 0.25 * v.x); }   // * i/4

// W(m, n) of order t and column q from the records: the curl parts of the four
// panel pairs with the signs of the slopes, and the rest
__device__ __forceinline__ cdbl record_W(const cdbl* __restrict__ E, int ncol, int nvd, int t0, int q, int m, int n, int N) {
    const int m1 = m == 0 ? N - 1 : m - 1, n1 = n == 0 ? N - 1 : n - 1;
    auto rec = [&](int i, int j) { return (size_t)(i >= j ? tri_ll(i, j) : tri_ll(j, i)); };
    auto at = [&](size_t r, int v) { return E[(r * nvd + t0 + v) * ncol + q]; };
    const size_t mn = rec(m, n);
    const cdbl a00 = at(rec(m1, n1), 4), a01 = at(rec(m1, n), 4), a10 = at(rec(m, n1), 4), a11 = at(mn, 4);
    const cdbl w = at(mn, 2);
    // symmetric under m <-> n bit for bit: a01 and a10 exchange
    return mk(((a00.x + a11.x) - (a01.x + a10.x)) + w.x, ((a00.y + a11.y) - (a01.y + a10.y)) + w.y);
}

// Builder matrices of column q: out[layer][t] (N x N column-major)
__global__ __launch_bounds__(256) void k_gather_layers(const cdbl* __restrict__ E, int ncol, int nv, int q, int N, int D,
                                                       int layers, cdbl* __restrict__ Kout, cdbl* __restrict__ Wout,
                                                       cdbl* __restrict__ Vout) {
    const long long NN = (long long)N * N;
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= NN * (D + 1)) return;
    const int t = (int)(id / NN);
    const long long e = id - t * NN;
    const int m = (int)(e % N), n = (int)(e / N);
    const size_t rec = (size_t)(m >= n ? tri_ll(m, n) : tri_ll(n, m));
    const cdbl* r = E + (rec * (nv * (D + 1)) + nv * t) * ncol + q;
    if ((layers & 1) && Kout) Kout[id] = quarter_i(r[m >= n ? 0 : (size_t)ncol]);
    if ((layers & 4) && Wout) Wout[id] = quarter_i(record_W(E, ncol, nv * (D + 1), nv * t, q, m, n, N));
    if ((layers & 2) && Vout) Vout[id] = quarter_i(r[(size_t)(m < n && nv == 6 ? 5 : 3) * ncol]);
}

// Transmission matrix (assemble_operator, gen_sol_op.cpp:59-74, unprojected):
// T = [[K_i - K_o + M, V_o - V_i], [W_o - W_i, K_o - K_i + M^T]], M only for t = 0
// (P1: non-zero only for neighbouring hats), from records of differences
// (qo < 0: output b is column b) or of two slots (columns qi, qo; one output).
// T_t of output b is written at Tt + b ld^2.
// Workgroup = one pair of 8 x 8 tiles (I, J), I >= J, for 32 outputs; thread
// (i, jb) = (threadIdx & 7, threadIdx >> 3).  Each layer in turn: the tile's
// records are read (runs over the columns), written to tile (I, J) of T in
// runs of 8 rows, and through LDS to tile (J, I).  A record is read once, 64
// bytes per pair of hats, order and column, against the four local matrices'
// 256 an entry gathered from them takes (polygon2000, 128 k: 8.2 GB read where
// the gather read 66).
template <bool TWO>
__global__ __launch_bounds__(256) void k_form_T(const cdbl* __restrict__ E, int ncol, int nv, int qi, int qo, int nb, int N, int D,
                                                int Dout, const double* __restrict__ M, cdbl* __restrict__ T0,
                                                cdbl* __restrict__ T1, cdbl* __restrict__ T2, int ld,
                                                cflt* __restrict__ T32) {
    __shared__ cdbl sh[8][8][33];              // [column in tile (I, J)][row in tile (I, J)][output]
    const int nbc = (nb + 31) >> 5;
    const int bc = blockIdx.x % nbc, tile = blockIdx.x / nbc;
    int I, J;
    tri_mn(tile, I, J);
    const int i = threadIdx.x & 7, jb = threadIdx.x >> 3;
    const int b = bc * 32 + jb;
    const bool act = b < nb;                   // idle threads still reach every barrier
    const size_t NN = (size_t)ld * ld;
    const int ca = !act ? 0 : (TWO ? qi : b);
    const int m = 8 * I + i, r = 8 * J + i;
    const bool asym = nv == 6;
    auto mass = [&](int x, int y) {
        const int g = x >= y ? x - y : y - x;
        return g <= 1 || g == N - 1 ? M[x + (size_t)y * N] : 0.0;
    };
#pragma unroll 1
    for (int t = 0; t <= Dout; ++t) {
        cdbl* Tt = (t == 0 ? T0 : (t == 1 ? T1 : T2)) + (size_t)(act ? b : 0) * NN;
        // T and, when asked, its FP32 copy for the mixed-precision LU (each
        // entry rounded to nearest) in the same pass
        cflt* Ts = t == 0 && T32 ? T32 + (size_t)(act ? b : 0) * NN : nullptr;
        auto put = [&](size_t idx, cdbl v) {
            Tt[idx] = v;
            if (Ts) Ts[idx] = cflt{(float)v.x, (float)v.y};
        };
        // entry (x, y) of layer lay (0 K, 1 W, 2 V) in its blocks of T
        auto store = [&](int lay, int x, int y, cdbl v) {
            if (lay == 0) {
                cdbl k00 = v, k11 = mk(-v.x, -v.y);
                if (t == 0) {
                    k00.x += mass(x, y);
                    k11.x += mass(y, x);
                }
                put(x + (size_t)y * ld, k00);
                put((x + N) + (size_t)(y + N) * ld, k11);
            } else if (lay == 1) {
                put((x + N) + (size_t)y * ld, v);
            } else {
                put(x + (size_t)(y + N) * ld, v);
            }
        };
#pragma unroll 1
        for (int lay = 0; lay < 3; ++lay) {
            const bool two = lay == 0 || (lay == 2 && asym);
#pragma unroll 1
            for (int c0 = 0; c0 < 8; c0 += 4) {
                cdbl a[4], bt[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int n = 8 * J + c0 + c;
                    const bool in = act && m < N && n < N, low = m >= n;
                    const size_t rec = !in ? 0 : (size_t)(low ? tri_ll(m, n) : tri_ll(n, m));
                    const cdbl* e = E + (rec * (nv * (D + 1)) + nv * t) * ncol;
                    // entry (m, n), and entry (n, m) where it is not the same
                    const size_t s0 = (size_t)(lay == 0 ? (low ? 0 : 1) : (asym && !low ? 5 : 3)) * ncol;
                    const size_t s1 = (size_t)(lay == 0 ? (low ? 1 : 0) : (low ? 5 : 3)) * ncol;
                    if (lay == 1) {
                        a[c] = record_W(E, ncol, nv * (D + 1), nv * t, ca, in ? m : 0, in ? n : 0, N);
                        if (TWO) a[c] = record_W(E, ncol, nv * (D + 1), nv * t, qo, in ? m : 0, in ? n : 0, N) - a[c];
                        continue;
                    }
                    a[c] = e[s0 + ca];
                    if (two) bt[c] = e[s1 + ca];
                    if (TWO) {
                        const cdbl vo = e[s0 + qo];
                        a[c] = lay == 0 ? a[c] - vo : vo - a[c];
                        if (two) bt[c] = lay == 0 ? bt[c] - e[s1 + qo] : e[s1 + qo] - bt[c];
                    }
                }
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int n = 8 * J + c0 + c;
                    const cdbl v = quarter_i(a[c]);
                    if (I != J) sh[c0 + c][i][jb] = two ? quarter_i(bt[c]) : v;
                    if (act && m < N && n < N) store(lay, m, n, v);
                }
            }
            if (I == J) continue;
            __syncthreads();
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const int col = 8 * I + c;
                if (act && r < N && col < N) store(lay, r, col, sh[i][c][jb]);
            }
            __syncthreads();                   // the next layer overwrites sh
        }
    }
}

// Right-hand-side operator of the transmission solve (tp::direct_second_kind::
// A_rhs, solvers.cpp:116-122) from the outer operators of column o:
// A_o = [[-K_o + M/2, V_o], [W_o, K_o^T + M/2]] (2N x 2N, column-major).
// One thread per (m, n) writes the four block entries.
__global__ __launch_bounds__(256) void k_form_Ao(const cdbl* __restrict__ E, int ncol, int o, int N,
                                                 const double* __restrict__ M, cdbl* __restrict__ A) {
    const long long id = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= (long long)N * N) return;
    const int m = (int)(id % N), n = (int)(id / N);
    const size_t n2 = 2 * (size_t)N;
    const double hm = 0.5 * M[m + (size_t)n * N];
    const bool low = m >= n;
    const cdbl* e = E + (size_t)(low ? tri_ll(m, n) : tri_ll(n, m)) * kRecValues * ncol + o;
    const cdbl Ko = quarter_i(e[low ? 0 : (size_t)ncol]), KoT = quarter_i(e[low ? (size_t)ncol : 0]);
    A[m + (size_t)n * n2] = mk(-Ko.x + hm, -Ko.y);
    A[m + (size_t)(n + N) * n2] = quarter_i(e[3 * (size_t)ncol]);
    A[(m + N) + (size_t)n * n2] = quarter_i(record_W(E, ncol, kRecValues, 0, o, m, n, N));
    A[(m + N) + (size_t)(n + N) * n2] = mk(KoT.x + hm, KoT.y);
}

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------
static unsigned grid_of(long long n, int per = 256) { return (unsigned)((n + per - 1) / per); }

// Points of a band for kappa <= kmax.  Far: the coefficients of the radial
// functions on [c - a, c + a] fall like M(rho) rho^-p for every Bernstein
// ellipse rho inside the singularity's, rho0 = q + sqrt(q^2 - 1), q = c / a,
// where they grow at most like M = exp(kappa a (rho - 1 / rho) / 2) (with a
// factor 4 p next to the singularity); p is the least multiple of 4 for which
// the best such bound is below tol.  Near: the same for functions entire in
// r^2 on [0, a^2], whose ellipse is sigma^2 in r^2 for sigma in r, one point
// more for the factor r^2 of the k-derivatives.
int band_order(double c, double a, double kmax, double tol, bool near) {
    const double ka = kmax * a, q = c / a;
    const double rho0 = near ? 1e300 : q + std::sqrt(q * q - 1.0);
    for (int p = 8; p <= kBandMaxP; p += 4) {
        const double m = near ? 2.0 * (p - 1) : p;
        const double t = m / ka, ro = t + std::sqrt(t * t + 1.0);
        const double rho = std::min(ro, rho0);
        double e = 0.5 * ka * (rho - 1.0 / rho) - m * std::log(rho);
        if (rho == rho0) e += std::log(4.0 * p);
        if (e <= std::log(tol)) return p;
    }
    return 0;
}

void launch_radial_band(const double* gtab, int N, int ns, int npairs, double R, double first, double step, double width,
                        unsigned short* band, hipStream_t st) {
    hipLaunchKernelGGL(k_radial_band, dim3(grid_of(4LL * npairs)), dim3(256), 0, st, gtab, N, ns, npairs, R, first, step,
                       width, band);
}

void launch_radial_flags(const double* gtab, int ns, int npairs, unsigned char* flags, hipStream_t st) {
    hipLaunchKernelGGL(k_radial_flags, dim3(grid_of(npairs)), dim3(256), 0, st, gtab, ns, npairs, flags);
}

constexpr int kFarFewTiles = 512;
void launch_radial_far(const int* recs, const BandTile* tiles, int tile0, int ntile, const Band* bands, int pmax,
                       const double* gtab, const double* xg, const double* wg, int N, int ns, const unsigned char* flags,
                       const double* costab, double* tab, hipStream_t st) {
    if (ntile <= 0) return;
    const auto run = [&](auto kernel, int lanes) {
        const int pairs = 128 / lanes;
        hipLaunchKernelGGL(kernel, dim3((unsigned)ntile * (16 / pairs)), dim3(128), pairs * pmax * 5 * sizeof(double), st, recs,
                           tiles, tile0, bands, gtab, xg, wg, N, ns, flags, costab, tab, pmax);
    };
    // Up to two wavefronts a SIMD with 16 lanes a pair, 64 lanes shorten the chain of a
    // pair's nodes (us, 16 -> 64 lanes, order 11): 48 panels, kappa d = 4.5 128 -> 53; 64
    // panels, 0.5 82 -> 31; 100 panels 85 -> 63; 140 panels (over 600 tiles) 112 -> 117,
    // where the sums over more lanes only cost.
    if (ntile <= kFarFewTiles) run(k_radial_far<64>, 64);
    else run(k_radial_far<16>, 16);
}

void launch_radial_moments(int cls, const int* ent, int cnt, const double* panels, const double* coefs, const double* xc,
                           const double* wc, int nc, double R, double iS, const double* pts, int p, double* mom,
                           double* ext, hipStream_t st) {
    if (cnt <= 0) return;
    const dim3 g((unsigned)cnt, cls == 1 ? 2 : 1, (unsigned)((p + kMomQ - 1) / kMomQ));
    if (cls == 1)
        hipLaunchKernelGGL(k_radial_moments<1>, g, dim3(256), 0, st, ent, panels, coefs, xc, wc, nc, R, iS, pts, p,
                           mom, ext);
    else
        hipLaunchKernelGGL(k_radial_moments<0>, g, dim3(256), 0, st, ent, panels, coefs, xc, wc, nc, R, iS, pts, p,
                           mom, ext);
}

void launch_radial_near(const RadialNear* ent, int nent, const BandTile* tiles, const Band* bands, int p,
                        const double* gtab, const double* xg, const double* wg, int N, int ns, const unsigned char* flags,
                        const double* mom_c, const double* ext_c, const double* mom_a, const double* ext_a,
                        const double* costab, double iS, double curl_s, double curl_g, double* tab, double* ext,
                        hipStream_t st) {
    if (nent <= 0) return;
    // the nodes' products and logarithms are kept in LDS from the first points on
    // where two wavefronts' fit in 64 KB (orders up to 20)
    const size_t mu = (size_t)p * 10, nodes = (size_t)4 * ns * ns;
    const int cache = 2 * (mu + 2 * nodes) * sizeof(double) <= 65536 ? (int)nodes : 0;
    hipLaunchKernelGGL(k_radial_near, dim3((unsigned)((nent + 15) / 16 * 8)), dim3(128),
                       2 * (mu + 2 * cache) * sizeof(double), st, ent, nent, tiles, bands, gtab, xg, wg, N, ns, flags, mom_c,
                       ext_c, mom_a, ext_a, costab, iS, curl_s, curl_g, tab, ext, p, cache);
}

void launch_band_basis(const RadialParams& P, bool diff, const Band* bands, int nbands, int pmax, const double* costab,
                       hipStream_t st) {
    if (nbands <= 0 || P.ncolg <= 0) return;
    const int nslots = P.ncolg * (diff ? 2 : 1);
    hipLaunchKernelGGL(k_band_basis, dim3(grid_of((long long)pmax * nslots), (unsigned)nbands), dim3(256), 0, st, P, bands,
                       costab, nslots);
}

template <int D, bool DIFF, bool NEAR, class K>
static void band_eval(const RadialParams& P, const int* recs, const BandTile* tiles, int tile0, int ntile,
                      const Band* bands, const double* costab, const double* tab, const double* ext, hipStream_t st) {
    const long long waves = (long long)ntile * ((P.ncolg + 15) / 16);
    if (waves <= 0) return;
    hipLaunchKernelGGL((k_band_eval<D, DIFF, NEAR, K>), dim3(grid_of(waves, 4)), dim3(256), 0, st, P, recs, tiles, tile0,
                       ntile, bands, costab, tab, ext);
}
template <int D, bool DIFF>
static void band_eval_d(const RadialParams& P, bool near, const int* recs, const BandTile* tiles, int tile0, int ntile,
                        const Band* bands, const double* costab, const double* tab, const double* ext, hipStream_t st) {
    if (P.kapi && near) band_eval<D, DIFF, true, cdbl>(P, recs, tiles, tile0, ntile, bands, costab, tab, ext, st);
    else if (P.kapi) band_eval<D, DIFF, false, cdbl>(P, recs, tiles, tile0, ntile, bands, costab, tab, ext, st);
    else if (near) band_eval<D, DIFF, true, double>(P, recs, tiles, tile0, ntile, bands, costab, tab, ext, st);
    else band_eval<D, DIFF, false, double>(P, recs, tiles, tile0, ntile, bands, costab, tab, ext, st);
}

void launch_band_eval(int D, bool diff, bool near, const RadialParams& P, const int* recs, const BandTile* tiles, int tile0,
                      int ntile, const Band* bands, const double* costab, const double* tab, const double* ext,
                      hipStream_t st) {
    if (diff) {
        if (D == 0) band_eval_d<0, true>(P, near, recs, tiles, tile0, ntile, bands, costab, tab, ext, st);
        else if (D == 1) band_eval_d<1, true>(P, near, recs, tiles, tile0, ntile, bands, costab, tab, ext, st);
        else band_eval_d<2, true>(P, near, recs, tiles, tile0, ntile, bands, costab, tab, ext, st);
    } else {
        if (D == 0) band_eval_d<0, false>(P, near, recs, tiles, tile0, ntile, bands, costab, tab, ext, st);
        else if (D == 1) band_eval_d<1, false>(P, near, recs, tiles, tile0, ntile, bands, costab, tab, ext, st);
        else band_eval_d<2, false>(P, near, recs, tiles, tile0, ntile, bands, costab, tab, ext, st);
    }
}

void launch_records_from_locals(const cdbl* L, int lcols, int D, int lout, int npairs, const int* cols, int ncolg, int N,
                                cdbl* out, int ncol, int nv, hipStream_t st) {
    const long long n = (long long)npairs * ncolg;
    if (n <= 0) return;
    hipLaunchKernelGGL(k_records_from_locals, dim3(grid_of(n)), dim3(256), 0, st, L, lcols, D, lout, npairs, cols, ncolg, N,
                       out, ncol, nv);
}

void launch_gather_layers(const cdbl* E, int ncol, int nv, int q, int N, int D, int layers, cdbl* K, cdbl* W, cdbl* V,
                          hipStream_t st) {
    const long long n = (long long)N * N * (D + 1);
    hipLaunchKernelGGL(k_gather_layers, dim3(grid_of(n)), dim3(256), 0, st, E, ncol, nv, q, N, D, layers, K, W, V);
}

void launch_form_T(const cdbl* E, int ncol, int nv, int qi, int qo, int nb, int N, int D, const double* M, cdbl* T0, cdbl* T1,
                   cdbl* T2, hipStream_t st, int ld, cflt* T32, bool only0) {
    const unsigned mt = (unsigned)((N + 7) / 8);
    const dim3 grid(mt * (mt + 1) / 2 * (unsigned)((nb + 31) / 32));
    if (ld <= 0) ld = 2 * N;
    if (qo < 0)
        hipLaunchKernelGGL(k_form_T<false>, grid, dim3(256), 0, st, E, ncol, nv, qi, qo, nb, N, D, only0 ? 0 : D, M, T0, T1,
                           T2, ld, T32);
    else
        hipLaunchKernelGGL(k_form_T<true>, grid, dim3(256), 0, st, E, ncol, nv, qi, qo, nb, N, D, only0 ? 0 : D, M, T0, T1,
                           T2, ld, T32);
}

void launch_form_Ao(const cdbl* E, int ncol, int o, int N, const double* M, cdbl* A, hipStream_t st) {
    const long long n = (long long)N * N;
    if (n <= 0) return;
    hipLaunchKernelGGL(k_form_Ao, dim3(grid_of(n)), dim3(256), 0, st, E, ncol, o, N, M, A);
}

}  // namespace hbem
