// hbem_capi.hip -- geometry contexts and the C-ABI of include/hbem.h.
#include <algorithm>
#include <array>
#include <cmath>
#include <complex>
#include <cstdlib>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/hbem.h"
#include "hbem_internal.hpp"

using hbem::cdbl;
using hbem::cflt;

namespace {

thread_local std::string g_err;
int g_device = 0;

struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

void hip_check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw Error(HBEM_EDEVICE, std::string(what) + ": " + hipGetErrorString(e));
}
#define HIPC(x) hip_check((x), #x)

// Growable device buffer.
struct DBuf {
    void* p = nullptr;
    size_t n = 0;
    void* get(size_t bytes) {
        if (bytes > n) {
            if (p) (void)hipFree(p);
            p = nullptr;
            n = 0;
            if (bytes > 0) {
                if (hipMalloc(&p, bytes) != hipSuccess) { p = nullptr; throw Error(HBEM_ENOMEM, "device allocation failed"); }
            }
            n = bytes;
        }
        return p;
    }
    template <class T> T* as(size_t count) { return (T*)get(count * sizeof(T)); }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        n = 0;
    }
    ~DBuf() { release(); }
};

template <class T>
T* upload(DBuf& b, const std::vector<T>& v, hipStream_t st) {
    T* d = b.as<T>(std::max<size_t>(v.size(), 1));
    if (!v.empty()) HIPC(hipMemcpyAsync(d, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, st));
    return d;
}

constexpr size_t al256(size_t b) { return (b + 255) & ~(size_t)255; }

// Several host arrays laid out for one upload, each 256-byte aligned.
struct Packed {
    std::vector<char> bytes;
    template <class T> size_t add(const std::vector<T>& v) {
        const size_t at = al256(bytes.size());
        bytes.resize(at + v.size() * sizeof(T) + 8);
        if (!v.empty()) std::memcpy(bytes.data() + at, v.data(), v.size() * sizeof(T));
        return at;
    }
};

// Real sparse n x n matrix in compressed-row form on the device.
struct DCsr {
    DBuf rp, ci, v;
    // rows of op(A) for a dense column-major A (op = A or A^T); exact zeros are dropped
    void build(const std::vector<double>& A, int n, bool trans, hipStream_t st) {
        std::vector<int> r(n + 1, 0), c;
        std::vector<double> x;
        for (int i = 0; i < n; ++i) {
            for (int j = 0; j < n; ++j) {
                const double a = trans ? A[j + (size_t)i * n] : A[i + (size_t)j * n];
                if (a != 0.0) { c.push_back(j); x.push_back(a); }
            }
            r[i + 1] = (int)c.size();
        }
        upload(rp, r, st);
        upload(ci, c, st);
        upload(v, x, st);
    }
};

// The same rows in slices of 64 of similar length, entries [k][64] (zero-padded).
struct DSell {
    DBuf mem;
    const int *rows = nullptr, *off = nullptr, *col = nullptr;
    const double* val = nullptr;
    void build(const std::vector<double>& A, int n, hipStream_t st) {
        std::vector<std::vector<std::pair<int, double>>> r(n);
        for (int j = 0; j < n; ++j)
            for (int i = 0; i < n; ++i)
                if (A[i + (size_t)j * n] != 0.0) r[i].emplace_back(j, A[i + (size_t)j * n]);
        std::vector<int> ord(n), o(1, 0), c;
        std::vector<double> v;
        for (int i = 0; i < n; ++i) ord[i] = i;
        std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) { return r[a].size() > r[b].size(); });
        for (int s = 0; s < n; s += 64) {
            const size_t w = r[ord[s]].size();
            for (size_t k = 0; k < w; ++k)
                for (int l = 0; l < 64; ++l) {
                    // (a shorter row repeats its last column with a zero)
                    const auto& row = r[ord[std::min(s + l, n - 1)]];
                    const bool in = s + l < n && k < row.size();
                    c.push_back(row.empty() ? 0 : row[std::min(k, row.size() - 1)].first);
                    v.push_back(in ? row[k].second : 0.0);
                }
            o.push_back((int)c.size());
        }
        Packed pk;
        const size_t a = pk.add(ord), b = pk.add(o), d = pk.add(c), e = pk.add(v);
        char* p = (char*)mem.get(pk.bytes.size());
        HIPC(hipMemcpyAsync(p, pk.bytes.data(), pk.bytes.size(), hipMemcpyHostToDevice, st));
        HIPC(hipStreamSynchronize(st));       // the upload reads a host vector
        rows = (const int*)(p + a);
        off = (const int*)(p + b);
        col = (const int*)(p + d);
        val = (const double*)(p + e);
    }
};

// Algorithmic FP64 flops per node (frozen model): Hankel node (13 geometry + 171
// Bessel) and accumulation for P1 x P1, three layers, derivative order d.
double flops_per_node(int d) { return 184.0 + (d == 0 ? 108.0 : d == 1 ? 192.0 : 314.0); }

// Timed sections on a stream.  begin/end record a pair of events around
// device work; nothing waits for them until resolve(), which the caller runs
// after the timed work (so timing does not add host synchronisations to it).
struct EventLog {
    static constexpr int kSlots = 8;
    struct Rec { int slot; hipEvent_t a, b; double flops; };
    std::vector<Rec> pending;
    std::vector<hipEvent_t> pool;
    double ms[kSlots] = {};
    long long n[kSlots] = {};
    double flops[kSlots] = {};
    hipEvent_t take() {
        if (!pool.empty()) { hipEvent_t e = pool.back(); pool.pop_back(); return e; }
        hipEvent_t e = nullptr;
        HIPC(hipEventCreate(&e));
        return e;
    }
    hipEvent_t begin(hipStream_t st) {
        hipEvent_t e = take();
        HIPC(hipEventRecord(e, st));
        return e;
    }
    void end(hipStream_t st, int slot, hipEvent_t a, double fl = 0.0) {
        hipEvent_t b = take();
        HIPC(hipEventRecord(b, st));
        pending.push_back({slot, a, b, fl});
    }
    void resolve() {
        for (auto& r : pending) {
            HIPC(hipEventSynchronize(r.b));
            float t = 0.f;
            HIPC(hipEventElapsedTime(&t, r.a, r.b));
            ms[r.slot] += t;
            n[r.slot] += 1;
            flops[r.slot] += r.flops;
            pool.push_back(r.a);
            pool.push_back(r.b);
        }
        pending.clear();
    }
    void reset() {
        resolve();
        for (int i = 0; i < kSlots; ++i) { ms[i] = 0; n[i] = 0; flops[i] = 0; }
    }
    ~EventLog() {
        for (auto& r : pending) { (void)hipEventDestroy(r.a); (void)hipEventDestroy(r.b); }
        for (auto e : pool) (void)hipEventDestroy(e);
    }
};

// The LU's matrix-core launches recorded into an event log slot
struct GemmTimer : hbem::LaunchTimer {
    EventLog* log;
    int slot;
    hipEvent_t e = nullptr;
    GemmTimer(EventLog* l, int s) : log(l), slot(s) {}
    void begin(hipStream_t st) override { e = log->begin(st); }
    void end(hipStream_t st, double flops) override { log->end(st, slot, e, flops); }
};

// Profile slots of a geometry context (hbem_profile_query)
enum { kProfGeneral = 0, kProfAdjacent = 1, kProfCoinciding = 2, kProfLU = 3, kProfFormT = 4, kProfRsvd = 5,
       kProfGemm = 6 };
// randomized_svd timer slots (randsvd.cpp:27-47): LU, first solve + QR, subspace iterations, last solve + SVD
enum { kTimLU = 0, kTimQR = 1, kTimIter = 2, kTimSVD = 3 };

// Number of node chunks of the paired-lane kernel per singular pair (chunks of
// 2048 nodes; adjacent pairs chunk each of their two node halves on its own).
constexpr int kChunkNodes = 2048;
long long adj_chunks(int nc) { return 2 * (((long long)nc * nc + kChunkNodes - 1) / kChunkNodes); }
long long coi_chunks(int nc) { return ((long long)nc * nc + kChunkNodes - 1) / kChunkNodes; }

// Device bytes a sigma sweep needs per wavenumber of a batch: on the node loops
// the local matrices and chunk partials (lcols columns per k: 1 in the
// T-difference layout, 2 for the two refraction indices otherwise); T
// (factorised in place), T', T'', pivots and the thin blocks of the randomized SVD.
size_t locals_bytes_per_k(long long npairs, long long nadj, long long ncoi, int nc_rule, int D, int lcols) {
    const size_t nslot = 16 * (size_t)(D + 1);
    const size_t part = (size_t)std::max(nadj * adj_chunks(nc_rule), ncoi * coi_chunks(nc_rule));
    return (size_t)lcols * ((size_t)npairs + part) * nslot * sizeof(cdbl);
}
size_t dense_bytes_per_k(int n, int D, int ncols) {
    const size_t nn = (size_t)n * n;
    return (size_t)(D + 1) * nn * sizeof(cdbl) + 2 * (size_t)n * sizeof(int) + (4 * (size_t)ncols + 4) * n * sizeof(cdbl) +
           64;
}

// Sweeps of >= 32 real positive wavenumbers run every batch on the paired-lane
// kernel in the T-difference layout (AsmParams::tdiff), so a k's bits do not
// depend on the batch size the free memory allows.
bool sweep_tdiff(const double* ks, int nk) {
    bool allpos = nk >= 32;
    for (int j = 0; j < nk && allpos; ++j) allpos = ks[j] > 0.0;
    return allpos;
}

// Extra device bytes per wavenumber of the sigma'' stage: T_p, the bordered
// 2n x 2n matrix (which is also the projection's scratch), its pivots and
// the 2n-vectors of the two solves.
size_t der2_bytes_per_k(int n) {
    const size_t nn = (size_t)n * n;
    return 5 * nn * sizeof(cdbl) + 4 * (size_t)n * sizeof(int) + 16 * (size_t)n * sizeof(cdbl) + 64;
}

// Extra device bytes per wavenumber of the mixed-precision dense stage: the
// FP32 copy of T (factorised in place) and the refinement's thin blocks.
size_t mixed_bytes_per_k(int n, int ncols) {
    return (size_t)n * n * sizeof(cflt) + (2 * (size_t)ncols * n + hbem::residual_part_count(n, ncols, 1)) * sizeof(cdbl) +
           64;
}

// Refinement tolerance of the mixed-precision sweep: a k is recomputed in FP64
// when the estimated error left after a refined solve (the last correction
// times the observed contraction rate) exceeds this fraction of the solution.
constexpr double kMixedTol = 1e-10;

// Wavenumbers per sweep batch: as many as fit in `avail` bytes, at most 256
// (the dense stage then has about one matrix per CU; more only adds latency),
// and balanced so the batches of nk wavenumbers have equal sizes.
int sweep_batch(size_t per_k, size_t avail, int nk) {
    long long B = (long long)(avail / std::max<size_t>(per_k, 1));
    if (B > 256) B = 256;
    if (B < 1) B = 1;
    if (nk > 0) {
        const long long nbatch = (nk + B - 1) / B;
        B = (nk + nbatch - 1) / nbatch;
    }
    return (int)B;
}

// Work space of hbem_rsvd_sv_noalloc: a fixed device array, one per GPU (the
// runtime instantiates file-scope device variables on every device the
// library runs on, each at its own address).  Layout for order n <= kNaMaxN
// and nc <= kNaMaxCols columns, each part 256-byte aligned: the LU copy of T
// (n^2 complex), pivots, permutation (n ints each), X, Y (n nc complex each),
// thin-solve work (2 n nc complex).
constexpr int kNaMaxN = 2048;
constexpr int kNaMaxCols = 8;
constexpr size_t kNaBytes = al256(sizeof(cdbl) * (size_t)kNaMaxN * kNaMaxN) + 2 * al256(sizeof(int) * (size_t)kNaMaxN) +
                            4 * al256(sizeof(cdbl) * (size_t)kNaMaxN * kNaMaxCols);
static __device__ __align__(256) unsigned char scratch[kNaBytes];

// Device address of `scratch` on device `dev` (which must be current): the
// array's name is a host-side stand-in, so its address is looked up once per
// device and only that address is given to copies and kernels.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
void* scratch_on(int dev) {
    if (dev < 0 || dev >= kMaxDevices) throw Error(HBEM_EDEVICE, "device index beyond the library's table");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        HIPC(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) throw Error(HBEM_EDEVICE, "no device address for the work array");
        g_scratch_ptr[dev] = p;
    }
    return g_scratch_ptr[dev];
}

// Free device memory usable by a call that may regrow buffers currently
// holding `held` bytes, less a reserve of 2 GiB or 3% of the device.
size_t usable_device_bytes(size_t held) {
    size_t fr = 0, tot = 0;
    HIPC(hipMemGetInfo(&fr, &tot));
    const size_t reserve = std::max<size_t>((size_t)2 << 30, tot / 32);
    const size_t have = fr + held;
    return have > reserve ? have - reserve : 0;
}

}  // namespace

// Work space of an assembly call: the slots' tables and column lists ...
struct RecBufs {
    DBuf tab;                                    // slots and columns, one upload
};
// ... and what the groups use in turn
struct RecScratch {
    DBuf E, L, part;                             // E: the records, then a group's basis
};

struct hbem_geometry {
    int dev = 0;
    hipStream_t st = nullptr;
    int N = 0, order = 0, ns = 0, nc = 0, flags = 0;
    bool lines = true, straight = true, proj = true;   // straight: line and arc panels only
    long long npairs = 0;
    std::vector<double> panels, coefs, xg, wg, xc, wc;
    std::vector<double> M, F, Finv;
    std::vector<int> tr;
    // device geometry
    DBuf d_panels, d_coefs, d_xg, d_wg, d_xc, d_wc, d_gtab;
    std::vector<int> aent;                 // adjacent panel pairs (i, j, swap), i > j
    double dmax = 0.0;                     // largest diameter of a panel's bounding disc
    // Panel pairs by class (coinciding, adjacent, general) with their node tables,
    // for the node-loop kernels; built on first use.
    struct Loops {
        bool built = false;
        int cnt[3] = {0, 0, 0};
        DBuf ent[3], pidx[3], flags[3], ngeo[3];
    } loops;
    // Radial functionals (hbem_radial.hip): the pairs of hats by distance band,
    // and per tier of kappa dmax the bands' points and coefficient tables.
    struct Tier {
        bool built = false;
        int pmax = 0, pnear = 0, basis = 0;   // most points of a band; the near band's; basis records per slot
        double points = 0.0;               // points summed over the far pairs
        DBuf mem;                          // bands, tiles, transforms; coefficients; extra sums
        const hbem::Band* bands = nullptr;
        const hbem::BandTile* tiles = nullptr;
        const double *costab = nullptr, *tab = nullptr, *ext = nullptr;
    };
    static constexpr int kTiers = 6, kFarTiers = kTiers;   // then the same edges at the separated pairs' tolerance
    struct Radial {
        bool usable = false;
        int nbands = 0, ntile = 0, ntile_near = 0;
        long long nfar = 0;
        double R = 0.0, first = 0.0, step = 0.0, width = 0.0;
        std::vector<hbem::RadialNear> near;
        std::vector<int> tile_band;
        DBuf plan, flagmem;                // near pairs, tiles' pairs; bands, skip flags
        const unsigned char* flags = nullptr;
        const hbem::RadialNear* d_near = nullptr;
        const int* recs = nullptr;
        Tier tier[kTiers + kFarTiers];
    };
    std::unique_ptr<Radial> rad;           // null until it is complete
    DBuf d_M;
    DCsr s_F, s_FT, s_FinvT, s_Finv;   // F, F^T, Finv^T and Finv of the projection
    DSell l_Finv;                      // Finv once more, in slices
    // work space
    DBuf w_Ao, w_U, w_rhs, w_flag;
    DBuf w_Tp, w_B, w_mv, w_bpiv, w_bperm, w_bvec, w_d2;   // bordered system of sv_der2 (sweeps)
    DBuf w_T32, w_rb, w_rr, w_rpart, w_flag2, w_rprev;       // mixed-precision dense stage
    DBuf w_T0, w_T1, w_T2, w_piv, w_perm, w_X, w_Y, w_work, w_R, w_u, w_v, w_a, w_b, w_sig, w_dsig, w_tmp, w_out;
    RecBufs w_rec;
    RecScratch w_scr;
    // profiling (hbem_profile_enable / query)
    bool prof = false;
    EventLog plog;
    std::mutex mu;
    // bytes held by the per-batch work buffers of the sweep
    size_t work_held() const {
        const DBuf* bs[] = {&w_scr.E, &w_scr.L, &w_scr.part, &w_T0, &w_T1, &w_T2, &w_piv, &w_perm, &w_X, &w_Y, &w_work, &w_u, &w_v, &w_a, &w_b,
                            &w_Tp, &w_B, &w_bpiv, &w_bperm, &w_bvec, &w_T32, &w_rb, &w_rr, &w_rpart, &w_rprev};
        size_t s = 0;
        for (auto* b : bs) s += b->n;
        return s;
    }
};

// drops the multi-instance graphs that name g (defined with the multi-instance sweep)
void multi_forget(hbem_geometry* g);

namespace {

int fail(const std::exception& e) {
    g_err = e.what();
    if (auto* he = dynamic_cast<const Error*>(&e)) return he->code;
    return HBEM_EINVAL;
}

#define API_BEGIN try {
#define API_END \
    }                                              \
    catch (const std::exception& e) { return fail(e); } \
    return HBEM_OK;

// GalerkinBuilder::initialize_constants' validation (galerkin_builder.cpp:899-916)
void check_k(double k_re, double k_im, double c) {
    if (c < 1.0) throw Error(HBEM_EINVAL, "Refraction index must not be smaller than 1");
    if (k_im < 0.0)
        throw Error(HBEM_EINVAL, "Wavenumber does not meet conditions for uniqueness of the solution (Im(k) >= 0)");
    if (!std::isfinite(k_re) || !std::isfinite(k_im)) throw Error(HBEM_EINVAL, "wavenumber must be finite");
}

// k_rp of initialize_constants: the real Hankel path
bool real_positive(double k_re, double k_im) { return k_im == 0.0 && k_re > 0.0; }

// ---------------------------------------------------------------------------
// Pairs of hats by distance band, and the bands' tables per tier of kappa dmax
// ---------------------------------------------------------------------------
// Upper edges of kappa dmax.  A tier serves every kappa up to its edge, so each
// doubling of the mesh width in wavelengths adds points to the bands (0.625, ten
// panels a wavelength: 20 points, 2.5: 32, 20: 108); beyond the last edge, where
// no rule resolves the panels, the node loops take over.
constexpr double kTierEdge[hbem_geometry::kTiers] = {0.625, 1.25, 2.5, 5.0, 10.0, 20.0};
// Interpolation error of the far bands relative to the radial function, and of
// separated line and arc panels on contexts with HBEM_FLAG_FAR_FIELD at real positive
// wavenumbers (up to kappa dmax = 5: half of the flag's 1e-13).
constexpr double kBandTol = 1e-16, kBandTolFar = 5e-14, kNearTol = 1e-17;
// Near radius, band step and largest interval width in units of dmax.  A hat's
// support is at most 2 dmax wide, so a pair's distances spread over 4 dmax at
// most; R = 10 puts the first far band at c / a = 3 (24 points at the first
// tier, 20 from c / a = 5 on), and step 2 makes the bands half as wide again as
// the widest interval.
constexpr double kNearRadius = 10.0, kBandStep = 2.0, kBandWidth = 4.0;

int tier_of(double kd) {
    if (!(kd > 0.0)) return -1;
    for (int t = 0; t < hbem_geometry::kTiers; ++t)
        if (kd <= kTierEdge[t]) return t;
    return -1;
}

int class_nodes(const hbem_geometry* g, int cls) {
    return cls == 2 ? g->ns * g->ns : (cls == 1 ? 2 * g->nc * g->nc : g->nc * g->nc);
}

long long tri_index(int i, int j) { return i >= j ? (long long)i * (i + 1) / 2 + j : (long long)j * (j + 1) / 2 + i; }

// Bands and tiles of the geometry (independent of kappa), built on first use; not
// usable with fewer than 8 panels or where consecutive panels lie so far apart that
// a pair of hats leaves its band (hbem_radial.hip).
hbem_geometry::Radial& radial_base(hbem_geometry* g) {
    if (g->rad) return *g->rad;
    // (an allocation that fails on the way leaves the context without a plan)
    auto plan_ptr = std::make_unique<hbem_geometry::Radial>();
    auto& r = *plan_ptr;
    auto done = [&]() -> hbem_geometry::Radial& { return *(g->rad = std::move(plan_ptr)); };
    const int N = g->N;
    // too few panels for disjoint supports: the node loops
    if (N < 8 || g->npairs > 0x7fffffffLL || !(g->dmax > 0.0)) return done();
    r.R = kNearRadius * g->dmax;
    r.width = kBandWidth * g->dmax * (1.0 + 1e-12);
    r.step = kBandStep * g->dmax;
    r.first = r.R - r.width;
    // pairs of hats over a coinciding or adjacent panel pair
    std::vector<unsigned short> band((size_t)g->npairs, 0);
    std::vector<std::vector<std::pair<int, int>>> adj(N);      // adjacent lower-numbered panels, their entries
    auto touch = [&](int P, int Q) {
        for (int a = 0; a < 2; ++a)
            for (int b = 0; b < 2; ++b) band[tri_index((P + a) % N, (Q + b) % N)] = 1;
    };
    for (int P = 0; P < N; ++P) touch(P, P);
    for (size_t e = 0; e < g->aent.size(); e += 3) {
        touch(g->aent[e], g->aent[e + 1]);
        adj[std::max(g->aent[e], g->aent[e + 1])].emplace_back(std::min(g->aent[e], g->aent[e + 1]), (int)(e / 3));
    }
    // bands and skip flags in one buffer
    const size_t obf = al256(band.size() * sizeof(band[0]));
    unsigned short* db = (unsigned short*)r.flagmem.get(obf + g->npairs);
    HIPC(hipMemcpyAsync(db, band.data(), band.size() * sizeof(band[0]), hipMemcpyHostToDevice, g->st));
    hbem::launch_radial_band((const double*)g->d_gtab.p, N, g->ns, (int)g->npairs, r.R, r.first, r.step, r.width, db,
                             g->st);
    unsigned char* fl = (unsigned char*)db + obf;
    r.flags = fl;
    HIPC(hipMemcpyAsync(band.data(), db, band.size() * sizeof(band[0]), hipMemcpyDeviceToHost, g->st));
    HIPC(hipStreamSynchronize(g->st));
    hbem::launch_radial_flags((const double*)g->d_gtab.p, g->ns, (int)g->npairs, fl, g->st);
    HIPC(hipGetLastError());
    int top = 0;
    for (unsigned short b : band) top = std::max<int>(top, b);
    if (top == hbem::kBandOutside) {
        // panels that do not follow one another: every call of this context takes
        // the node loops, which sum each panel pair by itself
        HIPC(hipStreamSynchronize(g->st));
        r.flagmem.release();
        return done();
    }
    r.nbands = top + 1;
    // tiles of 16 pairs, band by band (the last of a band padded with -1)
    std::vector<long long> count(r.nbands, 0), pos(r.nbands, 0);
    for (unsigned short b : band) ++count[b];
    long long slots = 0;
    for (int b = 0; b < r.nbands; ++b) {
        pos[b] = slots;
        const long long nt = (count[b] + 15) / 16;
        slots += nt * 16;
        for (long long t = 0; t < nt; ++t) r.tile_band.push_back(b);
    }
    r.ntile = (int)r.tile_band.size();
    r.ntile_near = (int)((count[0] + 15) / 16);
    r.nfar = g->npairs - count[0];
    std::vector<int> recs((size_t)slots, -1);
    long long rec = 0;
    for (int m = 0; m < N; ++m)
        for (int n = 0; n <= m; ++n, ++rec) {
            const int b = band[rec];
            recs[pos[b]++] = (int)rec;
            if (b) continue;
            hbem::RadialNear e = {m, n, {0, 0, 0, 0}};
            for (int q = 0; q < 4; ++q) {
                const int P = (m + N - 1 + (q & 1)) % N, Q = (n + N - 1 + (q >> 1)) % N;
                e.type[q] = P == Q ? 4 * P : 3;
                for (const auto& a : adj[std::max(P, Q)])
                    if (a.first == std::min(P, Q)) e.type[q] = 1 + 4 * a.second;
            }
            r.near.push_back(e);
        }
    Packed pk;
    const size_t on = pk.add(r.near), orec = pk.add(recs);
    const char* plan = (const char*)r.plan.get(pk.bytes.size());
    HIPC(hipMemcpyAsync(r.plan.p, pk.bytes.data(), pk.bytes.size(), hipMemcpyHostToDevice, g->st));
    r.d_near = (const hbem::RadialNear*)(plan + on);
    r.recs = (const int*)(plan + orec);
    HIPC(hipStreamSynchronize(g->st));        // the upload reads a host vector
    r.usable = true;
    return done();
}

// Whether a wavenumber of tier t takes the separated pairs' tolerance: real positive
// ones of contexts with HBEM_FLAG_FAR_FIELD on line and arc panels.
bool far_tolerance(const hbem_geometry* g, int t, bool cplx) { return g->straight && (g->flags & HBEM_FLAG_FAR_FIELD) && !cplx && kTierEdge[t] <= 5.0; }

// The power of two with R^2 near_scale(R) in [1, 4).
double near_scale(double R) { return std::ldexp(1.0, -2 * std::ilogb(R)); }
// r^2 near_scale(R) of point j of the near band's p, Chebyshev in r^2 on [0, R^2]; the
// point is the one this double names, whose last bit is clear (near_node).
double near_u(double R, int p, int j) {
    const long double x = R * cosl(acosl(-1.0L) * (2 * j + 1) / (4.0L * p));
    const double u = (double)(x * x * near_scale(R));
    unsigned long long b;
    std::memcpy(&b, &u, sizeof(b));
    b &= ~1ull;
    double v;
    std::memcpy(&v, &b, sizeof(v));
    return v;
}

// The power series of series_comp (hbem_radial.hip) in y = x^2 / 64, A&S 9.1.10-9.1.13:
// J0, J1 / x, the entire part of Y0 and that of Y1 over x; doubles, then residuals.
std::vector<double> entire_series() {
    constexpr int n = hbem::kSeriesDeg + 1;
    const long double g = 0.57721566490153286060651209008240243L, pi = acosl(-1.0L);
    std::vector<double> out(8 * n);
    long double a = 1.0L, b = 0.5L, h = 0.0L;            // (-16)^k / k!^2, half of (-16)^k / (k! (k + 1)!), H_k
    for (int k = 0; k < n; ++k) {
        if (k > 0) {
            a *= -16.0L / ((long double)k * k);
            b *= -16.0L / ((long double)k * (k + 1));
            h += 1.0L / k;
        }
        const long double c[4] = {a, b, 2.0L / pi * (g - h) * a, -b / pi * (2.0L * h + 1.0L / (k + 1) - 2.0L * g)};
        for (int f = 0; f < 4; ++f) {
            out[4 * k + f] = (double)c[f];
            out[4 * (n + k) + f] = (double)(c[f] - (double)c[f]);
        }
    }
    return out;
}

// Points and coefficient tables of tier t (kTiers + t: at the separated pairs'
// tolerance), built on first use (null: a band would need more than kBandMaxP points).
hbem_geometry::Tier* radial_tier(hbem_geometry* g, int t) {
    auto& r = radial_base(g);
    if (!r.usable || t < 0) return nullptr;
    auto& T = r.tier[t];
    if (T.built) return T.pmax > 0 ? &T : nullptr;
    const double tol = t >= hbem_geometry::kTiers ? kBandTolFar : kBandTol;
    const double kmax = kTierEdge[t % hbem_geometry::kTiers] / g->dmax;
    std::vector<hbem::Band> bands(r.nbands);
    std::vector<double> cosv = entire_series();
    std::map<int, int> cosoff;
    std::map<int, std::vector<long double>> points;
    int pmax = 0, basis = 0;
    for (int b = 0; b < r.nbands; ++b) {
        hbem::Band& B = bands[b];
        if (b == 0) {
            B.c = 0.0;
            B.a = r.R;
        } else {
            const double lo = r.first + (b - 1) * r.step;
            B.c = lo + 0.5 * (r.step + r.width);
            B.a = 0.5 * (r.step + r.width);
        }
        B.p = hbem::band_order(B.c, B.a, kmax, b == 0 ? kNearTol : tol, b == 0);
        if (B.p == 0) {
            T.built = true;
            return nullptr;
        }
        const int p = B.p;
        if (b == 0) {
            // the points' r^2 in units of a power of two, and the reciprocal
            // products of their differences
            const int P = hbem::near_stride(p);
            B.cos = (int)cosv.size();
            cosv.resize(B.cos + (size_t)P, -1.0);
            cosv.resize(B.cos + 2 * (size_t)P, 0.0);
            double* u = &cosv[B.cos];
            for (int j = 0; j < p; ++j) u[j] = near_u(r.R, p, j);
            for (int j = 0; j < p; ++j) {
                long double v = 1.0L;
                for (int k = 0; k < p; ++k)
                    if (k != j) v *= (long double)u[j] - u[k];
                u[P + j] = (double)(1.0L / v);
            }
        }
        auto it = cosoff.find(p);
        if (b > 0 && it == cosoff.end()) {
            it = cosoff.emplace(p, (int)cosv.size()).first;
            for (int j = 0; j < p; ++j) points[p].push_back(cosl(acosl(-1.0L) * (2 * j + 1) / (2.0L * p)));
            std::vector<double> c4(4 * p);        // cos of the multiples of pi / (2 p)
            for (int k = 0; k < 4 * p; ++k) c4[k] = std::cos(M_PI * k / (2.0 * p));
            for (int j = 0; j < p; ++j)
                for (int q = 0; q < p; ++q) cosv.push_back((q == 0 ? 1.0 : 2.0) / p * c4[q * (2 * j + 1) % (4 * p)]);
        }
        if (b > 0) B.cos = it->second;
        B.rad = (int)cosv.size();
        std::vector<double> res;              // the points' radii, then what rounding took from them
        for (int j = 0; j < p; ++j) {
            const long double x = b == 0 ? sqrtl(near_u(r.R, p, j) / (long double)near_scale(r.R)) : B.c + B.a * points[p][j];
            cosv.push_back((double)x);
            res.push_back((double)(x - (double)x));
        }
        cosv.insert(cosv.end(), res.begin(), res.end());
        B.basis = basis;
        basis += 2 * p;
        pmax = std::max(pmax, p);
    }
    std::vector<hbem::BandTile> tiles(r.ntile);
    long long off = 0;
    double npoints = 0.0;
    for (int i = 0; i < r.ntile; ++i) {
        const int b = r.tile_band[i];
        tiles[i] = {off, b, 0};
        off += (long long)bands[b].p * (b == 0 ? 10 : 5) * 16;
        if (b) npoints += 16.0 * bands[b].p;
    }
    std::vector<int> cent;
    for (int i = 0; i < g->N; ++i) cent.insert(cent.end(), {i, i, 0});
    const std::vector<int>* ents[2] = {&cent, &g->aent};
    // one upload: bands, tiles, transforms, and the singular pairs' lists
    Packed pk;
    const size_t ob = pk.add(bands), ot = pk.add(tiles), oc = pk.add(cosv), oe[2] = {pk.add(*ents[0]), pk.add(*ents[1])};
    // ... and one buffer for these, the coefficients, the extra sums and the
    // singular pairs' moments (which the tier does not need later)
    const int pn = bands[0].p;
    size_t need = al256(pk.bytes.size());
    auto place = [&](size_t bytes) {
        const size_t at = need;
        need += al256(bytes);
        return at;
    };
    size_t omom[2], oext[2];
    const size_t otab = place((size_t)off * sizeof(double));
    const size_t osum = place(std::max<size_t>(1, (size_t)r.ntile_near * 7 * 16) * sizeof(double));
    for (int cls = 0; cls < 2; ++cls) {
        const size_t cnt = ents[cls]->size() / 3 * (1 + cls);
        omom[cls] = place(cnt * pn * hbem::kRadialMoments * sizeof(double));
        oext[cls] = place(cnt * hbem::kRadialSums * sizeof(double));
    }
    char* plan = (char*)T.mem.get(need);
    HIPC(hipMemcpyAsync(plan, pk.bytes.data(), pk.bytes.size(), hipMemcpyHostToDevice, g->st));
    const hbem::Band* db = T.bands = (const hbem::Band*)(plan + ob);
    const hbem::BandTile* dt = T.tiles = (const hbem::BandTile*)(plan + ot);
    const double* dc = T.costab = (const double*)(plan + oc);
    double *tab = (double*)(plan + otab), *ext = (double*)(plan + osum);
    T.tab = tab;
    T.ext = ext;
    const double* gtab = (const double*)g->d_gtab.p;
    const double *xg = (const double*)g->d_xg.p, *wg = (const double*)g->d_wg.p;
    const double iS = near_scale(r.R);
    // the quadrature rules' integrals of 1 over a panel pair, less one
    long double c0 = 0.0L, c1 = 0.0L, gs = 0.0L;
    for (int i = 0; i < g->nc; ++i) {
        c0 += g->wc[i];
        c1 += (long double)g->xc[i] * g->wc[i];
    }
    for (int i = 0; i < g->ns; ++i) gs += g->wg[i];
    const double curl_s = (double)(2.0L * c0 * c1 - 1.0L), curl_g = (double)(gs * gs - 1.0L);
    for (int cls = 0; cls < 2; ++cls)
        hbem::launch_radial_moments(cls, (const int*)(plan + oe[cls]), (int)ents[cls]->size() / 3,
                                    (const double*)g->d_panels.p, (const double*)g->d_coefs.p, (const double*)g->d_xc.p,
                                    (const double*)g->d_wc.p, g->nc, r.R, iS, dc + bands[0].cos, pn, (double*)(plan + omom[cls]),
                                    (double*)(plan + oext[cls]), g->st);
    hbem::launch_radial_near(r.d_near, (int)r.near.size(), dt, db, pn, gtab, xg, wg, g->N, g->ns,
                             r.flags, (const double*)(plan + omom[0]), (const double*)(plan + oext[0]),
                             (const double*)(plan + omom[1]), (const double*)(plan + oext[1]), dc, iS, curl_s, curl_g, tab,
                             ext, g->st);
    hbem::launch_radial_far(r.recs, dt, r.ntile_near, r.ntile - r.ntile_near, db, pmax, gtab, xg, wg, g->N,
                            g->ns, r.flags, dc, tab, g->st);
    HIPC(hipGetLastError());
    HIPC(hipStreamSynchronize(g->st));        // the uploads above read host vectors; other streams may use the tables
    T.points = npoints;
    T.pmax = pmax;
    T.pnear = pn;
    T.basis = basis;
    T.built = true;
    return &T;
}

// Classes and node tables of all panel pairs.
hbem_geometry::Loops& node_loops(hbem_geometry* g) {
    auto& s = g->loops;
    if (s.built) return s;
    const int N = g->N;
    std::vector<int> ent[3];
    std::vector<long long> pidx[3];
    auto add = [&](int cls, int i, int j, int swap) {
        ent[cls].insert(ent[cls].end(), {i, j, swap});
        pidx[cls].push_back(tri_index(i, j));
    };
    std::vector<std::vector<int>> nb(N);      // adjacent lower-numbered panels
    for (int i = 0; i < N; ++i) add(0, i, i, 0);
    for (size_t e = 0; e < g->aent.size(); e += 3) {
        add(1, g->aent[e], g->aent[e + 1], g->aent[e + 2]);
        nb[g->aent[e]].push_back(g->aent[e + 1]);
    }
    for (int i = 0; i < N; ++i)
        for (int j = 0; j < i; ++j)
            if (std::find(nb[i].begin(), nb[i].end(), j) == nb[i].end()) add(2, i, j, 0);
    for (int c = 0; c < 3; ++c) {
        s.cnt[c] = (int)pidx[c].size();
        const int* de = upload(s.ent[c], ent[c], g->st);
        upload(s.pidx[c], pidx[c], g->st);
        unsigned char* fl = (unsigned char*)s.flags[c].get(std::max(1, s.cnt[c]));
        double* ng = s.ngeo[c].as<double>(std::max<size_t>(1, (size_t)s.cnt[c] * class_nodes(g, c) * hbem::kNodeStride));
        if (c == 2)
            hbem::launch_setup_general(de, s.cnt[c], (const double*)g->d_gtab.p, g->ns, ng, fl, g->st);
        else
            hbem::launch_setup_singular(c, de, s.cnt[c], (const double*)g->d_panels.p, (const double*)g->d_coefs.p,
                                        (const double*)g->d_xc.p, g->nc, ng, fl, g->st);
    }
    HIPC(hipGetLastError());
    HIPC(hipStreamSynchronize(g->st));
    s.built = true;
    return s;
}

// The tier of a column with |kappa| between lo and hi and Im kappa at most im, or -1
// for the node loops: kappa = 0, beyond the last tier, or so far from the real
// axis that J and iY of the near band, each of size e^{Im kappa r}, would leave
// H with fewer digits (kNearImag: e^{2 Im kappa R} below 3).  cplx: it is evaluated as
// a complex one.  sweep: of a sweep; the single matrices' calls at real wavenumbers take
// the node loops from kappa dmax = 5 on (kBuilderEdge), where a panel holds most of a
// wavelength and the tables' many points cost a context's first call far more than any
// later call saves: made and called once, with the bands 400 panels at kappa dmax = 15
// took 21.4 ms (node loops 12.5), 100 panels 2.4 (1.15); their second calls 0.84 (1.22) and
// 0.22 (0.22).  At complex ones the loops are ten times as long (100 panels at 9 + 0.04 i:
// 3.4 ms made and called once, with the bands 2.6).
constexpr double kNearImag = 0.5, kBuilderEdge = 5.0;
int record_tier(hbem_geometry* g, double lo, double hi, double im, bool cplx, bool sweep) {
    int t = lo > 0.0 ? tier_of(hi * g->dmax) : -1;
    if (t >= 0 && !sweep && !cplx && kTierEdge[t] > kBuilderEdge) t = -1;
    if (t >= 0 && far_tolerance(g, t, cplx)) t += hbem_geometry::kTiers;
    if (t < 0 || !radial_tier(g, t)) return -1;
    if (im > 0.0 && (im * g->rad->R > kNearImag || hi * g->rad->R > hbem::kEntireMax)) return -1;
    return t;
}

// ---------------------------------------------------------------------------
// Assembly of the records of a call's columns.  prepare_records does what needs
// the host (tables, uploads, buffers), launch_records only launches, so that it
// can stand in a captured graph.
// ---------------------------------------------------------------------------
// A group of columns that take the same way: tier >= 0: the bands' tables of that
// tier; tier < 0: the node loops.
struct RecGroup {
    int tier, start, count;
    const double *kap = nullptr, *kr = nullptr, *cv = nullptr, *kapi = nullptr, *kri = nullptr;   // node loops: the group's slots
    int nslots = 0;
};
// Values per order of the records of a call (see hbem_radial.hip).
int record_values(const hbem_geometry* g, int D) { return (g->flags & HBEM_FLAG_QUIRK_SLP_COINC_DER) && D >= 1 ? hbem::kRecValues + 1 : hbem::kRecValues; }

struct RecJob {
    hbem_geometry* g = nullptr;
    RecScratch* w = nullptr;
    int D = 0, ncol = 0, nslot2 = 0, nv = 4;
    bool diff = false, cplx = false, tdiff = false, sweep = false, prof = false;   // prof: time into the context's log
    hipStream_t st = nullptr;
    const double *kap = nullptr, *kapi = nullptr, *kr = nullptr, *kri = nullptr, *cv = nullptr;
    const int* cols = nullptr;
    size_t obasis = 0;                           // the basis' place behind the records
    std::vector<RecGroup> groups;
};

// lanes per item of the node loops for ns slots: 0 = the paired-lane kernel
// (32 wavenumbers x 2 nodes per wavefront), else groups of lanes per item (in the
// single matrices' calls one size, so that a matrix of a batch of fewer than 64 is the
// one of a call of its own)
void loop_lanes(int ns, bool cplx, bool tdiff, bool sweep, int& general, int& singular) {
    general = cplx ? 16 : (ns >= 64 || tdiff ? 0 : (sweep && ns >= 16 ? 4 : 16));
    singular = (ns >= 64 || tdiff) && !cplx ? 0 : 64;
}

// chunks of a class's nodes: singular pairs chunks of 2048 nodes (paired-lane
// kernel, 16 staging rounds; for adjacent pairs each of the two node halves is
// chunked on its own) or 64 x 48 nodes (one wavefront per item)
void loop_chunks(int cls, int G, int nodes, int& chunk, int& nchunk) {
    chunk = cls == 2 ? nodes : (G == 0 ? kChunkNodes : 64 * 48);
    nchunk = (nodes + chunk - 1) / chunk;
    if (cls == 1 && G == 0) nchunk = 2 * ((nodes / 2 + chunk - 1) / chunk);
}

// Node loops of one group: local matrices of all panel pairs, then the records.
void launch_loops(const RecJob& J, const RecGroup& r) {
    hbem_geometry* g = J.g;
    const auto& set = g->loops;
    const int nslot = 16 * (J.D + 1), nko = J.tdiff ? r.count : r.nslots;
    cdbl* L = (cdbl*)J.w->L.p;
    hbem::AsmParams P;
    std::memset(&P, 0, sizeof(P));
    P.xg = (const double*)g->d_xg.p;
    P.wg = (const double*)g->d_wg.p;
    P.xc = (const double*)g->d_xc.p;
    P.wc = (const double*)g->d_wc.p;
    P.npairs_total = g->npairs;
    P.ns = g->ns;
    P.nc = g->nc;
    P.qflags = g->flags;
    P.tdiff = J.tdiff ? 1 : 0;
    P.nkt = J.tdiff ? r.count : 0;
    P.nk = r.nslots;
    P.kap = r.kap;
    P.kr = r.kr;
    P.cv = r.cv;
    P.kapi = r.kapi;
    P.kri = r.kri;
    int Gg, Gs;
    loop_lanes(r.nslots, J.cplx, J.tdiff, J.sweep, Gg, Gs);
    const int which[3] = {kProfCoinciding, kProfAdjacent, kProfGeneral};
    for (int cls = 2; cls >= 0; --cls) {
        if (set.cnt[cls] == 0) continue;
        const int G = cls == 2 ? Gg : Gs, nodes = class_nodes(g, cls);
        P.nent = set.cnt[cls];
        P.ent = (const int*)set.ent[cls].p;
        P.ngeo = (const double*)set.ngeo[cls].p;
        P.flags = (const unsigned char*)set.flags[cls].p;
        P.pidx = (const long long*)set.pidx[cls].p;
        loop_chunks(cls, G, nodes, P.chunk, P.nchunk);
        cdbl* part = (cdbl*)J.w->part.p;
        P.out = P.nchunk > 1 ? part : L;
        // the class's kernel alone is timed: the chunk sums are a separate launch
        hipEvent_t e0 = J.prof ? g->plog.begin(J.st) : nullptr;
        hbem::launch_assemble(cls, J.D, P, G, J.st);
        if (J.prof) g->plog.end(J.st, which[cls], e0, (double)P.nent * P.nk * nodes * flops_per_node(J.D));
        if (P.nchunk > 1) hbem::launch_chunk_sum(part, P.nent, P.nchunk, nko, nslot, P.pidx, g->npairs, L, J.st);
    }
    const int lout = J.diff && !J.tdiff ? r.count : 0;
    hbem::launch_records_from_locals(L, nko, J.D, lout, (int)g->npairs, J.cols + r.start, r.count, g->N, (cdbl*)J.w->E.p,
                                     J.ncol, J.nv, J.st);
}

// Slot tables kap = k sqrt(c), k, c (imaginary parts kapi, kri: any slot is not
// real positive) of a call with ncol columns: ncol slots, or (diff) 2 ncol, the
// inner slots then the outer, whose differences T is formed from.  tdiff: the
// node loops take the paired-lane kernel in the difference layout whatever the
// width (sweeps of >= 32 wavenumbers, so that a wavenumber's bits do not depend
// on its batch).  sweep: see record_tier.  together: the columns are one system's and
// take one way, that of the largest kappa.
RecJob prepare_records(hbem_geometry* g, RecBufs& b, RecScratch& w, hipStream_t st, const std::vector<double>& kap,
                       const std::vector<double>& kr, const std::vector<double>& cv, int D, bool diff,
                       const std::vector<double>& kapi = {}, const std::vector<double>& kri = {}, bool sweep = false,
                       bool tdiff = false, bool together = false) {
    RecJob J;
    J.sweep = sweep;
    J.g = g;
    J.w = &w;
    J.st = st;
    J.D = D;
    J.diff = diff;
    J.cplx = !kapi.empty();
    J.tdiff = tdiff && diff && !J.cplx;
    J.ncol = (int)kap.size() / (diff ? 2 : 1);
    J.nslot2 = diff ? J.ncol : 0;
    const int n = J.ncol;
    // a column's way depends on its own kappa
    J.nv = record_values(g, D);
    const bool quirk = J.nv != hbem::kRecValues;
    std::map<int, std::vector<int>> by;
    double lo = 1e300, hi = 0.0, im = 0.0;
    auto reach = [&](int q) {
        const double m = J.cplx ? std::hypot(kap[q], kapi[q]) : std::fabs(kap[q]);
        lo = std::min(lo, m);
        hi = std::max(hi, m);
        if (J.cplx) im = std::max(im, kapi[q]);
    };
    for (int q = 0; q < (int)kap.size() && together; ++q) reach(q);
    for (int c = 0; c < n; ++c) {
        if (!together) {
            lo = 1e300;
            hi = im = 0.0;
            for (int h = 0; h < (diff ? 2 : 1); ++h) reach(c + h * n);
        }
        by[quirk ? -1 : record_tier(g, lo, hi, im, J.cplx, sweep)].push_back(c);
    }
    std::vector<int> cols;
    size_t nL = 0, npart = 0, nbasis = 0;
    Packed pk;
    std::vector<std::array<size_t, 5>> places;   // of the groups' slot tables in pk
    for (auto& kv : by) {
        RecGroup r;
        r.tier = kv.first;
        r.start = (int)cols.size();
        r.count = (int)kv.second.size();
        cols.insert(cols.end(), kv.second.begin(), kv.second.end());
        if (r.tier >= 0)
            nbasis = std::max(nbasis, (size_t)(g->rad->tier[r.tier].basis + (J.cplx ? 2 * g->rad->tier[r.tier].pnear : 0)) *
                                          r.count * (diff ? 2 : 1));
        if (r.tier < 0) {
            // the group's slots: blocks of 32 wavenumbers, inner and outer in turn
            // (tdiff), or in the order of its columns, inner then outer
            std::vector<int> slot;
            if (J.tdiff) {
                const int nblk = (r.count + 31) / 32;
                for (int q = 0; q < 64 * nblk; ++q) {
                    const int blk = q >> 5, c = kv.second[std::min(r.count - 1, (blk >> 1) * 32 + (q & 31))];
                    slot.push_back((blk & 1) ? c + n : c);
                }
            } else {
                for (int h = 0; h < (diff ? 2 : 1); ++h)
                    for (int c : kv.second) slot.push_back(c + h * n);
            }
            r.nslots = (int)slot.size();
            std::array<size_t, 5> at;
            const std::vector<double>* tabs[5] = {&kap, &kr, &cv, &kapi, &kri};
            for (int i = 0; i < 5; ++i) {
                std::vector<double> x;
                if (!tabs[i]->empty())
                    for (int q : slot) x.push_back((*tabs[i])[q]);
                at[i] = pk.add(x);
            }
            places.push_back(at);
            auto& set = node_loops(g);
            const size_t rows = (size_t)16 * (D + 1) * (J.tdiff ? r.count : r.nslots);
            nL = std::max(nL, rows * (size_t)g->npairs);
            int G[2];
            loop_lanes(r.nslots, J.cplx, J.tdiff, J.sweep, G[0], G[1]);
            for (int cls = 0; cls < 3; ++cls) {
                int chunk, nchunk;
                loop_chunks(cls, cls == 2 ? G[0] : G[1], class_nodes(g, cls), chunk, nchunk);
                if (nchunk > 1) npart = std::max(npart, rows * set.cnt[cls] * nchunk);
            }
        }
        J.groups.push_back(r);
    }
    const std::vector<double>* tabs[5] = {&kap, &kr, &cv, &kapi, &kri};
    const double** dst[5] = {&J.kap, &J.kr, &J.cv, &J.kapi, &J.kri};
    size_t at[5];
    for (int i = 0; i < 5; ++i) at[i] = pk.add(*tabs[i]);
    const size_t ocols = pk.add(cols);
    const char* d = (const char*)b.tab.get(pk.bytes.size());
    HIPC(hipMemcpyAsync(b.tab.p, pk.bytes.data(), pk.bytes.size(), hipMemcpyHostToDevice, st));
    for (int i = 0; i < 5; ++i) *dst[i] = tabs[i]->empty() ? nullptr : (const double*)(d + at[i]);
    J.cols = (const int*)(d + ocols);
    size_t np = 0;
    for (RecGroup& r : J.groups)
        if (r.tier < 0) {
            const std::array<size_t, 5>& p = places[np++];
            const double** own[5] = {&r.kap, &r.kr, &r.cv, &r.kapi, &r.kri};
            for (int i = 0; i < 5; ++i) *own[i] = tabs[i]->empty() ? nullptr : (const double*)(d + p[i]);
        }
    J.obasis = al256((size_t)g->npairs * J.nv * (D + 1) * n * sizeof(cdbl));
    w.E.get(J.obasis + nbasis * sizeof(cdbl));
    if (nL) w.L.get(nL * sizeof(cdbl));
    if (npart) w.part.get(npart * sizeof(cdbl));
    HIPC(hipGetLastError());
    return J;
}

cdbl* launch_records(const RecJob& J) {
    hbem_geometry* g = J.g;
    cdbl* E = (cdbl*)J.w->E.p;
    for (const RecGroup& r : J.groups) {
        if (r.tier >= 0) {
            const auto& R = *g->rad;
            const auto& T = R.tier[r.tier];
            hbem::RadialParams P;
            P.kap = J.kap;
            P.kapi = J.kapi;
            P.kr = J.kr;
            P.kri = J.kri;
            P.cv = J.cv;
            P.cols = J.cols + r.start;
            P.ncolg = r.count;
            P.nslot2 = J.nslot2;
            P.ncol = J.ncol;
            P.nv = J.nv;
            P.nbasis = T.basis;
            P.basis = (cdbl*)((char*)E + J.obasis);
            P.out = E;
            const auto* bands = T.bands;
            const auto* tiles = T.tiles;
            const auto* recs = R.recs;
            const double *cs = T.costab, *tab = T.tab, *ext = T.ext;
            hipEvent_t e0 = J.prof ? g->plog.begin(J.st) : nullptr;
            hbem::launch_band_basis(P, J.diff, bands, R.nbands, T.pmax, cs, J.st);
            hbem::launch_band_eval(J.D, J.diff, false, P, recs, tiles, R.ntile_near, R.ntile - R.ntile_near, bands, cs, tab,
                                   ext, J.st);
            if (J.prof)
                g->plog.end(J.st, kProfGeneral, e0, 20.0 * (J.D + 1) * T.points * r.count * (J.diff ? 2.0 : 1.0));
            if (J.prof) e0 = g->plog.begin(J.st);
            hbem::launch_band_eval(J.D, J.diff, true, P, recs, tiles, 0, R.ntile_near, bands, cs, tab, ext, J.st);
            if (J.prof)
                g->plog.end(J.st, kProfAdjacent, e0,
                            (J.cplx ? 40.0 : 30.0) * (J.D + 1) * 16.0 * R.ntile_near * T.pnear * r.count * (J.diff ? 2.0 : 1.0));
        } else {
            launch_loops(J, r);
        }
    }
    return E;
}

// Records of a call on the context's own buffers and stream.
cdbl* assemble_records(hbem_geometry* g, const std::vector<double>& kap, const std::vector<double>& kr,
                       const std::vector<double>& cv, int D, bool diff, const std::vector<double>& kapi = {},
                       const std::vector<double>& kri = {}, bool sweep = false, bool tdiff = false, bool together = false) {
    RecJob J = prepare_records(g, g->w_rec, g->w_scr, g->st, kap, kr, cv, D, diff, kapi, kri, sweep, tdiff, together);
    J.prof = g->prof;
    cdbl* E = launch_records(J);
    HIPC(hipGetLastError());
    return E;
}

// Device bytes per column of a call with these kappa (the larger one of each
// column) and `slots` kappa a column: its records and basis, and where one of them
// takes the node loops for every pair their local matrices and partials too.  Builds
// the tables the call needs, so that the free memory seen afterwards is what its
// batches can use.
size_t records_bytes_per_k(hbem_geometry* g, const std::vector<double>& kap, int D, int lcols, int slots, bool sweep) {
    const bool quirk = record_values(g, D) != hbem::kRecValues;
    bool loops = false, cplx = false;
    size_t basis = 0;
    // (a batch with a wavenumber that is not positive is evaluated as complex)
    for (double v : kap) cplx = cplx || !(v > 0.0);
    for (double v : kap) {
        const double m = std::fabs(v);
        if (cplx && !quirk) record_tier(g, m, m, 0.0, true, sweep);
        const int t = quirk ? -1 : record_tier(g, m, m, 0.0, false, sweep);
        if (t < 0) loops = true;
        else basis = std::max(basis, (size_t)(g->rad->tier[t].basis + 2 * g->rad->tier[t].pnear) * slots * sizeof(cdbl));
    }
    if (loops) node_loops(g);
    return (size_t)g->npairs * record_values(g, D) * (D + 1) * sizeof(cdbl) + basis +
           (loops ? locals_bytes_per_k(g->npairs, (long long)g->aent.size() / 3, g->N, g->nc, D, lcols) : 0);
}

// Dense stage shared by sv, sv_der and the sweep: given LU factors of the
// unprojected T (batch matrices), the projection factor (sparse F and F^T, or
// none) and R, returns sigma and the singular pair (u, v) of
// T_p = F^{-1} T F^{-T} in d_u / d_v.
struct DenseCtx {
    hipStream_t st;
    int n, batch, nc, q;
    const cdbl* LU;
    long long ms;        // matrix stride of LU
    const int* perm;
    const DCsr* F;       // projection factor, null = no projection
    const DCsr* FT;      // its transpose
    // or, for a batch of zero-padded matrices of several scatterers, the
    // factor of each matrix's scatterer (device arrays of batch entries)
    const hbem::CsrDesc* Fm = nullptr;
    const hbem::CsrDesc* FTm = nullptr;
    cdbl* X;             // n x nc x batch
    cdbl* Y;
    cdbl* work;          // 2 n nc batch: thin-solve scratch, then the projected right-hand sides
    EventLog* tim = nullptr;   // randomized_svd timers (kTim*), or null
    // mixed precision (LU32 set): the factors are FP32 (LU32, stride ms) and
    // every solve with T is refined `refine` times against T64 (the FP64 T,
    // stride ms): residual in FP64, correction from the FP32 factors
    const cflt* LU32 = nullptr;
    const cdbl* T64 = nullptr;
    int refine = 0;         // steps of the final solve of the randomized SVD
    int refine_inner = 0;   // steps of the solves before it
    bool last_solve = false;
    double* rprev = nullptr;   // per matrix: the previous correction's size
    double rtol = 0.0;   // a matrix whose last correction exceeds rtol of its solution is flagged
    int* flag = nullptr; // per matrix
    cdbl* rb = nullptr;  // n nc batch: the right-hand side
    cdbl* rr = nullptr;  // n nc batch: residual, then correction
    cdbl* rpart = nullptr;
};

// Z <- op(T)^{-1} Z with the context's factors (op = T or T^H): FP64 factors,
// or FP32 factors plus `refine` steps of FP64 iterative refinement.
void t_solve(DenseCtx& c, cdbl* Z, bool adj) {
    if (!c.LU32) {
        hbem::lu_solve_thin_batched(c.LU, c.ms, c.perm, c.n, c.batch, Z, c.nc, adj, c.work, c.st);
        return;
    }
    const size_t cnt = (size_t)c.n * c.nc;
    const int steps = c.last_solve ? c.refine : c.refine_inner;
    if (steps > 0) HIPC(hipMemcpyAsync(c.rb, Z, sizeof(cdbl) * cnt * c.batch, hipMemcpyDeviceToDevice, c.st));
    hbem::lu_solve_thin_batched_f32(c.LU32, c.ms, c.perm, c.n, c.batch, Z, c.nc, adj, c.work, c.st);
    // the final solve, whose vectors give sigma, must reach the tolerance; the
    // solves before it only move the subspace and must contract
    const int check_last = c.last_solve ? 2 : 1;
    for (int it = 0; it < steps; ++it) {
        hbem::residual_thin_batched(c.T64, c.ms, Z, c.rb, c.rr, c.n, c.nc, c.batch, adj, c.rpart, c.st);
        hbem::lu_solve_thin_batched_f32(c.LU32, c.ms, c.perm, c.n, c.batch, c.rr, c.nc, adj, c.work, c.st);
        hbem::refine_update_batched(Z, c.rr, (int)cnt, c.batch, c.rtol, it == steps - 1 ? check_last : 0, it == 0,
                                    c.rprev, c.flag, c.st);
    }
}

// Y <- T_p^{-1} X  or  T_p^{-H} X  (T_p^{-1} = F^T T^{-1} F, T_p^{-H} = F^T T^{-H} F); X is kept.
void tp_solve(DenseCtx& c, const cdbl* X, cdbl* Y, bool adj) {
    const long long cols = (long long)c.nc * c.batch;
    if (c.Fm) {
        cdbl* Z = c.work + (size_t)c.n * cols;
        hbem::csr_apply_multi(c.Fm, c.n, X, Z, c.nc, c.batch, c.st);
        t_solve(c, Z, adj);
        hbem::csr_apply_multi(c.FTm, c.n, Z, Y, c.nc, c.batch, c.st);
    } else if (c.F) {
        cdbl* Z = c.work + (size_t)c.n * cols;
        hbem::csr_apply_batched((const int*)c.F->rp.p, (const int*)c.F->ci.p, (const double*)c.F->v.p, c.n, X, Z, cols,
                                c.st);
        t_solve(c, Z, adj);
        hbem::csr_apply_batched((const int*)c.FT->rp.p, (const int*)c.FT->ci.p, (const double*)c.FT->v.p, c.n, Z, Y,
                                cols, c.st);
    } else {
        HIPC(hipMemcpyAsync(Y, X, sizeof(cdbl) * (size_t)c.n * cols, hipMemcpyDeviceToDevice, c.st));
        t_solve(c, Y, adj);
    }
}

// randomized_svd::sv (randsvd.cpp:99-146) on the batch; X holds R replicated
// per matrix.  The power iteration alternates between X and Y.
void rsvd_core(DenseCtx& c, double* d_sigma, cdbl* d_u, cdbl* d_v) {
    hipEvent_t e = c.tim ? c.tim->begin(c.st) : nullptr;
    tp_solve(c, c.X, c.Y, false);                              // Y = T_p^{-1} R
    hbem::orthonormalize_thin_batched(c.Y, c.n, c.batch, c.nc, c.st);   // Q
    if (c.tim) { c.tim->end(c.st, kTimQR, e); e = c.tim->begin(c.st); }
    for (int it = 0; it < c.q; ++it) {
        tp_solve(c, c.Y, c.X, true);
        hbem::orthonormalize_thin_batched(c.X, c.n, c.batch, c.nc, c.st);
        tp_solve(c, c.X, c.Y, false);
        hbem::orthonormalize_thin_batched(c.Y, c.n, c.batch, c.nc, c.st);
    }
    if (c.tim) { c.tim->end(c.st, kTimIter, e); e = c.tim->begin(c.st); }
    // Q = Y, X = T_p^{-H} Q
    c.last_solve = true;
    tp_solve(c, c.Y, c.X, true);
    c.last_solve = false;
    hbem::sigma_from_thin_batched(c.X, c.Y, c.n, c.batch, c.nc, d_sigma, d_u, d_v, c.st);
    if (c.tim) c.tim->end(c.st, kTimSVD, e);
}

void copy_out_square(const cdbl* d, void* h, size_t count, hipStream_t st) {
    if (h) HIPC(hipMemcpyAsync(h, d, count * sizeof(cdbl), hipMemcpyDeviceToHost, st));
}

// T_p = Finv T Finv^T for `count` matrices (in place through tmp: count n^2
// entries, the context's buffer when null)
void project_inplace(hbem_geometry* g, cdbl* T, int count, cdbl* tmp = nullptr) {
    const int n = 2 * g->N;
    const long long s = (long long)n * n;
    if (!tmp) tmp = g->w_tmp.as<cdbl>((size_t)s * count);
    const DCsr& F = g->s_Finv;
    const DSell& l = g->l_Finv;
    hbem::sparse_congruence((const int*)F.rp.p, (const int*)F.ci.p, (const double*)F.v.p, l.rows, l.off, l.col, l.val, n, T, tmp,
                            count, g->st);
}

// The linear system of tp::direct_second_kind::A_rhs (solvers.cpp:106-131) on
// the device: both wavenumber slots (c_i, c_o) are assembled in one pass, T is
// gen_sol_op's unprojected operator, and rhs = A_o U for the nrhs host columns
// U (2N x nrhs) with A_o = [[-K_o + M/2, V_o], [W_o, K_o^T + M/2]].
void tp_system(hbem_geometry* g, double k_re, double k_im, double c_o, double c_i, const void* U, int nrhs,
               cdbl*& T, cdbl*& rhs) {
    const double si = std::sqrt(c_i), so = std::sqrt(c_o);
    // the outer operators are wanted by themselves: one column per refraction index
    std::vector<double> kapi, kri;
    if (!real_positive(k_re, k_im)) {
        kapi = {k_im * si, k_im * so};
        kri = {k_im, k_im};
    }
    cdbl* E = assemble_records(g, {k_re * si, k_re * so}, {k_re, k_re}, {c_i, c_o}, 0, false, kapi, kri, false, false, true);
    const int N = g->N, n = 2 * N;
    const size_t nn = (size_t)n * n;
    const double* dM = (const double*)g->d_M.p;
    T = g->w_T0.as<cdbl>(nn);
    hbem::launch_form_T(E, 2, hbem::kRecValues, 0, 1, 1, N, 0, dM, T, nullptr, nullptr, g->st);
    HIPC(hipGetLastError());
    cdbl* Ao = g->w_Ao.as<cdbl>(nn);
    hbem::launch_form_Ao(E, 2, 1, N, dM, Ao, g->st);
    HIPC(hipGetLastError());
    cdbl* dU = g->w_U.as<cdbl>((size_t)n * nrhs);
    HIPC(hipMemcpyAsync(dU, U, sizeof(cdbl) * (size_t)n * nrhs, hipMemcpyHostToDevice, g->st));
    rhs = g->w_rhs.as<cdbl>((size_t)n * nrhs);
    hbem::zgemm_batched(n, nrhs, n, hbem::mk(1, 0), Ao, n, 0, dU, n, 0, hbem::mk(0, 0), rhs, n, 0, 1, g->st);
    HIPC(hipGetLastError());
}

void check_tp_args(hbem_geometry* g, const void* U, int nrhs) {
    if (!g || !U) throw Error(HBEM_EINVAL, "null argument");
    if (nrhs < 1) throw Error(HBEM_EINVAL, "number of right-hand sides must be positive");
}

}  // namespace

extern "C" {

int hbem_last_error(char* buf, size_t len) {
    if (buf && len > 0) {
        std::strncpy(buf, g_err.c_str(), len - 1);
        buf[len - 1] = 0;
    }
    return (int)g_err.size();
}

int hbem_init(int device) {
    API_BEGIN
    int n = 0;
    HIPC(hipGetDeviceCount(&n));
    if (device < 0 || device >= n) throw Error(HBEM_EINVAL, "invalid device index");
    g_device = device;
    HIPC(hipSetDevice(device));
    scratch_on(device);          // resolve hbem_rsvd_sv_noalloc's array on this device now
    API_END
}

int hbem_geometry_create(const double* panels, int npanels, const double* coefs, int ncoefs, int order, int proj,
                         int flags, hbem_geometry_t* out) {
    hbem_geometry* g = nullptr;
    API_BEGIN
    if (!out) throw Error(HBEM_EINVAL, "null output handle");
    if (npanels < 3) throw Error(HBEM_EINVAL, "a closed P1 mesh needs at least 3 panels");
    if (order < 1 || order > 40) throw Error(HBEM_EINVAL, "quadrature order out of range");
    if (flags & ~(HBEM_FLAG_QUIRK_SLP_COINC_DER | HBEM_FLAG_FAR_FIELD)) throw Error(HBEM_EINVAL, "unknown geometry flags");
    for (int i = 0; i < npanels; ++i) {
        int t = (int)panels[8 * i];
        if (t < 0 || t > 3 || panels[8 * i] != (double)t) throw Error(HBEM_EINVAL, "invalid panel type");
        if (t == 2) {
            int c0 = (int)panels[8 * i + 3], nc = (int)panels[8 * i + 4];
            if (c0 < 0 || nc < 1 || c0 + nc > ncoefs) throw Error(HBEM_EINVAL, "trig-curve panel coefficients out of range");
        }
        if (t == 3) {
            const long long c0 = (long long)panels[8 * i + 3], np = (long long)panels[8 * i + 4];
            if (c0 < 0 || np < 1 || c0 + 3 * np + 1 > ncoefs)
                throw Error(HBEM_EINVAL, "spline panel coefficients out of range");
            if (!(panels[8 * i + 1] < panels[8 * i + 2])) throw Error(HBEM_EINVAL, "spline panel needs tmin < tmax");
        }
    }
    g = new hbem_geometry;
    g->dev = g_device;
    HIPC(hipSetDevice(g->dev));
    HIPC(hipStreamCreateWithFlags(&g->st, hipStreamNonBlocking));
    g->N = npanels;
    g->order = order;
    g->ns = order;
    g->nc = order * (order + 1) / 2 - 1;
    g->flags = flags;
    g->proj = proj != 0;
    g->panels.assign(panels, panels + 8 * (size_t)npanels);
    if (ncoefs > 0) g->coefs.assign(coefs, coefs + 3 * (size_t)ncoefs);
    g->lines = true;
    for (int i = 0; i < npanels; ++i) {
        if ((int)panels[8 * i] != 0) g->lines = false;
        if ((int)panels[8 * i] >= 2) g->straight = false;
    }
    g->xg.resize(g->ns); g->wg.resize(g->ns); g->xc.resize(g->nc); g->wc.resize(g->nc);
    hbem::gauss_rule(0.0, 1.0, g->ns, g->xg.data(), g->wg.data());
    hbem::composite_rule(order, g->xc.data(), g->wc.data());
    const int N = npanels;
    g->npairs = (long long)N * (N + 1) / 2;
    // adjacent pairs (galerkin_builder.cpp:872-897; adjacency test 189-201)
    const double* cptr = g->coefs.empty() ? nullptr : g->coefs.data();
    std::vector<double> ends(4 * (size_t)N);
    std::vector<double> disc(3 * (size_t)N);   // bounding discs: centre, radius
    hbem::panel_endpoints(g->panels.data(), cptr, N, ends.data());
    hbem::panel_bounds(g->panels.data(), cptr, N, disc.data());
    for (int i = 0; i < N; ++i) g->dmax = std::max(g->dmax, 2.0 * disc[3 * (size_t)i + 2]);
    const double tol = 100.0 * hbem::kDblEps;
    auto meet = [&](const double* a, const double* b) {
        return std::fabs(a[0] - b[0]) < tol && std::fabs(a[1] - b[1]) < tol && std::hypot(a[0] - b[0], a[1] - b[1]) < tol;
    };
    for (int i = 0; i < N; ++i)
        for (int j = 0; j < i; ++j) {
            const double* ei = &ends[4 * (size_t)i];
            const double* ej = &ends[4 * (size_t)j];
            if (meet(ei + 2, ej)) g->aent.insert(g->aent.end(), {i, j, 0});           // end(i) == start(j)
            else if (meet(ei, ej + 2)) g->aent.insert(g->aent.end(), {i, j, 1});      // start(i) == end(j)
        }
    hipStream_t st = g->st;
    const double* dpan = upload(g->d_panels, g->panels, st);
    std::vector<double> cf = g->coefs.empty() ? std::vector<double>(3, 0.0) : g->coefs;
    const double* dcoef = upload(g->d_coefs, cf, st);
    const double* dxg = upload(g->d_xg, g->xg, st);
    upload(g->d_wg, g->wg, st);
    upload(g->d_xc, g->xc, st);
    upload(g->d_wc, g->wc, st);
    double* gtab = g->d_gtab.as<double>((size_t)N * g->ns * 5);
    hbem::launch_setup_gauss_table(dpan, dcoef, N, dxg, g->ns, gtab, st);
    HIPC(hipGetLastError());
    // mass matrix and projection factor (gen_sol_op.cpp:23-43)
    g->M.resize((size_t)N * N);
    hbem::mass_matrix_host(g->panels.data(), N, cptr, g->lines, order, g->M.data());
    upload(g->d_M, g->M, st);
    if (g->proj) {
        const int n = 2 * N;
        std::vector<double> A((size_t)n * n, 0.0);
        for (int j = 0; j < N; ++j)
            for (int i = 0; i < N; ++i) {
                A[i + (size_t)j * n] = g->M[i + (size_t)j * N];
                A[(N + i) + (size_t)(N + j) * n] = g->M[j + (size_t)i * N];
            }
        g->F.resize((size_t)n * n);
        g->tr.resize(n);
        hbem::ldlt_projection_factor(A.data(), n, g->F.data(), g->tr.data());
        g->Finv.resize((size_t)n * n);
        hbem::invert_projection_factor(g->F.data(), g->tr.data(), n, g->Finv.data());
        g->s_F.build(g->F, n, false, st);
        g->s_FT.build(g->F, n, true, st);
        g->s_FinvT.build(g->Finv, n, true, st);
        g->s_Finv.build(g->Finv, n, false, st);
        g->l_Finv.build(g->Finv, n, st);
    }
    HIPC(hipStreamSynchronize(st));
    *out = g;
    g = nullptr;
    }
    catch (const std::exception& e) {
        if (g) { if (g->st) (void)hipStreamDestroy(g->st); delete g; }
        return fail(e);
    }
    return HBEM_OK;
}

int hbem_geometry_destroy(hbem_geometry_t g) {
    API_BEGIN
    if (!g) return HBEM_OK;
    multi_forget(g);
    (void)hipStreamSynchronize(g->st);
    hipStream_t st = g->st;
    delete g;
    (void)hipStreamDestroy(st);
    API_END
}

int hbem_geometry_release_work(hbem_geometry_t g) {
    API_BEGIN
    if (!g) throw Error(HBEM_EINVAL, "null geometry");
    multi_forget(g);
    std::lock_guard<std::mutex> lk(g->mu);
    HIPC(hipSetDevice(g->dev));
    HIPC(hipStreamSynchronize(g->st));
    std::vector<DBuf*> bs = {&g->w_Ao, &g->w_U, &g->w_rhs, &g->w_flag, &g->w_Tp, &g->w_B, &g->w_mv, &g->w_bpiv, &g->w_bperm,
                             &g->w_bvec, &g->w_d2, &g->w_T32, &g->w_rb, &g->w_rr, &g->w_rpart, &g->w_flag2, &g->w_rprev,
                             &g->w_T0, &g->w_T1, &g->w_T2, &g->w_piv, &g->w_perm, &g->w_X, &g->w_Y, &g->w_work,
                             &g->w_R, &g->w_u, &g->w_v, &g->w_a, &g->w_b, &g->w_sig, &g->w_dsig, &g->w_tmp, &g->w_out,
                             &g->w_rec.tab,
                             &g->w_scr.E, &g->w_scr.L, &g->w_scr.part};
    for (DBuf* b : bs) b->release();
    API_END
}

int hbem_geometry_info(hbem_geometry_t g, int* npanels, int* order, int* corder, int* lines) {
    API_BEGIN
    if (!g) throw Error(HBEM_EINVAL, "null geometry");
    if (npanels) *npanels = g->N;
    if (order) *order = g->ns;
    if (corder) *corder = g->nc;
    if (lines) *lines = g->lines ? 1 : 0;
    API_END
}

int hbem_assemble_dense(hbem_geometry_t g, double k_re, double k_im, double c, int layers, int d, void* K, void* W,
                        void* V) {
    API_BEGIN
    if (!g) throw Error(HBEM_EINVAL, "null geometry");
    if (d < 0 || d > 2) throw Error(HBEM_EINVAL, "Invalid order of derivative");
    check_k(k_re, k_im, c);
    std::lock_guard<std::mutex> lk(g->mu);
    HIPC(hipSetDevice(g->dev));
    const double sc = std::sqrt(c);
    cdbl* E = real_positive(k_re, k_im) ? assemble_records(g, {k_re * sc}, {k_re}, {c}, d, false)
                                        : assemble_records(g, {k_re * sc}, {k_re}, {c}, d, false, {k_im * sc}, {k_im});
    const int N = g->N;
    const size_t NN = (size_t)N * N * (d + 1);
    cdbl* out = g->w_out.as<cdbl>(3 * NN);
    hbem::launch_gather_layers(E, 1, record_values(g, d), 0, N, d, layers, out, out + NN, out + 2 * NN, g->st);
    HIPC(hipGetLastError());
    if (layers & HBEM_LAYER_DOUBLE) copy_out_square(out, K, NN, g->st);
    if (layers & HBEM_LAYER_HYPERSINGULAR) copy_out_square(out + NN, W, NN, g->st);
    if (layers & HBEM_LAYER_SINGLE) copy_out_square(out + 2 * NN, V, NN, g->st);
    HIPC(hipStreamSynchronize(g->st));
    API_END
}

int hbem_assemble_dense_batch(hbem_geometry_t g, const double* ks, int nk, double c, int layers, int d, void* K,
                              void* W, void* V) {
    API_BEGIN
    if (!g || (nk > 0 && !ks)) throw Error(HBEM_EINVAL, "null argument");
    if (nk < 0) throw Error(HBEM_EINVAL, "negative number of wavenumbers");
    if (d < 0 || d > 2) throw Error(HBEM_EINVAL, "Invalid order of derivative");
    for (int i = 0; i < nk; ++i) check_k(ks[i], 0.0, c);
    std::lock_guard<std::mutex> lk(g->mu);
    HIPC(hipSetDevice(g->dev));
    const double sc = std::sqrt(c);
    const int N = g->N;
    const size_t NN = (size_t)N * N * (d + 1);
    cdbl* out = g->w_out.as<cdbl>(3 * NN);
    // one wavenumber slot per k: its records, and its local matrices where it takes the node loops
    std::vector<double> all(nk);
    for (int i = 0; i < nk; ++i) all[i] = ks[i] * sc;
    const size_t per = records_bytes_per_k(g, all, d, 1, 1, false);
    const int B = sweep_batch(per, usable_device_bytes(g->w_scr.E.n + g->w_scr.L.n + g->w_scr.part.n), nk);
    for (int k0 = 0; k0 < nk; k0 += B) {
        const int nb = std::min(B, nk - k0);
        std::vector<double> kap(nb), kr(nb), cv(nb, c);
        bool allpos = true;
        for (int b = 0; b < nb; ++b) {
            kap[b] = ks[k0 + b] * sc;
            kr[b] = ks[k0 + b];
            allpos = allpos && ks[k0 + b] > 0.0;
        }
        const std::vector<double> zero(allpos ? 0 : nb, 0.0);
        cdbl* E = assemble_records(g, kap, kr, cv, d, false, zero, zero);
        for (int b = 0; b < nb; ++b) {
            hbem::launch_gather_layers(E, nb, record_values(g, d), b, N, d, layers, out, out + NN, out + 2 * NN, g->st);
            HIPC(hipGetLastError());
            const size_t off = (size_t)(k0 + b) * NN * sizeof(cdbl);
            if ((layers & HBEM_LAYER_DOUBLE) && K) copy_out_square(out, (char*)K + off, NN, g->st);
            if ((layers & HBEM_LAYER_HYPERSINGULAR) && W) copy_out_square(out + NN, (char*)W + off, NN, g->st);
            if ((layers & HBEM_LAYER_SINGLE) && V) copy_out_square(out + 2 * NN, (char*)V + off, NN, g->st);
        }
    }
    HIPC(hipStreamSynchronize(g->st));
    API_END
}

int hbem_mass_matrix(hbem_geometry_t g, double* M) {
    API_BEGIN
    if (!g || !M) throw Error(HBEM_EINVAL, "null argument");
    std::memcpy(M, g->M.data(), sizeof(double) * g->M.size());
    API_END
}

int hbem_projection_factor(hbem_geometry_t g, double* F, int* transpositions) {
    API_BEGIN
    if (!g) throw Error(HBEM_EINVAL, "null geometry");
    if (!g->proj) throw Error(HBEM_EINVAL, "geometry was created without projection");
    if (F) std::memcpy(F, g->F.data(), sizeof(double) * g->F.size());
    if (transpositions) std::memcpy(transpositions, g->tr.data(), sizeof(int) * g->tr.size());
    API_END
}

int hbem_gen_sol_op(hbem_geometry_t g, double k_re, double k_im, double c_o, double c_i, int d, void* T, void* Td,
                    void* Tdd) {
    API_BEGIN
    if (!g) throw Error(HBEM_EINVAL, "null geometry");
    if (d < 0 || d > 2) throw Error(HBEM_EINVAL, "Invalid order of derivative");
    check_k(k_re, k_im, c_i);
    check_k(k_re, k_im, c_o);
    std::lock_guard<std::mutex> lk(g->mu);
    HIPC(hipSetDevice(g->dev));
    const double si = std::sqrt(c_i), so = std::sqrt(c_o);
    cdbl* E = real_positive(k_re, k_im)
                  ? assemble_records(g, {k_re * si, k_re * so}, {k_re, k_re}, {c_i, c_o}, d, true)
                  : assemble_records(g, {k_re * si, k_re * so}, {k_re, k_re}, {c_i, c_o}, d, true,
                                     {k_im * si, k_im * so}, {k_im, k_im});
    const int n = 2 * g->N;
    const size_t nn = (size_t)n * n;
    cdbl* T0 = g->w_T0.as<cdbl>(nn);
    cdbl* T1 = d >= 1 ? g->w_T1.as<cdbl>(nn) : nullptr;
    cdbl* T2 = d >= 2 ? g->w_T2.as<cdbl>(nn) : nullptr;
    hbem::launch_form_T(E, 1, record_values(g, d), 0, -1, 1, g->N, d, (const double*)g->d_M.p, T0, T1, T2, g->st);
    HIPC(hipGetLastError());
    cdbl* Ts[3] = {T0, T1, T2};
    void* hs[3] = {T, Td, Tdd};
    for (int t = 0; t <= d; ++t) {
        if (!hs[t]) continue;
        if (g->proj) project_inplace(g, Ts[t], 1);
        copy_out_square(Ts[t], hs[t], nn, g->st);
    }
    HIPC(hipStreamSynchronize(g->st));
    API_END
}

int hbem_projection(hbem_geometry_t g, const void* T, void* Tp) {
    API_BEGIN
    if (!g || !T || !Tp) throw Error(HBEM_EINVAL, "null argument");
    if (!g->proj) throw Error(HBEM_EINVAL, "geometry was created without projection");
    std::lock_guard<std::mutex> lk(g->mu);
    HIPC(hipSetDevice(g->dev));
    const int n = 2 * g->N;
    const size_t nn = (size_t)n * n;
    cdbl* d = g->w_T0.as<cdbl>(nn);
    HIPC(hipMemcpyAsync(d, T, nn * sizeof(cdbl), hipMemcpyHostToDevice, g->st));
    project_inplace(g, d, 1);
    copy_out_square(d, Tp, nn, g->st);
    HIPC(hipStreamSynchronize(g->st));
    API_END
}

int hbem_tp_A_rhs(hbem_geometry_t g, double k_re, double k_im, double c_o, double c_i, const void* u_inc_N, int nrhs,
                  void* A, void* rhs) {
    API_BEGIN
    check_tp_args(g, u_inc_N, nrhs);
    check_k(k_re, k_im, c_i);
    check_k(k_re, k_im, c_o);
    std::lock_guard<std::mutex> lk(g->mu);
    HIPC(hipSetDevice(g->dev));
    cdbl *T = nullptr, *r = nullptr;
    tp_system(g, k_re, k_im, c_o, c_i, u_inc_N, nrhs, T, r);
    const int n = 2 * g->N;
    if (A) {
        if (g->proj) project_inplace(g, T, 1);
        copy_out_square(T, A, (size_t)n * n, g->st);
    }
    if (rhs) copy_out_square(r, rhs, (size_t)n * nrhs, g->st);
    HIPC(hipStreamSynchronize(g->st));
    API_END
}

int hbem_tp_solve(hbem_geometry_t g, double k_re, double k_im, double c_o, double c_i, const void* u_inc_N, int nrhs,
                  void* sol) {
    API_BEGIN
    check_tp_args(g, u_inc_N, nrhs);
    if (!sol) throw Error(HBEM_EINVAL, "null argument");
    check_k(k_re, k_im, c_i);
    check_k(k_re, k_im, c_o);
    std::lock_guard<std::mutex> lk(g->mu);
    HIPC(hipSetDevice(g->dev));
    cdbl *T = nullptr, *r = nullptr;
    tp_system(g, k_re, k_im, c_o, c_i, u_inc_N, nrhs, T, r);
    const int n = 2 * g->N;
    const size_t nn = (size_t)n * n;
    // solve (solvers.cpp:133-152): finiteness of rhs and T, then zgesv
    int* flag = g->w_flag.as<int>(3);
    HIPC(hipMemsetAsync(flag, 0, 3 * sizeof(int), g->st));
    hbem::flag_nonfinite((const double*)r, 2LL * n * nrhs, flag, g->st);
    hbem::flag_nonfinite((const double*)T, 2LL * (long long)nn, flag + 1, g->st);
    HIPC(hipGetLastError());
    int hf[3] = {0, 0, 0};
    HIPC(hipMemcpyAsync(hf, flag, 2 * sizeof(int), hipMemcpyDeviceToHost, g->st));
    HIPC(hipStreamSynchronize(g->st));
    if (hf[0]) throw Error(HBEM_ENUMERIC, "Failed to solve for traces, right-hand side is undefined");
    if (hf[1]) throw Error(HBEM_ENUMERIC, "Failed to solve for traces, solutions operator is undefined");
    int* piv = g->w_piv.as<int>(n);
    int* perm = g->w_perm.as<int>(n);
    hbem::lu_factor_batched(T, n, 1, piv, perm, g->st);
    hbem::flag_zero_diag(T, n, flag + 2, g->st);
    cdbl* work = g->w_work.as<cdbl>((size_t)n * 8);
    for (int j = 0; j < nrhs; j += 8) {
        const int nc = std::min(8, nrhs - j);
        hbem::lu_solve_thin_batched(T, (long long)n * n, perm, n, 1, r + (size_t)j * n, nc, false, work, g->st);
    }
    HIPC(hipGetLastError());
    HIPC(hipMemcpyAsync(hf + 2, flag + 2, sizeof(int), hipMemcpyDeviceToHost, g->st));
    HIPC(hipStreamSynchronize(g->st));
    if (hf[2]) throw Error(HBEM_ENUMERIC, "zgesv: LU is singular");
    copy_out_square(r, sol, (size_t)n * nrhs, g->st);
    HIPC(hipStreamSynchronize(g->st));
    API_END
}

}  // extern "C"

namespace {

// Standalone dense context for randomized_svd::* on caller matrices.  The
// reference keeps the randomized_svd timers in file-scope statics shared by
// every call (randsvd.cpp:27-47); here they are this context's event log,
// filled while benchmarking is on and read when a timer is queried.
struct Standalone {
    std::mutex mu;
    hipStream_t st = nullptr;
    DBuf T, T1, T2, piv, perm, X, Y, work, u, v, sig, out, W, Wpiv, Wperm, p, p2, ud, tmp, Wq, cpn, cps, cpl;
    bool bench = false;
    EventLog tim;
    void init() {
        if (!st) {
            HIPC(hipSetDevice(g_device));
            HIPC(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
        }
    }
};
Standalone g_sa;

// The eigenvector of the Wielandt matrix W = [[0, T], [T^H, 0]] for sigma as
// randomized_svd::sv_der / sv_der2 take it: the last column of Q of the
// column-pivoted QR of W - sigma I (randsvd.cpp:160-162).  That column is
// orthogonal to every column of the Hermitian W - sigma I but the last
// pivot p, so it is (W - sigma I)^{-1} e_p normalised (up to a phase, which
// neither sigma' nor sigma'' sees): the pivot order comes from
// colpiv_last_pivot_batched, the solve from the blocked LU.  T is the
// caller's host matrix; s.T is overwritten.
void reference_wielandt_vector(Standalone& s, const void* T, int n, double sigma, std::vector<cdbl>& x) {
    const size_t nn = (size_t)n * n;
    const int m2 = 2 * n;
    const size_t mm = (size_t)m2 * m2;
    cdbl* dT = s.T.as<cdbl>(nn);
    HIPC(hipMemcpyAsync(dT, T, nn * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    cdbl* Wq = s.Wq.as<cdbl>(mm);
    hbem::wielandt_build(dT, n, sigma, Wq, s.st);
    int* dl = s.cpl.as<int>(1);
    hbem::colpiv_last_pivot_batched(Wq, (long long)mm, m2, 1, s.cpn.as<double>(2 * (size_t)m2),
                                    s.cps.as<int>(2 * (size_t)m2), dl, s.st);
    int p = 0;
    HIPC(hipMemcpyAsync(&p, dl, sizeof(int), hipMemcpyDeviceToHost, s.st));
    HIPC(hipStreamSynchronize(s.st));
    if (p < 0 || p >= m2) throw Error(HBEM_ENUMERIC, "pivoted QR of the Wielandt matrix failed");
    hbem::wielandt_build(dT, n, sigma, Wq, s.st);
    int* wpiv = s.Wpiv.as<int>(m2);
    int* wperm = s.Wperm.as<int>(m2);
    hbem::lu_factor_batched(Wq, m2, 1, wpiv, wperm, s.st);
    std::vector<cdbl> e(m2, hbem::mk(0, 0));
    e[p] = hbem::mk(1, 0);
    cdbl* de = s.ud.as<cdbl>(m2);
    HIPC(hipMemcpyAsync(de, e.data(), m2 * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    cdbl* wk = s.work.as<cdbl>(2 * (size_t)m2);
    hbem::lu_solve_thin_batched(Wq, (long long)mm, wperm, m2, 1, de, 1, false, wk, s.st);
    x.resize(m2);
    HIPC(hipMemcpyAsync(x.data(), de, m2 * sizeof(cdbl), hipMemcpyDeviceToHost, s.st));
    HIPC(hipStreamSynchronize(s.st));
    double nrm = 0.0;
    for (const auto& z : x) nrm += z.x * z.x + z.y * z.y;
    nrm = std::sqrt(nrm);
    if (!(nrm > 0.0) || !std::isfinite(nrm)) throw Error(HBEM_ENUMERIC, "singular Wielandt matrix");
    for (auto& z : x) z = hbem::mk(z.x / nrm, z.y / nrm);
}

void check_dense_args(const void* T, int n, const void* R, int nc, int q) {
    if (!T || !R) throw Error(HBEM_EINVAL, "null matrix");
    if (n < 1) throw Error(HBEM_EINVAL, "matrix order must be positive");
    if (nc < 1 || nc > 8 || nc > n) throw Error(HBEM_EINVAL, "number of random columns must be in [1, min(8, n)]");
    if (q < 0) throw Error(HBEM_EINVAL, "number of subspace iterations must be >= 0");
}

// Runs LU + rsvd on one host matrix; leaves LU/u/v on the device.
double standalone_sv(const void* T, int n, const void* R, int nc, int q, bool want_vectors) {
    Standalone& s = g_sa;
    s.init();
    const size_t nn = (size_t)n * n;
    cdbl* dT = s.T.as<cdbl>(nn);
    HIPC(hipMemcpyAsync(dT, T, nn * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    int* piv = s.piv.as<int>(n);
    int* perm = s.perm.as<int>(n);
    hipEvent_t e = s.bench ? s.tim.begin(s.st) : nullptr;
    hbem::lu_factor_batched(dT, n, 1, piv, perm, s.st);
    if (s.bench) s.tim.end(s.st, kTimLU, e, (8.0 / 3.0) * (double)n * n * n);
    DenseCtx c;
    c.st = s.st; c.n = n; c.batch = 1; c.nc = nc; c.q = q; c.LU = dT; c.ms = (long long)n * n; c.perm = perm;
    c.F = nullptr; c.FT = nullptr;
    c.tim = s.bench ? &s.tim : nullptr;
    c.X = s.X.as<cdbl>((size_t)n * nc);
    c.Y = s.Y.as<cdbl>((size_t)n * nc);
    c.work = s.work.as<cdbl>(2 * (size_t)n * nc);
    HIPC(hipMemcpyAsync(c.X, R, (size_t)n * nc * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    double* dsig = s.sig.as<double>(1);
    cdbl* du = want_vectors ? s.u.as<cdbl>(n) : nullptr;
    cdbl* dv = want_vectors ? s.v.as<cdbl>(n) : nullptr;
    rsvd_core(c, dsig, du, dv);
    HIPC(hipGetLastError());
    double sigma = 0.0;
    HIPC(hipMemcpyAsync(&sigma, dsig, sizeof(double), hipMemcpyDeviceToHost, s.st));
    HIPC(hipStreamSynchronize(s.st));
    return sigma;
}

}  // namespace

extern "C" {

int hbem_rsvd_sv(const void* T, int n, const void* R, int nc, int q, double* sigma) {
    API_BEGIN
    check_dense_args(T, n, R, nc, q);
    if (!sigma) throw Error(HBEM_EINVAL, "null output");
    std::lock_guard<std::mutex> lk(g_sa.mu);
    *sigma = standalone_sv(T, n, R, nc, q, false);
    API_END
}

// The kernels of hbem_rsvd_sv with every work buffer carved out of this
// device's `scratch`: a device-to-device copy of T, the blocked LU, the
// randomized iteration, sigma written to the caller's device double.  Only
// enqueues work on `stream`; nothing here allocates or waits.  Every buffer is
// written before it is read, so the array needs no clearing between calls.
int hbem_rsvd_sv_noalloc(const void* T_dev, int n, const void* R_dev, int nc, int q, double* sigma_dev, void* stream) {
    API_BEGIN
    check_dense_args(T_dev, n, R_dev, nc, q);
    if (!sigma_dev) throw Error(HBEM_EINVAL, "null output");
    if (n > kNaMaxN) throw Error(HBEM_EINVAL, "matrix order exceeds the no-allocation limit of 2048");
    int dev = 0;
    HIPC(hipGetDevice(&dev));
    unsigned char* base = (unsigned char*)scratch_on(dev);
    const hipStream_t st = (hipStream_t)stream;
    const size_t nn = (size_t)n * n;
    cdbl* LU = (cdbl*)base;
    base += al256(sizeof(cdbl) * nn);
    int* piv = (int*)base;
    base += al256(sizeof(int) * (size_t)n);
    int* perm = (int*)base;
    base += al256(sizeof(int) * (size_t)n);
    const size_t thin = al256(sizeof(cdbl) * (size_t)n * nc);
    DenseCtx c;
    c.st = st; c.n = n; c.batch = 1; c.nc = nc; c.q = q; c.LU = LU; c.ms = (long long)nn; c.perm = perm;
    c.F = nullptr; c.FT = nullptr;
    c.X = (cdbl*)base;
    c.Y = (cdbl*)(base + thin);
    c.work = (cdbl*)(base + 2 * thin);
    HIPC(hipMemcpyAsync(LU, T_dev, nn * sizeof(cdbl), hipMemcpyDeviceToDevice, st));
    hbem::lu_factor_batched(LU, n, 1, piv, perm, st);
    HIPC(hipMemcpyAsync(c.X, R_dev, (size_t)n * nc * sizeof(cdbl), hipMemcpyDeviceToDevice, st));
    rsvd_core(c, sigma_dev, nullptr, nullptr);
    HIPC(hipGetLastError());
    API_END
}

int hbem_rsvd_sv_der(const void* T, const void* Td, int n, const void* R, int nc, int q, double* out2) {
    API_BEGIN
    check_dense_args(T, n, R, nc, q);
    if (!Td || !out2) throw Error(HBEM_EINVAL, "null argument");
    std::lock_guard<std::mutex> lk(g_sa.mu);
    Standalone& s = g_sa;
    double sigma = standalone_sv(T, n, R, nc, q, true);
    const size_t nn = (size_t)n * n;
    const int m2 = 2 * n;
    cdbl* dT1 = s.T1.as<cdbl>(nn);
    HIPC(hipMemcpyAsync(dT1, Td, nn * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    std::vector<cdbl> x;
    reference_wielandt_vector(s, T, n, sigma, x);
    // sigma' = Re(x^H [T' x_2; T'^H x_1]) (randsvd.cpp:163-167)
    cdbl* dx = s.p.as<cdbl>(m2);
    cdbl* dp = s.p2.as<cdbl>(m2);
    HIPC(hipMemcpyAsync(dx, x.data(), m2 * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    hbem::gemv_batched(dT1, 0, dx + n, dp, n, 1, false, s.st);
    hbem::gemv_batched(dT1, 0, dx, dp + n, n, 1, true, s.st);
    std::vector<cdbl> hp(m2);
    HIPC(hipMemcpyAsync(hp.data(), dp, m2 * sizeof(cdbl), hipMemcpyDeviceToHost, s.st));
    HIPC(hipStreamSynchronize(s.st));
    double der = 0.0;
    for (int l = 0; l < m2; ++l) der += x[l].x * hp[l].x + x[l].y * hp[l].y;
    out2[0] = sigma;
    out2[1] = der;
    API_END
}

// randomized_svd::sv_der2 (randsvd.cpp:171-216): the eigenvector x of the
// Wielandt matrix W = [[0,T],[T^H,0]] for sigma as the reference takes it
// (reference_wielandt_vector); the bordered system follows the reference.
int hbem_rsvd_sv_der2(const void* T, const void* Td, const void* Tdd, int n, const void* R, int nc, int q,
                      double* out3) {
    API_BEGIN
    check_dense_args(T, n, R, nc, q);
    if (!Td || !Tdd || !out3) throw Error(HBEM_EINVAL, "null argument");
    std::lock_guard<std::mutex> lk(g_sa.mu);
    Standalone& s = g_sa;
    double sigma = standalone_sv(T, n, R, nc, q, true);
    const size_t nn = (size_t)n * n;
    const int m2 = 2 * n;
    cdbl* dT1 = s.T1.as<cdbl>(nn);
    cdbl* dT2 = s.T2.as<cdbl>(nn);
    HIPC(hipMemcpyAsync(dT1, Td, nn * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    HIPC(hipMemcpyAsync(dT2, Tdd, nn * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    std::vector<cdbl> x;
    reference_wielandt_vector(s, T, n, sigma, x);
    // sigma' = Re(x^H [T' x_2; T'^H x_1]); then u = x normalised by its
    // largest-modulus entry (randsvd.cpp:185-198)
    cdbl* dx = s.p.as<cdbl>(m2);
    cdbl* dpx = s.p2.as<cdbl>(m2);
    HIPC(hipMemcpyAsync(dx, x.data(), m2 * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    hbem::gemv_batched(dT1, 0, dx + n, dpx, n, 1, false, s.st);
    hbem::gemv_batched(dT1, 0, dx, dpx + n, n, 1, true, s.st);
    std::vector<cdbl> hpx(m2);
    HIPC(hipMemcpyAsync(hpx.data(), dpx, m2 * sizeof(cdbl), hipMemcpyDeviceToHost, s.st));
    HIPC(hipStreamSynchronize(s.st));
    double der = 0.0;
    for (int l = 0; l < m2; ++l) der += x[l].x * hpx[l].x + x[l].y * hpx[l].y;
    double best = 0.0;
    int m = 5 < m2 ? 5 : 0;
    for (int l = 0; l < m2; ++l) {
        double a = std::sqrt(x[l].x * x[l].x + x[l].y * x[l].y);
        if (a > best) { best = a; m = l; }
    }
    const std::complex<double> xm(x[m].x, x[m].y);
    std::vector<cdbl> u(m2);
    for (int l = 0; l < m2; ++l) {
        std::complex<double> z = std::complex<double>(x[l].x, x[l].y) / xm;
        u[l] = hbem::mk(z.real(), z.imag());
    }
    cdbl* W = s.W.as<cdbl>((size_t)m2 * m2);
    // s.T holds the LU factors of T; W is built from the caller's T
    HIPC(hipMemcpyAsync(s.T.p, T, nn * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    hbem::wielandt_build((const cdbl*)s.T.p, n, sigma, W, s.st);
    cdbl* du = s.p.as<cdbl>(m2);
    HIPC(hipMemcpyAsync(du, u.data(), m2 * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    std::vector<cdbl> negu(m2);
    for (int l = 0; l < m2; ++l) negu[l] = hbem::mk(-u[l].x, -u[l].y);
    HIPC(hipMemcpyAsync(W + (size_t)m * m2, negu.data(), m2 * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    int* wpiv = s.Wpiv.as<int>(m2);
    int* wperm = s.Wperm.as<int>(m2);
    hbem::lu_factor_batched(W, m2, 1, wpiv, wperm, s.st);
    // p = [T' u2; T'^H u1]
    cdbl* p = s.p2.as<cdbl>(m2);
    hbem::gemv_batched(dT1, 0, du + n, p, n, 1, false, s.st);
    hbem::gemv_batched(dT1, 0, du, p + n, n, 1, true, s.st);
    cdbl* wk = s.work.as<cdbl>(2 * (size_t)m2);
    hbem::lu_solve_thin_batched(W, (long long)m2 * m2, wperm, m2, 1, p, 1, false, wk, s.st);   // p <- W^{-1} p
    std::vector<cdbl> ud(m2);
    HIPC(hipMemcpyAsync(ud.data(), p, m2 * sizeof(cdbl), hipMemcpyDeviceToHost, s.st));
    HIPC(hipStreamSynchronize(s.st));
    for (auto& z : ud) z = hbem::mk(-z.x, -z.y);   // u_der = -W^{-1} p
    const std::complex<double> t(ud[m].x, ud[m].y);
    ud[m] = hbem::mk(0, 0);
    cdbl* dud = s.ud.as<cdbl>(m2);
    HIPC(hipMemcpyAsync(dud, ud.data(), m2 * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    cdbl* pp = s.tmp.as<cdbl>(2 * (size_t)m2);
    cdbl* p2 = pp + m2;
    hbem::gemv_batched(dT1, 0, dud + n, pp, n, 1, false, s.st);
    hbem::gemv_batched(dT1, 0, dud, pp + n, n, 1, true, s.st);
    hbem::gemv_batched(dT2, 0, du + n, p2, n, 1, false, s.st);
    hbem::gemv_batched(dT2, 0, du, p2 + n, n, 1, true, s.st);
    std::vector<cdbl> hp(m2), hp2(m2);
    HIPC(hipMemcpyAsync(hp.data(), pp, m2 * sizeof(cdbl), hipMemcpyDeviceToHost, s.st));
    HIPC(hipMemcpyAsync(hp2.data(), p2, m2 * sizeof(cdbl), hipMemcpyDeviceToHost, s.st));
    HIPC(hipStreamSynchronize(s.st));
    std::vector<cdbl> rhs(m2);
    for (int l = 0; l < m2; ++l) {
        std::complex<double> v = std::complex<double>(hp2[l].x, hp2[l].y) +
                                 2.0 * (std::complex<double>(hp[l].x, hp[l].y) - t * std::complex<double>(ud[l].x, ud[l].y));
        rhs[l] = hbem::mk(v.real(), v.imag());
    }
    HIPC(hipMemcpyAsync(p, rhs.data(), m2 * sizeof(cdbl), hipMemcpyHostToDevice, s.st));
    hbem::lu_solve_thin_batched(W, (long long)m2 * m2, wperm, m2, 1, p, 1, false, wk, s.st);
    cdbl sol;
    HIPC(hipMemcpyAsync(&sol, p + m, sizeof(cdbl), hipMemcpyDeviceToHost, s.st));
    HIPC(hipStreamSynchronize(s.st));
    out3[0] = sigma;
    out3[1] = der;
    out3[2] = -sol.x;
    API_END
}

}  // extern "C"

namespace {

// out_head = T_p^(t) x_tail, out_tail = T_p^(t)H x_head for the 2n-vectors X of
// the batch (2n x nb), with T_p^(t) = F^{-1} Tt F^{-T} (Tt: n x n x nb) or Tt
// itself without projection.  h: scratch of 4 n nb complex.
void apply_pair_op(hbem_geometry* g, const cdbl* Tt, const cdbl* X, cdbl* out, int nb, cdbl* h) {
    const int n = 2 * g->N;
    const long long nn = (long long)n * n, m2 = 2LL * n;
    cdbl *xh = h, *xt = h + (size_t)n * nb, *z = h + 2 * (size_t)n * nb, *y = h + 3 * (size_t)n * nb;
    hbem::copy_blocks_batched(X, m2, 0, xh, n, 0, n, nb, g->st);
    hbem::copy_blocks_batched(X, m2, n, xt, n, 0, n, nb, g->st);
    for (int part = 0; part < 2; ++part) {
        const cdbl* src = part == 0 ? xt : xh;
        const bool adj = part == 1;
        const long long off = part == 0 ? 0 : n;
        if (g->proj) {
            const DCsr& A = g->s_FinvT;
            const DCsr& Bm = g->s_Finv;
            hbem::csr_apply_batched((const int*)A.rp.p, (const int*)A.ci.p, (const double*)A.v.p, n, src, z, nb, g->st);
            hbem::gemv_batched(Tt, nn, z, y, n, nb, adj, g->st);
            hbem::csr_apply_batched((const int*)Bm.rp.p, (const int*)Bm.ci.p, (const double*)Bm.v.p, n, y, z, nb, g->st);
            hbem::copy_blocks_batched(z, n, 0, out, m2, off, n, nb, g->st);
        } else {
            hbem::gemv_batched(Tt, nn, src, y, n, nb, adj, g->st);
            hbem::copy_blocks_batched(y, n, 0, out, m2, off, n, nb, g->st);
        }
    }
}

// The sweep shared by hbem_sigma_sweep and hbem_sigma_sweep_der2: sigma for
// every k, dsigma/dk when dsigma is given (operators of order D >= 1), and
// d2sigma/dk2 when d2sigma is given (D = 2).
// sigma of the matrices idx of a batch from their FP64 T (T0, stride n^2) with
// the FP64 factorisation: the fallback of the mixed-precision sweep
void sweep_fp64_subset(hbem_geometry* g, const cdbl* T0, const std::vector<int>& idx, const cdbl* dR, int nc, int q,
                       double* sigma_host) {
    const int n = 2 * g->N, m = (int)idx.size();
    const size_t nn = (size_t)n * n;
    if (m == 0) return;
    cdbl* Tf = g->w_T1.as<cdbl>(nn * m);
    for (int j = 0; j < m; ++j)
        HIPC(hipMemcpyAsync(Tf + j * nn, T0 + (size_t)idx[j] * nn, nn * sizeof(cdbl), hipMemcpyDeviceToDevice, g->st));
    int* piv = g->w_bpiv.as<int>((size_t)n * m);
    int* perm = g->w_bperm.as<int>((size_t)n * m);
    hbem::lu_factor_batched(Tf, n, m, piv, perm, g->st);
    DenseCtx c;
    c.st = g->st; c.n = n; c.batch = m; c.nc = nc; c.q = q; c.LU = Tf; c.ms = (long long)nn; c.perm = perm;
    c.F = g->proj ? &g->s_F : nullptr;
    c.FT = g->proj ? &g->s_FT : nullptr;
    c.X = g->w_X.as<cdbl>((size_t)n * nc * m);
    c.Y = g->w_Y.as<cdbl>((size_t)n * nc * m);
    c.work = g->w_work.as<cdbl>(2 * (size_t)n * nc * m);
    hbem::replicate_batched(dR, (long long)n * nc, m, c.X, g->st);
    double* dsig = g->w_d2.as<double>(m);
    rsvd_core(c, dsig, nullptr, nullptr);
    std::vector<double> out(m);
    HIPC(hipMemcpyAsync(out.data(), dsig, m * sizeof(double), hipMemcpyDeviceToHost, g->st));
    HIPC(hipStreamSynchronize(g->st));
    for (int j = 0; j < m; ++j) sigma_host[idx[j]] = out[j];
}

// mixed >= 0 (D = 0 only): the dense stage in mixed precision with `mixed`
// refinement steps per solve; fp64_used (may be null) marks the k recomputed
// in FP64.
void sweep_run(hbem_geometry* g, const double* ks, int nk, double c_o, double c_i, const void* R, int nc, int q, int D,
               double* sigma, double* dsigma, double* d2sigma, int mixed = -1, int* fp64_used = nullptr,
               int mixed_inner = -1) {
    const int n = 2 * g->N;
    const size_t nn = (size_t)n * n;
    const bool mx = mixed >= 0 && D == 0 && !d2sigma;
    // Batches of B <= 256 wavenumbers give the dense stage (one workgroup per
    // matrix in the panel factorisation and the thin solves) up to one matrix
    // per CU.  B is bounded by the free device memory: records (and local
    // matrices and chunk partials where a wavenumber takes the node loops) and
    // T, T', T'' per wavenumber (and the bordered systems of the sigma'' stage).
    const bool tdiff = sweep_tdiff(ks, nk);
    const double si = std::sqrt(c_i), so = std::sqrt(c_o);
    std::vector<double> all;
    for (int i = 0; i < nk; ++i) all.push_back(ks[i] * std::max(si, so));
    const size_t per = records_bytes_per_k(g, all, D, tdiff ? 1 : 2, 2, true) + dense_bytes_per_k(n, D, nc) +
                       (d2sigma ? der2_bytes_per_k(n) : 0) + (mx ? mixed_bytes_per_k(n, nc) : 0);
    const int B = sweep_batch(per, usable_device_bytes(g->work_held()), nk);
    cdbl* dR = g->w_R.as<cdbl>((size_t)n * nc);
    HIPC(hipMemcpyAsync(dR, R, (size_t)n * nc * sizeof(cdbl), hipMemcpyHostToDevice, g->st));
    for (int k0 = 0; k0 < nk; k0 += B) {
        const int nb = std::min(B, nk - k0);
        bool allpos = true;
        for (int b = 0; b < nb; ++b) allpos = allpos && ks[k0 + b] > 0.0;
        // inner slots 0..nb-1, outer nb..2nb-1
        std::vector<double> kap(2 * nb), kr(2 * nb), cv(2 * nb);
        for (int b = 0; b < nb; ++b) {
            const double k = ks[k0 + b];
            kap[b] = k * si; kr[b] = k; cv[b] = c_i;
            kap[nb + b] = k * so; kr[nb + b] = k; cv[nb + b] = c_o;
        }
        const std::vector<double> zero(allpos ? 0 : kap.size(), 0.0);
        cdbl* E = assemble_records(g, kap, kr, cv, D, true, zero, zero, true, tdiff);
        cdbl* T0 = g->w_T0.as<cdbl>(nn * nb);
        cdbl* T1 = D >= 1 ? g->w_T1.as<cdbl>(nn * nb) : nullptr;
        cdbl* T2 = D >= 2 ? g->w_T2.as<cdbl>(nn * nb) : nullptr;
        // mixed precision: T formed in FP64 (kept for the residuals) and in FP32
        // (factorised on the FP32 matrix cores) in one pass
        cflt* T32 = mx ? g->w_T32.as<cflt>(nn * nb) : nullptr;
        hipEvent_t e0 = g->prof ? g->plog.begin(g->st) : nullptr;
        hbem::launch_form_T(E, nb, record_values(g, D), 0, -1, nb, g->N, D, (const double*)g->d_M.p, T0, T1, T2, g->st, 0, T32);
        if (g->prof) g->plog.end(g->st, kProfFormT, e0);
        int* piv = g->w_piv.as<int>((size_t)n * nb);
        int* perm = g->w_perm.as<int>((size_t)n * nb);
        if (g->prof) e0 = g->plog.begin(g->st);
        GemmTimer gt(&g->plog, kProfGemm);
        if (mx) {
            hbem::lu_factor_batched_f32(T32, n, nb, piv, perm, g->st, g->prof ? &gt : nullptr);
        } else {
            hbem::lu_factor_batched(T0, n, nb, piv, perm, g->st, g->prof ? &gt : nullptr);
        }
        if (g->prof) {
            g->plog.end(g->st, kProfLU, e0, (8.0 / 3.0) * (double)n * n * n * nb);
            e0 = g->plog.begin(g->st);
        }
        DenseCtx c;
        c.st = g->st; c.n = n; c.batch = nb; c.nc = nc; c.q = q; c.LU = T0; c.ms = (long long)nn; c.perm = perm;
        c.F = g->proj ? &g->s_F : nullptr;
        c.FT = g->proj ? &g->s_FT : nullptr;
        c.X = g->w_X.as<cdbl>((size_t)n * nc * nb);
        c.Y = g->w_Y.as<cdbl>((size_t)n * nc * nb);
        c.work = g->w_work.as<cdbl>(2 * (size_t)n * nc * nb);
        int* flag = nullptr;
        if (mx) {
            c.LU32 = T32;
            c.T64 = T0;
            c.refine = mixed;
            c.refine_inner = mixed_inner < 0 ? mixed : mixed_inner;
            c.rtol = kMixedTol;
            flag = g->w_flag2.as<int>(nb);
            hbem::fill_int(flag, nb, mixed > 0 ? 0 : 1, g->st);   // no refinement: nothing certifies the solves
            c.flag = flag;
            c.rprev = g->w_rprev.as<double>(nb);
            c.rb = g->w_rb.as<cdbl>((size_t)n * nc * nb);
            c.rr = g->w_rr.as<cdbl>((size_t)n * nc * nb);
            c.rpart = g->w_rpart.as<cdbl>(hbem::residual_part_count(n, nc, nb));
        }
        hbem::replicate_batched(dR, (long long)n * nc, nb, c.X, g->st);
        double* dsig = g->w_sig.as<double>(nb);
        cdbl* du = D ? g->w_u.as<cdbl>((size_t)n * nb) : nullptr;
        cdbl* dv = D ? g->w_v.as<cdbl>((size_t)n * nb) : nullptr;
        rsvd_core(c, dsig, du, dv);
        HIPC(hipMemcpyAsync(sigma + k0, dsig, nb * sizeof(double), hipMemcpyDeviceToHost, g->st));
        if (mx) {
            // k whose refinement did not converge: sigma again with the FP64 factorisation
            std::vector<int> hf(nb);
            HIPC(hipMemcpyAsync(hf.data(), flag, nb * sizeof(int), hipMemcpyDeviceToHost, g->st));
            HIPC(hipStreamSynchronize(g->st));
            std::vector<int> idx;
            for (int b = 0; b < nb; ++b) {
                if (hf[b]) idx.push_back(b);
                if (fp64_used) fp64_used[k0 + b] = hf[b] ? 1 : 0;
            }
            sweep_fp64_subset(g, T0, idx, dR, nc, q, sigma + k0);
        }
        if (D) {
            cdbl* a = g->w_a.as<cdbl>((size_t)n * nb);
            cdbl* bb = g->w_b.as<cdbl>((size_t)n * nb);
            if (g->proj) {
                const DCsr& S = g->s_FinvT;
                hbem::csr_apply_batched((const int*)S.rp.p, (const int*)S.ci.p, (const double*)S.v.p, n, du, a, nb, g->st);
                hbem::csr_apply_batched((const int*)S.rp.p, (const int*)S.ci.p, (const double*)S.v.p, n, dv, bb, nb, g->st);
            } else {
                HIPC(hipMemcpyAsync(a, du, (size_t)n * nb * sizeof(cdbl), hipMemcpyDeviceToDevice, g->st));
                HIPC(hipMemcpyAsync(bb, dv, (size_t)n * nb * sizeof(cdbl), hipMemcpyDeviceToDevice, g->st));
            }
            double* dd = g->w_dsig.as<double>((size_t)nb * (1 + hbem::kBilinearParts));
            hbem::bilinear_re_batched(T1, (long long)nn, a, bb, n, nb, dd, dd + nb, g->st);
            if (dsigma) HIPC(hipMemcpyAsync(dsigma + k0, dd, nb * sizeof(double), hipMemcpyDeviceToHost, g->st));
        }
        if (d2sigma) {
            // randomized_svd::sv_der2's bordered system (randsvd.cpp:171-216) for
            // every k of the batch, on T_p formed explicitly: T again from the
            // records (T0 holds its LU factors), projected through the
            // bordered matrix's storage.
            const int m2 = 2 * n;
            cdbl* Tp = g->w_Tp.as<cdbl>(nn * nb);
            cdbl* Bw = g->w_B.as<cdbl>(4 * nn * nb);
            hbem::launch_form_T(E, nb, record_values(g, D), 0, -1, nb, g->N, D, (const double*)g->d_M.p, Tp, nullptr, nullptr, g->st, 0, nullptr,
                                true);
            if (g->proj) project_inplace(g, Tp, nb, Bw);
            int* mv = g->w_mv.as<int>(nb);
            cdbl* vec = g->w_bvec.as<cdbl>(16 * (size_t)n * nb);
            cdbl *X = vec, *P = vec + (size_t)m2 * nb, *Pd = vec + 2 * (size_t)m2 * nb, *P2 = vec + 3 * (size_t)m2 * nb;
            cdbl *h = vec + 4 * (size_t)m2 * nb, *wk = vec + 6 * (size_t)m2 * nb, *tv = vec + 7 * (size_t)m2 * nb;
            hbem::border_prep_batched(du, dv, n, nb, mv, X, g->st);
            hbem::border_build_batched(Tp, n, nb, dsig, mv, X, Bw, g->st);
            int* bpiv = g->w_bpiv.as<int>((size_t)m2 * nb);
            int* bperm = g->w_bperm.as<int>((size_t)m2 * nb);
            hbem::lu_factor_batched(Bw, m2, nb, bpiv, bperm, g->st);
            apply_pair_op(g, T1, X, P, nb, h);                       // p = [T_p' u_2; T_p'^H u_1]
            hbem::lu_solve_thin_batched(Bw, 4LL * (long long)nn, bperm, m2, nb, P, 1, false, wk, g->st);
            hbem::border_negate_pick_batched(P, n, nb, mv, tv, g->st);   // P = u', tv = t
            apply_pair_op(g, T1, P, Pd, nb, h);                      // [T_p' u'_2; T_p'^H u'_1]
            apply_pair_op(g, T2, X, P2, nb, h);                      // [T_p'' u_2; T_p''^H u_1]
            hbem::border_rhs_batched(Pd, P2, P, tv, n, nb, Pd, g->st);
            hbem::lu_solve_thin_batched(Bw, 4LL * (long long)nn, bperm, m2, nb, Pd, 1, false, wk, g->st);
            double* d2 = g->w_d2.as<double>(nb);
            hbem::border_final_batched(Pd, n, nb, mv, d2, g->st);
            HIPC(hipMemcpyAsync(d2sigma + k0, d2, nb * sizeof(double), hipMemcpyDeviceToHost, g->st));
        }
        if (g->prof) g->plog.end(g->st, kProfRsvd, e0);
        HIPC(hipGetLastError());
    }
    HIPC(hipStreamSynchronize(g->st));
}

void check_sweep_args(hbem_geometry* g, const double* ks, int nk, double c_o, double c_i, const void* R, int nc, int q,
                      const double* sigma) {
    if (!g || !ks || !R || !sigma) throw Error(HBEM_EINVAL, "null argument");
    if (nk < 0) throw Error(HBEM_EINVAL, "negative number of wavenumbers");
    check_dense_args(ks, 2 * g->N, R, nc, q);
    for (int i = 0; i < nk; ++i) { check_k(ks[i], 0.0, c_i); check_k(ks[i], 0.0, c_o); }
}

}  // namespace

extern "C" {

int hbem_sigma_sweep(hbem_geometry_t g, const double* ks, int nk, double c_o, double c_i, const void* R, int nc, int q,
                     int want_der, double* sigma, double* dsigma) {
    API_BEGIN
    check_sweep_args(g, ks, nk, c_o, c_i, R, nc, q, sigma);
    if (want_der && !dsigma) throw Error(HBEM_EINVAL, "null dsigma");
    std::lock_guard<std::mutex> lk(g->mu);
    HIPC(hipSetDevice(g->dev));
    const int D = want_der ? (want_der >= 2 ? 2 : 1) : 0;
    sweep_run(g, ks, nk, c_o, c_i, R, nc, q, D, sigma, D ? dsigma : nullptr, nullptr);
    API_END
}

int hbem_sigma_sweep_der2(hbem_geometry_t g, const double* ks, int nk, double c_o, double c_i, const void* R, int nc,
                          int q, double* sigma, double* dsigma, double* d2sigma) {
    API_BEGIN
    check_sweep_args(g, ks, nk, c_o, c_i, R, nc, q, sigma);
    if (!dsigma || !d2sigma) throw Error(HBEM_EINVAL, "null argument");
    std::lock_guard<std::mutex> lk(g->mu);
    HIPC(hipSetDevice(g->dev));
    sweep_run(g, ks, nk, c_o, c_i, R, nc, q, 2, sigma, dsigma, d2sigma);
    API_END
}

int hbem_sigma_sweep_mixed(hbem_geometry_t g, const double* ks, int nk, double c_o, double c_i, const void* R, int nc,
                           int q, int refine, int refine_inner, double* sigma, int* fp64_used) {
    API_BEGIN
    check_sweep_args(g, ks, nk, c_o, c_i, R, nc, q, sigma);
    if (refine < 0 || refine > 20 || refine_inner > 20)
        throw Error(HBEM_EINVAL, "number of refinement steps must be in [0, 20]");
    std::lock_guard<std::mutex> lk(g->mu);
    HIPC(hipSetDevice(g->dev));
    sweep_run(g, ks, nk, c_o, c_i, R, nc, q, 0, sigma, nullptr, nullptr, refine, fp64_used, refine_inner);
    API_END
}

}  // extern "C"

namespace {

// Work space of hbem_sigma_sweep_multi (one per process; calls are serialised),
// and the hipGraphs of its device phases, one per subset shape: a subset's
// device work (entry concatenation, assembly, T, LU, randomized SVD) is
// captured on first use and replayed by later calls with the same instances,
// sizes and buffers.  Everything a replay reads from the host side is
// uploaded before the launch into buffers the graph reads in place.
struct GraphEntry {
    std::vector<const void*> key;
    hipGraphExec_t exec = nullptr;
};
struct MultiWork {
    std::mutex mu;
    DBuf T, piv, perm, X, Y, work, sig, desc, descT, roff, nrow, Rall;
    std::vector<std::unique_ptr<RecBufs>> rec;   // per instance of a subset
    RecScratch scr;
    std::vector<GraphEntry> graphs;
    void drop_graphs() {
        for (auto& e : graphs) (void)hipGraphExecDestroy(e.exec);
        graphs.clear();
    }
};
MultiWork g_multi;

}  // namespace

// Graphs that name a geometry being destroyed (or released) are dropped: a
// later context may reuse its addresses.
void multi_forget(hbem_geometry* g) {
    std::lock_guard<std::mutex> lk(g_multi.mu);
    auto& v = g_multi.graphs;
    for (size_t i = 0; i < v.size();) {
        if (std::find(v[i].key.begin(), v[i].key.end(), (const void*)g) != v[i].key.end()) {
            (void)hipGraphExecDestroy(v[i].exec);
            v.erase(v.begin() + i);
        } else {
            ++i;
        }
    }
}

namespace {

bool graphs_enabled() {
    const char* e = std::getenv("HBEM_NO_GRAPH");
    return !(e && e[0] && e[0] != '0');
}

// One bucket subset of hbem_sigma_sweep_multi: instances `ids` (all padded to
// order n_pad, all factorised in steps of `panels` sub-panels by their own order),
// their nk wavenumbers each.  T of instance i, k j is matrix i_local nk + j of one
// batch of order n_pad (identity in the padding), factorised and reduced to sigma by
// the batched dense stage.
void multi_subset(const std::vector<hbem_geometry*>& G, const std::vector<int>& ids, int n_pad, int panels, const double* ks, int nk,
                  double c_o, const double* c_i, const void* const* R, int nc, int q, double* sigma) {
    MultiWork& w = g_multi;
    hbem_geometry* g0 = G[ids[0]];
    const hipStream_t st = g0->st;
    const int m = (int)ids.size();
    const size_t nn = (size_t)n_pad * n_pad;
    const int batch = m * nk;
    // ---- host side: every table the device phase reads, uploaded first ----
    std::vector<RecJob> jobs;
    while ((int)w.rec.size() < m) w.rec.push_back(std::make_unique<RecBufs>());
    for (int a = 0; a < m; ++a) {
        const int i = ids[a];
        std::vector<double> kap(2 * nk), kr(2 * nk), cv(2 * nk);
        for (int j = 0; j < nk; ++j) {
            const double k = ks[(size_t)i * nk + j];
            kap[j] = k * std::sqrt(c_i[i]); kr[j] = k; cv[j] = c_i[i];
            kap[nk + j] = k * std::sqrt(c_o); kr[nk + j] = k; cv[nk + j] = c_o;
        }
        jobs.push_back(prepare_records(G[i], *w.rec[a], w.scr, st, kap, kr, cv, 0, true, {}, {}, true,
                                       sweep_tdiff(ks + (size_t)i * nk, nk)));
    }
    std::vector<hbem::CsrDesc> desc(batch), descT(batch);
    std::vector<long long> roff(batch);
    std::vector<int> nrow(batch);
    std::vector<cdbl> Rall;
    for (int a = 0; a < m; ++a) {
        hbem_geometry* g = G[ids[a]];
        const int n = 2 * g->N;
        const long long off = (long long)Rall.size();
        const cdbl* Rh = (const cdbl*)R[ids[a]];
        Rall.insert(Rall.end(), Rh, Rh + (size_t)n * nc);
        for (int j = 0; j < nk; ++j) {
            const int b = a * nk + j;
            if (g->proj) {
                desc[b] = {(const int*)g->s_F.rp.p, (const int*)g->s_F.ci.p, (const double*)g->s_F.v.p, n};
                descT[b] = {(const int*)g->s_FT.rp.p, (const int*)g->s_FT.ci.p, (const double*)g->s_FT.v.p, n};
            }
            roff[b] = off;
            nrow[b] = n;
        }
    }
    const hbem::CsrDesc* dF = g0->proj ? upload(w.desc, desc, st) : nullptr;
    const hbem::CsrDesc* dFT = g0->proj ? upload(w.descT, descT, st) : nullptr;
    const cdbl* dRall = upload(w.Rall, Rall, st);
    const long long* droff = upload(w.roff, roff, st);
    const int* dnrow = upload(w.nrow, nrow, st);
    // ---- every device buffer at its final size before the device phase ----
    cdbl* T = w.T.as<cdbl>(nn * batch);
    int* piv = w.piv.as<int>((size_t)n_pad * batch);
    int* perm = w.perm.as<int>((size_t)n_pad * batch);
    cdbl* X = w.X.as<cdbl>((size_t)n_pad * nc * batch);
    cdbl* Y = w.Y.as<cdbl>((size_t)n_pad * nc * batch);
    cdbl* work = w.work.as<cdbl>(2 * (size_t)n_pad * nc * batch);
    double* dsig = w.sig.as<double>(batch);
    HIPC(hipStreamSynchronize(st));   // uploads done; nothing below reads host memory
    // ---- device phase ----
    auto device_phase = [&]() {
        for (int a = 0; a < m; ++a) {
            hbem_geometry* g = G[ids[a]];
            const int n = 2 * g->N;
            const cdbl* E = launch_records(jobs[a]);
            hbem::launch_form_T(E, nk, hbem::kRecValues, 0, -1, nk, g->N, 0, (const double*)g->d_M.p, T + (size_t)a * nk * nn, nullptr,
                                nullptr, st, n_pad);
            if (n < n_pad) hbem::launch_pad_identity(T + (size_t)a * nk * nn, n, n_pad, nk, st);
        }
        hbem::lu_factor_batched(T, n_pad, batch, piv, perm, st, nullptr, panels);
        DenseCtx c;
        c.st = st; c.n = n_pad; c.batch = batch; c.nc = nc; c.q = q; c.LU = T; c.ms = (long long)nn; c.perm = perm;
        c.F = nullptr;
        c.FT = nullptr;
        c.Fm = dF;
        c.FTm = dFT;
        c.X = X;
        c.Y = Y;
        c.work = work;
        hbem::replicate_padded(dRall, droff, dnrow, n_pad, nc, batch, c.X, st);
        rsvd_core(c, dsig, nullptr, nullptr);
    };
    if (graphs_enabled()) {
        std::vector<const void*> key;
        for (int a = 0; a < m; ++a) key.push_back(G[ids[a]]);
        key.push_back((const void*)(size_t)nk);
        key.push_back((const void*)(size_t)nc);
        key.push_back((const void*)(size_t)q);
        key.push_back((const void*)(size_t)n_pad);
        key.push_back((const void*)(size_t)panels);
        const void* bufs[] = {dF, dFT, dRall, droff, dnrow, T, piv, perm, X, Y, work, dsig, w.scr.E.p, w.scr.L.p,
                              w.scr.part.p};
        // the ways its columns take, and the tables each reads
        for (const RecJob& J : jobs) {
            key.push_back((const void*)(size_t)J.tdiff);
            for (const void* p : {(const void*)J.kap, (const void*)J.kr, (const void*)J.cv, (const void*)J.cols}) key.push_back(p);
            for (const RecGroup& r : J.groups)
                for (const void* p : {(const void*)(size_t)(r.tier + 1), (const void*)(size_t)r.start, (const void*)(size_t)r.count,
                                      (const void*)r.kap, (const void*)r.kr, (const void*)r.cv})
                    key.push_back(p);
        }
        key.insert(key.end(), std::begin(bufs), std::end(bufs));
        GraphEntry* ge = nullptr;
        for (auto& e : w.graphs)
            if (e.key == key) ge = &e;
        if (!ge) {
            hipGraph_t graph = nullptr;
            HIPC(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
            device_phase();
            const hipError_t ec = hipStreamEndCapture(st, &graph);
            HIPC(ec);
            hipGraphExec_t exec = nullptr;
            const hipError_t ei = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
            (void)hipGraphDestroy(graph);
            HIPC(ei);
            if (w.graphs.size() >= 16) w.drop_graphs();
            w.graphs.push_back({key, exec});
            ge = &w.graphs.back();
        }
        HIPC(hipGraphLaunch(ge->exec, st));
    } else {
        device_phase();
    }
    HIPC(hipGetLastError());
    std::vector<double> out(batch);
    HIPC(hipMemcpyAsync(out.data(), dsig, batch * sizeof(double), hipMemcpyDeviceToHost, st));
    HIPC(hipStreamSynchronize(st));
    for (int a = 0; a < m; ++a)
        for (int j = 0; j < nk; ++j) sigma[(size_t)ids[a] * nk + j] = out[(size_t)a * nk + j];
}

}  // namespace

extern "C" {

int hbem_sigma_sweep_multi(const hbem_geometry_t* geoms, int ninst, const double* ks, int nk, double c_o,
                           const double* c_i, const void* const* R, int nc, int q, int bucket, double* sigma) {
    API_BEGIN
    if (!geoms || !ks || !c_i || !R || !sigma) throw Error(HBEM_EINVAL, "null argument");
    if (ninst < 1 || nk < 1) throw Error(HBEM_EINVAL, "need at least one instance and one wavenumber");
    if (bucket < 0 || bucket % 32 != 0 || bucket > 4096) throw Error(HBEM_EINVAL, "bucket must be a multiple of 32 in [0, 4096]");
    const int gran = bucket == 0 ? 256 : bucket;
    std::vector<hbem_geometry*> G(geoms, geoms + ninst);
    for (int i = 0; i < ninst; ++i) {
        if (!G[i] || !R[i]) throw Error(HBEM_EINVAL, "null geometry or test matrix");
        if (G[i]->ns != G[0]->ns || G[i]->proj != G[0]->proj || G[i]->flags != G[0]->flags || G[i]->dev != G[0]->dev)
            throw Error(HBEM_EINVAL, "instances must share quadrature order, projection, flags and device");
        if (G[i]->flags & HBEM_FLAG_FAR_FIELD)
            throw Error(HBEM_EINVAL, "the multi-instance sweep takes contexts without HBEM_FLAG_FAR_FIELD");
        check_dense_args(ks, 2 * G[i]->N, R[i], nc, q);
        for (int j = 0; j < nk; ++j) { check_k(ks[(size_t)i * nk + j], 0.0, c_i[i]); check_k(ks[(size_t)i * nk + j], 0.0, c_o); }
    }
    // every instance's context is locked for the call (in address order), then the work space
    std::vector<hbem_geometry*> order(G);
    std::sort(order.begin(), order.end());
    order.erase(std::unique(order.begin(), order.end()), order.end());
    std::vector<std::unique_lock<std::mutex>> locks;
    for (auto* g : order) locks.emplace_back(g->mu);
    std::lock_guard<std::mutex> lk(g_multi.mu);
    HIPC(hipSetDevice(G[0]->dev));
    // buckets of equal padded order, in increasing order; a bucket is split by the
    // LU's step width, which follows the instance's own order (1024 and 2048 may lie
    // inside a bucket), and into subsets whose work space fits the free device memory
    typedef std::pair<std::pair<int, int>, int> Key;
    std::vector<Key> key(ninst);
    for (int i = 0; i < ninst; ++i)
        key[i] = {{(2 * G[i]->N + gran - 1) / gran * gran, hbem::lu_step_panels(2 * G[i]->N, true)}, i};
    std::sort(key.begin(), key.end());
    // (the instances' tables first: the free memory is what is left beside them)
    std::vector<size_t> need(ninst);
    for (int i = 0; i < ninst; ++i) {
        const double cm = std::sqrt(std::max(c_i[i], c_o));
        std::vector<double> kap;
        for (int j = 0; j < nk; ++j) kap.push_back(ks[(size_t)i * nk + j] * cm);
        const size_t n_pad = (2 * (size_t)G[i]->N + gran - 1) / gran * gran;
        need[i] = (size_t)nk * records_bytes_per_k(G[i], kap, 0, sweep_tdiff(ks + (size_t)i * nk, nk) ? 1 : 2, 2, true) +
                  (size_t)nk * (n_pad * n_pad * sizeof(cdbl) + n_pad * (8 + (4 * nc + 4) * sizeof(cdbl)));
    }
    size_t held = 0;
    {
        MultiWork& w = g_multi;
        const DBuf* bs[] = {&w.scr.E, &w.scr.L, &w.scr.part, &w.T, &w.piv, &w.perm, &w.X, &w.Y, &w.work};
        for (auto* b : bs) held += b->n;
    }
    const size_t avail = usable_device_bytes(held);
    size_t a = 0;
    while (a < key.size()) {
        const std::pair<int, int> form = key[a].first;
        std::vector<int> ids;
        size_t used = 0;
        while (a < key.size() && key[a].first == form) {
            const int i = key[a].second;
            if (!ids.empty() && used + need[i] > avail) break;
            ids.push_back(i);
            used += need[i];
            ++a;
        }
        multi_subset(G, ids, form.first, form.second, ks, nk, c_o, c_i, R, nc, q, sigma);
    }
    API_END
}

int hbem_profile_enable(hbem_geometry_t g, int enable) {
    API_BEGIN
    if (!g) throw Error(HBEM_EINVAL, "null geometry");
    std::lock_guard<std::mutex> lk(g->mu);
    g->plog.reset();
    g->prof = enable != 0;
    API_END
}

int hbem_profile_query(hbem_geometry_t g, int which, double* ms, long long* launches, double* flops) {
    API_BEGIN
    if (!g || which < 0 || which > kProfGemm) throw Error(HBEM_EINVAL, "invalid argument");
    std::lock_guard<std::mutex> lk(g->mu);
    g->plog.resolve();
    if (ms) *ms = g->plog.ms[which];
    if (launches) *launches = g->plog.n[which];
    if (flops) *flops = g->plog.flops[which];
    API_END
}

int hbem_sweep_batch_size(int npanels, int order, int d, int nc, unsigned long long avail_bytes, int nk, int* B) {
    API_BEGIN
    if (!B) throw Error(HBEM_EINVAL, "null output");
    if (npanels < 3 || order < 1 || order > 40 || d < 0 || d > 2 || nc < 1 || nk < 0)
        throw Error(HBEM_EINVAL, "invalid argument");
    // a closed curve of N panels: N coinciding, N adjacent pairs
    const long long N = npanels;
    const int ncr = order * (order + 1) / 2 - 1;
    *B = sweep_batch(locals_bytes_per_k(N * (N + 1) / 2, N, N, ncr, d, nk >= 32 ? 1 : 2) +
                         dense_bytes_per_k(2 * npanels, d, nc),
                     (size_t)avail_bytes, nk);
    API_END
}

int hbem_rsvd_benchmarking(int yes) {
    API_BEGIN
    std::lock_guard<std::mutex> lk(g_sa.mu);
    g_sa.bench = yes != 0;
    API_END
}

int hbem_rsvd_timers(double* seconds4) {
    API_BEGIN
    if (!seconds4) throw Error(HBEM_EINVAL, "null output");
    std::lock_guard<std::mutex> lk(g_sa.mu);
    g_sa.tim.resolve();
    for (int i = 0; i < 4; ++i) seconds4[i] = g_sa.tim.ms[i] * 1e-3;
    API_END
}

int hbem_rsvd_reset_timer(void) {
    API_BEGIN
    std::lock_guard<std::mutex> lk(g_sa.mu);
    g_sa.tim.reset();
    API_END
}

}  // extern "C"
