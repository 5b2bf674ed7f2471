// pk_fock.hip — host side of the MI355X Fock-build engine and its C ABI
// (include/pk_fock.h).  Per-lane class kernels live in eri_kernels.h (instantiated
// in pk_kernels.hip), the row kernels of the large classes in eri_rows.h, the
// cooperative kernel for ERI output in eri_generic.h; this file builds the shell
// pairs, the Schwarz table and the screened quartet work lists, and launches the
// kernels on the context's stream.
//
// Reference path replaced: src/integrals/base.h:57-93 (_compute_2e_fock[_uhf]),
// src/integrals/os.cpp:1435-1625 and rys.cpp:701-824 (the Fock builds),
// os.cpp:1703-1752 (Schwarz table), shellpair.cpp:7-22 (pairs).
#include "pk_fock.h"
#include "pk_internal.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <numeric>
#include <string>
#include <thread>
#include <unordered_map>
#include <vector>

#include "eri_classes.h"
#include "eri_generic.h"
#include "eri_grad.h"
#include "grad_table.h"
#include "rows_table.h"
#include "small_table.h"

// per-class launchers, defined in pk_kernels.hip
#define PK_DECL(a, b, c, d, shard)                                                             \
    void pk_launch_jk_rys_##a##b##c##d(const pk::JKArgs &, int, int, hipStream_t, int &);           \
    void pk_launch_jk_os_##a##b##c##d(const pk::JKArgs &, int, int, hipStream_t, int &);            \
    void pk_launch_jk_rys32_##a##b##c##d(const pk::JKArgs &, int, int, hipStream_t, int &);         \
    void pk_launch_jk_os32_##a##b##c##d(const pk::JKArgs &, int, int, hipStream_t, int &);         \
    void pk_launch_jk_os_uhf_##a##b##c##d(const pk::JKArgs &, int, int, hipStream_t, int &);          \
    void pk_launch_jk_os_seg_##a##b##c##d(const pk::JKArgs &, int, int, hipStream_t, int &);          \
    void pk_launch_jk_os32_seg_##a##b##c##d(const pk::JKArgs &, int, int, hipStream_t, int &);        \
    void pk_launch_jk_os_uhf_seg_##a##b##c##d(const pk::JKArgs &, int, int, hipStream_t, int &);
PK_FOR_EACH_CLASS(PK_DECL)
#undef PK_DECL

namespace {

thread_local std::string g_err;

int fail(int code, const std::string &msg) {
    g_err = msg;
    return code;
}

#define PK_HIP(expr)                                                                            \
    do {                                                                                        \
        hipError_t e_ = (expr);                                                                 \
        if (e_ != hipSuccess)                                                                   \
            return fail(PK_ERR_HIP, std::string(#expr ": ") + hipGetErrorString(e_));           \
    } while (0)

constexpr int kMaxL = PK_MAX_L;
constexpr double kPrimCut = 1e-17;  // primitive-pair screening bound (see add_molecule)
// Class kernels of one build run on the context stream and up to kSideQueues
// more streams when the build holds at least kSideMinQuartets shell quartets
// (GPU_MAX_HW_QUEUES is 4: one queue per stream).
constexpr int kSideQueues = 3;
constexpr int64_t kSideMinQuartets = 1 << 20;
// Segment mode of the per-lane kernels (see k_jk): at most kSegWaves waves of one
// bra per segment, fewer (kSegWavesMin at least) where a list would have less than
// kSegs of them or one would take more than 1/kSegs of the list's primitive steps,
// and at most kSegLdsMax bytes of LDS exchange rows.  The waves of a segment run
// one after another on its workgroup: with workgroups of two waves on n-C10H22 /
// cc-pVTZ, 16 -> 4 waves: (pp|ss) 2.7 -> 1.6 ms, (fs|ss) 1.5 -> 1.0, but (dp|ps)
// 6.5 -> 7.0 (every segment flushes its rows).
constexpr size_t kSegWaves = 16, kSegWavesMin = 4, kSegs = 4096;
// Row kernels: a list is cut into about kRowItems work items (workgroups) of at
// most kRowKetsMax kets; measured on n-C10H22 / cc-pVTZ, 8192 items: the same or
// up to 1.6x slower (a workgroup flushes its exchange rows once).
constexpr size_t kRowItems = 4096, kRowKetsMax = 1024;
constexpr size_t kGradItems = 8192;  // gradient work items (one wave each) of a class, about
constexpr size_t kLdsMax = 160 * 1024;  // LDS of a CU, and of one workgroup
// Waves are cut along the bra's primitives above 1/kCutWaves of their list's
// steps (items of the row kernels: four times the average), and kCutSteps
// primitive quartets (see build_work).
constexpr double kCutWaves = 8192.0, kCutSteps = 32.0;
// quartets below which the list of a class with a per-lane Rys and a row kernel
// takes the row kernel (fewer than the lanes of two waves per SIMD)
constexpr size_t kRowsFew = 2 * 64 * 4 * 256;
// A build whose lists hold at most kSmallWaves waves and work items in all is
// short: its lists go out in one launch (k_small).  H2O / 6-31G* 0.76 -> 0.08 ms,
// three waters 1.47 -> 0.32 ms, H2O / cc-pVTZ 4.3 -> 0.72 ms; above it the lists
// win by themselves (n-C2H6 / cc-pVTZ, 60 thousand waves, 2.6 ms against 4.9 ms).
constexpr int64_t kSmallWaves = 32768;
constexpr int kMinSegs = 256;  // segments below which a list runs in plain mode
// A list with fewer quartets than lanes of two waves per SIMD (quartet slots of
// one, for the row kernels) and at least kSplitPrims primitive quartets each has
// its kets cut along their primitives too, in at most kSplitMost parts.
constexpr size_t kSplitLanes = 2 * 64 * 4 * 256, kSplitSlots = 4 * 256, kSplitMost = 16, kSplitPrims = 8;
// primitive quartets per shell quartet below which a list of a pk::seg_alt_class
// runs in segment mode (6-31G* water clusters: 11-13; cc-pVTZ alkanes: 40-80)
constexpr double kSegAltPrim = 24.0;
constexpr size_t kSegLdsMax = 64 * 1024;
// lanes per workgroup of a class list until pk_ctx_autotune picks its own;
// one wave per workgroup for the segment-mode lists of a batch with at most
// kSegOneWaveLds bytes of exchange rows (see launch_list).  128 against 256 lanes: the
// lists one after another take the same time (n-C10H22 / cc-pVTZ 131 ms both), a
// build over the side queues, where workgroups of several lists share a CU,
// 117 ms against 121 (n-C20H42 / cc-pVDZ 31.5 ms against 33.9).
constexpr int kDefaultBlock = 128;
constexpr int kRowWavesMax = 4;  // waves per workgroup of the row kernels
constexpr size_t kSegOneWaveLds = 24 * 1024;
constexpr int kPairClasses = (kMaxL + 1) * (kMaxL + 2) / 2;
constexpr int kQuartClasses = kPairClasses * (kPairClasses + 1) / 2;

struct ClassFns {
    int la, lb, lc, ld;
    bool has_os;    // Obara-Saika per-lane kernel
    bool has_tmpl;  // Rys per-lane kernel (else the row kernel, pk::rows_class)
    bool few_rows;  // short lists of the class run in a row kernel (pk::small_rows)
    int small_set;  // k_small set that covers the class (-1: none)
    bool seg;       // the per-lane kernels run in segment mode (pk::seg_class)
    bool seg_alt;   // the OS kernel also exists in segment mode (pk::seg_alt_class)
    void (*jk_os)(const pk::JKArgs &, int, int, hipStream_t, int &);
    void (*jk_rys)(const pk::JKArgs &, int, int, hipStream_t, int &);
    void (*jk_os32)(const pk::JKArgs &, int, int, hipStream_t, int &);  // FP32 integrals
    void (*jk_rys32)(const pk::JKArgs &, int, int, hipStream_t, int &);
    void (*jk_os_uhf)(const pk::JKArgs &, int, int, hipStream_t, int &);  // FP64, two exchange densities
    void (*jk_os_seg)(const pk::JKArgs &, int, int, hipStream_t, int &);  // segment-mode variants
    void (*jk_os32_seg)(const pk::JKArgs &, int, int, hipStream_t, int &);
    void (*jk_os_uhf_seg)(const pk::JKArgs &, int, int, hipStream_t, int &);
};

#define PK_ENTRY(a, b, c, d, shard)                                                             \
    ClassFns{a, b, c, d, pk::os_available(a, b, c, d), pk::rys_tmpl_available(a, b, c, d),      \
             pk::small_rows(a, b, c, d), pk::small_class(a, b, c, d) ? ((a) == 3 ? 1 : 0) : -1,     \
             pk::seg_class(a, b, c, d), pk::os_available(a, b, c, d) && pk::seg_alt_class(a, b, c, d), \
             &pk_launch_jk_os_##a##b##c##d, &pk_launch_jk_rys_##a##b##c##d,                     \
             &pk_launch_jk_os32_##a##b##c##d, &pk_launch_jk_rys32_##a##b##c##d,                 \
             &pk_launch_jk_os_uhf_##a##b##c##d, &pk_launch_jk_os_seg_##a##b##c##d,                   \
             &pk_launch_jk_os32_seg_##a##b##c##d, &pk_launch_jk_os_uhf_seg_##a##b##c##d},
// Quartet classes (bra class >= ket class), indexed cb (cb + 1) / 2 + ck with
// pair classes (0,0) (1,0) (1,1) (2,0) (2,1) (2,2) (3,0) (3,1) (3,2) (3,3).
const ClassFns kClasses[kQuartClasses] = {PK_FOR_EACH_CLASS(PK_ENTRY)};
#undef PK_ENTRY

// row kernels by quartet class
const pk::RowsEntry *rows_table() {
    static const std::vector<pk::RowsEntry> t = [] {
        std::vector<pk::RowsEntry> v(kQuartClasses);
        pk_rows_register<0>(v.data());
        pk_rows_register<1>(v.data());
        pk_rows_register<2>(v.data());
        pk_rows_register<3>(v.data());
        pk_rows_register<4>(v.data());
        pk_rows_register<5>(v.data());
        pk_rows_register<6>(v.data());
        pk_rows_register<7>(v.data());
        return v;
    }();
    return t.data();
}

// gradient kernels by ordered class (bra pair class, ket pair class)
static_assert(PK_GRAD_PAIRS == kPairClasses, "gradient kernels cover every pair class");
const pk::GradEntry *grad_table() {
    static const std::vector<pk::GradEntry> t = [] {
        std::vector<pk::GradEntry> v(PK_GRAD_PAIRS * PK_GRAD_PAIRS);
        pk_grad_register<0>(v.data());
        pk_grad_register<1>(v.data());
        pk_grad_register<2>(v.data());
        pk_grad_register<3>(v.data());
        pk_grad_register<4>(v.data());
        pk_grad_register<5>(v.data());
        pk_grad_register<6>(v.data());
        pk_grad_register<7>(v.data());
        return v;
    }();
    return t.data();
}

int quart_class(int cb, int ck) { return cb * (cb + 1) / 2 + ck; }
int class_la(int c) {
    int l = 0;
    while ((l + 1) * (l + 2) / 2 <= c) ++l;
    return l;
}
int class_lb(int c) { return c - class_la(c) * (class_la(c) + 1) / 2; }

// ---------------------------------------------------------------- small kernels
// Packed matrices: molecule m (blockIdx.y) has nb = mol_nb[m] functions, its
// nb x nb block at mol_off[m].  Inside the engine a molecule's functions are
// in the internal order: shells grouped by angular momentum (s, p, d, f), in
// basis order within a group, components contiguous.  Kets of one bra that
// share their first shell then have second shells of one type at neighbouring
// positions, so a wave's atomic adds into a row of J or K land in a few cache
// lines (the L2 executes a 64-lane FP64 atomic per cache line touched: ~24 G
// lines/s, against ~180 G lanes/s when the lanes share lines).  pos[foff[m] +
// f] is the internal position of the caller's function f; the component
// norms nrm[foff[m] + x] are stored by internal position x.
struct MolTab {
    const long long *off;
    const int *nb;
    const int *foff;
    const int *pos;
};

// Pn (internal order) = n n^T o P (caller's order)
__global__ void k_scale_density(const double *__restrict__ P, const double *__restrict__ nrm,
                                double *__restrict__ Pn, MolTab t) {
    const int m = blockIdx.y, nb = t.nb[m];
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)nb * nb) return;
    const int r = (int)(i / nb), c = (int)(i % nb);
    const int *ps = t.pos + t.foff[m];
    const int pr = ps[r], pc = ps[c];
    const double *n = nrm + t.foff[m];
    const size_t o = (size_t)t.off[m];
    Pn[o + (size_t)pr * nb + pc] = n[pr] * n[pc] * P[o + i];
}

// The same, and the accumulators of the build cleared
__global__ void k_prepare(const double *__restrict__ P, const double *__restrict__ nrm, double *__restrict__ Pn,
                          double *__restrict__ A, double *__restrict__ B, MolTab t) {
    const int m = blockIdx.y, nb = t.nb[m];
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)nb * nb) return;
    const int r = (int)(i / nb), c = (int)(i % nb);
    const int *ps = t.pos + t.foff[m];
    const int pr = ps[r], pc = ps[c];
    const double *n = nrm + t.foff[m];
    const size_t o = (size_t)t.off[m];
    Pn[o + (size_t)pr * nb + pc] = n[pr] * n[pc] * P[o + i];
    A[o + i] = 0.0;
    B[o + i] = 0.0;
}

// out (caller's order) = in (internal order)
__global__ void k_unpermute(const double *__restrict__ in, double *__restrict__ out, MolTab t) {
    const int m = blockIdx.y, nb = t.nb[m];
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)nb * nb) return;
    const int r = (int)(i / nb), c = (int)(i % nb);
    const int *ps = t.pos + t.foff[m];
    const size_t o = (size_t)t.off[m];
    out[o + i] = in[o + (size_t)ps[r] * nb + ps[c]];
}

// y = (float) x
__global__ void k_to_f32(const double *__restrict__ x, float *__restrict__ y, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = (float)x[i];
}

// z = x + y
__global__ void k_sum2(const double *__restrict__ x, const double *__restrict__ y, double *__restrict__ z, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) z[i] = x[i] + y[i];
}

__global__ void k_fill(double *__restrict__ x, size_t n, double v) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = v;
}

// J = n n^T o (A + A^T), K = n n^T o (B + B^T) (A, B internal order; J, K, G
// caller's order); optional G = J - K/2
__global__ void k_finalize(const double *__restrict__ A, const double *__restrict__ B,
                           const double *__restrict__ nrm, double *J, double *K, double *G, MolTab t) {
    const int m = blockIdx.y, nb = t.nb[m];
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)nb * nb) return;
    const int r = (int)(i / nb), c = (int)(i % nb);
    const int *ps = t.pos + t.foff[m];
    const int pr = ps[r], pc = ps[c];
    const double *n = nrm + t.foff[m];
    const size_t o = (size_t)t.off[m];
    const double s = n[pr] * n[pc];
    const size_t x = o + (size_t)pr * nb + pc, y = o + (size_t)pc * nb + pr;
    const double j = s * (A[x] + A[y]);
    const double k = s * (B[x] + B[y]);
    if (J) J[o + i] = j;
    if (K) K[o + i] = k;
    if (G) G[o + i] = j - 0.5 * k;
}

// Autotuned launch shape of a class list.  A class of pk::small_rows runs its short
// lists in another kernel than its long ones, so a choice holds for lists of its kind.
struct TuneEntry {
    int cls, prec;
    bool rows;
    int block, remap, alt;
};

struct ClassWork {
    int cls = 0;
    int prec = PK_PREC_FP64;  // PK_PREC_MIXED: the FP32 list of the class
    int block = 0;            // lanes per workgroup (autotuned or PK_BLOCK; 0: the default of the launch)
    int block_run = 0;        // lanes per workgroup of the last launch
    int remap = 0;            // XCD-contiguous wave ranges (autotuned)
    int alt = 0;              // alternative kernel (autotuned, see has_alt): FP64 integrals for an
                              // FP32 list, the cooperative kernel for a per-lane Rys list
    int nwaves = 0;
    int64_t nquart = 0;
    int64_t nprimq = 0;
    double flops = 0.0;
    int *d_wave = nullptr;  // [4][nwaves]: bra, start, count, molecule
    int *d_kets = nullptr;
    int row_waves[2] = {0, 0};  // row kernels: waves per workgroup, one and two exchange densities (0: not chosen yet)
    int nseg = 0;          // segments: runs of at most kSegWaves waves of one bra
    int *d_seg = nullptr;  // [2 nseg] first wave and end of each segment, most expensive first
    int kcols = 0;         // LDS columns of an exchange row (largest molecule)
    bool rows = false;     // runs in the class's row kernel
    int group = 0;         // row kernels: most kets of a work item
    int kernels = 0;
    double ms_total = 0.0;
    int64_t builds = 0;
    double cost_ms = 0.0;  // measured time of the list in the last timed build (0: not yet)
    hipEvent_t e0 = nullptr, e1 = nullptr;
};

// Gradient work of one ordered class: items (bra, first ket, kets, bra primitives)
// into the context's gradient order.
struct GradWork {
    int cls = 0;  // bra class * kPairClasses + ket class
    int nitems = 0;
    double cost = 0.0;
    int *d_items = nullptr;  // [4][nitems]
};

template <typename T>
int dev_upload(T **dst, const T *src, size_t n, hipStream_t s) {
    *dst = nullptr;
    if (n == 0) return PK_OK;
    PK_HIP(hipMalloc((void **)dst, n * sizeof(T)));
    PK_HIP(hipMemcpyAsync(*dst, src, n * sizeof(T), hipMemcpyHostToDevice, s));
    return PK_OK;
}

template <typename T>
int dev_upload(T **dst, const std::vector<T> &src, hipStream_t s) {
    return dev_upload(dst, src.data(), src.size(), s);
}

}  // namespace

struct pk_ctx {
    int nb = 0, ns = 0;  // functions and shells over all molecules
    int nmol = 1;
    std::vector<int> mol_nb, mol_foff;  // functions per molecule, first function
    std::vector<int> tblk;              // [5 * nmol]: first function of type s, p, d, f (internal order), nb
    int *d_tblk = nullptr;
    bool seg_on = true;                 // segment mode of the per-lane kernels (PK_EXCHANGE_ROWS=0: off)
    std::vector<long long> mol_off;     // offset of the molecule's nb x nb block
    size_t n2 = 0;                      // packed matrix length
    int nbmax = 0;
    std::vector<int> pair_mol;
    long long *d_mol_off = nullptr;
    int *d_mol_nb = nullptr, *d_mol_foff = nullptr;
    bool graph_on = false, graph_ok = false;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    double *d_G = nullptr;
    std::vector<TuneEntry> tuned;  // autotuned launch shape per (class, precision)
    std::vector<int> sh_l, sh_np, sh_poff, sh_f0;
    std::vector<double> sh_c, ex, co, pn;
    std::vector<double> fnorm;  // component norms by internal position
    std::vector<int> fpos;      // internal position of each caller's function (per molecule)
    std::vector<int> fnat;      // caller's function at each internal position
    int *d_fpos = nullptr;
    std::vector<pk::PairDev> pairs;
    std::vector<int> pair_cls;
    std::vector<double> pair_q;
    std::vector<pk::PrimDev> prims;
    std::vector<double> palpha;  // exponent on the pair's first shell, per primitive pair
    std::vector<double> hz;      // 1/(2 zeta) per primitive pair
    std::vector<int> pair_sh;    // first and second shell of each pair
    std::vector<double> Q;  // packed nb x nb blocks, normalised functions, internal order
    pk::PairDev *d_pairs = nullptr;
    pk::PairDev *d_wpairs = nullptr;  // pairs of the work lists: the pairs, then parts of them (build_work)
    pk::PrimDev *d_prims = nullptr;
    double *d_Q = nullptr, *d_fnorm = nullptr, *d_P = nullptr, *d_Pn = nullptr, *d_A = nullptr, *d_B = nullptr;
    double *d_J = nullptr, *d_K = nullptr;
    double *d_J2 = nullptr;  // UHF: J of the second density
    double *d_hz = nullptr;
    double *d_palpha = nullptr, *d_Pk1n = nullptr, *d_Pk2n = nullptr, *d_gsh = nullptr;  // gradient, UHF
    double *d_B2 = nullptr;  // one-pass UHF: second exchange accumulator
    float *d_P32 = nullptr;  // mixed precision: FP32 copy of the scaled density
    int *d_pair_sh = nullptr;
    std::vector<ClassWork> work;
    bool work_ok = false;
    pk::SmallList *d_small = nullptr;  // the lists, for k_small; null when the build is not short
    pk::SmallTab small_tab[2];
    int small_blocks[2] = {0, 0};
    size_t small_lds[2] = {0, 0};
    bool lists_win = false;  // the tuned lists of a short build beat its one launch (pk_ctx_autotune)
    std::vector<GradWork> gwork;  // gradient work items, built by the first gradient at a tolerance
    int *d_gorder = nullptr;
    double gwork_tol = -1.0;
    int engine = PK_ENGINE_OS;
    double tol = 1e-10;
    int precision = PK_PREC_FP64;
    double cutoff = 0.0;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // side queues of a build: the class kernels are spread over the context
    // stream and these (default priority), forked and joined by events
    hipStream_t side[kSideQueues] = {};
    hipEvent_t fork_ev = nullptr, join_ev[kSideQueues] = {};
    bool side_ok = false;
    bool side_off = false;  // PK_SIDE_QUEUES=0
    double seg_alt_prim = kSegAltPrim;  // PK_SEG_ALT_PRIM
    int block0 = kDefaultBlock;         // PK_BLOCK: lanes per workgroup of every list before autotuning
    bool block_forced = false;          // PK_BLOCK given: no per-list default
    bool cost_learned = false;  // the lists' times have been measured (first large build)
    bool learning = false;      // the current build records per-list events for that
    bool profile = false;
    pk_stats st{};
};

namespace {

// OS kernels where they exist unless the Rys engine is forced
bool use_os(const pk_ctx *c, const ClassFns &f) { return f.has_os && c->engine != PK_ENGINE_RYS; }

// Kernels that run a class list (pk_class_stats.kind): 0 / 3 per-lane OS in
// FP64 / FP32, 1 / 4 per-lane Rys in FP64 / FP32, 2 row or cooperative kernel (FP64).
int list_kind(const pk_ctx *c, const ClassWork &w) {
    const ClassFns &f = kClasses[w.cls];
    const bool fp32 = w.prec == PK_PREC_MIXED && !w.alt;
    if (use_os(c, f)) return fp32 ? 3 : 0;
    if (!w.rows && !(w.alt && w.prec == PK_PREC_FP64)) return fp32 ? 4 : 1;
    return 2;
}

// lists with an alternative kernel (ClassWork::alt)
bool has_alt(const pk_ctx *c, const ClassWork &w) {
    return w.prec == PK_PREC_MIXED || (!w.rows && !use_os(c, kClasses[w.cls]));
}

// lists that k_small takes: Obara-Saika classes and rows (in FP64)
bool small_covers(const ClassWork &w) {
    const ClassFns &f = kClasses[w.cls];
    return f.small_set >= 0 && (w.rows || f.has_os) && w.prec == PK_PREC_FP64;
}

// The build goes out in one launch (k_small): a short one whose tuned lists, if any,
// are not the faster.  k_small holds the FP64 Obara-Saika and row kernels of one
// exchange density; UHF, mixed precision and the Rys engine run their lists.
bool one_launch(const pk_ctx *c, const double *B2) {
    return c->d_small && !c->lists_win && c->engine != PK_ENGINE_RYS && !B2;
}

void drop_graph(pk_ctx *c) {
    if (c->gexec) (void)hipGraphExecDestroy(c->gexec);
    if (c->graph) (void)hipGraphDestroy(c->graph);
    c->gexec = nullptr;
    c->graph = nullptr;
    c->graph_ok = false;
}

void free_grad(pk_ctx *c) {
    for (GradWork &w : c->gwork)
        if (w.d_items) (void)hipFree(w.d_items);
    c->gwork.clear();
    if (c->d_gorder) (void)hipFree(c->d_gorder);
    c->d_gorder = nullptr;
    c->gwork_tol = -1.0;
}

void free_work(pk_ctx *c) {
    for (ClassWork &w : c->work) {
        if (w.d_wave) (void)hipFree(w.d_wave);
        if (w.d_kets) (void)hipFree(w.d_kets);
        if (w.d_seg) (void)hipFree(w.d_seg);
        if (w.e0) (void)hipEventDestroy(w.e0);
        if (w.e1) (void)hipEventDestroy(w.e1);
    }
    c->work.clear();
    if (c->d_wpairs) (void)hipFree(c->d_wpairs);
    c->d_wpairs = nullptr;
    if (c->d_small) (void)hipFree(c->d_small);
    c->d_small = nullptr;
    c->work_ok = false;
    c->cost_learned = false;
    drop_graph(c);
}

// Raw contracted ERIs (no component norms) of the quartets (bra[i] | ket[i]),
// all of class (cb, ck) with cb >= ck.  out gets NA NB NC ND values per quartet.
// One 64-lane workgroup per item; the dynamic LDS holds the transferred 1-D
// factors and the quartet's accumulators (at most 123 KB for (ff|ff)).
int launch_generic(const pk::GenArgs &a, hipStream_t s) {
    if (a.nitems <= 0) return PK_OK;
    static const hipError_t attr = hipFuncSetAttribute((const void *)pk::k_generic, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       (int)pk::generic_lds_bytes(kMaxL, kMaxL, kMaxL, kMaxL));
    PK_HIP(attr);
    hipLaunchKernelGGL(pk::k_generic, dim3(a.nitems), dim3(64), pk::generic_lds_bytes(a.la, a.lb, a.lc, a.ld), s, a);
    PK_HIP(hipGetLastError());
    return PK_OK;
}

int run_eri_class(pk_ctx *c, int cb, int ck, const std::vector<int> &bra, const std::vector<int> &ket,
                  std::vector<double> &out) {
    const ClassFns &f = kClasses[quart_class(cb, ck)];
    const int nabcd = pk::ncart(f.la) * pk::ncart(f.lb) * pk::ncart(f.lc) * pk::ncart(f.ld);
    const int nq = (int)bra.size();
    out.assign((size_t)nq * nabcd, 0.0);
    if (nq == 0) return PK_OK;
    int *d_b = nullptr, *d_k = nullptr;
    double *d_o = nullptr;
    int rc;
    if ((rc = dev_upload(&d_b, bra, c->stream)) != PK_OK) return rc;
    if ((rc = dev_upload(&d_k, ket, c->stream)) != PK_OK) return rc;
    PK_HIP(hipMalloc((void **)&d_o, out.size() * sizeof(double)));
    pk::GenArgs a{};
    a.qbra = d_b;
    a.qket = d_k;
    a.pairs = c->d_pairs;
    a.prims = c->d_prims;
    a.hz = c->d_hz;
    a.out = d_o;
    a.nitems = nq;
    a.la = f.la;
    a.lb = f.lb;
    a.lc = f.lc;
    a.ld = f.ld;
    a.eri_mode = 1;
    if ((rc = launch_generic(a, c->stream)) != PK_OK) return rc;
    PK_HIP(hipMemcpyAsync(out.data(), d_o, out.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    PK_HIP(hipStreamSynchronize(c->stream));
    (void)hipFree(d_b);
    (void)hipFree(d_k);
    (void)hipFree(d_o);
    return PK_OK;
}

int build_schwarz(pk_ctx *c) {
    c->Q.assign(c->n2, 0.0);
    for (int cls = 0; cls < kPairClasses; ++cls) {
        std::vector<int> idx;
        for (int p = 0; p < (int)c->pairs.size(); ++p)
            if (c->pair_cls[p] == cls) idx.push_back(p);
        if (idx.empty()) continue;
        std::vector<double> out;
        int rc = run_eri_class(c, cls, cls, idx, idx, out);
        if (rc != PK_OK) return rc;
        const int la = class_la(cls), lb = class_lb(cls);
        const int na = pk::ncart(la), nbb = pk::ncart(lb), nab = na * nbb;
        for (size_t q = 0; q < idx.size(); ++q) {
            const pk::PairDev &p = c->pairs[idx[q]];
            const int m = c->pair_mol[idx[q]], nb = c->mol_nb[m];
            const double *fn = c->fnorm.data() + c->mol_foff[m];
            double *Qm = c->Q.data() + c->mol_off[m];
            double qmax = 0.0, qmin = 1e300;
            for (int ia = 0; ia < na; ++ia)
                for (int ib = 0; ib < nbb; ++ib) {
                    const int i = p.f0 + ia, j = p.f1 + ib;
                    const double raw = out[q * (size_t)nab * nab + (size_t)(ia * nbb + ib) * nab + ia * nbb + ib];
                    const double v = fn[i] * fn[j] * std::sqrt(std::fabs(raw));
                    Qm[(size_t)i * nb + j] = Qm[(size_t)j * nb + i] = v;
                    qmax = std::max(qmax, v);
                    qmin = std::min(qmin, v);
                }
            c->pair_q[idx[q]] = qmax;
            c->pairs[idx[q]].qmin = qmin;
        }
    }
    return PK_OK;
}

// Runs f(i) for i in [0, n) on up to 16 host threads (dynamic chunks of 64), one
// thread per `grain` of them (starting a thread costs tens of microseconds).
template <typename F>
void parallel_for(size_t n, F f, size_t grain = 64) {
    const unsigned hw = std::max(1u, std::min(16u, std::thread::hardware_concurrency()));
    const unsigned nt = (unsigned)std::min<size_t>(hw, (n + grain - 1) / grain);
    if (nt <= 1) {
        for (size_t i = 0; i < n; ++i) f(i);
        return;
    }
    std::atomic<size_t> next{0};
    std::vector<std::thread> th;
    for (unsigned t = 0; t < nt; ++t)
        th.emplace_back([&] {
            for (size_t i0; (i0 = next.fetch_add(64)) < n;)
                for (size_t i = i0; i < std::min(n, i0 + 64); ++i) f(i);
        });
    for (std::thread &t : th) t.join();
}

// Screened work lists: for every quartet class (cb >= ck), every molecule and
// every bra pair, the ket pairs of the same molecule with
// qmax_bra * qmax_ket >= tol (and ket <= bra when cb == ck), sorted by
// primitive count and shells, cut into waves of at most 64 kets; the waves of all
// molecules form one list per class.  In mixed precision the kets with
// qmax_bra * qmax_ket < cutoff form a second, FP32 list of the class (classes
// of the row kernels stay FP64).
int ensure_side(pk_ctx *c);

int build_work(pk_ctx *c) {
    free_work(c);
    const int np = (int)c->pairs.size();
    // by_cls[m][class]: pairs of molecule m, q descending
    std::vector<std::vector<std::vector<int>>> by_cls(c->nmol, std::vector<std::vector<int>>(kPairClasses));
    for (int p = 0; p < np; ++p) by_cls[c->pair_mol[p]][c->pair_cls[p]].push_back(p);
    for (auto &mv : by_cls)
        for (auto &v : mv)
            std::stable_sort(v.begin(), v.end(), [&](int x, int y) { return c->pair_q[x] > c->pair_q[y]; });
    // ket order inside a wave: ordering group descending, then first and
    // second function (one 64-bit key per pair)
    std::vector<uint64_t> okey(np);
    for (int p = 0; p < np; ++p)
        okey[p] = ((uint64_t)(2047 - c->pairs[p].grp) << 40) | ((uint64_t)c->pairs[p].f0 << 20) | (uint64_t)c->pairs[p].f1;
    c->st.quartets = 0;
    c->st.primitive_quartets = 0;
    c->st.model_flops = 0.0;
    const bool mixed = c->precision == PK_PREC_MIXED;
    // ord[m][class]: positions in by_cls[m][class] in ket order (okey
    // ascending), so that a bra's kets -- a prefix range of the q order -- come
    // out in ket order by one pass over it instead of a sort per bra
    std::vector<std::vector<std::vector<int>>> ord(c->nmol, std::vector<std::vector<int>>(kPairClasses));
    parallel_for((size_t)c->nmol, [&](size_t m) {
        for (int cl = 0; cl < kPairClasses; ++cl) {
            const std::vector<int> &v = by_cls[m][cl];
            std::vector<int> &o = ord[m][cl];
            o.resize(v.size());
            for (size_t i = 0; i < v.size(); ++i) o[i] = (int)i;
            std::sort(o.begin(), o.end(), [&](int x, int y) { return okey[v[x]] < okey[v[y]]; });
        }
    });
    // records of parts of pairs (primitives [p0, p1)), indexed after the pairs
    std::vector<pk::PairDev> vpairs;
    std::unordered_map<uint64_t, int> vindex;
    std::vector<int> npr(np);  // primitive counts beside the records (one per quartet is read)
    for (int p = 0; p < np; ++p) npr[p] = c->pairs[p].nprim;
    // arrays of the list at hand, kept from list to list (page faults; an upload from
    // pageable memory has read its source when it returns): the kets,
    // one index per quartet, not value-initialised (up to GBs for large batches);
    // the steps of its waves before the cuts, and their primitive pairs (row kernels);
    // after the cuts the steps of its waves, or the costs of its row items; the first
    // wave and the order of its segments
    std::unique_ptr<int[]> kets;
    size_t kets_cap = 0;
    auto need_kets = [&](size_t n) {
        if (n <= kets_cap) return;
        kets.reset();
        kets.reset(new int[n]);
        kets_cap = n;
    };
    std::vector<double> steps, ksum, wsteps;
    std::vector<int> cut_at;
    std::vector<unsigned char> cut_key;
    std::vector<int> part_base;  // first of a ket's parts, of the list at hand
    auto add_part = [&](int p, int p0, int p1) {
        pk::PairDev v = c->pairs[p];
        v.prim_off += p0;
        v.nprim = p1 - p0;
        vpairs.push_back(v);
        return np + (int)vpairs.size() - 1;
    };
    auto part_of = [&](int p, int p0, int p1) {
        if (p1 - p0 >= c->pairs[p].nprim) return p;
        const uint64_t key = ((uint64_t)p << 24) | ((uint64_t)p0 << 12) | (uint64_t)p1;  // nprim < 2048
        const auto it = vindex.find(key);
        if (it != vindex.end()) return it->second;
        return vindex[key] = add_part(p, p0, p1);
    };
    struct BraRange {
        size_t k0 = 0, k1 = 0;  // positions [k0, k1) of the q-ordered kets
        int64_t nprimq = 0;
        double flops = 0.0;
    };
    for (int cb = 0; cb < kPairClasses; ++cb)
        for (int ck = 0; ck <= cb; ++ck) {
            const int cls = quart_class(cb, ck);
            const ClassFns &f = kClasses[cls];
            const bool split = mixed && f.has_tmpl;
            // bra tasks of every molecule, in order
            std::vector<std::pair<int, int>> tasks;
            for (int m = 0; m < c->nmol; ++m)
                if (!by_cls[m][cb].empty() && !by_cls[m][ck].empty())
                    for (int ib = 0; ib < (int)by_cls[m][cb].size(); ++ib) tasks.emplace_back(m, ib);
            if (tasks.empty()) continue;
            for (int prec : {PK_PREC_FP64, PK_PREC_MIXED}) {
                if (prec == PK_PREC_MIXED && !split) continue;
                // pass 1: each bra's ket range (binary searches only)
                std::vector<BraRange> outs(tasks.size());
                parallel_for(tasks.size(), [&](size_t t) {
                    const int m = tasks[t].first, ib = tasks[t].second;
                    const std::vector<int> &B = by_cls[m][cb], &Kl = by_cls[m][ck];
                    const double qb = c->pair_q[B[ib]];
                    // number of kets (q descending) with qb * qk >= thr
                    auto count = [&](double thr) {
                        size_t lo = 0, hi = Kl.size();
                        while (lo < hi) {
                            const size_t mid = (lo + hi) / 2;
                            if (qb * c->pair_q[Kl[mid]] >= thr)
                                lo = mid + 1;
                            else
                                hi = mid;
                        }
                        return cb == ck ? std::min(lo, (size_t)ib + 1) : lo;
                    };
                    const size_t n_tol = count(c->tol);
                    const size_t n_hi = split ? std::min(count(c->cutoff), n_tol) : n_tol;
                    BraRange &o = outs[t];
                    o.k0 = prec == PK_PREC_FP64 ? 0 : n_hi;
                    o.k1 = std::max(o.k0, prec == PK_PREC_FP64 ? n_hi : n_tol);
                }, 1024);
                // kets per work item: a wave of 64 lanes for the per-lane kernels; for
                // the row kernels a workgroup's share of a bra's kets (below)
                size_t group = 64;
                // row kernel: by class, or a short list of a class that has both
                bool rows = !f.has_tmpl;
                if (f.few_rows && !mixed) {
                    size_t tot = 0;
                    for (const BraRange &o : outs) tot += o.k1 - o.k0;
                    rows = rows || tot < kRowsFew;
                }
                if (rows) {
                    // about kRowItems work items of equal ket counts, whole groups
                    size_t tot = 0;
                    for (const BraRange &o : outs) tot += o.k1 - o.k0;
                    const size_t qw = rows_table()[cls].qw;
                    group = std::min<size_t>(kRowKetsMax, std::max<size_t>(1, tot / kRowItems));
                    group = (group + qw - 1) / qw * qw;
                }
                ClassWork w;
                w.cls = cls;
                w.prec = prec;
                w.rows = rows;
                w.block = c->block_forced ? c->block0 : 0;
                // offsets of every bra's kets and waves (prefix sums), then the
                // flat arrays filled in parallel
                std::vector<size_t> koff(tasks.size() + 1, 0);
                for (size_t t = 0; t < tasks.size(); ++t) koff[t + 1] = koff[t] + (outs[t].k1 - outs[t].k0);
                if (koff.back() > (size_t)INT32_MAX) return fail(PK_ERR_ARG, "build_work: more than 2^31 quartets in one class");
                need_kets(koff.back());
                auto nprim = [&](int p) { return p < np ? npr[p] : vpairs[p - np].nprim; };
                auto bra_of = [&](size_t t) { return by_cls[tasks[t].first][cb][tasks[t].second]; };
                // waves of up to `group` kets before the cuts, a bra's steps, its longest
                // wave.  Steps of a wave: the primitive quartets of its first ket (the
                // longest within the ordering ratio), per group of slots.
                const size_t per = rows ? (size_t)rows_table()[cls].qw : 64;
                std::vector<size_t> uoff(tasks.size() + 1, 0);
                std::vector<double> tsteps(tasks.size()), tmost(tasks.size());
                auto count_waves = [&]() {
                    for (size_t t = 0; t < tasks.size(); ++t)
                        uoff[t + 1] = uoff[t] + (koff[t + 1] - koff[t] + group - 1) / group;
                    if (steps.size() < uoff.back()) steps.resize(uoff.back());
                    if (rows && ksum.size() < uoff.back()) ksum.resize(uoff.back());
                };
                auto count_steps = [&](size_t t) {
                    const int kb = npr[bra_of(t)];
                    double sum = 0.0, most = 0.0;
                    for (size_t u = uoff[t]; u < uoff[t + 1]; ++u) {
                        const size_t k0 = koff[t] + (u - uoff[t]) * group, m = std::min(group, koff[t + 1] - k0);
                        steps[u] = (double)kb * nprim(kets[k0]) * ((m + per - 1) / per);
                        sum += steps[u];
                        most = std::max(most, steps[u]);
                        if (rows) {
                            int64_t nk = 0;
                            for (size_t k = k0; k < k0 + m; ++k) nk += nprim(kets[k]);
                            ksum[u] = (double)nk;
                        }
                    }
                    tsteps[t] = sum;
                    tmost[t] = most;
                };
                count_waves();
                // quartets that fill the chip; a list of at most half as many may have its
                // kets cut below, and its steps are counted after that
                const size_t fill_quart = rows ? kSplitSlots * per : kSplitLanes;
                const bool few = 2 * koff.back() <= fill_quart;
                // pass 2: every bra's kets in ket order (ordering group
                // descending, then first and second function) straight into the
                // flat array, and, while they are in the cache, the steps of its waves
                parallel_for(tasks.size(), [&](size_t t) {
                    BraRange &o = outs[t];
                    const size_t n = o.k1 - o.k0;
                    if (n == 0) return;
                    const int m = tasks[t].first;
                    const std::vector<int> &Kl = by_cls[m][ck];
                    int *dst = kets.get() + koff[t];
                    if (Kl.size() <= 16 * n + 64) {
                        size_t j = 0;
                        for (const int i : ord[m][ck])
                            if ((size_t)i >= o.k0 && (size_t)i < o.k1) {
                                dst[j++] = Kl[i];
                                if (j == n) break;
                            }
                    } else {
                        std::vector<std::pair<uint64_t, int>> kk(n);
                        for (size_t i = o.k0; i < o.k1; ++i) kk[i - o.k0] = {okey[Kl[i]], Kl[i]};
                        std::sort(kk.begin(), kk.end());
                        for (size_t i = 0; i < n; ++i) dst[i] = kk[i].second;
                    }
                    int64_t nk = 0;
                    for (size_t i = 0; i < n; ++i) nk += npr[dst[i]];
                    o.nprimq = npr[bra_of(t)] * nk;
                    if (!few) count_steps(t);
                    // the model is linear in the primitive quartets of a quartet
                    const double f0 = pk::model_flops(f.la, f.lb, f.lc, f.ld, 0.0);
                    o.flops = (double)n * f0 + (double)o.nprimq * (pk::model_flops(f.la, f.lb, f.lc, f.ld, 1.0) - f0);
                });
                for (size_t t = 0; t < tasks.size(); ++t) {
                    w.nquart += (int64_t)(outs[t].k1 - outs[t].k0);
                    w.nprimq += outs[t].nprimq;
                    w.flops += outs[t].flops;
                }
                if (w.nquart == 0) continue;
                const size_t parts =
                    w.nprimq < (int64_t)kSplitPrims * w.nquart
                        ? 1
                        : std::min<size_t>(kSplitMost, fill_quart / (size_t)w.nquart);
                if (parts > 1) {
                    // few quartets for the chip: every ket as its parts, neighbours
                    std::vector<int> ex;
                    std::vector<size_t> off(1, 0);
                    ex.reserve(koff.back() * parts);
                    part_base.assign(np, -1);
                    for (size_t t = 0; t < tasks.size(); ++t) {
                        for (size_t k = koff[t]; k < koff[t + 1]; ++k) {
                            const int nk = c->pairs[kets[k]].nprim, m = std::max(1, std::min((int)parts, nk));
                            if (m == 1) {
                                ex.push_back(kets[k]);
                                continue;
                            }
                            int &b0 = part_base[kets[k]];  // the pair's m parts, neighbours
                            if (b0 < 0) {
                                b0 = np + (int)vpairs.size();
                                for (int i = 0; i < m; ++i) add_part(kets[k], nk * i / m, nk * (i + 1) / m);
                            }
                            for (int i = 0; i < m; ++i) ex.push_back(b0 + i);
                        }
                        off.push_back(ex.size());
                    }
                    if (ex.size() > (size_t)INT32_MAX) return fail(PK_ERR_ARG, "build_work: more than 2^31 quartets in one class");
                    need_kets(ex.size());
                    std::copy(ex.begin(), ex.end(), kets.get());
                    koff.swap(off);
                    count_waves();
                }
                // a thread per 32768 waves (one takes about 0.1 ms for them, and tens of
                // microseconds to start)
                const size_t grain = std::max<size_t>(64, tasks.size() * 32768 / std::max<size_t>(1, uoff.back()));
                if (few) parallel_for(tasks.size(), count_steps, grain);
                // Waves are cut along the bra's primitives where one would take more than
                // about 1/kCutWaves of the list's steps.
                std::vector<size_t> woff(tasks.size() + 1, 0);
                const double most = std::max(kCutSteps, std::accumulate(tsteps.begin(), tsteps.end(), 0.0) /
                                                            (rows ? kRowItems / 4 : kCutWaves));
                auto cuts = [&](int kb, size_t u) { return std::max(1, std::min(kb, (int)(steps[u] / most))); };
                if (*std::max_element(tmost.begin(), tmost.end()) < 2.0 * most) {
                    woff = uoff;  // no wave is cut
                } else {
                    parallel_for(tasks.size(), [&](size_t t) {
                        const int kb = c->pairs[bra_of(t)].nprim;
                        size_t n = uoff[t + 1] - uoff[t];
                        if (tmost[t] >= 2.0 * most) {
                            n = 0;
                            for (size_t u = uoff[t]; u < uoff[t + 1]; ++u) n += cuts(kb, u);
                        }
                        woff[t + 1] = n;
                    }, grain);
                    for (size_t t = 0; t < tasks.size(); ++t) woff[t + 1] += woff[t];
                }
                const size_t nw = woff.back();
                std::vector<int> packed(4 * nw);
                if (wsteps.size() < nw) wsteps.resize(nw);
                auto fill = [&](size_t t) {
                    const int b = bra_of(t), kb = c->pairs[b].nprim;
                    size_t wi = woff[t];
                    for (size_t u = uoff[t]; u < uoff[t + 1]; ++u) {
                        const size_t k0 = koff[t] + (u - uoff[t]) * group;
                        const int nc = cuts(kb, u);
                        for (int k = 0; k < nc; ++k, ++wi) {
                            packed[wi] = nc == 1 ? b : part_of(b, kb * k / nc, kb * (k + 1) / nc);
                            packed[nw + wi] = (int)k0;
                            packed[2 * nw + wi] = (int)std::min(group, koff[t + 1] - k0);
                            packed[3 * nw + wi] = tasks[t].first;
                            wsteps[wi] = rows ? packed[2 * nw + wi] + (double)nprim(packed[wi]) * ksum[u] : steps[u] / nc;
                        }
                    }
                };
                auto whole = [&](size_t t) { return woff[t + 1] - woff[t] == uoff[t + 1] - uoff[t]; };
                parallel_for(tasks.size(), [&](size_t t) {
                    if (whole(t)) fill(t);
                }, grain);
                for (size_t t = 0; t < tasks.size(); ++t)
                    if (!whole(t)) fill(t);  // part_of adds records
                w.nwaves = (int)nw;
                std::vector<int> seg;
                if (!rows) {
                    // segments of the per-lane kernels: each bra's waves in runs of at
                    // most segw, shorter where they take more than 1/kSegs of the
                    // list's steps; LDS columns: the two ket shell types of the largest
                    // molecule.  The segments of bra task t from woff[t] on.
                    const size_t segw = std::min<size_t>(kSegWaves, std::max<size_t>(kSegWavesMin, nw / kSegs));
                    const double seg_most = std::accumulate(tsteps.begin(), tsteps.end(), 0.0) / kSegs;
                    if (cut_at.size() < nw) cut_at.resize(nw), cut_key.resize(nw);
                    std::vector<int> nseg(tasks.size(), 0);
                    parallel_for(tasks.size(), [&](size_t t) {
                        size_t i = woff[t], n = 0;
                        double sum = 0.0;
                        // order among the segments: the steps' binary exponent, descending
                        auto close = [&]() {
                            if (i > woff[t]) cut_key[i - 1] = (unsigned char)(255 - std::min(255, std::max(0, std::ilogb(sum))));
                        };
                        for (size_t u = woff[t]; u < woff[t + 1]; ++u, ++n) {
                            if (u == woff[t] || n == segw || (n >= kSegWavesMin && sum + wsteps[u] > seg_most)) {
                                close();
                                cut_at[i++] = (int)u;
                                n = 0;
                                sum = 0.0;
                            }
                            sum += wsteps[u];
                        }
                        close();
                        nseg[t] = (int)(i - woff[t]);
                    }, grain);
                    for (size_t t = 0; t < tasks.size(); ++t) {
                        w.nseg += nseg[t];
                        if (woff[t + 1] > woff[t]) {
                            const int *tb = &c->tblk[5 * tasks[t].first];
                            const int ncol = tb[f.lc + 1] - tb[f.lc] + (f.lc == f.ld ? 0 : tb[f.ld + 1] - tb[f.ld]);
                            w.kcols = std::max(w.kcols, ncol);
                        }
                    }
                    // counting sort
                    std::array<int, 257> at{};
                    for (size_t t = 0; t < tasks.size(); ++t)
                        for (int i = 0; i < nseg[t]; ++i) ++at[1 + cut_key[woff[t] + i]];
                    std::partial_sum(at.begin(), at.end(), at.begin());
                    seg.resize(2 * (size_t)w.nseg);
                    for (size_t t = 0; t < tasks.size(); ++t)
                        for (int i = 0; i < nseg[t]; ++i) {
                            const size_t n = at[cut_key[woff[t] + i]]++;
                            seg[2 * n] = cut_at[woff[t] + i];
                            seg[2 * n + 1] = i + 1 < nseg[t] ? cut_at[woff[t] + i + 1] : (int)woff[t + 1];
                        }
                }
                // Most expensive work first, so that no segment or work item ends the list
                // alone: segments, to a factor of two (their neighbours share the
                // bra's densities), and the items of the row kernels.  n-C10H22 / cc-pVTZ,
                // segments: (ps|ps) 5.4 -> 3.9 ms, (dp|ps) 7.5 -> 6.7, (fp|ps) 4.0 -> 3.2,
                // (ds|ss) 3.7 -> 3.1; items: (dd|dp) 5.2 -> 3.4, (fd|dp) 3.1 -> 2.1.  The waves
                // stay in bra order, which plain lists are run in: (ps|ss) 6.7 ms against 7.4
                // in cost order.
                if (rows) {
                    std::vector<int> o(nw), q(4 * nw);
                    std::iota(o.begin(), o.end(), 0);
                    std::stable_sort(o.begin(), o.end(), [&](int x, int y) { return wsteps[x] > wsteps[y]; });
                    for (int k = 0; k < 4; ++k)
                        for (size_t i = 0; i < nw; ++i) q[k * nw + i] = packed[k * nw + o[i]];
                    packed.swap(q);
                }
                int rc;
                if ((rc = dev_upload(&w.d_wave, packed, c->stream)) != PK_OK) return rc;
                if ((rc = dev_upload(&w.d_kets, kets.get(), koff.back(), c->stream)) != PK_OK) return rc;
                if (!rows) {
                    if ((rc = dev_upload(&w.d_seg, seg, c->stream)) != PK_OK) return rc;
                } else {
                    // LDS columns of the row kernels: the ket's second shell type
                    w.group = (int)group;
                    for (size_t t = 0; t < tasks.size(); ++t) {
                        const int *tb = &c->tblk[5 * tasks[t].first];
                        if (woff[t + 1] > woff[t]) w.kcols = std::max(w.kcols, tb[f.ld + 1] - tb[f.ld]);
                    }
                }
                c->st.quartets += w.nquart;
                c->st.primitive_quartets += w.nprimq;
                c->st.model_flops += w.flops;
                c->work.push_back(w);
            }
        }
    // the lists' pairs: the context's, then the parts
    vpairs.insert(vpairs.begin(), c->pairs.begin(), c->pairs.end());
    {
        int rc;
        if ((rc = dev_upload(&c->d_wpairs, vpairs, c->stream)) != PK_OK) return rc;
    }
    // largest classes first
    std::sort(c->work.begin(), c->work.end(), [](const ClassWork &x, const ClassWork &y) { return x.flops > y.flops; });
    // launch shapes chosen by pk_ctx_autotune for this context, if any
    for (ClassWork &w : c->work)
        for (const TuneEntry &t : c->tuned)
            if (t.cls == w.cls && t.prec == w.prec && t.rows == w.rows) {
                w.block = t.block;
                w.remap = t.remap;
                w.alt = t.alt;
            }
    // a short build: its lists for k_small
    int64_t waves = 0;
    for (const ClassWork &w : c->work) waves += w.nwaves;
    std::vector<pk::SmallList> small;  // uploaded from here until the synchronisation below
    if (waves <= kSmallWaves && !mixed && !c->block_forced) {
        c->small_tab[0].n = c->small_tab[1].n = 0;
        c->small_blocks[0] = c->small_blocks[1] = 0;
        c->small_lds[0] = c->small_lds[1] = 0;
        for (size_t i = 0; i < c->work.size(); ++i) {
            const ClassWork &w = c->work[i];
            const ClassFns &f = kClasses[w.cls];
            const pk::RowsEntry &r = rows_table()[w.cls];
            pk::SmallList l{w.d_wave, w.d_kets, w.nwaves, w.cls, 1};
            if (w.rows) l.chunk = std::max(1, std::min(8, (w.group + r.qw - 1) / r.qw / 2));
            small.push_back(l);
            if (!small_covers(w)) continue;
            pk::SmallTab &t = c->small_tab[f.small_set];
            t.first[t.n] = c->small_blocks[f.small_set];
            t.list[t.n++] = (int)i;
            c->small_blocks[f.small_set] += w.nwaves * (w.rows ? r.rc : 1);
            if (w.rows)
                c->small_lds[f.small_set] = std::max(
                    c->small_lds[f.small_set], (size_t)r.wave_bytes[0] + (size_t)pk::ncart(f.la) * pk::ncart(f.lb) * sizeof(double));
        }
        int rc;
        if ((rc = dev_upload(&c->d_small, small, c->stream)) != PK_OK) return rc;
    }
    PK_HIP(hipStreamSynchronize(c->stream));
    if (c->st.quartets >= kSideMinQuartets) {
        int rc;
        if ((rc = ensure_side(c)) != PK_OK) return rc;
    }
    c->work_ok = true;
    return PK_OK;
}

// Work items of the gradient (one molecule): for every ordered pair of pair
// classes and every bra, all kets with qmax_bra qmax_ket >= tol.  The pairs of a
// class are ordered by ordering group, then Schwarz bound, so the kets of a bra
// are one range per group (neighbouring ranges joined) and no list per bra is
// needed.
int build_grad(pk_ctx *c) {
    if (c->gwork_tol == c->tol) return PK_OK;
    free_grad(c);
    const int np = (int)c->pairs.size();
    std::vector<int> order;
    std::vector<int> cbeg(kPairClasses + 1, 0);
    std::vector<std::vector<int>> gseg(kPairClasses);  // starts of the groups in order, and the end
    for (int cl = 0; cl < kPairClasses; ++cl) {
        const size_t o0 = order.size();
        for (int p = 0; p < np; ++p)
            if (c->pair_cls[p] == cl) order.push_back(p);
        std::sort(order.begin() + o0, order.end(), [&](int x, int y) {
            if (c->pairs[x].grp != c->pairs[y].grp) return c->pairs[x].grp > c->pairs[y].grp;
            return c->pair_q[x] > c->pair_q[y];
        });
        for (size_t i = o0; i < order.size(); ++i)
            if (i == o0 || c->pairs[order[i]].grp != c->pairs[order[i - 1]].grp) gseg[cl].push_back((int)i);
        cbeg[cl + 1] = (int)order.size();
        gseg[cl].push_back((int)order.size());
    }
    int rc;
    if ((rc = dev_upload(&c->d_gorder, order, c->stream)) != PK_OK) return rc;
    struct Range {
        int start, count;
    };
    for (int cb = 0; cb < kPairClasses; ++cb)
        for (int ck = 0; ck < kPairClasses; ++ck) {
            const int nbra = cbeg[cb + 1] - cbeg[cb];
            if (nbra == 0 || cbeg[ck + 1] == cbeg[ck]) continue;
            std::vector<std::vector<Range>> rg(nbra);
            parallel_for((size_t)nbra, [&](size_t t) {
                const double qb = c->pair_q[order[cbeg[cb] + t]];
                for (size_t g = 0; g + 1 < gseg[ck].size(); ++g) {
                    int lo = gseg[ck][g], hi = gseg[ck][g + 1];
                    const int g0 = lo;
                    while (lo < hi) {
                        const int mid = (lo + hi) / 2;
                        if (qb * c->pair_q[order[mid]] >= c->tol)
                            lo = mid + 1;
                        else
                            hi = mid;
                    }
                    if (lo == g0) continue;
                    if (!rg[t].empty() && rg[t].back().start + rg[t].back().count == g0)
                        rg[t].back().count += lo - g0;
                    else
                        rg[t].push_back({g0, lo - g0});
                }
            });
            size_t tot = 0;
            for (const auto &v : rg)
                for (const Range &r : v) tot += r.count;
            if (tot == 0) continue;
            const pk::GradEntry &e = grad_table()[cb * kPairClasses + ck];
            const size_t group = (std::min<size_t>(kRowKetsMax, std::max<size_t>(1, tot / kGradItems)) + e.qw - 1) / e.qw * e.qw;
            std::vector<int> it[4];
            std::vector<double> cost;
            GradWork w;
            w.cls = cb * kPairClasses + ck;
            // steps of the item (n kets from s0): primitive quartets of the largest
            // quartet, and the densities' share, per group of slots
            auto steps = [&](int np, int s0, int n) {
                return (1.0 + (double)np * c->pairs[order[s0]].nprim) * ((n + e.qw - 1) / e.qw);
            };
            double total = 0.0;
            for (int t = 0; t < nbra; ++t)
                for (const Range &r : rg[t]) total += steps(c->pairs[order[cbeg[cb] + t]].nprim, r.start, r.count);
            const double most = std::max(32.0, total / kGradItems);  // steps of one item, about
            for (int t = 0; t < nbra; ++t)
                for (const Range &r : rg[t])
                    for (int s0 = 0; s0 < r.count; s0 += (int)group) {
                        const int n = std::min<int>((int)group, r.count - s0), b = order[cbeg[cb] + t];
                        const int np = c->pairs[b].nprim;
                        const double st = steps(np, r.start + s0, n);
                        const int cuts = std::max(1, std::min(np, (int)std::ceil(st / (2.0 * most))));
                        for (int k = 0; k < cuts; ++k) {
                            const int p0 = (int)((int64_t)np * k / cuts), p1 = (int)((int64_t)np * (k + 1) / cuts);
                            it[0].push_back(b);
                            it[1].push_back(r.start + s0);
                            it[2].push_back(n);
                            it[3].push_back(p0 | (p1 << 16));
                            cost.push_back(steps(p1 - p0, r.start + s0, n));
                        }
                    }
            const int ni = (int)cost.size();
            std::vector<int> o(ni), items(4 * (size_t)ni);
            std::iota(o.begin(), o.end(), 0);
            std::stable_sort(o.begin(), o.end(), [&](int x, int y) { return cost[x] > cost[y]; });
            for (int k = 0; k < 4; ++k)
                for (int i = 0; i < ni; ++i) items[(size_t)k * ni + i] = it[k][o[i]];
            // queue balance: longest lists first
            const int la = class_la(cb), lb = class_lb(cb), lc = class_la(ck), ld = class_lb(ck);
            const double per = 20.0 + 12.0 * (la + lb + lc + ld + 1) + 6.0 * pk::nlev(lc, lc + ld);
            for (double x : cost) w.cost += x * per * ((la + lb + lc + ld + 1) / 2 + 1);
            w.nitems = ni;
            if ((rc = dev_upload(&w.d_items, items, c->stream)) != PK_OK) return rc;
            PK_HIP(hipStreamSynchronize(c->stream));  // items leaves its scope
            c->gwork.push_back(w);
        }
    std::sort(c->gwork.begin(), c->gwork.end(), [](const GradWork &x, const GradWork &y) { return x.cost > y.cost; });
    PK_HIP(hipStreamSynchronize(c->stream));
    c->gwork_tol = c->tol;
    return PK_OK;
}

int ensure_buffers(pk_ctx *c) {
    const size_t n2 = c->n2 * sizeof(double);
    if (!c->d_P) PK_HIP(hipMalloc((void **)&c->d_P, n2));
    if (!c->d_Pn) PK_HIP(hipMalloc((void **)&c->d_Pn, n2));
    if (!c->d_A) PK_HIP(hipMalloc((void **)&c->d_A, n2));
    if (!c->d_B) PK_HIP(hipMalloc((void **)&c->d_B, n2));
    if (!c->d_J) PK_HIP(hipMalloc((void **)&c->d_J, n2));
    if (!c->d_K) PK_HIP(hipMalloc((void **)&c->d_K, n2));
    if (!c->d_G) PK_HIP(hipMalloc((void **)&c->d_G, n2));
    if (!c->d_P32 && c->precision == PK_PREC_MIXED) PK_HIP(hipMalloc((void **)&c->d_P32, c->n2 * sizeof(float)));
    return PK_OK;
}

// Enqueue the kernels of one build on the context stream: P (device) -> A, B
// accumulators -> J, K, G (any may be null).  Class events only when profiling
// (never while the stream is being captured).
// Per-build scratch: the scaled density and the J, K accumulators (packed,
// c->n2 doubles each).
// One-pass UHF adds the scaled exchange densities PKa, PKb and the second K
// accumulator B2 (all null for RHF; Pn then holds Pa + Pb).
// P32 is an FP32 copy of Pn for the FP32 kernels of the mixed precision.
struct BuildBufs {
    double *Pn, *A, *B;
    float *P32 = nullptr;
    double *PKa = nullptr, *PKb = nullptr, *B2 = nullptr;
};

BuildBufs ctx_bufs(pk_ctx *c) { return BuildBufs{c->d_Pn, c->d_A, c->d_B, c->d_P32}; }

// Enqueue the class kernels of one build (the density already scaled into
// sb.Pn, the accumulators cleared); nl counts the launches.  With sb.B2 set
// (one-pass UHF) every list runs FP64 two-density digestion: the per-lane OS
// or row kernels where the class has them, else the per-lane Rys kernels twice.
int launch_list(pk_ctx *c, ClassWork &w, const BuildBufs &sb, bool events, hipStream_t s, int &nl);

// Side streams and events of a context, created on first use.
int ensure_side(pk_ctx *c) {
    if (c->side_ok) return PK_OK;
    if (!c->fork_ev) PK_HIP(hipEventCreateWithFlags(&c->fork_ev, hipEventDisableTiming));
    for (int i = 0; i < kSideQueues; ++i) {
        if (!c->side[i]) PK_HIP(hipStreamCreateWithFlags(&c->side[i], hipStreamNonBlocking));
        if (!c->join_ev[i]) PK_HIP(hipEventCreateWithFlags(&c->join_ev[i], hipEventDisableTiming));
    }
    c->side_ok = true;
    return PK_OK;
}

// Side queues of the work at hand: q[0] is the context stream, the others wait for
// what it holds so far.
int fork_side(pk_ctx *c, hipStream_t (&q)[kSideQueues + 1]) {
    q[0] = c->stream;
    PK_HIP(hipEventRecord(c->fork_ev, c->stream));
    for (int i = 0; i < kSideQueues; ++i) {
        q[i + 1] = c->side[i];
        PK_HIP(hipStreamWaitEvent(c->side[i], c->fork_ev, 0));
    }
    return PK_OK;
}

// The context stream waits for the side queues.  Called after a failed launch as well
// (status rc, returned): kernels already on them still use the context's buffers.
int join_side(pk_ctx *c, int rc) {
    for (int i = 0; i < kSideQueues; ++i) {
        hipError_t e = hipEventRecord(c->join_ev[i], c->side[i]);
        if (e == hipSuccess) e = hipStreamWaitEvent(c->stream, c->join_ev[i], 0);
        if (e != hipSuccess && rc == PK_OK) rc = fail(PK_ERR_HIP, std::string("side queue join: ") + hipGetErrorString(e));
    }
    return rc;
}

// kernel arguments of a build, without those of a list
pk::JKArgs build_args(const pk_ctx *c, const BuildBufs &sb) {
    pk::JKArgs a{};
    a.pairs = c->d_wpairs;
    a.prims = c->d_prims;
    a.hz = c->d_hz;
    a.mol_off = c->d_mol_off;
    a.mol_nb = c->d_mol_nb;
    a.P = sb.Pn;
    a.P32 = sb.P32;
    a.PK = sb.PKa;
    a.PK2 = sb.PKb;
    a.Q = c->d_Q;
    a.A = sb.A;
    a.B = sb.B;
    a.B2 = sb.B2;
    a.tol = c->tol;
    a.tblk = c->d_tblk;
    return a;
}

// The lists of a short build that k_small covers, in one launch (two with f
// shells); the rest one by one.
int launch_small(pk_ctx *c, const BuildBufs &sb, int &nl) {
    static const void *const kernel[2] = {pk_small_kernel<0>(), pk_small_kernel<1>()};
    static const hipError_t attr[2] = {
        hipFuncSetAttribute(kernel[0], hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsMax),
        hipFuncSetAttribute(kernel[1], hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsMax)};
    pk::JKArgs a = build_args(c, sb);
    const pk::SmallList *lists = c->d_small;
    for (int k = 0; k < 2; ++k) {
        if (c->small_tab[k].n == 0) continue;
        PK_HIP(attr[k]);
        void *args[] = {&a, &lists, &c->small_tab[k]};
        PK_HIP(hipLaunchKernel(kernel[k], dim3(c->small_blocks[k]), dim3(64), args, c->small_lds[k], c->stream));
        ++nl;
    }
    int rc;
    for (ClassWork &w : c->work) {
        if (small_covers(w))
            w.kernels = 1, w.block_run = 64;  // the launch it shares
        else if ((rc = launch_list(c, w, sb, false, c->stream, nl)) != PK_OK)
            return rc;
    }
    return PK_OK;
}

int launch_classes(pk_ctx *c, const BuildBufs &sb, bool events, int &nl) {
    int rc;
    hipStream_t s = c->stream;
    if (!events && one_launch(c, sb.B2)) return launch_small(c, sb, nl);
    // Concurrent queues (not while profiling: the class events time one list
    // at a time): lists in descending model cost, each to the queue with the
    // least cost so far, so that the small classes fill the tails of the
    // large ones.  All lists add into the same accumulators with atomics.
    if (!events && c->side_ok && !c->side_off && c->st.quartets >= kSideMinQuartets && c->work.size() > 1) {
        hipStream_t q[kSideQueues + 1];
        if ((rc = fork_side(c, q)) != PK_OK) return rc;
        std::vector<size_t> order(c->work.size());
        for (size_t i = 0; i < order.size(); ++i) order[i] = i;
        // cost of a list: its measured time when the context has one (the first
        // large build of a context times every list, one at a time), else the
        // model flops over a typical rate of its kernel (TFLOP/s: per-lane OS
        // ~10, per-lane Rys ~3, row kernels ~6)
        std::vector<double> cost(c->work.size());
        for (size_t i = 0; i < cost.size(); ++i) {
            const ClassWork &w = c->work[i];
            const int kind = list_kind(c, w) % 3;  // 0 OS, 1 Rys, 2 rows
            cost[i] = w.cost_ms > 0.0 ? w.cost_ms : w.flops * 1e-9 / (kind == 0 ? 10.0 : kind == 1 ? 3.0 : 6.0);
        }
        std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) { return cost[x] > cost[y]; });
        double load[kSideQueues + 1] = {};
        for (size_t i : order) {
            int k = 0;
            for (int j = 1; j <= kSideQueues; ++j)
                if (load[j] < load[k]) k = j;
            load[k] += cost[i];
            if ((rc = launch_list(c, c->work[i], sb, false, q[k], nl)) != PK_OK) break;
        }
        return join_side(c, rc);
    }
    for (ClassWork &w : c->work)
        if ((rc = launch_list(c, w, sb, events, s, nl)) != PK_OK) return rc;
    return PK_OK;
}

// Enqueue the kernels of one class list on stream s.
int launch_list(pk_ctx *c, ClassWork &w, const BuildBufs &sb, bool events, hipStream_t s, int &nl) {
    int rc;
    {
        const int *wv = w.d_wave;
        pk::JKArgs a = build_args(c, sb);
        a.wave_bra = wv;
        a.wave_start = wv + w.nwaves;
        a.wave_count = wv + 2 * w.nwaves;
        a.wave_mol = wv + 3 * w.nwaves;
        a.kets = w.d_kets;
        a.nwaves = w.nwaves;
        a.remap = w.remap;
        a.seg = w.d_seg;
        a.nseg = w.nseg;
        a.kcols = w.kcols;
        const bool uhf = sb.B2 != nullptr;
        if (events) {
            if (!w.e0) PK_HIP(hipEventCreate(&w.e0));
            if (!w.e1) PK_HIP(hipEventCreate(&w.e1));
            PK_HIP(hipEventRecord(w.e0, s));
        }
        const int before = nl;
        const ClassFns &f = kClasses[w.cls];
        const bool fp32 = w.prec == PK_PREC_MIXED && !w.alt;
        // segment mode when the exchange rows of the call fit the LDS budget
        // (two rows sets for the one-pass UHF OS kernels); the low-L OS classes
        // compiled both ways take it for lists of few primitive quartets per
        // shell quartet (atomic-bound), the plain kernel otherwise
        const bool seg_alt = f.seg_alt && use_os(c, f) && (double)w.nprimq <= c->seg_alt_prim * (double)w.nquart;
        if (w.rows) {
            const pk::RowsEntry &r = rows_table()[w.cls];
            const int rk = uhf ? 2 : 1;
            const size_t wave_bytes = r.wave_bytes[rk - 1];
            const void *k = uhf ? r.k2 : r.k1;
            // exchange rows of the kets' second shells in LDS, beside at least one
            // wave.  Even where they leave room for few waves they win as a whole:
            // 40 waters 6 Angstrom apart / cc-pVTZ (2600 functions, rows of up to 134 KB)
            // 319 ms against 462 without rows, (fd|dp) 3.4 / 7.9, (fd|pp) 3.7 / 11.5;
            // only lists of few kets per row column lose, (ff|fp) 2.2 / 1.1, (fd|fd)
            // 1.0 / 0.5, (ff|ff) 0.4 / 0.2, (ff|fs) 1.5 / 1.2, (fs|fs) 2.4 / 2.1.
            const size_t jrow = (size_t)pk::ncart(f.la) * pk::ncart(f.lb) * sizeof(double);
            size_t krow = (size_t)rk * (pk::ncart(f.la) + pk::ncart(f.lb)) * w.kcols * sizeof(double) + jrow;
            a.segmode = c->seg_on && krow + wave_bytes <= kLdsMax;
            if (!a.segmode) krow = jrow;
            static std::atomic<int> attr_done[2 * kQuartClasses];  // zero-initialised
            std::atomic<int> &done = attr_done[2 * w.cls + rk - 1];
            if (!done.load()) {
                PK_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsMax));
                done.store(1);
            }
            const int groups = (w.group + r.qw - 1) / r.qw;  // of the largest work item
            if (w.row_waves[rk - 1] == 0) {
                // Waves per workgroup: as few as keep the most waves resident on a CU
                // (they share the exchange rows in LDS), two at least.  A workgroup's
                // waves wait for its last one before the flush; n-C10H22 / cc-pVTZ, two
                // waves against four where both keep eight resident: (dp|pp) 4.3 / 4.8 ms,
                // (pp|pp) 1.9 / 2.2, (fs|pp) 2.4 / 2.7; six against eight: (fp|dp) 3.0 / 2.5,
                // (fd|dp) 2.6 / 2.2; one against two (five against eight): (dp|pp) 5.5 / 4.3
                int best = 0, most = 0;
                for (int n = kRowWavesMax; n >= 2; n /= 2) {
                    int wgs = 0;
                    if (krow + (size_t)n * wave_bytes > kLdsMax) continue;
                    PK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&wgs, k, 64 * n, krow + (size_t)n * wave_bytes));
                    if (wgs * n >= most) {
                        most = wgs * n;
                        best = n;
                    }
                }
                w.row_waves[rk - 1] = std::max(1, best);
            }
            int waves = w.block > 0 ? w.block / 64 : w.row_waves[rk - 1];
            while (waves > 1 && (waves / 2 >= groups || krow + (size_t)waves * wave_bytes > kLdsMax)) waves /= 2;
            // eight groups per turn of a wave, fewer where the item has fewer
            a.chunk = std::max(1, std::min(8, groups / (2 * waves)));
            w.block_run = 64 * waves;
            int grid = w.nwaves;
            if (w.remap) grid = (grid + 7) / 8 * 8;
            void *args[] = {&a};
            PK_HIP(hipLaunchKernel(k, dim3(grid, r.rc), dim3(64 * waves), args, krow + (size_t)waves * wave_bytes, s));
            w.kernels = 1;
            ++nl;
            if (events) PK_HIP(hipEventRecord(w.e1, s));
            return PK_OK;
        }
        const int nk = uhf && use_os(c, f) ? 2 : 1;
        {
            const size_t rows = (size_t)nk * (pk::ncart(f.la) + pk::ncart(f.lb)) * w.kcols +
                                (size_t)pk::ncart(f.la) * pk::ncart(f.lb);
            a.segmode = c->seg_on && (f.seg || seg_alt) && w.nseg > 0 && rows * sizeof(double) <= kSegLdsMax;
        }
        if (w.nseg < kMinSegs) a.segmode = 0;  // the waves of a segment run one after another
        const bool alt = seg_alt && a.segmode;  // the segment-mode variant of a plain OS class
        // lanes per workgroup: the autotuned (or PK_BLOCK) shape, else one wave
        // per workgroup for the segment-mode lists of a batch of molecules whose
        // exchange rows leave room for at least 6 such workgroups per CU (256 water
        // clusters, rows of 2-19 KB: every list is faster with one wave, 356 -> 256 ms
        // for the build), and kDefaultBlock otherwise (one molecule, segments of
        // many kets: n-C10H22 / cc-pVTZ (pp|ss) 7.4 -> 3.5 ms with four waves for one)
        const bool one_wave =
            a.segmode && c->nmol > 1 && pk::jk_lds_bytes(a, f.la, f.lb, nk) <= kSegOneWaveLds;
        const int block = w.block > 0 ? w.block : (one_wave ? 64 : kDefaultBlock);
        w.block_run = block;
        const int wpb = block / 64;
        int grid = a.segmode ? w.nseg : (w.nwaves + wpb - 1) / wpb;
        if (w.remap) grid = (grid + 7) / 8 * 8;
        if (uhf && use_os(c, f)) {
            (alt ? f.jk_os_uhf_seg : f.jk_os_uhf)(a, grid, block, s, nl);
        } else if (uhf) {
            // per-lane Rys kernels once per spin density: J of each into A
            // (summing to J of Pa + Pb), exchange into B and B2
            pk::JKArgs x = a;
            x.P = sb.PKa;
            f.jk_rys(x, grid, block, s, nl);
            x.P = sb.PKb;
            x.B = sb.B2;
            f.jk_rys(x, grid, block, s, nl);
        } else if (use_os(c, f)) {
            if (alt)
                (fp32 ? f.jk_os32_seg : f.jk_os_seg)(a, grid, block, s, nl);
            else
                (fp32 ? f.jk_os32 : f.jk_os)(a, grid, block, s, nl);
        } else if (!(w.alt && w.prec == PK_PREC_FP64)) {
            (fp32 ? f.jk_rys32 : f.jk_rys)(a, grid, block, s, nl);
        }
        if (!uhf && !use_os(c, f) && w.alt && w.prec == PK_PREC_FP64) {
            pk::GenArgs g{};
            g.wave_bra = a.wave_bra;
            g.wave_start = a.wave_start;
            g.wave_count = a.wave_count;
            g.wave_mol = a.wave_mol;
            g.kets = a.kets;
            g.mol_off = a.mol_off;
            g.mol_nb = a.mol_nb;
            g.pairs = a.pairs;
            g.prims = a.prims;
            g.hz = a.hz;
            g.P = a.P;
            g.Q = a.Q;
            g.A = a.A;
            g.B = a.B;
            g.tol = a.tol;
            g.nitems = w.nwaves;
            g.la = f.la;
            g.lb = f.lb;
            g.lc = f.lc;
            g.ld = f.ld;
            if ((rc = launch_generic(g, s)) != PK_OK) return rc;
            ++nl;
        }
        w.kernels = nl - before;
        if (events) PK_HIP(hipEventRecord(w.e1, s));
    }
    return PK_OK;
}

int launch_build(pk_ctx *c, const double *dP, double *dJ, double *dK, double *dG, const BuildBufs &sb,
                 bool events) {
    int rc;
    hipStream_t s = c->stream;
    const MolTab t{c->d_mol_off, c->d_mol_nb, c->d_mol_foff, c->d_fpos};
    const dim3 g2((unsigned)(((size_t)c->nbmax * c->nbmax + 255) / 256), (unsigned)c->nmol);
    const int gf = (int)((c->n2 + 255) / 256);
    hipLaunchKernelGGL(k_prepare, g2, dim3(256), 0, s, dP, c->d_fnorm, sb.Pn, sb.A, sb.B, t);
    int nl = 1;
    if (c->precision == PK_PREC_MIXED) {
        if (!sb.P32) return fail(PK_ERR_STATE, "mixed precision build without an FP32 density buffer");
        hipLaunchKernelGGL(k_to_f32, dim3(gf), dim3(256), 0, s, sb.Pn, sb.P32, c->n2);
        ++nl;
    }
    if ((rc = launch_classes(c, sb, events, nl)) != PK_OK) return rc;
    hipLaunchKernelGGL(k_finalize, g2, dim3(256), 0, s, sb.A, sb.B, c->d_fnorm, dJ, dK, dG, t);
    ++nl;
    PK_HIP(hipGetLastError());
    c->st.kernel_launches = nl;
    return PK_OK;
}

// One-pass UHF build: Pn = n n^T o (Pa + Pb) for J, PKa, PKb the scaled spin
// densities for the two exchange matrices; each integral computed once.
int launch_build_uhf(pk_ctx *c, const double *dPa, const double *dPb, double *dJt, double *dKa, double *dKb,
                     const BuildBufs &sb, bool events) {
    int rc;
    hipStream_t s = c->stream;
    const MolTab t{c->d_mol_off, c->d_mol_nb, c->d_mol_foff, c->d_fpos};
    const dim3 g2((unsigned)(((size_t)c->nbmax * c->nbmax + 255) / 256), (unsigned)c->nmol);
    const int gf = (int)((c->n2 + 255) / 256);
    hipLaunchKernelGGL(k_scale_density, g2, dim3(256), 0, s, dPa, c->d_fnorm, sb.PKa, t);
    hipLaunchKernelGGL(k_scale_density, g2, dim3(256), 0, s, dPb, c->d_fnorm, sb.PKb, t);
    hipLaunchKernelGGL(k_sum2, dim3(gf), dim3(256), 0, s, sb.PKa, sb.PKb, sb.Pn, c->n2);
    hipLaunchKernelGGL(k_fill, dim3(gf), dim3(256), 0, s, sb.A, c->n2, 0.0);
    hipLaunchKernelGGL(k_fill, dim3(gf), dim3(256), 0, s, sb.B, c->n2, 0.0);
    hipLaunchKernelGGL(k_fill, dim3(gf), dim3(256), 0, s, sb.B2, c->n2, 0.0);
    int nl = 6;
    if ((rc = launch_classes(c, sb, events, nl)) != PK_OK) return rc;
    hipLaunchKernelGGL(k_finalize, g2, dim3(256), 0, s, sb.A, sb.B, c->d_fnorm, dJt, dKa, (double *)nullptr, t);
    hipLaunchKernelGGL(k_finalize, g2, dim3(256), 0, s, sb.A, sb.B2, c->d_fnorm, (double *)nullptr, dKb,
                       (double *)nullptr, t);
    nl += 2;
    PK_HIP(hipGetLastError());
    c->st.kernel_launches = nl;
    return PK_OK;
}

// One build.  With graphs enabled (and profiling off) the kernels of a build
// are captured once into a hipGraph that reads the context's own density
// buffer and writes its own J, K, G buffers, and every later build replays
// it; the caller's buffers are copied in and out around the replay.
int build_device(pk_ctx *c, const double *dP, double *dJ, double *dK, double *dG) {
    int rc;
    if (!c->work_ok && (rc = build_work(c)) != PK_OK) return rc;
    if ((rc = ensure_buffers(c)) != PK_OK) return rc;
    hipStream_t s = c->stream;
    const size_t bytes = c->n2 * sizeof(double);
    // the first build that would spread its lists over the side queues times every
    // list (one at a time), so that later builds balance the queues by measured cost
    c->learning = !c->cost_learned && !c->profile && c->side_ok && !c->side_off && !one_launch(c, nullptr) &&
                  c->st.quartets >= kSideMinQuartets && c->work.size() > 1;
    if (!c->graph_on || c->profile || c->learning) {
        PK_HIP(hipEventRecord(c->ev0, s));
        if ((rc = launch_build(c, dP, dJ, dK, dG, ctx_bufs(c), c->profile || c->learning)) != PK_OK) return rc;
        PK_HIP(hipEventRecord(c->ev1, s));
        return PK_OK;
    }
    if (!c->graph_ok) {
        drop_graph(c);
        PK_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
        const int rc_cap = launch_build(c, c->d_P, c->d_J, c->d_K, c->d_G, ctx_bufs(c), false);
        hipGraph_t g = nullptr;
        const hipError_t e = hipStreamEndCapture(s, &g);
        if (rc_cap != PK_OK) {
            if (g) (void)hipGraphDestroy(g);
            return rc_cap;
        }
        PK_HIP(e);
        c->graph = g;
        PK_HIP(hipGraphInstantiate(&c->gexec, g, nullptr, nullptr, 0));
        c->graph_ok = true;
    }
    PK_HIP(hipEventRecord(c->ev0, s));
    if (dP != c->d_P) PK_HIP(hipMemcpyAsync(c->d_P, dP, bytes, hipMemcpyDeviceToDevice, s));
    PK_HIP(hipGraphLaunch(c->gexec, s));
    if (dJ && dJ != c->d_J) PK_HIP(hipMemcpyAsync(dJ, c->d_J, bytes, hipMemcpyDeviceToDevice, s));
    if (dK && dK != c->d_K) PK_HIP(hipMemcpyAsync(dK, c->d_K, bytes, hipMemcpyDeviceToDevice, s));
    if (dG && dG != c->d_G) PK_HIP(hipMemcpyAsync(dG, c->d_G, bytes, hipMemcpyDeviceToDevice, s));
    PK_HIP(hipEventRecord(c->ev1, s));
    return PK_OK;
}

int finish_timing(pk_ctx *c) {
    PK_HIP(hipEventSynchronize(c->ev1));
    float ms = 0.f;
    PK_HIP(hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->st.last_build_ms = ms;
    c->st.last_eri_kernel_ms = ms;
    if (c->profile || c->learning) {
        double eri = 0.0;
        for (ClassWork &w : c->work) {
            float m = 0.f;
            PK_HIP(hipEventElapsedTime(&m, w.e0, w.e1));
            if (c->profile) {
                w.ms_total += m;
                w.builds += 1;
            }
            w.cost_ms = m;
            eri += m;
        }
        c->st.last_eri_kernel_ms = eri;
        c->cost_learned = true;
        c->learning = false;
    }
    return PK_OK;
}

}  // namespace

int pk_build_with_scratch(pk_ctx *c, const double *P, double *J, double *K, double *scratch, size_t each,
                          const char *caller) {
    const std::string who = caller ? caller : "pk_build_with_scratch";
    if (!c || !P || !scratch) return fail(PK_ERR_ARG, who + ": null context, density or scratch");
    if (c->n2 > each)
        return fail(PK_ERR_ARG, who + ": packed matrices of " + std::to_string(c->n2) +
                                    " elements exceed the scratch limit of " + std::to_string(each) + " elements");
    if (!c->work_ok)
        return fail(PK_ERR_STATE, who + ": the work lists of the current settings are not built "
                                        "(call pk_fock_jk once after pk_ctx_create / pk_ctx_set)");
    BuildBufs sb{scratch, scratch + each, scratch + 2 * each};
    sb.P32 = reinterpret_cast<float *>(scratch + 3 * each);
    return launch_build(c, P, J, K, nullptr, sb, false);
}

int pk_set_error(int code, const char *msg) { return fail(code, msg ? msg : ""); }

// ====================================================================== C ABI
extern "C" {

const char *pk_last_error(void) { return g_err.c_str(); }

}  // extern "C"

namespace {

// Ordering group of a pair with n primitive pairs: floor(log_1.5 n).  Kets of
// one group run the primitive loop for up to 1.5 times as many iterations as
// the group's smallest member (idle lanes), in exchange for longer runs of
// neighbouring second shells in a wave (fewer cache lines per atomic add).
// Measured on n-C20H42 / cc-pVDZ (ms per build): exact primitive counts 60.9,
// ratio 1.5 58.3; an earlier sweep gave 62.2 / 61.1 / 61.0 / 61.3 / 63.4 for
// exact / 1.25 / 1.5 / 2 / 3.
constexpr double kGroupRatio = 1.5;
int prim_group(int n) { return (int)std::floor(std::log((double)n) / std::log(kGroupRatio) + 1e-9); }

// Shells, component norms and shell pairs of molecule m (pairs within the
// molecule only), appended to the context's arrays.
int add_molecule(pk_ctx *c, const pk_basis_desc *d, int m) {
    if (!d || d->nshells <= 0 || !d->center || !d->l || !d->nprim || !d->exponent || !d->coef || !d->prim_norm)
        return fail(PK_ERR_ARG, "pk_ctx_create: null or empty basis description (molecule " + std::to_string(m) + ")");
    const int s0 = c->ns;
    int off = (int)c->ex.size(), f0 = 0;
    const int poff0 = off;
    for (int s = 0; s < d->nshells; ++s) {
        const int l = d->l[s];
        if (l < 0 || l > kMaxL)
            return fail(PK_ERR_UNSUPPORTED, "pk_ctx_create: shell " + std::to_string(s) + " has l=" + std::to_string(l) +
                                                "; this build supports l <= " + std::to_string(kMaxL));
        if (d->nprim[s] <= 0) return fail(PK_ERR_ARG, "pk_ctx_create: shell with no primitives");
    }
    // internal order: shells grouped by l, basis order within a group
    std::vector<int> spos(d->nshells), snat(d->nshells);
    {
        int pos = 0;
        for (int l = 0; l <= kMaxL; ++l) {
            c->tblk.push_back(pos);
            for (int s = 0; s < d->nshells; ++s)
                if (d->l[s] == l) {
                    spos[s] = pos;
                    pos += pk::ncart(l);
                }
        }
        c->tblk.push_back(pos);
        for (int s = 0, f = 0; s < d->nshells; ++s) {
            snat[s] = f;
            f += pk::ncart(d->l[s]);
        }
        const size_t fb = c->fnorm.size();
        c->fnorm.resize(fb + pos);
        c->fnat.resize(fb + pos);
        c->fpos.resize(fb + pos);
        for (int s = 0; s < d->nshells; ++s)
            for (int k = 0; k < pk::ncart(d->l[s]); ++k) {
                c->fpos[fb + snat[s] + k] = spos[s] + k;
                c->fnat[fb + spos[s] + k] = snat[s] + k;
            }
    }
    const size_t fbase = (size_t)c->nb;  // this molecule's first entry in fnorm / fpos / fnat
    for (int s = 0; s < d->nshells; ++s) {
        const int l = d->l[s], np = d->nprim[s];
        c->sh_l.push_back(l);
        c->sh_np.push_back(np);
        c->sh_poff.push_back(off);
        c->sh_f0.push_back(spos[s]);
        for (int q = 0; q < 3; ++q) c->sh_c.push_back(d->center[3 * s + q]);
        for (int k = 0; k < np; ++k) {
            c->ex.push_back(d->exponent[off - poff0 + k]);
            c->co.push_back(d->coef[off - poff0 + k]);
            c->pn.push_back(d->prim_norm[off - poff0 + k]);
        }
        // component norms 1/sqrt((2lx-1)!!(2ly-1)!!(2lz-1)!!)  (gaussian.cpp:286-298)
        for (int k = 0; k < pk::ncart(l); ++k) {
            auto df = [](int n) {
                int r = 1;
                while (n > 0) {
                    r *= n;
                    n -= 2;
                }
                return r;
            };
            const int x = pk::cart_x(l, k), y = pk::cart_y(l, k), z = pk::cart_z(l, k);
            c->fnorm[fbase + spos[s] + k] = 1.0 / std::sqrt((double)(df(2 * x - 1) * df(2 * y - 1) * df(2 * z - 1)));
        }
        off += np;
        f0 += pk::ncart(l);
    }
    // the kernels pack (pair primitive count, first function) into one int
    if (f0 >= (1 << 20)) return fail(PK_ERR_ARG, "pk_ctx_create: more than 2^20 functions in one molecule");
    for (int s = s0; s < s0 + d->nshells; ++s)
        if (c->sh_np[s] * c->sh_np[s] >= 2048) return fail(PK_ERR_ARG, "pk_ctx_create: shell with more than 45 primitives");
    c->ns += d->nshells;
    c->mol_foff.push_back(c->nb);
    c->mol_nb.push_back(f0);
    c->mol_off.push_back((long long)c->n2);
    c->nb += f0;
    c->n2 += (size_t)f0 * f0;
    c->nbmax = std::max(c->nbmax, f0);
    // shell pairs a >= b, first shell carries the larger l (types.h:606-675 pair data)
    const size_t pair0 = c->pairs.size();
    std::vector<std::vector<pk::PrimDev>> pp_all;
    std::vector<std::vector<double>> pa_all;
    double kmax = 0.0;  // max over primitive pairs of |kc| / sqrt(zeta)
    for (int A = s0; A < c->ns; ++A)
        for (int Bs = s0; Bs <= A; ++Bs) {
            const int sa = c->sh_l[A] >= c->sh_l[Bs] ? A : Bs, sb = sa == A ? Bs : A;
            pk::PairDev p{};
            p.f0 = c->sh_f0[sa];
            p.f1 = c->sh_f0[sb];
            p.diag = A == Bs;
            const double *Ac = &c->sh_c[3 * sa], *Bc = &c->sh_c[3 * sb];
            for (int q = 0; q < 3; ++q) p.ab[q] = Ac[q] - Bc[q];
            const double R2 = p.ab[0] * p.ab[0] + p.ab[1] * p.ab[1] + p.ab[2] * p.ab[2];
            std::vector<pk::PrimDev> pps;
            std::vector<double> pal;
            for (int i = 0; i < c->sh_np[sa]; ++i)
                for (int j = 0; j < c->sh_np[sb]; ++j) {
                    const double al = c->ex[c->sh_poff[sa] + i], be = c->ex[c->sh_poff[sb] + j];
                    const double ca = c->co[c->sh_poff[sa] + i] * c->pn[c->sh_poff[sa] + i];
                    const double cb = c->co[c->sh_poff[sb] + j] * c->pn[c->sh_poff[sb] + j];
                    pk::PrimDev pp{};
                    pp.zeta = al + be;
                    const double iz = 1.0 / pp.zeta;
                    // K_ab sqrt(zeta) (4/pi)^(1/4): two records and 1/sqrt(zeta+eta)
                    // give K_ab K_cd 2 sqrt(rho/pi)
                    pp.kc = std::pow(M_PI * iz, 1.5) * std::exp(-(al * be * iz) * R2) * ca * cb *
                            std::sqrt(pp.zeta) * 1.0622519320271969145;
                    for (int q = 0; q < 3; ++q) {
                        pp.p[q] = (al * Ac[q] + be * Bc[q]) * iz;
                        pp.pa[q] = pp.p[q] - Ac[q];
                    }
                    kmax = std::max(kmax, std::fabs(pp.kc) / std::sqrt(pp.zeta));
                    pps.push_back(pp);
                    pal.push_back(al);
                }
            // A shell pair on one centre: alpha_i + beta_j repeats with the roles of
            // the two exponents swapped (s and p contractions over one set of
            // exponents, and every shell with itself), and so do P and P - A = 0, so
            // such primitive pairs are one with the sum of their coefficients (the
            // gradient is linear in the exponent on A: its weighted mean).  Coefficients
            // that nearly cancel stay apart, the mean would lose digits.
            if (R2 == 0.0) {
                size_t n = 0;
                for (size_t i = 0; i < pps.size(); ++i) {
                    size_t j = 0;
                    for (; j < n; ++j) {
                        const double sum = pps[j].kc + pps[i].kc;
                        if (pps[j].zeta == pps[i].zeta && pps[j].p[0] == pps[i].p[0] && pps[j].p[1] == pps[i].p[1] &&
                            pps[j].p[2] == pps[i].p[2] &&
                            std::fabs(sum) >= 0.5 * std::max(std::fabs(pps[j].kc), std::fabs(pps[i].kc))) {
                            pal[j] = (pps[j].kc * pal[j] + pps[i].kc * pal[i]) / sum;
                            pps[j].kc = sum;
                            break;
                        }
                    }
                    if (j == n) {
                        pps[n] = pps[i];
                        pal[n++] = pal[i];
                    }
                }
                pps.resize(n);
                pal.resize(n);
                for (const pk::PrimDev &pp : pps) kmax = std::max(kmax, std::fabs(pp.kc) / std::sqrt(pp.zeta));
            }
            pp_all.push_back(std::move(pps));
            pa_all.push_back(std::move(pal));
            c->pair_sh.push_back(sa);
            c->pair_sh.push_back(sb);
            c->pairs.push_back(p);
            c->pair_cls.push_back(pk::pair_class(c->sh_l[sa], c->sh_l[sb]));
            c->pair_q.push_back(0.0);
            c->pair_mol.push_back(m);
        }
    // Primitive screening: a primitive pair whose prefactor bound
    // |kc_p| max_q |kc_q| / sqrt(eta_q) (>= |kc_p kc_q| / sqrt(zeta_p + eta_q))
    // is below kPrimCut cannot move any integral by more than that times its
    // angular factors; it is dropped (distant tight primitives: e^{-ab R^2/z}).
    for (size_t k = 0; k < pp_all.size(); ++k) {
        pk::PairDev &p = c->pairs[pair0 + k];
        p.prim_off = (int)c->prims.size();
        for (size_t i = 0; i < pp_all[k].size(); ++i)
            if (std::fabs(pp_all[k][i].kc) * kmax >= kPrimCut) {
                c->prims.push_back(pp_all[k][i]);
                c->palpha.push_back(pa_all[k][i]);
                c->hz.push_back(0.5 / pp_all[k][i].zeta);
            }
        p.nprim = (int)c->prims.size() - p.prim_off;
        p.grp = prim_group(p.nprim);
    }
    return PK_OK;
}

int ctx_build(const pk_basis_desc *descs, int nmol, pk_ctx **out) {
    if (!descs || !out || nmol <= 0) return fail(PK_ERR_ARG, "pk_ctx_create: null or empty basis description");
    *out = nullptr;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
        return fail(PK_ERR_HIP, "pk_ctx_create: no HIP device visible");
    pk_ctx *c = new pk_ctx;
    c->nmol = nmol;
    for (int m = 0; m < nmol; ++m) {
        const int rc = add_molecule(c, &descs[m], m);
        if (rc != PK_OK) {
            delete c;
            return rc;
        }
    }
    if (c->prims.size() > (size_t)INT32_MAX || c->n2 > (size_t)1 << 40) {
        delete c;
        return fail(PK_ERR_ARG, "pk_ctx_create: batch too large");
    }
    c->st.nbasis = c->nb;
    c->st.nshells = c->ns;
    // diagnostic switch: PK_EXCHANGE_ROWS=0 runs the per-lane kernels without
    // the LDS exchange rows (one global atomic per exchange contribution)
    if (const char *e = std::getenv("PK_EXCHANGE_ROWS")) c->seg_on = std::atoi(e) != 0;
    // diagnostic switch: PK_SIDE_QUEUES=0 keeps every class kernel of a build
    // on the context stream (one kernel at a time, as a kernel trace times them)
    if (const char *e = std::getenv("PK_SIDE_QUEUES")) c->side_off = std::atoi(e) == 0;
    // diagnostic knob: PK_SEG_ALT_PRIM overrides the primitive quartets per
    // shell quartet below which the low-L OS lists run in segment mode
    if (const char *e = std::getenv("PK_SEG_ALT_PRIM")) c->seg_alt_prim = std::atof(e);
    // diagnostic knob: PK_BLOCK = 64, 128 or 256 lanes per workgroup of every
    // class list until pk_ctx_autotune chooses per list
    if (const char *e = std::getenv("PK_BLOCK")) {
        const int b = std::atoi(e);
        if (b == 64 || b == 128 || b == 256) c->block0 = b, c->block_forced = true;
    }
    c->st.shell_pairs = (int64_t)c->pairs.size();
    int rc = PK_OK;
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess) {
        pk_ctx_destroy(c);
        return fail(PK_ERR_HIP, "pk_ctx_create: stream/event creation failed");
    }
    c->own_stream = true;
    if ((rc = dev_upload(&c->d_mol_off, c->mol_off, c->stream)) != PK_OK ||
        (rc = dev_upload(&c->d_mol_nb, c->mol_nb, c->stream)) != PK_OK ||
        (rc = dev_upload(&c->d_mol_foff, c->mol_foff, c->stream)) != PK_OK ||
        (rc = dev_upload(&c->d_tblk, c->tblk, c->stream)) != PK_OK ||
        (rc = dev_upload(&c->d_pairs, c->pairs, c->stream)) != PK_OK ||
        (rc = dev_upload(&c->d_prims, c->prims, c->stream)) != PK_OK ||
        (rc = dev_upload(&c->d_palpha, c->palpha, c->stream)) != PK_OK ||
        (rc = dev_upload(&c->d_hz, c->hz, c->stream)) != PK_OK ||
        (rc = dev_upload(&c->d_pair_sh, c->pair_sh, c->stream)) != PK_OK ||
        (rc = dev_upload(&c->d_fnorm, c->fnorm, c->stream)) != PK_OK ||
        (rc = dev_upload(&c->d_fpos, c->fpos, c->stream)) != PK_OK || (rc = build_schwarz(c)) != PK_OK ||
        (rc = dev_upload(&c->d_Q, c->Q, c->stream)) != PK_OK ||
        hipMemcpyAsync(c->d_pairs, c->pairs.data(), c->pairs.size() * sizeof(pk::PairDev), hipMemcpyHostToDevice,
                       c->stream) != hipSuccess) {
        if (rc == PK_OK) rc = fail(PK_ERR_HIP, "pk_ctx_create: pair upload failed");
        const std::string msg = g_err;
        pk_ctx_destroy(c);
        return fail(rc, msg);
    }
    if (hipStreamSynchronize(c->stream) != hipSuccess) {
        pk_ctx_destroy(c);
        return fail(PK_ERR_HIP, "pk_ctx_create: device error during setup");
    }
    *out = c;
    return PK_OK;
}

}  // namespace

extern "C" {

int pk_ctx_create(const pk_basis_desc *d, pk_ctx **out) { return ctx_build(d, 1, out); }

int pk_batch_create(const pk_basis_desc *descs, int nmol, pk_ctx **out) { return ctx_build(descs, nmol, out); }

int pk_ctx_nmol(const pk_ctx *c) { return c ? c->nmol : -1; }

int pk_ctx_mol_layout(const pk_ctx *c, int32_t *nb, int64_t *offset) {
    if (!c) return fail(PK_ERR_ARG, "pk_ctx_mol_layout: null context");
    for (int m = 0; m < c->nmol; ++m) {
        if (nb) nb[m] = c->mol_nb[m];
        if (offset) offset[m] = c->mol_off[m];
    }
    return PK_OK;
}

// Launch-shape autotuner: every class list is timed (HIP events, `reps` builds
// per candidate after one untimed build) under each candidate shape --
// workgroups of 1, 2 or 4 waves, with and without XCD-contiguous wave ranges
// -- and keeps the fastest; a short build then takes its lists so tuned or the one
// launch, whichever is faster.  The choices persist for the context and are
// re-applied when the work lists are rebuilt.
int pk_ctx_autotune(pk_ctx *c, int reps) {
    if (!c) return fail(PK_ERR_ARG, "pk_ctx_autotune: null context");
    if (reps < 1) reps = 1;
    int rc;
    if (!c->work_ok && (rc = build_work(c)) != PK_OK) return rc;
    if ((rc = ensure_buffers(c)) != PK_OK) return rc;
    hipStream_t s = c->stream;
    hipLaunchKernelGGL(k_fill, dim3((unsigned)((c->n2 + 255) / 256)), dim3(256), 0, s, c->d_P, c->n2, 0.01);
    const bool prof = c->profile;
    c->profile = true;
    // launch shapes (lanes per workgroup, XCD remap) of the class kernels, and
    // the alternative kernel of the list (see ClassWork::alt) in its own shape
    constexpr int kCand = 7;
    const int cand[kCand][3] = {{64, 0, 0}, {128, 0, 0}, {256, 0, 0}, {64, 1, 0}, {128, 1, 0}, {256, 1, 0}, {256, 0, 1}};
    const size_t nw = c->work.size();
    std::vector<double> best(nw, 1e300);
    std::vector<int> pick(nw, 2);
    auto run = [&](int k, int nrep, bool keep) -> int {
        for (ClassWork &w : c->work) {
            w.block = cand[k][0];
            w.remap = cand[k][1];
            w.alt = cand[k][2] && has_alt(c, w);
        }
        std::vector<double> t(nw, 0.0);
        for (int r = 0; r < nrep; ++r) {
            int rc2;
            if ((rc2 = launch_build(c, c->d_P, c->d_J, c->d_K, nullptr, ctx_bufs(c), true)) != PK_OK) return rc2;
            PK_HIP(hipStreamSynchronize(s));
            for (size_t i = 0; i < nw; ++i) {
                float ms = 0.f;
                PK_HIP(hipEventElapsedTime(&ms, c->work[i].e0, c->work[i].e1));
                t[i] += ms;
            }
        }
        if (keep)
            for (size_t i = 0; i < nw; ++i)
                if (t[i] < best[i] && c->work[i].alt == cand[k][2]) {
                    best[i] = t[i];
                    pick[i] = k;
                }
        return PK_OK;
    };
    rc = run(2, 1, false);
    for (int k = 0; k < kCand && rc == PK_OK; ++k) rc = run(k, reps, true);
    c->profile = prof;
    if (rc != PK_OK) return rc;
    c->tuned.clear();
    for (size_t i = 0; i < nw; ++i) {
        ClassWork &w = c->work[i];
        w.block = cand[pick[i]][0];
        w.remap = cand[pick[i]][1];
        w.alt = cand[pick[i]][2];
        w.ms_total = 0.0;
        w.builds = 0;
        c->tuned.push_back(TuneEntry{w.cls, w.prec, w.rows, w.block, w.remap, w.alt});
    }
    drop_graph(c);
    // a short build: its lists as tuned against the one launch for all of them
    if (c->d_small && c->engine != PK_ENGINE_RYS) {
        float ms[2] = {0.f, 0.f};
        auto time_build = [&](float &t) -> int {
            PK_HIP(hipEventRecord(c->ev0, s));
            int rc2;
            if ((rc2 = launch_build(c, c->d_P, c->d_J, c->d_K, nullptr, ctx_bufs(c), false)) != PK_OK) return rc2;
            PK_HIP(hipEventRecord(c->ev1, s));
            PK_HIP(hipEventSynchronize(c->ev1));
            PK_HIP(hipEventElapsedTime(&t, c->ev0, c->ev1));
            return PK_OK;
        };
        for (int r = 0; r <= reps && rc == PK_OK; ++r)  // the first of each untimed
            for (int lists = 0; lists < 2 && rc == PK_OK; ++lists) {
                c->lists_win = lists != 0;
                float t = 0.f;
                rc = time_build(t);
                if (r > 0) ms[lists] += t;
            }
        c->lists_win = rc == PK_OK && ms[1] < ms[0];
        if (rc != PK_OK) return rc;
    }
    return PK_OK;
}

int pk_ctx_set_graph(pk_ctx *c, int enable) {
    if (!c) return fail(PK_ERR_ARG, "pk_ctx_set_graph: null context");
    c->graph_on = enable != 0;
    if (!c->graph_on) drop_graph(c);
    return PK_OK;
}

int pk_ctx_destroy(pk_ctx *c) {
    if (!c) return PK_OK;
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    free_work(c);
    free_grad(c);
    for (void *p : {(void *)c->d_pairs, (void *)c->d_prims, (void *)c->d_Q, (void *)c->d_fnorm, (void *)c->d_P,
                    (void *)c->d_Pn, (void *)c->d_A, (void *)c->d_B, (void *)c->d_J, (void *)c->d_K, (void *)c->d_G, (void *)c->d_J2,
                    (void *)c->d_palpha, (void *)c->d_hz, (void *)c->d_B2, (void *)c->d_P32, (void *)c->d_Pk1n, (void *)c->d_Pk2n, (void *)c->d_gsh, (void *)c->d_pair_sh,
                    (void *)c->d_mol_off, (void *)c->d_mol_nb, (void *)c->d_mol_foff, (void *)c->d_tblk, (void *)c->d_fpos})
        if (p) (void)hipFree(p);
    if (c->ev0) (void)hipEventDestroy(c->ev0);
    if (c->ev1) (void)hipEventDestroy(c->ev1);
    if (c->fork_ev) (void)hipEventDestroy(c->fork_ev);
    for (int i = 0; i < kSideQueues; ++i) {
        if (c->join_ev[i]) (void)hipEventDestroy(c->join_ev[i]);
        if (c->side[i]) (void)hipStreamDestroy(c->side[i]);
    }
    if (c->own_stream && c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
    return PK_OK;
}

int pk_ctx_set(pk_ctx *c, int engine, double tol, int precision, double cutoff) {
    if (!c) return fail(PK_ERR_ARG, "pk_ctx_set: null context");
    if (engine < PK_ENGINE_OS || engine > PK_ENGINE_AUTO) return fail(PK_ERR_ARG, "pk_ctx_set: unknown engine");
    if (!(tol >= 0.0)) return fail(PK_ERR_ARG, "pk_ctx_set: tol_eri must be >= 0");
    if (precision != PK_PREC_FP64 && precision != PK_PREC_MIXED)
        return fail(PK_ERR_ARG, "pk_ctx_set: unknown precision");
    if (precision == PK_PREC_MIXED && !(cutoff >= 0.0))
        return fail(PK_ERR_ARG, "pk_ctx_set: the FP32 cutoff must be >= 0");
    if (precision == PK_PREC_FP64) cutoff = 0.0;
    // the kernel of each class (OS or Rys) is chosen at launch time, so a
    // captured graph holds the previous engine's kernels
    if (engine != c->engine) drop_graph(c);
    c->engine = engine;
    if (tol != c->tol || precision != c->precision || cutoff != c->cutoff) {
        c->tol = tol;
        c->precision = precision;
        c->cutoff = cutoff;
        c->work_ok = false;
    }
    return PK_OK;
}

int pk_ctx_set_stream(pk_ctx *c, void *stream) {
    if (!c) return fail(PK_ERR_ARG, "pk_ctx_set_stream: null context");
    (void)hipStreamSynchronize(c->stream);
    if (c->own_stream && c->stream) (void)hipStreamDestroy(c->stream);
    if (stream) {
        c->stream = (hipStream_t)stream;
        c->own_stream = false;
    } else {
        PK_HIP(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
        c->own_stream = true;
    }
    return PK_OK;
}

int pk_ctx_nbasis(const pk_ctx *c) { return c ? c->nb : -1; }

int pk_ctx_profile(pk_ctx *c, int enable) {
    if (!c) return fail(PK_ERR_ARG, "pk_ctx_profile: null context");
    c->profile = enable != 0;
    if (c->profile)
        for (ClassWork &w : c->work) {
            w.ms_total = 0.0;
            w.builds = 0;
        }
    return PK_OK;
}

int pk_ctx_class_count(const pk_ctx *c) { return c ? (int)c->work.size() : -1; }

int pk_ctx_class_stats(const pk_ctx *c, int i, pk_class_stats *o) {
    if (!c || !o || i < 0 || i >= (int)c->work.size()) return fail(PK_ERR_ARG, "pk_ctx_class_stats: bad index");
    const ClassWork &w = c->work[i];
    const ClassFns &f = kClasses[w.cls];
    o->la = f.la;
    o->lb = f.lb;
    o->lc = f.lc;
    o->ld = f.ld;
    o->kernels = w.kernels;
    o->quartets = w.nquart;
    o->primitive_quartets = w.nprimq;
    o->model_flops = w.flops;
    o->ms_total = w.ms_total;
    o->builds = w.builds;
    o->precision = w.prec;
    o->block = w.block > 0 ? w.block : w.block_run;
    o->remap = w.remap;
    o->alt = w.alt;
    o->kind = list_kind(c, w);
    o->waves = w.nwaves;
    return PK_OK;
}

int pk_ctx_stats(const pk_ctx *c, pk_stats *out) {
    if (!c || !out) return fail(PK_ERR_ARG, "pk_ctx_stats: null argument");
    *out = c->st;
    return PK_OK;
}

static int fock_common(pk_ctx *c, const double *P, double *J, double *K, double *G, int memkind) {
    if (!c || !P) return fail(PK_ERR_ARG, "pk_fock: null context or density");
    if (memkind != PK_MEM_HOST && memkind != PK_MEM_DEVICE) return fail(PK_ERR_ARG, "pk_fock: bad memkind");
    int rc;
    if ((rc = ensure_buffers(c)) != PK_OK) return rc;
    const size_t n2 = c->n2 * sizeof(double);
    if (memkind == PK_MEM_DEVICE) {
        if ((rc = build_device(c, P, J, K, G)) != PK_OK) return rc;
        return finish_timing(c);
    }
    PK_HIP(hipMemcpyAsync(c->d_P, P, n2, hipMemcpyHostToDevice, c->stream));
    double *dJ = J ? c->d_J : nullptr, *dK = K ? c->d_K : nullptr, *dG = G ? c->d_G : nullptr;
    if ((rc = build_device(c, c->d_P, dJ, dK, dG)) != PK_OK) return rc;
    if (J) PK_HIP(hipMemcpyAsync(J, c->d_J, n2, hipMemcpyDeviceToHost, c->stream));
    if (K) PK_HIP(hipMemcpyAsync(K, c->d_K, n2, hipMemcpyDeviceToHost, c->stream));
    if (G) PK_HIP(hipMemcpyAsync(G, c->d_G, n2, hipMemcpyDeviceToHost, c->stream));
    PK_HIP(hipStreamSynchronize(c->stream));
    return finish_timing(c);
}

int pk_fock_jk(pk_ctx *c, const double *P, double *J, double *K, int memkind) {
    return fock_common(c, P, J, K, nullptr, memkind);
}

int pk_fock_2e(pk_ctx *c, const double *P, double *G, int memkind) {
    if (!G) return fail(PK_ERR_ARG, "pk_fock_2e: null G");
    return fock_common(c, P, nullptr, nullptr, G, memkind);
}

int pk_fock_jk_uhf(pk_ctx *c, const double *Pa, const double *Pb, double *Jt, double *Ka, double *Kb, int memkind) {
    if (!c || !Pa || !Pb) return fail(PK_ERR_ARG, "pk_fock_jk_uhf: null argument");
    if (memkind != PK_MEM_HOST && memkind != PK_MEM_DEVICE) return fail(PK_ERR_ARG, "pk_fock_jk_uhf: bad memkind");
    int rc;
    if (!c->work_ok && (rc = build_work(c)) != PK_OK) return rc;
    if ((rc = ensure_buffers(c)) != PK_OK) return rc;
    const size_t n2 = c->n2 * sizeof(double);
    if (!c->d_J2) PK_HIP(hipMalloc((void **)&c->d_J2, n2));
    if (!c->d_Pk1n) PK_HIP(hipMalloc((void **)&c->d_Pk1n, n2));
    if (!c->d_Pk2n) PK_HIP(hipMalloc((void **)&c->d_Pk2n, n2));
    if (!c->d_B2) PK_HIP(hipMalloc((void **)&c->d_B2, n2));
    hipStream_t s = c->stream;
    // one pass over the integrals: J of Pa + Pb, the exchange of each spin
    // density from the same integrals (two exchange accumulators)
    BuildBufs sb = ctx_bufs(c);
    sb.PKa = c->d_Pk1n;
    sb.PKb = c->d_Pk2n;
    sb.B2 = c->d_B2;
    PK_HIP(hipEventRecord(c->ev0, s));
    if (memkind == PK_MEM_DEVICE) {
        if ((rc = launch_build_uhf(c, Pa, Pb, Jt, Ka, Kb, sb, c->profile)) != PK_OK) return rc;
        PK_HIP(hipEventRecord(c->ev1, s));
        PK_HIP(hipStreamSynchronize(s));
        return finish_timing(c);
    }
    // host memory: staged through the context's buffers
    PK_HIP(hipMemcpyAsync(c->d_P, Pa, n2, hipMemcpyHostToDevice, s));
    PK_HIP(hipMemcpyAsync(c->d_J2, Pb, n2, hipMemcpyHostToDevice, s));
    if ((rc = launch_build_uhf(c, c->d_P, c->d_J2, c->d_J, c->d_K, c->d_G, sb, c->profile)) != PK_OK) return rc;
    PK_HIP(hipEventRecord(c->ev1, s));
    if (Jt) PK_HIP(hipMemcpyAsync(Jt, c->d_J, n2, hipMemcpyDeviceToHost, s));
    if (Ka) PK_HIP(hipMemcpyAsync(Ka, c->d_K, n2, hipMemcpyDeviceToHost, s));
    if (Kb) PK_HIP(hipMemcpyAsync(Kb, c->d_G, n2, hipMemcpyDeviceToHost, s));
    PK_HIP(hipStreamSynchronize(s));
    return finish_timing(c);
}

// Two-electron gradient: the densities are scaled into the internal order,
// then every ordered class (same screening as the energy build) runs through its
// derivative kernel; the per-shell sums leave through the context's buffer.
int pk_eri_gradient(pk_ctx *c, const double *Pj, const double *Pk1, const double *Pk2, double kx, double *grad,
                    int memkind) {
    if (!c || !Pj || !Pk1 || !grad) return fail(PK_ERR_ARG, "pk_eri_gradient: null argument");
    if (memkind != PK_MEM_HOST && memkind != PK_MEM_DEVICE) return fail(PK_ERR_ARG, "pk_eri_gradient: bad memkind");
    if (c->nmol != 1) return fail(PK_ERR_ARG, "pk_eri_gradient: one molecule only");
    int rc;
    if (!c->work_ok && (rc = build_work(c)) != PK_OK) return rc;
    if ((rc = ensure_buffers(c)) != PK_OK) return rc;
    const size_t n2 = c->n2 * sizeof(double);
    if (!c->d_Pk1n) PK_HIP(hipMalloc((void **)&c->d_Pk1n, n2));
    if (!c->d_Pk2n) PK_HIP(hipMalloc((void **)&c->d_Pk2n, n2));
    if (!c->d_gsh) PK_HIP(hipMalloc((void **)&c->d_gsh, 3 * (size_t)c->ns * sizeof(double)));
    if ((rc = build_grad(c)) != PK_OK) return rc;
    hipStream_t s = c->stream;
    const double *src[3] = {Pj, Pk1, Pk2};
    if (memkind == PK_MEM_HOST) {
        // staging through the context's P, J and K buffers
        double *stage[3] = {c->d_P, c->d_J, c->d_K};
        for (int i = 0; i < 3; ++i)
            if (src[i]) {
                PK_HIP(hipMemcpyAsync(stage[i], src[i], n2, hipMemcpyHostToDevice, s));
                src[i] = stage[i];
            }
    }
    const MolTab t{c->d_mol_off, c->d_mol_nb, c->d_mol_foff, c->d_fpos};
    const dim3 g2((unsigned)(((size_t)c->nbmax * c->nbmax + 255) / 256), 1);
    double *dst[3] = {c->d_Pn, c->d_Pk1n, c->d_Pk2n};
    for (int i = 0; i < 3; ++i)
        if (src[i]) hipLaunchKernelGGL(k_scale_density, g2, dim3(256), 0, s, src[i], c->d_fnorm, dst[i], t);
    hipLaunchKernelGGL(k_fill, dim3((unsigned)((3 * c->ns + 255) / 256)), dim3(256), 0, s, c->d_gsh,
                       (size_t)3 * c->ns, 0.0);
    // the class lists are independent: longest first to the least loaded of the
    // context stream and the side queues
    hipStream_t q[kSideQueues + 1] = {s};
    int nq = 1;
    if (!c->side_off && c->gwork.size() > 1) {
        if ((rc = ensure_side(c)) != PK_OK || (rc = fork_side(c, q)) != PK_OK) return rc;
        nq = kSideQueues + 1;
    }
    double load[kSideQueues + 1] = {};
    const int nk = Pk2 ? 2 : 1;
    auto launch = [&](const GradWork &w, hipStream_t on) -> int {
        const pk::GradEntry &e = grad_table()[w.cls];
        pk::GradArgs a{};
        a.item_bra = w.d_items;
        a.item_start = w.d_items + w.nitems;
        a.item_count = w.d_items + 2 * (size_t)w.nitems;
        a.item_prim = w.d_items + 3 * (size_t)w.nitems;
        a.order = c->d_gorder;
        a.pairs = c->d_pairs;
        a.prims = c->d_prims;
        a.palpha = c->d_palpha;
        a.hz = c->d_hz;
        a.pair_sh = c->d_pair_sh;
        a.Pj = c->d_Pn;
        a.Pk1 = c->d_Pk1n;
        a.Pk2 = c->d_Pk2n;
        a.Q = c->d_Q;
        a.g = c->d_gsh;
        a.tol = c->tol;
        a.kx = kx;
        a.nb = c->nb;
        a.nitems = w.nitems;
        const void *k = nk == 2 ? e.k2 : e.k1;
        static std::atomic<int> attr_done[2 * kPairClasses * kPairClasses];  // zero-initialised
        std::atomic<int> &done = attr_done[2 * w.cls + nk - 1];
        if (!done.load()) {
            PK_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsMax));
            done.store(1);
        }
        void *args[] = {&a};
        PK_HIP(hipLaunchKernel(k, dim3(w.nitems, e.rc), dim3(64), args, e.lds[nk - 1], on));
        return PK_OK;
    };
    for (const GradWork &w : c->gwork) {
        int j = 0;
        for (int i = 1; i < nq; ++i)
            if (load[i] < load[j]) j = i;
        load[j] += w.cost;
        if ((rc = launch(w, q[j])) != PK_OK) break;
    }
    if (nq > 1) rc = join_side(c, rc);
    if (rc != PK_OK) return rc;
    PK_HIP(hipGetLastError());
    const size_t gb = 3 * (size_t)c->ns * sizeof(double);
    PK_HIP(hipMemcpyAsync(grad, c->d_gsh, gb, memkind == PK_MEM_HOST ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice, s));
    PK_HIP(hipStreamSynchronize(s));
    return PK_OK;
}

int pk_schwarz(pk_ctx *c, double *Q, int memkind) {
    if (!c || !Q) return fail(PK_ERR_ARG, "pk_schwarz: null argument");
    if (memkind == PK_MEM_DEVICE) {
        const MolTab t{c->d_mol_off, c->d_mol_nb, c->d_mol_foff, c->d_fpos};
        const dim3 g2((unsigned)(((size_t)c->nbmax * c->nbmax + 255) / 256), (unsigned)c->nmol);
        hipLaunchKernelGGL(k_unpermute, g2, dim3(256), 0, c->stream, c->d_Q, Q, t);
        PK_HIP(hipGetLastError());
        PK_HIP(hipStreamSynchronize(c->stream));
    } else {
        for (int m = 0; m < c->nmol; ++m) {
            const int nb = c->mol_nb[m];
            const int *ps = c->fpos.data() + c->mol_foff[m];
            const double *in = c->Q.data() + c->mol_off[m];
            double *out = Q + c->mol_off[m];
            for (int r = 0; r < nb; ++r)
                for (int q = 0; q < nb; ++q) out[(size_t)r * nb + q] = in[(size_t)ps[r] * nb + ps[q]];
        }
    }
    return PK_OK;
}

int pk_eri_tensor(pk_ctx *c, double *out) {
    if (!c || !out) return fail(PK_ERR_ARG, "pk_eri_tensor: null argument");
    if (c->nmol != 1) return fail(PK_ERR_ARG, "pk_eri_tensor: one molecule only");
    const size_t nb = c->nb, nb2 = nb * nb, nb3 = nb2 * nb;
    if ((double)nb3 * nb * 8.0 > 2147483648.0) return fail(PK_ERR_ARG, "pk_eri_tensor: nb^4 tensor exceeds 2 GiB");
    std::fill(out, out + nb3 * nb, 0.0);
    const int np = (int)c->pairs.size();
    std::vector<std::vector<int>> qb(kQuartClasses), qk(kQuartClasses);
    for (int p = 0; p < np; ++p)
        for (int q = 0; q <= p; ++q) {
            int b = p, k = q;
            if (c->pair_cls[b] < c->pair_cls[k]) std::swap(b, k);
            const int cls = quart_class(c->pair_cls[b], c->pair_cls[k]);
            qb[cls].push_back(b);
            qk[cls].push_back(k);
        }
    for (int cls = 0; cls < kQuartClasses; ++cls) {
        if (qb[cls].empty()) continue;
        const ClassFns &f = kClasses[cls];
        std::vector<double> v;
        int rc = run_eri_class(c, pk::pair_class(f.la, f.lb), pk::pair_class(f.lc, f.ld), qb[cls], qk[cls], v);
        if (rc != PK_OK) return rc;
        const int na = pk::ncart(f.la), nbs = pk::ncart(f.lb), nc = pk::ncart(f.lc), nd = pk::ncart(f.ld);
        for (size_t q = 0; q < qb[cls].size(); ++q) {
            const pk::PairDev &B = c->pairs[qb[cls][q]], &K = c->pairs[qk[cls][q]];
            for (int ia = 0; ia < na; ++ia)
                for (int ib = 0; ib < nbs; ++ib)
                    for (int ic = 0; ic < nc; ++ic)
                        for (int id = 0; id < nd; ++id) {
                            // internal positions (screening, norms), then the caller's order
                            size_t i = B.f0 + ia, j = B.f1 + ib, k = K.f0 + ic, l = K.f1 + id;
                            if (c->Q[i * nb + j] * c->Q[k * nb + l] < c->tol) continue;
                            const double val = c->fnorm[i] * c->fnorm[j] * c->fnorm[k] * c->fnorm[l] *
                                               v[q * (size_t)na * nbs * nc * nd + ((ia * nbs + ib) * nc + ic) * nd + id];
                            i = c->fnat[i];
                            j = c->fnat[j];
                            k = c->fnat[k];
                            l = c->fnat[l];
                            const size_t idx[8] = {i * nb3 + j * nb2 + k * nb + l, j * nb3 + i * nb2 + k * nb + l,
                                                   i * nb3 + j * nb2 + l * nb + k, j * nb3 + i * nb2 + l * nb + k,
                                                   k * nb3 + l * nb2 + i * nb + j, l * nb3 + k * nb2 + i * nb + j,
                                                   k * nb3 + l * nb2 + j * nb + i, l * nb3 + k * nb2 + j * nb + i};
                            for (size_t x : idx) out[x] = val;
                        }
        }
    }
    return PK_OK;
}

}  // extern "C"
