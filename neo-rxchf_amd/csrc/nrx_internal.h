// nrx_internal.h -- declarations shared by the translation units of
// libneorx_hip.so (nrx_lib.hip: integral kernels, builders and the
// reference-semantics contractions; nrx_scf.hip: the device-resident XCHF
// Fock build and SCF).  Nothing here is part of the C ABI: the functions are
// hidden from the shared library's symbol table.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/neorx.h"
#include "nrx_engine.h"

typedef int64_t i64;
#define NRX_DI __device__ inline __attribute__((always_inline))
#define NRX_HIDDEN __attribute__((visibility("hidden")))
using namespace nrx;

// error status of the calling thread (neorx_last_error); returns code
NRX_HIDDEN int fail(int code, const char *fmt, ...);

#define HIPCHK(x)                                                                                                  \
    do {                                                                                                           \
        hipError_t _e = (x);                                                                                       \
        if (_e != hipSuccess) return fail(NEORX_E_HIP, "%s failed: %s", #x, hipGetErrorString(_e));              \
    } while (0)

// NEORX_VERBOSE > 0: long builds report their progress on stderr
NRX_HIDDEN extern int g_verbose;

// neorx_init(0) unless a device is already selected
NRX_HIDDEN int ensure_init();

// ------------------------------------------------------------------
// system handle
// ------------------------------------------------------------------
struct DevSys {
    i64 nebf, npebf, npbf, nat, ngtg;
    i64 nebf1, npebf1;        // first electron basis; the rest is the special-electron basis (RXCHFmult)
    double pmass;
    const double *cat, *zan, *bcoef, *gamma, *agebfcc, *agnbfcc;
    const i64 *kpestr, *kpeend, *ampeb2c;
    const i64 *eord, *pord;   // enumeration order -> original primitive index
    const PairRec *ep, *pp;   // bra*ket tables [i][j] over primitives (npebf^2, npbf^2)
    const double *bt;         // Boys table (BT_N x BT_M)
    int lmax;                 // largest primitive angular momentum (3: f functions present)
};

// Distinct pairs of a one-basis system (device arrays).  A contracted pair is
// {I <= J}, number J(J+1)/2 + I; its primitive pairs (i of I, j of J; i <= j
// when I = J, the off-diagonal ones counted twice in their coefficient) are
// consecutive in the pair list.  Slots: the pair list sorted by angular
// momentum and padded to groups of 64, one per lane of a wave.
struct PairPlan {
    i64 ncp, npl, nslot, nq;  // contracted pairs, primitive pairs, slots, distinct nuclear pairs
    int le, lp;               // largest angular momentum, electronic and nuclear
    const int *cp_start;      // ncp + 1: pair-list range of a contracted pair
    const int *pl_idx, *pl_deg; // entry of ep; bra + ket powers per direction, a byte each
    const int *slot;          // pair-list entry per slot, -1 for padding
    const int *gdeg, *gL;     // per 64 slots: largest degree per direction, largest total degree
    const int *pp_idx, *pp_deg; // nuclear pair q = j(j+1)/2 + i: entry of pp, powers
    const double *pl_coef, *pp_coef;
    // geminal terms: every ordered (k,l) with b_k b_l; then the one-geminal
    // terms gamma_k with b_k and the k <= l terms gamma_k + gamma_l with
    // b_k b_l / 2 (k < l: twice that); {1, 0}
    const double *gk, *gl, *wkl, *gx, *wx, *one;
};

struct System {
    DevSys d;
    std::vector<void *> allocs;
    std::vector<i64> eord, pord;
    // host copies: contraction ranges (1-based), powers, coefficients, geminal
    std::vector<i64> kpestr, kpeend, elcam, nucam;
    std::vector<double> agebfcc, agnbfcc, bcoef, gamma;
    int maxl;
    // the pair plan, formed by the first builder that works from pairs
    // (nrx_plan): a handle that serves primitive tuples or two-basis routines
    // never pays for it (neorx_system_create at 60 primitives 354 us, 237 so)
    PairPlan plan{};
    std::vector<i64> cp_start; // host copy
    std::mutex plan_mu;
    bool planned = false;
    i64 nuc_pairs() const { return d.npbf * (d.npbf + 1) / 2; }
};

NRX_HIDDEN System *get_sys(i64 h);
// forms s->plan if it is not there yet (l <= 2); any thread
NRX_HIDDEN int nrx_plan(System *s);

// ------------------------------------------------------------------
// primitive tuples (nrx_prims.hip)
// ------------------------------------------------------------------
// values of tuples start .. start + ntup - 1 of class cls 1..10 from source src
// (nrx_tuples.h), up to four outputs (os, ox, oy may be null)
NRX_HIDDEN int nrx_prims(int cls, int src, const DevSys &d, i64 start, i64 ntup, const i64 *idx, double *oe, double *os,
                         hipStream_t st, double *ox = nullptr, double *oy = nullptr);

// ------------------------------------------------------------------
// the l <= 3 build of the engine (nrx_wide.hip)
// ------------------------------------------------------------------
// Tuples beyond the l <= 2 capacities (an f function on some particle) are
// binned by the tier kernels into the wide bin wbin of a launch's sorted
// list; this evaluates that bin (class cls, tuple source src) on stream st.
// n bounds the bin's size (the launch's tuple count).
NRX_HIDDEN int nrx_wide_prims(int cls, int src, const DevSys &d, i64 start, const i64 *idx, double *oe, double *os,
                              double *ox, double *oy, const unsigned *list, const unsigned *counts, int wbin, i64 n,
                              hipStream_t st);
// GAM1_OMP_MD (cls 1) / RXCHFmult_GAM1_MD (cls 8) and calc_GAM_ee at l <= 3
// capacities
NRX_HIDDEN int nrx_wide_gam1(int cls, const DevSys &d, double *G, double *Gs, hipStream_t st);
NRX_HIDDEN int nrx_wide_gam_ee(const DevSys &d, double *G, hipStream_t st);

// most blocks of a grid-stride launch (NEORX_GRID_CAP lowers it)
NRX_HIDDEN extern i64 g_grid_cap;

static inline unsigned nblocks(i64 n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// Blocks for a grid-stride kernel over n items: at most g_grid_cap blocks, so
// that the grid's work-item count stays far below 2^32 whatever n is (the
// in-core GAM_3 of a 24-function basis with 8 nuclear functions has 1.2e10
// entries).
static inline unsigned grid_blocks(i64 n, int bs) { return (unsigned)std::min<i64>((n + bs - 1) / bs, g_grid_cap); }

// hipMalloc that gives up the scratch kept between calls (Work) before it
// fails; no error is left behind
NRX_HIDDEN hipError_t nrx_malloc(void **p, size_t bytes);
NRX_HIDDEN void nrx_release_work();

// device buffer released when it goes out of scope
struct DevBuf {
    void *p = nullptr;
    bool own = true; // false: a resident tensor's memory, borrowed (not freed)
    ~DevBuf()
    {
        if (p && own) (void)hipFree(p);
    }
    int alloc(size_t bytes)
    {
        hipError_t e = nrx_malloc(&p, bytes ? bytes : 8);
        if (e != hipSuccess) {
            p = nullptr;
            return fail(NEORX_E_NOMEM, "hipMalloc(%zu) failed: %s", bytes, hipGetErrorString(e));
        }
        return NEORX_OK;
    }
    double *d() { return (double *)p; }
};

// stream-ordered scratch, freed on its stream when it goes out of scope
struct StreamBuf {
    void *p = nullptr;
    hipStream_t st = 0;
    ~StreamBuf()
    {
        if (p) (void)hipFreeAsync(p, st);
    }
    int alloc(size_t bytes, hipStream_t s)
    {
        st = s;
        hipError_t e = hipMallocAsync(&p, bytes, s);
        if (e != hipSuccess) { // as nrx_malloc
            (void)hipGetLastError();
            nrx_release_work();
            e = hipMallocAsync(&p, bytes, s);
        }
        if (e != hipSuccess) {
            (void)hipGetLastError();
            p = nullptr;
            return fail(NEORX_E_NOMEM, "hipMallocAsync(%zu) failed: %s", bytes, hipGetErrorString(e));
        }
        return NEORX_OK;
    }
};

// Scratch of one call that ends by synchronising its stream.  The blocks go
// back to a process-wide free list (at most WORK_KEEP bytes in all, the oldest
// released first; larger blocks are freed) once the stream has drained,
// so no two calls in flight share one, whatever their threads and streams.
// neorx_release_resident, neorx_finalize and an allocation of this library
// that would fail otherwise empty the list.  A device
// allocation costs 0.1 ms or more, as much as a small builder's kernels.
struct Work {
    hipStream_t st;
    struct Block {
        int dev;
        void *p;
        size_t n;
    };
    std::vector<Block> held;
    explicit Work(hipStream_t s) : st(s) {}
    Work(const Work &) = delete;
    Work &operator=(const Work &) = delete;
    NRX_HIDDEN ~Work();
    NRX_HIDDEN int get(void **p, size_t bytes);
    int get(double *&p, i64 n) { return get((void **)&p, (size_t)n * 8); }
};

// storage type of an in-core tensor read by the contractions
enum { NRX_F64 = 0, NRX_F32 = 1, NRX_BF16 = 2 };

// ------------------------------------------------------------------
// launchers defined in nrx_lib.hip, used by nrx_scf.hip.  They enqueue on st
// and neither allocate nor synchronise.
// ------------------------------------------------------------------
// GAM_ee (calc_GAM_ee) into d_gee (nebf^4)
NRX_HIDDEN int nrx_gam_ee_launch(System *s, double *d_gee, hipStream_t st);
// GAM_1, GAM_1s (GAM1_OMP_MD) into d_g1, d_g1s (nebf^2 npbf^2 each)
NRX_HIDDEN int nrx_gam1_launch(System *s, double *d_g1, double *d_g1s, hipStream_t st);
// EG3IC1 slab partials of nblk slabs (ip,jp,i1): part[blk][0..ne-1] = the FE
// row before the DP(ip,jp) weight, part[blk][ne] = its DE-weighted sum / 3;
// g in FP64 or FP32
NRX_HIDDEN int nrx_eg3_slabs(i64 ne, i64 nblk, const double *d_de, const void *g, int dtype, double *part,
                             double *split, hipStream_t st);
// doubles of the split scratch of such a launch (0: not used)
NRX_HIDDEN i64 nrx_eg3_split_doubles(i64 ne, i64 nblk);
// the rows of the symmetric bilinear form T(X, Y) of two densities (X on the
// (i2,j2) pair, Y on the (i3,j3) pair; T(DE, DE) are EG3IC1's rows), and
// part[blk][ne] = sum_x Z(i1,x) F[x] / 3, or 0 when d_z is null, over tensors
// packed in the (i3,j3) pair (nrx_gam3_pairs with pack), slabs (q,i1); u:
// loads in flight per lane, 0 for the tuned or default one
NRX_HIDDEN int nrx_eg3_packed(i64 ne, i64 nblk, const double *d_x, const double *d_y, const double *d_z, const void *g,
                              int dtype, int u, double *part, double *split, hipStream_t st);
// launch(u) at u = 8, 12, 16 and 24 loads in flight: ms a launch (the mean of
// reps, after a first one) and the fastest u
NRX_HIDDEN int nrx_time_depths(const std::function<int(int u)> &launch, i64 reps, hipStream_t st, int *best,
                               double *ms);
// doubles of scratch nrx_eg3_packed takes in `split`
NRX_HIDDEN i64 nrx_eg3_packed_split_doubles(i64 ne, i64 nblk);
// EG2IC1 slab partials of nblk slabs (ip,jp,i1): part[blk][4][ne] = dir, ex,
// dirS, exS (gs may be NULL: the S rows stay zero)
NRX_HIDDEN int nrx_eg2_slabs(i64 ne, i64 nblk, const double *d_de, const double *g, const double *gs, double *part,
                             hipStream_t st);

// ------------------------------------------------------------------
// tensors from distinct pairs (nrx_stars.hip), l <= 2.  Enqueued on W's
// stream, with scratch from W.
// ------------------------------------------------------------------
// GAM3_IC1 (mult: RXCHFmult_GAM3_XCHF) of every distinct nuclear pair.  npbf
// > 0: into the full tensor G, both orders of each pair; npbf = 0: one block
// of nebf^6 per pair, from G on.  nb > 0 (with npbf = 0): at most nb pairs at
// a time, each batch [q0, q1) from the start of G, and sink called after it --
// the scratch of one batch serves them all, and what does not depend on the
// nuclear pair is formed once.  pack: the third electron's index pair over its
// distinct values only, [i1 j1][i2 j2][J(J+1)/2 + I].
using PairSink = std::function<int(i64 q0, i64 q1)>;
NRX_HIDDEN int nrx_gam3_pairs(System *s, bool mult, i64 npbf, double *G, Work &W, bool pack = false, i64 nb = 0,
                              const PairSink &sink = {});
// GAM2_IC1 (G = GM2ICR, Gs = GM2sICR) or, with rxne, RXCHFne_GAM2_IC1 (GM2ICR,
// GM2exICR), nuclear pairs, blocks and batches as above
NRX_HIDDEN int nrx_gam2_pairs(System *s, bool rxne, i64 npbf, double *G, double *Gs, Work &W, i64 nb = 0,
                              const PairSink &sink = {});
