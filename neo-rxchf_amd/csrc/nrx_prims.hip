// nrx_prims.hip -- evaluation of primitive tuples (the tier kernels).
#include "nrx_tuples.h"

namespace {

// tuple t of a launch from source src (uniform); false for a list entry out
// of range
template <int CLS> NRX_DI bool any_tuple(const DevSys &S, int src, const i64 *idx, i64 start, i64 t, i64 *x)
{
    if (src == SRC_LIST) return load_tuple<CLS>(S, idx, t, x);
    if constexpr (!two_basis<CLS>()) {
        if (src == SRC_SORTED) {
            range_tuple<CLS, true>(S, start + t, x);
            return true;
        }
    }
    range_tuple<CLS, false>(S, start + t, x);
    return true;
}

// Tuples of a launch are sorted by bin, a counting sort in two passes:
// k_prim_bin gives each tuple its bin (capacity tier tuple_tier, and for the
// classes whose Coulomb terms take the hub-cycle path also the proton pair's
// largest per-direction degree, which bounds that path's series) and counts
// the bins, one atomic per wave and bin; k_prim_scatter writes the tuple
// positions bin by bin into one list; k_prim_tiers evaluates every bin with
// its tier's capacities, one lane per listed tuple, so that every wave runs
// at the capacity its tuples need.  Both passes count in LDS per block and
// touch each global counter once per block.  Out-of-range list entries are
// flagged (NaN results) and left out.
template <int CLS> constexpr int hub_bins() { return (CLS == 2 || CLS == 4 || CLS == 5 || CLS == 9) ? 5 : 1; }
template <int CLS> constexpr int n_bins() { return Tier<CLS>::N * hub_bins<CLS>(); }

template <int CLS> NRX_DI int tuple_bin(const PairRec *const *q)
{
    int k = tuple_tier<CLS>(q);
    if (k == Tier<CLS>::N) return n_bins<CLS>(); // the wide bin (l <= 3 build)
    if constexpr (hub_bins<CLS>() == 1) {
        return k;
    } else {
        const PairRec &P = *q[nel<CLS>()];
        int m = 0;
        NRX_UNROLL for (int d = 0; d < 3; ++d) m = max(m, P.la[d] + P.lb[d]);
        return k * hub_bins<CLS>() + min(m, hub_bins<CLS>() - 1);
    }
}

template <int CLS>
__global__ void __launch_bounds__(256) k_prim_bin(DevSys S, int src, i64 start, i64 ntup, const i64 *__restrict__ idx,
                                                  double *__restrict__ outE, double *__restrict__ outS,
                                                  double *__restrict__ outX, double *__restrict__ outY,
                                                  unsigned char *__restrict__ code, unsigned *__restrict__ counts)
{
    __shared__ unsigned lc[32];
    if (threadIdx.x < 32) lc[threadIdx.x] = 0u;
    __syncthreads();
    i64 t = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    int bin = -1;
    if (t < ntup) {
        i64 x[2 * nel<CLS>() + 2];
        const bool ok = any_tuple<CLS>(S, src, idx, start, t, x);
        if (ok) {
            const PairRec *q[nel<CLS>() + 1];
            tuple_pairs<CLS>(S, x, q);
            bin = tuple_bin<CLS>(q);
        } else { // out-of-range primitive index: flag the entry
            outE[t] = __builtin_nan("");
            if (outS) outS[t] = __builtin_nan("");
            if (outX) outX[t] = __builtin_nan("");
            if (outY) outY[t] = __builtin_nan("");
        }
        code[t] = (unsigned char)(bin < 0 ? 255 : bin);
    }
    if (bin >= 0) atomicAdd(&lc[bin], 1u);
    __syncthreads();
    if (threadIdx.x < n_bins<CLS>() + 1 && lc[threadIdx.x]) atomicAdd(&counts[threadIdx.x], lc[threadIdx.x]);
}

template <int CLS>
__global__ void __launch_bounds__(256) k_prim_scatter(i64 ntup, const unsigned char *__restrict__ code,
                                                      const unsigned *__restrict__ counts,
                                                      unsigned *__restrict__ cursors, unsigned *__restrict__ list)
{
    __shared__ unsigned lc[32], lbase[32];
    if (threadIdx.x < 32) lc[threadIdx.x] = 0u;
    __syncthreads();
    i64 t = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    int bin = -1;
    if (t < ntup) {
        int c = code[t];
        bin = (c == 255) ? -1 : c;
    }
    unsigned loc = 0;
    if (bin >= 0) loc = atomicAdd(&lc[bin], 1u); // rank within the block's share of the bin
    __syncthreads();
    if (threadIdx.x < n_bins<CLS>() + 1)
        lbase[threadIdx.x] = bin_offset(counts, threadIdx.x) +
                             (lc[threadIdx.x] ? atomicAdd(&cursors[threadIdx.x], lc[threadIdx.x]) : 0u);
    __syncthreads();
    if (bin >= 0) list[lbase[bin] + loc] = (unsigned)t;
}

// Lanes per block of the tier kernel: one wavefront, so that blocks are
// scheduled per SIMD (the kernels run at one wave per SIMD), measured ~1 %
// faster than 256-lane blocks.
constexpr int TIER_BS = 64;

// One listed tuple of tier K: its pair records are staged in LDS (the
// evaluation reads them many times; at one wave per SIMD, the register use
// of these kernels, the LDS footprint costs no occupancy), then it is
// evaluated with the tier's capacities.
template <int CLS, int K>
NRX_DI void tier_item(const DevSys &S, int src, i64 start, const i64 *__restrict__ idx, double *__restrict__ outE,
                      double *__restrict__ outS, double *__restrict__ outX, double *__restrict__ outY, i64 t,
                      PairRec (*stage)[TIER_BS])
{
    constexpr int NP = nel<CLS>() + 1;
    i64 x[2 * NP];
    any_tuple<CLS>(S, src, idx, start, t, x); // a list was validated by k_prim_bin
    const PairRec *q[NP];
    tuple_pairs<CLS>(S, x, q);
    NRX_UNROLL for (int i = 0; i < NP; ++i) {
        stage[i][threadIdx.x] = *q[i];
        q[i] = &stage[i][threadIdx.x];
    }
    double e, s, xx, yy;
    tuple_eval<CLS, Tier<CLS>::NL[K], Tier<CLS>::NB[K]>(d_params(S), q, e, s, xx, yy);
    outE[t] = e;
    if (outS) outS[t] = s;
    if (outX) outX[t] = xx;
    if (outY) outY[t] = yy;
}

// block b of the fused launch: the bins are laid out from the last tier and
// the highest proton degree down (their tuples take longest, so they start
// first).  Locates the block's bin; -1 past the last bin.
template <int CLS> NRX_DI int block_bin(const unsigned *__restrict__ counts, i64 b, i64 &k0)
{
    for (int bin = n_bins<CLS>() - 1; bin >= 0; --bin) {
        i64 nb = ((i64)counts[bin] + TIER_BS - 1) / TIER_BS;
        if (b < nb) {
            k0 = b * TIER_BS;
            return bin;
        }
        b -= nb;
    }
    return -1;
}

// one inlined evaluation per tier: tier K of the bin's tuple
template <int CLS, int K>
NRX_DI void tier_eval(int tier, const DevSys &S, int src, i64 start, const i64 *__restrict__ idx, double *__restrict__ outE,
                      double *__restrict__ outS, double *__restrict__ outX, double *__restrict__ outY, i64 t,
                      PairRec (*stage)[TIER_BS])
{
    if constexpr (K >= 0) {
        if (tier == K) {
            tier_item<CLS, K>(S, src, start, idx, outE, outS, outX, outY, t, stage);
            return;
        }
        tier_eval<CLS, K - 1>(tier, S, src, start, idx, outE, outS, outX, outY, t, stage);
    }
}

// Every bin of a launch in one kernel, so that the bins' tails overlap:
// lane per listed tuple, blocks past the bins exit.
template <int CLS>
__global__ void __launch_bounds__(TIER_BS) k_prim_tiers(DevSys S, int src, i64 start, const i64 *__restrict__ idx,
                                                    double *__restrict__ outE, double *__restrict__ outS,
                                                    double *__restrict__ outX, double *__restrict__ outY,
                                                    const unsigned *__restrict__ list,
                                                    const unsigned *__restrict__ counts)
{
    __shared__ PairRec stage[nel<CLS>() + 1][TIER_BS];
    i64 k0 = 0;
    const int bin = block_bin<CLS>(counts, (i64)blockIdx.x, k0);
    if (bin < 0) return;
    const i64 k = k0 + threadIdx.x;
    if (k >= (i64)counts[bin]) return;
    const i64 t = (i64)list[bin_offset(counts, bin) + k];
    tier_eval<CLS, Tier<CLS>::N - 1>(bin / hub_bins<CLS>(), S, src, start, idx, outE, outS, outX, outY, t, stage);
}

__global__ void k_zero_u32n(unsigned *p, int n)
{
    if ((int)threadIdx.x < n) p[threadIdx.x] = 0u;
}


// tuples per launch of the primitive kernels (bounds the sorted list, whose
// entries are 32-bit positions, and the bin counters)
const i64 PRIM_CHUNK = (i64)1 << 24;

template <int CLS>
int launch_class(int src, const DevSys &d, i64 start, i64 ntup, const i64 *idx, double *oe, double *os, double *ox,
                 double *oy, hipStream_t st)
{
    constexpr int NBN = n_bins<CLS>();
    static_assert(NBN + 1 <= 32, "bin counters (with the wide bin) and cursors fit the 256-byte header");
    if constexpr (two_basis<CLS>())
        if (src != SRC_LIST && (d.npebf1 <= 0 || d.npebf1 >= d.npebf))
            return fail(NEORX_E_ARG, "class %d enumerates two electron bases; this handle has one", CLS);
    if (ntup <= 0) return NEORX_OK;
    i64 cap = std::min(ntup, PRIM_CHUNK);
    // stream-ordered scratch: bin counters, the sorted tuple list and the bin codes
    StreamBuf ws; // header: counts[32], cursors[32]; list: cap x u32; codes: cap x u8
    int rc = ws.alloc(256 + cap * sizeof(unsigned) + cap, st);
    if (rc) return rc;
    unsigned *counts = (unsigned *)ws.p, *cursors = counts + 32, *list = (unsigned *)((char *)ws.p + 256);
    unsigned char *code = (unsigned char *)(list + cap);
    for (i64 off = 0; off < ntup; off += PRIM_CHUNK) {
        i64 n = std::min(ntup - off, PRIM_CHUNK);
        const i64 *ix = src == SRC_LIST ? idx + off * (2 * nel<CLS>() + 2) : nullptr;
        double *e = oe + off, *s = os ? os + off : nullptr, *x = ox ? ox + off : nullptr;
        double *y = oy ? oy + off : nullptr;
        hipLaunchKernelGGL(k_zero_u32n, dim3(1), dim3(64), 0, st, counts, 64);
        hipLaunchKernelGGL((k_prim_bin<CLS>), dim3(nblocks(n, 256)), dim3(256), 0, st, d, src, start + off, n, ix, e, s,
                           x, y, code, counts);
        HIPCHK(hipGetLastError());
        hipLaunchKernelGGL((k_prim_scatter<CLS>), dim3(nblocks(n, 256)), dim3(256), 0, st, n, code, counts, cursors,
                           list);
        HIPCHK(hipGetLastError());
        hipLaunchKernelGGL((k_prim_tiers<CLS>), dim3(nblocks(n, TIER_BS) + NBN), dim3(TIER_BS), 0, st, d, src,
                           start + off, ix,
                           e, s, x, y, list, counts);
        HIPCHK(hipGetLastError());
        if (d.lmax > 2) { // tuples with f functions: the wide bin
            rc = nrx_wide_prims(CLS, src, d, start + off, ix, e, s, x, y, list, counts, NBN, n, st);
            if (rc) return rc;
        }
    }
    return NEORX_OK;
}

} // namespace

int nrx_prims(int cls, int src, const DevSys &d, i64 start, i64 ntup, const i64 *idx, double *oe, double *os,
              hipStream_t st, double *ox, double *oy)
{
    switch (cls) {
    case 1: return launch_class<1>(src, d, start, ntup, idx, oe, os, ox, oy, st);
    case 2: return launch_class<2>(src, d, start, ntup, idx, oe, os, ox, oy, st);
    case 3: return launch_class<3>(src, d, start, ntup, idx, oe, os, ox, oy, st);
    case 4: return launch_class<4>(src, d, start, ntup, idx, oe, os, ox, oy, st);
    case 5: return launch_class<5>(src, d, start, ntup, idx, oe, os, ox, oy, st);
    case 6: return launch_class<6>(src, d, start, ntup, idx, oe, os, ox, oy, st);
    case 7: return launch_class<7>(src, d, start, ntup, idx, oe, os, ox, oy, st);
    case 8: return launch_class<8>(src, d, start, ntup, idx, oe, os, ox, oy, st);
    case 9: return launch_class<9>(src, d, start, ntup, idx, oe, os, ox, oy, st);
    case 10: return launch_class<10>(src, d, start, ntup, idx, oe, os, ox, oy, st);
    default: return fail(NEORX_E_ARG, "unknown tuple class %d", cls);
    }
}
