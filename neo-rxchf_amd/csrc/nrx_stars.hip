// nrx_stars.hip -- the contracted tensors GAM_2, GAM_3 and the RXCHF-ne GAM_2
// from the distinct primitive pairs of their particles (l <= 2).
//
// GAM_3.  Every term of the e-e-e-p value is the product of a star -- two electrons
// and the proton joined by their geminals -- or a part of one, with a lone
// electron that only the Coulomb and one-electron operators reach.  Averaged
// over the six electron permutations (gam3_IC1_OMP.f:149-263) the tensor is
//   GM3(1,2,3) = 1/3 sum_c [ T(a,b; c) + X(c) V(a,b) ],   {a,b,c} = {1,2,3},
//   T(a,b; c)  = sum_kl b_k b_l [ Y_kl(a,b) h(c) - <1/r_pc> + <1/r_ac> + <1/r_bc> ],
// g(a,p) = gamma_k and g(b,p) = gamma_l, Y the star's overlap, h the
// one-electron value of c, V the electron repulsion and X(c) the (c,p)
// overlaps of the one-geminal terms.  All of it is unchanged when a particle's
// bra and ket are exchanged (the operators multiply, and the one-electron
// kinetic operator is Hermitian), and T when a and b are.  So one evaluation
// per distinct pair of functions of each particle, and per distinct {a,b},
// gives every entry: of n^6 p^2 primitive tuples about 1/32 are left, and a
// tuple's terms need no absorption of their own, because the densities that
// the star leaves at p, a and b serve every lone electron.
//
//   k_star     the star densities: per primitive star and geminal pair, the
//              Hermite-Gaussian coefficients of the density at p, a and b
//   k_lone     their Coulomb integrals with the lone electron's pairs: a lane
//              per lone primitive pair, a wave per contracted star
//   k_lone_sum the lone electron's contraction
//   k_gam3_expand   the sum over c and the full tensor in the reference packing
//
// GAM_2 has the same parts.  Averaged over the electrons (gam2_IC1_OMP.f:
// 141-177),
//   GM2(a,b) = L(a; b) + L(b; a) + B(a,b),
//   L(c; a)  = sum_t w_t [ O_t(a,p) h(c) - <1/r_pc> + <1/r_ac> ]
// over the terms t of X above: a star of one electron with a lone one, again
// through k_star and k_lone.  B holds what both geminals bond:
//   B(a,b) = sum_kl b_k b_l [ T + V_p - V_a - V_b - <1/r_ap> - <1/r_bp> + <1/r_ab> ]
// with g(a,p) = gamma_k and g(b,p) = gamma_l, V the nuclear attractions of the
// star's members.  The kinetic part T of the average
// (star_kin) needs no derivative of a geminal under the kinetic operator of the
// other side: for an electron the two forms of the reference, g g T and g T g, are
// each other's transpose, and for the proton
//   (g_a T g_b + g_b T g_a)/2 = (T g_a g_b + g_a g_b T)/2 + (1/2m) grad g_a . grad g_b,
// so T is the mean of the operator on the bra and on the ket -- one polynomial
// per pair and direction (k_pair_kin) -- plus (2 gamma_k gamma_l / m)
// <(r_p - r_a).(r_p - r_b)>.  k_bond evaluates the seven terms, a lane per
// star, geminal pair and term, at the capacity of the star's powers.
// RXCHF-ne: GM2 is L with the lone electron second and without h, GM2ex the
// <1/r_ab> of B.
//
// k_lone takes about 150 FMAs per density and lone pair (27 densities per star
// with three geminals), its operands in scalar registers (the star's
// coefficients are wave-uniform) and LDS.  Lanes over the lone pairs rather
// than over stars for that reason: a lane per star would read 200 bytes per
// 150 FMAs.  The vector units issue 47 % of the time; half of the wave cycles
// wait, mostly on scalar loads of the records, 37 % of which miss their cache.
// k_bond is bound by FP64 issue (68 % of the time).
// GAM3_IC1 over 8 contracted functions (16 s/p primitives), 4 nuclear ones:
// 491 ms a tuple at a time, 6.1 ms here, of it 5.7 ms in k_lone; 7 functions in
// GAM3_DSCF + GAM2_DSCF: 4.38 ms, 0.44 ms.  GAM2_IC1 over 24 functions (36 s/p
// primitives), 8 nuclear: 504 ms, 46.5 ms, of it 41 ms in k_bond and 2.8 ms in
// k_lone; RXCHFne_GAM2_IC1 over 24 s/p/d functions, 4 nuclear: 12.6 ms, 0.75 ms.
#include "nrx_tuples.h"

#include <chrono>

namespace {

constexpr double TWO_PI_2P5 = 34.986836655249725; // 2 pi^(5/2)

// lower-triangle index of a pair of positions
NRX_DI i64 tri_index(i64 a, i64 b) { return a > b ? a * (a + 1) / 2 + b : b * (b + 1) / 2 + a; }

// row b and column a <= b of triangle entry t
NRX_DI void tri_decode(i64 t, i64 &b, i64 &a)
{
    i64 r = (i64)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while (r * (r + 1) / 2 > t) --r;
    while ((r + 1) * (r + 2) / 2 <= t) ++r;
    b = r;
    a = t - r * (r + 1) / 2;
}

// per-direction degrees packed in bytes (x lowest)
NRX_DI int deg_of(int packed, int d) { return (packed >> (8 * d)) & 255; }

// ------------------------------------------------------------------
// star densities
// ------------------------------------------------------------------
// KIND: the star's particles -- 3 (a, b, p), 2 (a, p), 1 (a alone: the plain
// density of a pair).  A record holds one density:
//   [0] exponent w  [1..3] centre  [4] prefactor  [5] overlap (density at p)
//   [6 + d NE + t] Hermite coefficients of direction d
// The prefactor carries the geminal weights, the sign of the Coulomb term (-
// at the proton), 2 pi^(5/2) / w and the Gaussian factors.  Records of one
// star are consecutive: geminal term by geminal term, p, a, b.
constexpr int REC_HEAD = 6;

struct StarJob {
    i64 st0, nst;     // primitive stars st0 .. st0 + nst - 1 (triangle over the pair list, or the list)
    i64 q0, nq;       // distinct nuclear pairs q0 .. q0 + nq - 1
    int nterm, NE;    // geminal terms, coefficients per direction
    const double *gk, *gl, *w; // geminal exponents at a and b, weight, per term
};

template <int KIND, int NL>
__global__ void __launch_bounds__(64) k_star(DevSys S, PairPlan P, StarJob J, double *__restrict__ rec)
{
    const i64 nrec = (i64)J.nterm * KIND, total = J.nst * J.nq * nrec;
    const int RS = REC_HEAD + 3 * J.NE;
    for (i64 t = (i64)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (i64)gridDim.x * blockDim.x) {
        const int r = (int)(t % nrec), k = r / KIND, dens = r % KIND;
        const i64 u = t / nrec, q = J.q0 + u / J.nst;
        i64 a = J.st0 + u % J.nst, b = 0;
        if constexpr (KIND == 3) tri_decode(J.st0 + u % J.nst, b, a);
        const PairRec *qa = S.ep + P.pl_idx[a], *qb = KIND == 3 ? S.ep + P.pl_idx[b] : nullptr;
        const PairRec *qp = KIND > 1 ? S.pp + P.pp_idx[q] : nullptr;
        SysParams SP = d_params(S);
        Sys s = KIND == 3 ? mksys(SP, 3, qa, qb, qp, 0, J.gk[k], J.gl[k], 0)
                          : KIND == 2 ? mksys(SP, 2, qa, qp, 0, 0, J.gk[k], 0, 0) : mksys(SP, 1, qa, 0, 0, 0, 0, 0, 0);
        const int core = dens == 0 ? KIND - 1 : dens - 1; // p (or a alone), then a, b
        double *o = rec + t * RS;
        double fac = J.w[k], w = 1.0, e0 = 1.0;
        NRX_UNROLL for (int i = 0; i < KIND; ++i) fac *= s.q[i]->K;
        NRX_DIRS for (int d = 0; d < 3; ++d) {
            PolyT<NL> e;
            double X;
            fac *= nuc_core<NL>(s, core, d, e, X, w, PI);
            o[1 + d] = X;
            NRX_UNROLL for (int i = 0; i < NL; ++i)
                if (i < J.NE) o[REC_HEAD + d * J.NE + i] = e.c[i];
            e0 *= e.c[0];
        }
        const double iw = rcp(w), rw = rsqrt(w);
        o[0] = w;
        o[4] = (KIND > 1 && dens == 0 ? -fac : fac) * TWO_PI_2P5 * iw;
        o[5] = KIND > 1 && dens == 0 ? fac * e0 * (PI * sqrt(PI)) * iw * rw : 0.0;
    }
}

// ------------------------------------------------------------------
// the lone electron
// ------------------------------------------------------------------
// Lone-pair data, a column per slot of the sorted order: exponent, centre,
// coefficient / exponent (with K), one-electron value times coefficient, and
// the Hermite coefficients with the sign (-1)^u of the second particle.
constexpr int LONE_HEAD = 6;
constexpr int LONE_NC = 5; // coefficients per direction (l <= 2)
constexpr int LONE_F = LONE_HEAD + 3 * LONE_NC;

__global__ void __launch_bounds__(64) k_lone_prep(DevSys S, PairPlan P, double *__restrict__ lone)
{
    const i64 k = (i64)blockIdx.x * blockDim.x + threadIdx.x, n = P.nslot;
    if (k >= n) return;
    const int pl = P.slot[k];
    const PairRec *q = S.ep + P.pl_idx[pl < 0 ? 0 : pl];
    const double cf = pl < 0 ? 0.0 : P.pl_coef[pl];
    SysParams SP = d_params(S);
    Sys s = mksys(SP, 1, q, 0, 0, 0, 0, 0, 0);
    const double h = kin<7>(s, 0, -1, 0.0, 1.0) - nuc_sum<5, 5>(s, 0, S.nat, S.cat, S.zan, false);
    lone[k] = q->p;
    for (int d = 0; d < 3; ++d) {
        lone[(1 + d) * n + k] = q->P[d];
        PolyT<LONE_NC> f, e;
        fpoly(*q, d, f);
        p_hermite(f, q->p, e);
        NRX_UNROLL for (int u = 0; u < LONE_NC; ++u)
            lone[(LONE_HEAD + d * LONE_NC + u) * n + k] = (u & 1) ? -e.c[u] : e.c[u];
    }
    lone[4 * n + k] = cf * q->K * rcp(q->p);
    lone[5 * n + k] = cf * h;
}

// One direction of a Coulomb integral: the star's coefficients e (degree <=
// M, wave-uniform) and the lane's ec (degree <= N) convolved, h, and
//   P(v) = sum_j v^j sum_k (j+k)! h_{j+k} (2D)^{j-k} / ((j-k)! k!),
// the closed form of the derivatives of exp(-rho u^2 D^2) with v = -rho u^2,
// multiplied into the running product cc (capacity LC; FIRST: cc = P).
template <int M, int N, int LC, bool FIRST>
NRX_DI void dir_step(const double *__restrict__ e, const double *ec, double D, double (&cc)[LC])
{
    constexpr int NT = M + N < LC ? M + N : LC - 1; // product terms past LC vanish
    double h[NT + 1], dd[NT + 1], Pj[NT + 1];
    NRX_UNROLL for (int t = 0; t <= NT; ++t) h[t] = 0.0;
    NRX_UNROLL for (int u = 0; u <= N; ++u) {
        const double x = ec[u * 64];
        NRX_UNROLL for (int t = 0; t <= M; ++t)
            if (t + u <= NT) h[t + u] += e[t] * x;
    }
    const double D2 = 2.0 * D;
    dd[0] = 1.0;
    NRX_UNROLL for (int i = 1; i <= NT; ++i) dd[i] = i == 1 ? D2 : dd[i - 1] * (D2 * (1.0 / i));
    NRX_UNROLL for (int t = 2; t <= NT; ++t) h[t] *= factc(t);
    NRX_UNROLL for (int j = 0; j <= NT; ++j) {
        double acc = h[j] * dd[j];
        NRX_UNROLL for (int k = 1; k <= j && j + k <= NT; ++k)
            acc += (k == 1 ? h[j + k] : h[j + k] * (1.0 / factc(k))) * dd[j - k];
        Pj[j] = acc;
    }
    if constexpr (FIRST) {
        NRX_UNROLL for (int j = 0; j < LC; ++j) cc[j] = j <= NT ? Pj[j] : 0.0;
    } else {
        NRX_UNROLL for (int j = LC - 1; j >= 0; --j) {
            double acc = cc[j] * Pj[0];
            NRX_UNROLL for (int i = 1; i <= NT && i <= j; ++i) acc += cc[j - i] * Pj[i];
            cc[j] = acc;
        }
    }
}

// dispatch of dir_step on the wave-uniform degrees m (star) and n (lone);
// large star degrees round up (the records hold zeros there)
template <int M, int LC, int NC, bool FIRST>
NRX_DI void dir_n(int n, const double *__restrict__ e, const double *ec, double D, double (&cc)[LC])
{
    if (n == 0)
        dir_step<M, 0, LC, FIRST>(e, ec, D, cc);
    else if (n == 1)
        dir_step<M, 1, LC, FIRST>(e, ec, D, cc);
    else if (NC == 2 || n == 2)
        dir_step<M, 2, LC, FIRST>(e, ec, D, cc);
    else
        dir_step<M, NC, LC, FIRST>(e, ec, D, cc);
}
template <int LC, int NC, bool FIRST>
NRX_DI void dir_mn(int m, int n, const double *__restrict__ e, const double *ec, double D, double (&cc)[LC])
{
    if (m == 0)
        dir_n<0, LC, NC, FIRST>(n, e, ec, D, cc);
    else if (LC <= 2 || m == 1)
        dir_n<1, LC, NC, FIRST>(n, e, ec, D, cc);
    else if (m == 2)
        dir_n<2, LC, NC, FIRST>(n, e, ec, D, cc);
    else if (LC <= 3 || m == 3)
        dir_n<(LC <= 3 ? 2 : 3), LC, NC, FIRST>(n, e, ec, D, cc);
    else if (m == 4)
        dir_n<4, LC, NC, FIRST>(n, e, ec, D, cc);
    else if (LC <= 7 || m <= 6)
        dir_n<(LC <= 5 ? 4 : 6), LC, NC, FIRST>(n, e, ec, D, cc);
    else if (LC <= 11 || m <= 8)
        dir_n<8, LC, NC, FIRST>(n, e, ec, D, cc);
    else
        dir_n<12, LC, NC, FIRST>(n, e, ec, D, cc);
}

// sum_n c_n mr^n F_n(T), T = rho D^2, mr = -rho: the reference's two-branch
// Boys function (see boys_dot), with exp(-T) from the table's grid value
template <int LC> NRX_DI double boys_lone(const double (&c)[LC], double T, double D2, double mr, const double *bt)
{
    if (T > 20.0) {
        const double rT = rsqrt(T), z = -rcp(D2); // mr / T
        double s = c[LC - 1];
        NRX_UNROLL for (int n = LC - 1; n >= 1; --n) s = c[n - 1] + s * ((n - 0.5) * z);
        return 0.88622692545275801365 * rT * s;
    }
    const int i = (int)(T * (1.0 / BT_H) + 0.5);
    const double dt = T - i * BT_H, *row = bt + i * BT_M + (LC - 1);
    double f = row[BT_K - 1];
    NRX_UNROLL for (int k = BT_K - 1; k >= 1; --k) f = row[k - 1] - dt * f * (1.0 / k);
    double s = c[LC - 1] * f;
    if constexpr (LC > 1) {
        const double ex = exp(-T), t2 = 2.0 * T;
        NRX_UNROLL for (int n = LC - 2; n >= 0; --n) {
            f = (t2 * f + ex) * (1.0 / (2 * n + 1));
            s = s * mr + c[n] * f;
        }
    }
    return s;
}

// the Coulomb sum of one star's nrec records with the wave's lone pairs
template <int LC, int NC>
NRX_DI void star_sum(const double *__restrict__ rec, int nrec, int RS, int NE, int m, int n, const double *ld,
                     double wc, const double *bt, double &acc, double &ov)
{
    for (int r = 0; r < nrec; ++r) {
        const double *R = rec + (i64)r * RS;
        const double rs = rsqrt(R[0] + wc), rho = R[0] * wc * (rs * rs);
        double cc[LC], D2;
        {
            const double D = R[1] - ld[0];
            D2 = D * D;
            dir_mn<LC, NC, true>(deg_of(m, 0), deg_of(n, 0), R + REC_HEAD, ld + 3 * 64, D, cc);
        }
        NRX_DIRS for (int d = 1; d < 3; ++d) {
            const double D = R[1 + d] - ld[d * 64];
            D2 += D * D;
            dir_mn<LC, NC, false>(deg_of(m, d), deg_of(n, d), R + REC_HEAD + d * NE, ld + (3 + d * (NC + 1)) * 64, D,
                                  cc);
        }
        acc += (R[4] * rs) * boys_lone<LC>(cc, rho * D2, D2, -rho, bt);
        ov += R[5];
    }
}

// A wave per contracted star (unit) and group of 64 lone pairs.  KIND 3: unit
// = triangle entry {A,B} of the contracted pairs and nuclear pair, KIND 2:
// contracted pair and nuclear pair, KIND 1: contracted pair.  NC: the lone
// pairs' largest degree per direction, LMAX: the largest total degree.
struct LoneJob {
    i64 u0, nu;       // contracted stars u0 .. u0 + nu - 1 of this launch
    i64 q0, st0, nst; // as the StarJob that filled rec
    int nterm, NE;
    i64 oq;           // output rows between nuclear pairs
    double hs;        // factor of the overlap x one-electron term (1, or 0 without it)
};

template <int KIND, int NC, int LMAX>
__global__ void __launch_bounds__(64) k_lone(DevSys S, PairPlan P, LoneJob J, const double *__restrict__ rec,
                                             const double *__restrict__ lone, double *__restrict__ out)
{
    // centre and Hermite coefficients of the lane's pair: [3][64], [3][NC+1][64]
    __shared__ double ls[(3 + 3 * (NC + 1)) * 64];
    const int lane = threadIdx.x;
    const i64 k = (i64)blockIdx.y * 64 + lane, ns = P.nslot;
    double *ld = ls + lane;
    const double wc = lone[k], kc = lone[4 * ns + k], hc = lone[5 * ns + k];
    NRX_UNROLL for (int d = 0; d < 3; ++d) {
        ld[d * 64] = lone[(1 + d) * ns + k];
        NRX_UNROLL for (int u = 0; u <= NC; ++u)
            ld[(3 + d * (NC + 1) + u) * 64] = lone[(LONE_HEAD + d * LONE_NC + u) * ns + k];
    }
    const int n = P.gdeg[blockIdx.y], nL = P.gL[blockIdx.y];
    const i64 u = J.u0 + blockIdx.x % (unsigned)J.nu, q = blockIdx.x / (unsigned)J.nu; // q relative to J.q0
    i64 A = u, B = 0;
    if constexpr (KIND == 3) {
        tri_decode(u, B, A);
        A = __builtin_amdgcn_readfirstlane((int)A); // wave-uniform, kept in scalar registers
        B = __builtin_amdgcn_readfirstlane((int)B);
    }
    const int RS = REC_HEAD + 3 * J.NE, nrec = J.nterm * KIND;
    const int mp = KIND > 1 ? P.pp_deg[J.q0 + q] : 0;
    double tot = 0.0, ovt = 0.0;
    const int b0 = KIND == 3 ? P.cp_start[B] : 0, b1 = KIND == 3 ? P.cp_start[B + 1] : 1;
    for (int b = b0; b < b1; ++b) {
        const int a0 = P.cp_start[A], a1 = KIND == 3 && A == B ? b + 1 : P.cp_start[A + 1];
        for (int a = a0; a < a1; ++a) {
            double cf = P.pl_coef[a];
            int m = mp + P.pl_deg[a];
            i64 st = a;
            if constexpr (KIND == 3) {
                cf *= P.pl_coef[b] * (A == B && a < b ? 2.0 : 1.0);
                m += P.pl_deg[b];
                st = (i64)b * (b + 1) / 2 + a;
            }
            const double *R = rec + (q * J.nst + st - J.st0) * nrec * RS;
            const int L = deg_of(m, 0) + deg_of(m, 1) + deg_of(m, 2) + nL;
            double acc = 0.0, ov = 0.0;
            if (L == 0)
                star_sum<1, NC>(R, nrec, RS, J.NE, m, n, ld, wc, S.bt, acc, ov);
            else if (L <= 2)
                star_sum<3, NC>(R, nrec, RS, J.NE, m, n, ld, wc, S.bt, acc, ov);
            else if (LMAX <= 4 || L <= 4)
                star_sum<5, NC>(R, nrec, RS, J.NE, m, n, ld, wc, S.bt, acc, ov);
            else if (L <= 6)
                star_sum<7, NC>(R, nrec, RS, J.NE, m, n, ld, wc, S.bt, acc, ov);
            else if (LMAX <= 8 || L <= 8)
                star_sum<9, NC>(R, nrec, RS, J.NE, m, n, ld, wc, S.bt, acc, ov);
            else if (LMAX <= 12 || L <= 12)
                star_sum<(LMAX < 12 ? LMAX : 12) + 1, NC>(R, nrec, RS, J.NE, m, n, ld, wc, S.bt, acc, ov);
            else
                star_sum<LMAX + 1, NC>(R, nrec, RS, J.NE, m, n, ld, wc, S.bt, acc, ov);
            tot += cf * acc;
            ovt += cf * ov;
        }
    }
    if (const int pl = P.slot[k]; pl >= 0) {
        const double cp = KIND > 1 ? P.pp_coef[J.q0 + q] : 1.0;
        out[(q * J.oq + u - J.u0) * P.npl + pl] = cp * (kc * tot + J.hs * (hc * ovt));
    }
}

// out[q][u][C] = sum of the lone primitive pairs of contracted pair C in
// in[q][u], u < nu, nuclear pairs oq rows apart in out
__global__ void __launch_bounds__(256) k_lone_sum(PairPlan P, i64 nu, i64 nq, i64 oq, const double *__restrict__ in,
                                                  double *__restrict__ out)
{
    const i64 n = nu * nq * P.ncp;
    for (i64 t = (i64)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (i64)gridDim.x * blockDim.x) {
        const i64 r = t / P.ncp, C = t % P.ncp;
        double v = 0.0;
        for (int i = P.cp_start[C]; i < P.cp_start[C + 1]; ++i) v += in[r * P.npl + i];
        out[(r / nu * oq + r % nu) * P.ncp + C] = v;
    }
}

// X[q][C] = sum over the terms of the (c,p) overlaps, contracted
__global__ void __launch_bounds__(64) k_star_ovl(DevSys S, PairPlan P, StarJob J, double *__restrict__ X)
{
    const i64 t = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= J.nq * P.ncp) return;
    const i64 q = J.q0 + t / P.ncp, C = t % P.ncp;
    SysParams SP = d_params(S);
    double acc = 0.0;
    for (int i = P.cp_start[C]; i < P.cp_start[C + 1]; ++i)
        for (int k = 0; k < J.nterm; ++k) {
            Sys s = mksys(SP, 2, S.ep + P.pl_idx[i], S.pp + P.pp_idx[q], 0, 0, J.gk[k], 0, 0);
            acc += P.pl_coef[i] * J.w[k] * ovl<9>(s);
        }
    X[t] = acc * P.pp_coef[q];
}

// Block per (contracted pairs p1 >= p2, nuclear pair): the row over p3 of
//   1/3 [ T(12;3) + T(13;2) + T(23;1) + X3 V12 + X2 V13 + X1 V23 ]
// in LDS, then every copy of it in the full tensor: both orders of p1, p2
// and of each one's bra and ket, and, where the tensor holds every (ip,jp),
// both nuclear orders.
struct Gam3Out {
    double *G;        // full tensor, or the first block
    i64 blk;          // entries of one (ip,jp) block
    i64 np;           // > 0: block of nuclear pair (i,j) at i*np + j and j*np + i; 0: at q
    int pack;         // the last index over the distinct pairs only
};

__global__ void __launch_bounds__(256) k_gam3_expand(PairPlan P, i64 ne, i64 q0, const double *__restrict__ T,
                                                     const double *__restrict__ V, const double *__restrict__ X,
                                                     Gam3Out O)
{
    extern __shared__ double row[];
    const i64 nc = P.ncp, ntri = nc * (nc + 1) / 2, q = blockIdx.y;
    const double *Tq = T + q * ntri * nc, *Xq = X + q * nc;
    i64 p1, p2;
    tri_decode(blockIdx.x, p1, p2);
    const double x1 = Xq[p1], x2 = Xq[p2], v12 = V[p1 * nc + p2];
    for (i64 c = threadIdx.x; c < nc; c += blockDim.x) {
        const double t = Tq[tri_index(p1, p2) * nc + c] + Tq[tri_index(p1, c) * nc + p2] + Tq[tri_index(p2, c) * nc + p1];
        const double v13 = V[max(p1, c) * nc + min(p1, c)], v23 = V[max(p2, c) * nc + min(p2, c)];
        row[c] = (t + Xq[c] * v12 + x2 * v13 + x1 * v23) / 3.0;
    }
    __syncthreads();
    i64 i1, j1, i2, j2; // contracted functions of the pairs
    tri_decode(p1, j1, i1);
    tri_decode(p2, j2, i2);
    const i64 ne2 = ne * ne;
    i64 r1[2] = {i1 * ne + j1, j1 * ne + i1}, r2[2] = {i2 * ne + j2, j2 * ne + i2};
    const int n1 = i1 == j1 ? 1 : 2, n2 = i2 == j2 ? 1 : 2, sw = p1 == p2 ? 1 : 2;
    i64 b[2] = {q, q};
    int nb = 1;
    if (O.np > 0) {
        i64 jp, ip;
        tri_decode(q0 + q, jp, ip);
        b[0] = ip * O.np + jp;
        b[1] = jp * O.np + ip;
        nb = ip == jp ? 1 : 2;
    }
    const i64 len = O.pack ? nc : ne2;
    for (i64 x = threadIdx.x; x < len; x += blockDim.x) {
        const double v = row[O.pack ? x : tri_index(x / ne, x % ne)];
        for (int k = 0; k < nb; ++k)
            for (int u = 0; u < n1; ++u)
                for (int w = 0; w < n2; ++w)
                    for (int z = 0; z < sw; ++z) {
                        const i64 P1 = z ? r2[w] : r1[u], P2 = z ? r1[u] : r2[w];
                        O.G[b[k] * O.blk + (P1 * ne2 + P2) * len + x] = v;
                    }
    }
}

// ------------------------------------------------------------------
// GAM_2: the terms that both geminals bond
// ------------------------------------------------------------------
constexpr int KT = 7;         // coefficients of a kinetic polynomial (degree <= 2 l + 2)

// kinetic polynomials of the pair list, then of the nuclear pairs (times 1/m):
// the mean of the operator on the bra and on the ket
__global__ void __launch_bounds__(64) k_pair_kin(DevSys S, PairPlan P, double *__restrict__ kt)
{
    const i64 t = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 3 * (P.npl + P.nq)) return;
    const i64 k = t / 3;
    const bool nuc = k >= P.npl;
    const double w = nuc ? 0.5 / S.pmass : 0.5;
    PolyT<KT> r;
    pair_kin_poly(nuc ? S.pp[P.pp_idx[k - P.npl]] : S.ep[P.pl_idx[k]], (int)(t % 3), w, w, r);
    NRX_UNROLL for (int i = 0; i < KT; ++i) kt[t * KT + i] = r.c[i];
}

// Capacity tiers of a star (largest degree per direction, total degree): the
// Coulomb terms need NL >= degree + 1 and NB >= total + 1.
constexpr int BT_N_TIERS = 5;
constexpr int BTIER_NL[BT_N_TIERS] = {3, 5, 7, 9, 13}, BTIER_NB[BT_N_TIERS] = {5, 7, 9, 13, 13};
NRX_DI int bond_tier(int m)
{
    const int dg = max(deg_of(m, 0), max(deg_of(m, 1), deg_of(m, 2))), L = deg_of(m, 0) + deg_of(m, 1) + deg_of(m, 2);
    int k = 0;
    while (k < BT_N_TIERS - 1 && (dg >= BTIER_NL[k] || L >= BTIER_NB[k])) ++k;
    return k;
}

__global__ void k_zero_counts(unsigned *p)
{
    if (threadIdx.x < 16) p[threadIdx.x] = 0u;
}

// the stars of a launch sorted by tier (count, then scatter): lists of star
// numbers, tier by tier from counts[]; cursors at counts + 8
__global__ void __launch_bounds__(256) k_bond_bin(PairPlan P, StarJob J, int scatter, unsigned *__restrict__ counts,
                                                  unsigned *__restrict__ list)
{
    __shared__ unsigned lc[BT_N_TIERS], lb[BT_N_TIERS];
    if (threadIdx.x < BT_N_TIERS) lc[threadIdx.x] = 0u;
    __syncthreads();
    const i64 t = (i64)blockIdx.x * blockDim.x + threadIdx.x;
    int tier = -1;
    unsigned pos = 0;
    if (t < J.nst * J.nq) {
        i64 a, b;
        tri_decode(J.st0 + t % J.nst, b, a);
        tier = bond_tier(P.pl_deg[a] + P.pl_deg[b] + P.pp_deg[J.q0 + t / J.nst]);
        pos = atomicAdd(&lc[tier], 1u);
    }
    __syncthreads();
    if (threadIdx.x < BT_N_TIERS) {
        const unsigned n = lc[threadIdx.x];
        if (!scatter) {
            if (n) atomicAdd(&counts[threadIdx.x], n);
        } else {
            lb[threadIdx.x] = bin_offset(counts, threadIdx.x) + (n ? atomicAdd(&counts[8 + threadIdx.x], n) : 0u);
        }
    }
    if (!scatter) return;
    __syncthreads();
    if (tier >= 0) list[lb[tier] + pos] = (unsigned)t;
}

// The rows of a launch's values: a row per term and geminal pair, the launch's
// stars along it.  All: every term of B and the overlap; rxne: <1/r_ab> alone.
enum { BT_KIN = 0, BT_AP, BT_BP, BT_AB, BT_NP, BT_NA, BT_NB, BT_OVL, BT_ROWS };

// Term blockIdx.y (or <1/r_ab>, rxne) of the tier's stars: a lane per star, the
// geminal pair uniform over most waves, striding over the tier's list.
// The kernel is bound by FP64 issue at one or two waves per SIMD: the
// polynomial tables of a term fill the registers.
template <int TIER>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(TIER < 2 ? 2 : 1)))
k_bond(DevSys S, PairPlan P, StarJob J, int rxne, const double *__restrict__ kt, const unsigned *__restrict__ counts,
       const unsigned *__restrict__ list, double *__restrict__ val)
{
    constexpr int NL = BTIER_NL[TIER], NBC = BTIER_NB[TIER];
    const unsigned off = bin_offset(counts, TIER);
    const i64 cnt = counts[TIER], nkl = J.nterm, row = J.nst * J.nq;
    const int term = rxne ? BT_AB : (int)blockIdx.y;
    for (i64 t = (i64)blockIdx.x * 64 + threadIdx.x; t < cnt * nkl; t += (i64)gridDim.x * 64) {
        const i64 star = list[off + t % cnt], k = t / cnt, q = J.q0 + star / J.nst;
        i64 a, b;
        tri_decode(J.st0 + star % J.nst, b, a);
        SysParams SP = d_params(S);
        Sys s = mksys(SP, 3, S.ep + P.pl_idx[a], S.ep + P.pl_idx[b], S.pp + P.pp_idx[q], 0, J.gk[k], J.gl[k], 0);
        double v;
        if (term == BT_KIN) {
            const double *kp[3] = {kt + a * 3 * KT, kt + b * 3 * KT, kt + (P.npl + q) * 3 * KT};
            double o;
            v = star_kin<NL + 2>(s, StarKin{{}, {}, 2.0 * J.gk[k] * J.gl[k] / S.pmass, 0.0, 0.0}, PI, o,
                                 [&](int i, int x, auto &f) {
                                     f.n = (int)(sizeof(f.c) / sizeof(double)); // at most KT
                                     NRX_UNROLL for (int c = 0; c < f.n; ++c) f.c[c] = kp[i][x * KT + c];
                                 });
            val[(BT_OVL * nkl + k) * row + star] = J.w[k] * o;
        } else if (term <= BT_BP) {
            v = -coul<NL, NBC>(s, term == BT_AP ? 0 : 1, 2);
        } else if (term == BT_AB) {
            v = coul<NL, NBC>(s, 0, 1);
        } else if (term == BT_NP) {
            v = nuc_sum<NL, NBC>(s, 2, S.nat, S.cat, S.zan, false);
        } else {
            v = -nuc_sum<NL, NBC>(s, term == BT_NA ? 0 : 1, S.nat, S.cat, S.zan, false);
        }
        val[((rxne ? 0 : term) * nkl + k) * row + star] = J.w[k] * v;
    }
}

// row 0 of the values becomes the sum of rows 0 .. nB-1 (B of a primitive
// star), row 1 that of the nO rows from rO on (its overlap)
__global__ void __launch_bounds__(256) k_bond_rows(i64 n, i64 nB, i64 rO, i64 nO, double *__restrict__ val)
{
    for (i64 t = (i64)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (i64)gridDim.x * blockDim.x) {
        double e = 0.0, y = 0.0;
        for (i64 k = 0; k < nB; ++k) e += val[k * n + t];
        for (i64 k = 0; k < nO; ++k) y += val[(rO + k) * n + t];
        val[t] = e;
        if (nO) val[n + t] = y;
    }
}

// contracted stars: B[q][u] and Y[q][u] (null to skip), sums over their
// primitive stars of the value rows 0 and 1
__global__ void __launch_bounds__(256) k_bond_sum(PairPlan P, StarJob J, LoneJob L, const double *__restrict__ val,
                                                  double *__restrict__ B, double *__restrict__ Y)
{
    const i64 n = L.nu * J.nq, row = J.nst * J.nq;
    for (i64 t = (i64)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (i64)gridDim.x * blockDim.x) {
        const i64 q = t / L.nu, u = L.u0 + t % L.nu;
        i64 Bc, Ac;
        tri_decode(u, Bc, Ac);
        double e = 0.0, y = 0.0;
        for (int b = P.cp_start[Bc]; b < P.cp_start[Bc + 1]; ++b)
            for (int a = P.cp_start[Ac]; a < (Ac == Bc ? b + 1 : P.cp_start[Ac + 1]); ++a) {
                const i64 star = q * J.nst + (i64)b * (b + 1) / 2 + a - J.st0;
                const double cf = P.pl_coef[a] * P.pl_coef[b] * (Ac == Bc && a < b ? 2.0 : 1.0);
                e += cf * val[star];
                if (Y) y += cf * val[row + star];
            }
        const double cp = P.pp_coef[J.q0 + q];
        B[q * L.oq + t % L.nu] = cp * e;
        if (Y) Y[q * L.oq + t % L.nu] = cp * y;
    }
}

// Full tensors of the nuclear pairs q0 ..: G = L(a;b) + L(b;a) + B, Gs = Y, or
// with rxne G = 2 L[a][b] (star electron first), Gs = B.  np > 0: every (ip,jp)
// of the full tensor; np = 0: one block per pair.
__global__ void __launch_bounds__(256) k_gam2_expand(i64 ne, i64 nc, i64 q0, i64 nq, i64 np, int rxne,
                                                     const double *__restrict__ Lq, const double *__restrict__ B,
                                                     const double *__restrict__ Y, double *__restrict__ G,
                                                     double *__restrict__ Gs)
{
    const i64 ne2 = ne * ne, ne4 = ne2 * ne2, ntri = nc * (nc + 1) / 2, nblk = np > 0 ? np * np : nq;
    for (i64 t = (i64)blockIdx.x * blockDim.x + threadIdx.x; t < nblk * ne4; t += (i64)gridDim.x * blockDim.x) {
        const i64 blk = t / ne4, p1 = t / ne2 % ne2, p2 = t % ne2;
        const i64 q = np > 0 ? tri_index(blk / np, blk % np) - q0 : blk;
        const i64 A = tri_index(p1 / ne, p1 % ne), C = tri_index(p2 / ne, p2 % ne), u = q * ntri + tri_index(A, C);
        const double l1 = Lq[(q * nc + A) * nc + C];
        if (rxne) {
            G[t] = 2.0 * l1;
            Gs[t] = B[u];
        } else {
            G[t] = l1 + Lq[(q * nc + C) * nc + A] + B[u];
            Gs[t] = Y[u];
        }
    }
}

// ------------------------------------------------------------------
// host side
// ------------------------------------------------------------------
// bytes of star records and lone partial sums of one launch, which then stay in
// the last-level cache; the primitive stars of one contracted row and nuclear
// pair are never divided, however many they are (24 functions of 6 s/p
// primitives each, three geminals: up to 2.2 GB)
constexpr i64 REC_BYTES = (i64)192 << 20;
// most blocks of one k_bond launch and term; the blocks stride over the list
constexpr i64 BOND_BLOCKS = 8192;
// bytes of contracted star values T held at once (at least one nuclear pair)
constexpr i64 T_BYTES = (i64)4 << 30;

template <int KIND> int star_launch(const DevSys &d, const PairPlan &P, const StarJob &J, double *rec, hipStream_t st)
{
    const i64 n = J.nst * J.nq * J.nterm * KIND;
    const dim3 grid(grid_blocks(n, 64)), blk(64);
    if (J.NE <= 7)
        hipLaunchKernelGGL((k_star<KIND, 7>), grid, blk, 0, st, d, P, J, rec);
    else if (J.NE <= 9)
        hipLaunchKernelGGL((k_star<KIND, 9>), grid, blk, 0, st, d, P, J, rec);
    else
        hipLaunchKernelGGL((k_star<KIND, 13>), grid, blk, 0, st, d, P, J, rec);
    HIPCHK(hipGetLastError());
    return NEORX_OK;
}

template <int KIND>
int lone_launch(const DevSys &d, const PairPlan &P, const LoneJob &J, i64 nq, const double *rec, const double *lone,
                double *out, hipStream_t st)
{
    const dim3 grid((unsigned)(J.nu * nq), (unsigned)(P.nslot / 64)), blk(64);
    // smallest capacities that hold the basis: l <= 1 or 2, total degree of
    // KIND - 1 (KIND 1: one) star electrons, the proton and the lone electron
    if constexpr (KIND == 1) {
        if (P.le <= 1)
            hipLaunchKernelGGL((k_lone<1, 2, 4>), grid, blk, 0, st, d, P, J, rec, lone, out);
        else
            hipLaunchKernelGGL((k_lone<1, 4, 8>), grid, blk, 0, st, d, P, J, rec, lone, out);
    } else {
        if (P.le <= 1 && 2 * KIND * P.le + 2 * P.lp <= 8)
            hipLaunchKernelGGL((k_lone<KIND, 2, 8>), grid, blk, 0, st, d, P, J, rec, lone, out);
        else if (P.le <= 1)
            hipLaunchKernelGGL((k_lone<KIND, 2, 10>), grid, blk, 0, st, d, P, J, rec, lone, out);
        else
            hipLaunchKernelGGL((k_lone<KIND, 4, 16>), grid, blk, 0, st, d, P, J, rec, lone, out);
    }
    HIPCHK(hipGetLastError());
    return NEORX_OK;
}

// coefficients per direction of a record: the star's largest degree, rounded
// up to one that dir_mn has
int rec_ne(int deg) { return (deg <= 4 ? deg : deg <= 6 ? 6 : deg <= 8 ? 8 : 12) + 1; }

} // namespace

// V, X and T of the distinct nuclear pairs, then G (see Gam3Out).  mult: the
// RXCHFmult form, without the one-geminal terms.
int nrx_gam3_pairs(System *s, bool mult, i64 np_full, double *G, Work &W, bool pack, i64 nb, const PairSink &sink)
{
    int rc = nrx_plan(s);
    if (rc) return rc;
    hipStream_t st = W.st;
    const DevSys &d = s->d;
    const PairPlan &P = s->plan;
    const i64 ne = d.nebf, nc = P.ncp, ntri = nc * (nc + 1) / 2;
    const int ng = (int)d.ngtg, nt = ng * ng;
    double *lone, *T, *rec;
    rc = W.get(lone, LONE_F * P.nslot + nc * nc + nc * P.nq + nc * P.npl);
    if (rc) return rc;
    double *V = lone + LONE_F * P.nslot, *X = V + nc * nc, *Vp = X + nc * P.nq;
    hipLaunchKernelGGL(k_lone_prep, dim3((unsigned)(P.nslot / 64)), dim3(64), 0, st, d, P, lone);
    HIPCHK(hipGetLastError());
    StarJob X1{0, P.npl, 0, P.nq, 0, 0, P.gx, nullptr, P.wx};
    X1.nterm = ng + ng * (ng + 1) / 2;
    if (mult) { // the two-geminal terms only: they follow the ng one-geminal ones
        X1.gk += ng;
        X1.w += ng;
        X1.nterm -= ng;
    }
    hipLaunchKernelGGL(k_star_ovl, dim3(nblocks(P.nq * nc, 64)), dim3(64), 0, st, d, P, X1, X);
    HIPCHK(hipGetLastError());
    const int NE = rec_ne(4 * P.le + 2 * P.lp), NE1 = rec_ne(2 * P.le), RS = REC_HEAD + 3 * NE;
    const i64 star_b = (i64)nt * 3 * RS * 8;
    // rows B0 .. B1-1 of the triangle for nq nuclear pairs: primitive stars,
    // contracted stars, bytes
    auto span = [&](i64 B0, i64 B1, i64 nq, i64 &nst, i64 &nu) {
        const i64 a = s->cp_start[B0], b = s->cp_start[B1];
        nst = b * (b + 1) / 2 - a * (a + 1) / 2;
        nu = B1 * (B1 + 1) / 2 - B0 * (B0 + 1) / 2;
        return nq * (nst * star_b + (P.npl > nc ? nu * P.npl * 8 : 0));
    };
    i64 nst = 0, nu = 0, big = 0;
    for (i64 B = 0; B < nc; ++B) big = std::max(big, span(B, B + 1, 1, nst, nu));
    const i64 nqt = std::max<i64>(1, std::min<i64>({nb ? nb : P.nq, P.nq, T_BYTES / (ntri * nc * 8), (i64)32768})); // nuclear pairs T holds
    const i64 nqr = std::max<i64>(1, std::min<i64>(nqt, REC_BYTES / big));               // and one launch takes
    const i64 vcap = P.npl * (REC_HEAD + 3 * NE1) * 8;
    if ((rc = W.get(T, nqt * ntri * nc))) return rc;
    const i64 all = std::min(REC_BYTES, span(0, nc, nqr, nst, nu));
    if ((rc = W.get(rec, (std::max({vcap, big * nqr, all}) + 7) / 8))) return rc;
    { // V: pair densities and lone pairs
        StarJob J{0, P.npl, 0, 1, 1, NE1, P.one + 1, P.one + 1, P.one};
        LoneJob L{0, nc, 0, 0, P.npl, 1, NE1, nc, 0.0};
        rc = star_launch<1>(d, P, J, rec, st);
        if (!rc) rc = lone_launch<1>(d, P, L, 1, rec, lone, Vp, st);
        if (rc) return rc;
        hipLaunchKernelGGL(k_lone_sum, dim3(grid_blocks(nc * nc, 256)), dim3(256), 0, st, P, nc, (i64)1, nc, Vp, V);
        HIPCHK(hipGetLastError());
    }
    using clock = std::chrono::steady_clock;
    const clock::time_point t0 = clock::now();
    clock::time_point said = t0;
    for (i64 q = 0; q < P.nq; q += nqt) {
        const i64 nqp = std::min(nqt, P.nq - q);
        for (i64 k = 0; k < nqp; k += nqr) {
            const i64 nq = std::min(nqr, nqp - k);
            for (i64 B0 = 0, B1; B0 < nc; B0 = B1) {
                B1 = B0 + 1;
                while (B1 < nc && span(B0, B1 + 1, nq, nst, nu) <= REC_BYTES && nu * nq < (i64)1 << 30) ++B1;
                span(B0, B1, nq, nst, nu);
                const i64 s0 = s->cp_start[B0], st0 = s0 * (s0 + 1) / 2, u0 = B0 * (B0 + 1) / 2;
                StarJob J{st0, nst, q + k, nq, nt, NE, P.gk, P.gl, P.wkl};
                rc = star_launch<3>(d, P, J, rec, st);
                if (rc) return rc;
                // T[q][u][C], straight from the lanes or through the sums over lone primitives
                double *part = rec + nq * nst * nt * 3 * RS, *o = T + (k * ntri + u0) * nc;
                const bool sum = P.npl > nc;
                LoneJob L{u0, nu, q + k, st0, nst, nt, NE, sum ? nu : ntri, 1.0};
                rc = lone_launch<3>(d, P, L, nq, rec, lone, sum ? part : o, st);
                if (rc) return rc;
                if (sum) {
                    hipLaunchKernelGGL(k_lone_sum, dim3(grid_blocks(nu * nq * nc, 256)), dim3(256), 0, st, P, nu, nq,
                                       ntri, part, o);
                    HIPCHK(hipGetLastError());
                }
                if (g_verbose) { // a line every second, and at the end
                    HIPCHK(hipStreamSynchronize(st));
                    const clock::time_point t = clock::now();
                    const bool last = B1 == nc && q + k + nq == P.nq;
                    if (last || t - said > std::chrono::seconds(1)) {
                        said = t;
                        fprintf(stderr, "neorx: e-e-e-p build, row %lld of %lld, nuclear pair %lld of %lld in %.1f s\n",
                                (long long)B1, (long long)nc, (long long)(q + k + nq), (long long)P.nq,
                                std::chrono::duration<double>(t - t0).count());
                    }
                }
            }
        }
        const i64 blk = ne * ne * ne * ne * (pack ? nc : ne * ne);
        Gam3Out O{np_full > 0 || nb ? G : G + q * blk, blk, np_full, pack};
        hipLaunchKernelGGL(k_gam3_expand, dim3((unsigned)ntri, (unsigned)nqp), dim3(256), nc * 8, st, P, ne, q, T, V,
                           X + q * nc, O);
        HIPCHK(hipGetLastError());
        if (nb && (rc = sink(q, q + nqp))) return rc;
    }
    return NEORX_OK;
}

// GAM_2 and its overlaps (rxne: the RXCHF-ne tensors) of the distinct nuclear pairs
int nrx_gam2_pairs(System *s, bool rxne, i64 np_full, double *G, double *Gs, Work &W, i64 nb, const PairSink &sink)
{
    int rc = nrx_plan(s);
    if (rc) return rc;
    hipStream_t st = W.st;
    const DevSys &d = s->d;
    const PairPlan &P = s->plan;
    const i64 ne = d.nebf, nc = P.ncp, ntri = nc * (nc + 1) / 2, nqa = nb ? std::min(nb, P.nq) : P.nq;
    const int ng = (int)d.ngtg, nt = ng * ng, nx = ng * (ng + 1) / 2 + (rxne ? 0 : ng);
    const int NE2 = rec_ne(2 * P.le + 2 * P.lp), nterms = rxne ? 1 : BT_OVL;
    const i64 nrows = (i64)nt * (rxne ? 1 : BT_ROWS);
    double *lone, *rec;
    rc = W.get(lone, LONE_F * P.nslot + 3 * KT * (P.npl + P.nq) + nqa * (nc * nc + 2 * ntri) + 8);
    if (rc) return rc;
    double *kt = lone + LONE_F * P.nslot, *L = kt + 3 * KT * (P.npl + P.nq),
           *B = L + nqa * nc * nc, *Y = B + nqa * ntri;
    unsigned *counts = (unsigned *)(Y + nqa * ntri);
    hipLaunchKernelGGL(k_lone_prep, dim3((unsigned)(P.nslot / 64)), dim3(64), 0, st, d, P, lone);
    hipLaunchKernelGGL(k_pair_kin, dim3(nblocks(3 * (P.npl + P.nq), 64)), dim3(64), 0, st, d, P, kt);
    HIPCHK(hipGetLastError());
    // bytes per primitive star of the bond terms (values, list entry; two rows
    // at least for the sums) and per nuclear pair of the lone part
    const i64 star_b = std::max<i64>(nrows, 2) * 8 + 4;
    const i64 lone_b = (P.npl * nx * 2 * (REC_HEAD + 3 * NE2) + (P.npl > nc ? nc * P.npl : 0)) * 8;
    auto span = [&](i64 B0, i64 B1, i64 &nst, i64 &nu) {
        const i64 a = s->cp_start[B0], b = s->cp_start[B1];
        nst = b * (b + 1) / 2 - a * (a + 1) / 2;
        nu = B1 * (B1 + 1) / 2 - B0 * (B0 + 1) / 2;
        return nst * star_b;
    };
    i64 nst = 0, nu = 0, big = 0;
    for (i64 k = 0; k < nc; ++k) big = std::max(big, span(k, k + 1, nst, nu));
    const i64 all = span(0, nc, nst, nu);
    const i64 nqr = std::max<i64>(1, std::min<i64>(nqa, REC_BYTES / big));
    const i64 nql = std::max<i64>(1, std::min<i64>(nqa, REC_BYTES / lone_b));
    if ((rc = W.get(rec, (std::max({nql * lone_b, nqr * big, std::min(nqr * all, REC_BYTES)}) + 7) / 8))) return rc;
    const int dmax = 4 * P.le + 2 * P.lp; // per direction and in total
    for (i64 q0 = 0; q0 < P.nq; q0 += nqa) {
        const i64 q1 = std::min(P.nq, q0 + nqa);
        for (i64 q = q0; q < q1; q += nql) { // L
            const i64 nq = std::min(nql, q1 - q);
            StarJob J{0, P.npl, q, nq, nx, NE2, P.gx + (rxne ? ng : 0), P.gx, P.wx + (rxne ? ng : 0)};
            LoneJob Lj{0, nc, q, 0, P.npl, nx, NE2, nc, rxne ? 0.0 : 1.0};
            double *part = rec + nq * P.npl * nx * 2 * (REC_HEAD + 3 * NE2), *o = L + (q - q0) * nc * nc;
            rc = star_launch<2>(d, P, J, rec, st);
            if (!rc) rc = lone_launch<2>(d, P, Lj, nq, rec, lone, P.npl > nc ? part : o, st);
            if (rc) return rc;
            if (P.npl > nc)
                hipLaunchKernelGGL(k_lone_sum, dim3(grid_blocks(nc * nq * nc, 256)), dim3(256), 0, st, P, nc, nq, nc, part,
                                   o);
            HIPCHK(hipGetLastError());
        }
        for (i64 q = q0; q < q1; q += nqr) { // B, Y
            const i64 nq = std::min(nqr, q1 - q);
            for (i64 B0 = 0, B1; B0 < nc; B0 = B1) {
                B1 = B0 + 1;
                while (B1 < nc && nq * span(B0, B1 + 1, nst, nu) <= REC_BYTES) ++B1;
                span(B0, B1, nst, nu);
                const i64 s0 = s->cp_start[B0], n = nst * nq;
                StarJob J{s0 * (s0 + 1) / 2, nst, q, nq, nt, 0, P.gk, P.gl, P.wkl};
                LoneJob U{B0 * (B0 + 1) / 2, nu, q, 0, 0, 0, 0, ntri, 0.0};
                unsigned *list = (unsigned *)(rec + std::max<i64>(nrows, 2) * n);
                hipLaunchKernelGGL(k_zero_counts, dim3(1), dim3(64), 0, st, counts);
                hipLaunchKernelGGL(k_bond_bin, dim3(nblocks(n, 256)), dim3(256), 0, st, P, J, 0, counts, list);
                hipLaunchKernelGGL(k_bond_bin, dim3(nblocks(n, 256)), dim3(256), 0, st, P, J, 1, counts, list);
                const dim3 g((unsigned)std::min<i64>(BOND_BLOCKS, (n * nt + 63) / 64), (unsigned)nterms);
#define NRX_BOND(K)                                                                                                   \
    if (K == 0 || dmax >= BTIER_NL[K ? K - 1 : 0] || dmax >= BTIER_NB[K ? K - 1 : 0])                                 \
    hipLaunchKernelGGL((k_bond<K>), g, dim3(64), 0, st, d, P, J, (int)rxne, kt, counts, list, rec)
                NRX_BOND(4);
                NRX_BOND(3);
                NRX_BOND(2);
                NRX_BOND(1);
                NRX_BOND(0);
#undef NRX_BOND
                hipLaunchKernelGGL(k_bond_rows, dim3(grid_blocks(n, 256)), dim3(256), 0, st, n, (i64)nterms * nt,
                                   (i64)BT_OVL * nt, rxne ? (i64)0 : (i64)nt, rec);
                const i64 o = (q - q0) * ntri + U.u0;
                hipLaunchKernelGGL(k_bond_sum, dim3(grid_blocks(nu * nq, 256)), dim3(256), 0, st, P, J, U, rec,
                                   B + o, rxne ? nullptr : Y + o);
                HIPCHK(hipGetLastError());
            }
        }
        const i64 nout = (np_full > 0 ? np_full * np_full : q1 - q0) * ne * ne * ne * ne;
        hipLaunchKernelGGL(k_gam2_expand, dim3(grid_blocks(nout, 256)), dim3(256), 0, st, ne, nc, q0, q1 - q0, np_full,
                           (int)rxne, L, B, Y, G, Gs);
        HIPCHK(hipGetLastError());
        if (nb && (rc = sink(q0, q1))) return rc;
    }
    return NEORX_OK;
}
