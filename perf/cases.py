"""The work that a NEO-XCHF / RXCHF calculation has this framework do, as
measurable cases: primitive integrals, the tensor builders, the Fock-build
contractions (in core, direct, mixed precision) and whole calculations.

A case is a dict of plain values.  ``kind`` picks the entry point:

  prim    primitive tuples of the four-centre s/p/d system: an index list
          (e-e-p, e-e-e-p) or a range of the enumeration (e-p)
  gam2    GAM2_IC1, the e-e-p tensors GM2ICR and GM2sICR
  gam3    GAM3_IC1, the e-e-e-p tensor GM3ICR
  ne2     RXCHFne_GAM2_IC1, the RXCHF-ne e-e-p tensors
  dscf    GAM2_DSCF and GAM3_DSCF, one direct-SCF Fock build
  fock    EG2IC1 and EG3IC1, one in-core Fock build, tensors in FP64 or FP32
  rxne    the closed-shell RXCHF-ne contractions in one pass over GM2 stored
          in FP64, FP32 or BF16
  xfock   one Fock build of a device-resident NEO-XCHF context
  inst    a whole small calculation: integrals and SCF of one instance of the
          proton scan

Everything lives in HBM before ``run``, as in a program that keeps its data
on the device.
"""
import itertools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "neo-rxchf_amd"))

import neorx  # noqa: E402
from neorx import synth, xchf  # noqa: E402

F64 = torch.float64
NSHELL = {"s": 1, "p": 3, "d": 6}
LSHELL = {"s": 0, "p": 1, "d": 2}


def listed():
    return [
        # the integral kernels on their own, over the benchmark's 60/16 system
        # and sampled as there: a slice of the e-p enumeration, and index
        # lists of the larger classes, one at the benchmark's own length
        dict(name="ep_range", kind="prim", cls=1, n=230401),
        dict(name="eep_list", kind="prim", cls=2, n=1 << 20),
        dict(name="eeep_list", kind="prim", cls=3, n=300007),
        # the e-e-p tensor of the 24/8 C-N-H system (36 contracted s/p
        # primitives): the ordinary integral build before an SCF
        dict(name="gam2_c1", kind="gam2", system="c1"),
        # the e-e-e-p tensor, the dominant cost of an XCHF calculation, over
        # contracted s/p shells on two centres
        dict(name="gam3_8", kind="gam3", centres=2, shells="sp", contract=2, pshells="sp", ngtg=3),
        # the RXCHF-ne tensor with d functions (24 electronic, 4 nuclear)
        dict(name="ne2_24", kind="ne2", centres=2, shells="ssspd", contract=1, pshells="sp", ngtg=3),
        # direct SCF at an odd, small size: integrals rebuilt per Fock build
        dict(name="dscf_7", kind="dscf", centres=1, shells="spp", contract=1, pshells="sp", ngtg=3),
        # in-core Fock builds: large and even in FP64, odd and ragged in FP32
        dict(name="fock_f64_20_8", kind="fock", ne=20, np=8, dtype=0),
        dict(name="fock_f32_17_5", kind="fock", ne=17, np=5, dtype=1),
        # RXCHF-ne contractions of the 48/12 system in mixed precision
        dict(name="rxne_bf16_48_12", kind="rxne", ne=48, np=12, dtype=2),
        # one Fock build inside a device-resident SCF, GAM_3 read in BF16
        dict(name="xfock_bf16_16", kind="xfock", centres=2, shells="sssssp", contract=1, pshells="sp", ngtg=3,
             nelec=10, prec="bf16"),
        # the smallest calls: one instance of the proton scan from its basis
        # to converged orbitals, where launches and latency count
        dict(name="inst_8_4", kind="inst", ne=8, np=4, mode="f64"),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["prim", "gam2", "gam3", "ne2", "dscf", "fock", "rxne", "xfock", "inst"])
    if kind == "prim":
        return dict(kind=kind, cls=rng.choice([1, 2, 3]), n=_logint(rng, 1, 900000))
    if kind == "fock":
        return dict(kind=kind, ne=rng.randint(3, 19), np=rng.randint(1, 8), dtype=rng.choice([0, 1]))
    if kind == "rxne":
        return dict(kind=kind, ne=rng.randint(3, 48), np=rng.randint(1, 12), dtype=rng.choice([0, 1, 2]))
    if kind == "inst":
        return dict(kind=kind, ne=rng.randint(5, 10), np=rng.choice([1, 4]), mode=rng.choice(["f64", "inc"]))
    # generated systems, no costlier than the listed ones
    while True:
        c = dict(kind=kind, centres=rng.choice([1, 2, 3]),
                 shells="".join(rng.choice("ssppd") for _ in range(rng.randint(1, 4))),
                 contract=rng.choice([1, 1, 2]), pshells=rng.choice(["s", "sp", "sd", "spd"]), ngtg=rng.choice([2, 3]))
        ne, pe, npb = _sizes(c)
        n2, n3 = pe ** 4 * npb ** 2, pe ** 6 * npb ** 2
        heavy = 4.0 if "d" in c["shells"] else 1.0
        if pe < 4 or pe > 36:
            continue
        if kind in ("gam2", "ne2") and heavy * n2 <= 4e7:
            return c
        if kind == "gam3" and heavy * n3 <= 2e8 and ne ** 6 * npb ** 2 <= 4e8:
            return c
        if kind == "dscf" and heavy * n3 <= 2e7:
            return c
        if kind == "xfock" and heavy * n3 <= 1e8:
            c.update(nelec=rng.choice([2, 4, 6]), prec=rng.choice(["f64", "f32", "bf16"]))
            if ne * 2 > c["nelec"]:
                return c


def _sizes(case):
    """(contracted functions, primitives, nuclear functions)"""
    if case.get("system") == "c1":
        return 24, 36, 8
    if case["kind"] == "prim":
        return 60, 60, 16
    if "ne" in case:
        return case["ne"], case["ne"], case["np"]
    ne = case["centres"] * sum(NSHELL[c] for c in case["shells"])
    return ne, ne * case["contract"], sum(NSHELL[c] for c in case["pshells"])


def _system(case, seed):
    if case["kind"] == "prim":
        return synth.config2(seed)
    if case.get("system") == "c1":
        return synth.config1(seed)
    if case["kind"] == "inst":  # the first instance of a scan with these basis sizes
        for s in itertools.count(seed):
            for k in range(64):
                d = synth.config5(k, 64, s)
                if (d["nebf"], d["npbf"]) == (case["ne"], case["np"]):
                    return d
    return synth.small(seed=seed, n_e_centres=case["centres"], e_shells=[LSHELL[c] for c in case["shells"]],
                       contract=(case["contract"],), p_shells=[LSHELL[c] for c in case["pshells"]],
                       ngtg=case["ngtg"])


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _dens(n, trace, seed):
    return _dev(synth.density(n, trace, seed).ravel(order="F"))


def _empty(n):
    return torch.empty(n, dtype=F64, device="cuda")


def _zeros(n):
    return torch.zeros(n, dtype=F64, device="cuda")


def _index_list(case, seed):
    """uniform tuples (ie1..ien, ip, je1..jen, jp) of the 60/16 system"""
    n, c = case["n"], case["cls"]
    rng = np.random.default_rng(seed + 17)
    return np.stack([rng.integers(0, 16 if k in (c, 2 * c + 1) else 60, n) for k in range(2 * c + 2)], axis=1)


def _tensor(n, dtype, gen):
    if dtype == 2:
        return torch.randn(n, dtype=torch.float32, device="cuda", generator=gen).to(torch.bfloat16)
    return torch.randn(n, dtype=torch.float32 if dtype else F64, device="cuda", generator=gen)


def prepare(case, seed):
    neorx.init(torch.cuda.current_device())
    kind = case["kind"]
    ne, pe, npb = _sizes(case)
    st = dict(case=case, ne=ne, np=npb)
    if kind in ("fock", "rxne"):
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        n2 = ne ** 4 * npb ** 2
        st["g2"] = _tensor(n2, case["dtype"], gen)
        if kind == "fock":
            st["g2s"] = _tensor(n2, case["dtype"], gen)
            st["g3"] = _tensor(n2 * ne * ne, case["dtype"], gen)
            st["de"], st["dp"] = _dens(ne, min(14.0, ne), seed + 1), _dens(npb, 1.0, seed + 2)
        else:
            st["dae"], st["dbe"], st["dp"] = _dens(ne, 20.0, seed + 1), _dens(ne, 2.0, seed + 2), _dens(npb, 1.0, seed + 3)
        return st
    st["sys"] = _system(case, seed)
    if kind == "inst":
        return st
    st["S"] = neorx.System(st["sys"])
    if kind == "prim" and case["cls"] > 1:
        st["idx"] = _dev(_index_list(case, seed))
    if kind in ("dscf", "xfock"):
        st["de"], st["dp"] = _dens(ne, float(case.get("nelec", min(4, ne))), seed + 1), _dens(npb, 1.0, seed + 2)
    if kind == "xfock":
        st["X"] = xchf.XCHF(st["S"], case["nelec"], store=("f64", case["prec"]))
    return st


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    ne, npb = state["ne"], state["np"]
    if kind == "prim":
        n, c = case["n"], case["cls"]
        e, s = _empty(n), _empty(n)
        if c == 1:
            state["S"].prim_range_dev(1, 0, n, e.data_ptr(), s.data_ptr())
        else:
            state["S"].prim_list_dev(c, n, state["idx"].data_ptr(), e.data_ptr(), s.data_ptr() if c == 2 else 0)
        return (e, s) if c < 3 else (e,)
    if kind in ("gam2", "ne2"):
        n2 = ne ** 4 * npb ** 2
        a, b = _empty(n2), _empty(n2)
        fn = "neorx_gam2_ic1_dev" if kind == "gam2" else "neorx_rxchfne_gam2_ic1_dev"
        neorx.call_dev(fn, state["S"].handle, a.data_ptr(), b.data_ptr(), 0)
        return a, b
    if kind == "gam3":
        a = _empty(ne ** 6 * npb ** 2)
        neorx.call_dev("neorx_gam3_ic1_dev", state["S"].handle, a.data_ptr(), 0)
        return (a,)
    if kind == "rxne":
        out = [_zeros(ne * ne), _zeros(npb * npb), _zeros(ne * ne), _zeros(1)]
        neorx.call_dev("neorx_rxchfne_omg2_dev", ne, npb, *[state[k].data_ptr() for k in ("dae", "dbe", "dp", "g2")],
                       case["dtype"], *[o.data_ptr() for o in out], 0)
        return out
    if kind == "xfock":
        fe, fp, comps = _empty(ne * ne), _empty(npb * npb), _empty(14)
        torch.cuda.current_stream().synchronize()  # the context has a stream of its own
        state["X"].fock_dev(state["de"].data_ptr(), state["dp"].data_ptr(), case["prec"], fe.data_ptr(), fp.data_ptr(),
                            comps.data_ptr(), torch.cuda.current_stream().cuda_stream)
        return fe, fp, comps
    if kind == "inst":
        s = state["sys"]
        S = neorx.System(s)
        X = xchf.XCHF(S, s["nelec"], store=("f64", "bf16") if case["mode"] == "inc" else ("f64",))
        r = X.scf(mode=case["mode"], diis=True, graph=True, maxit=100, tole=1e-6, tolp=1e-4, sw_hi=1e-3, sw_lo=1e-6)
        X.close()
        S.close()
        nocc = s["nelec"] // 2
        # orbitals have no fixed sign: the densities stand for them
        return dict(comps=np.array([r["comps"][k] for k in xchf.COMPS]), evE=r["evE"], evP=r["evP"],
                    DE=2.0 * r["CE"][:, :nocc] @ r["CE"][:, :nocc].T, DP=r["CP"][:, :1] @ r["CP"][:, :1].T)
    de, dp = state["de"].data_ptr(), state["dp"].data_ptr()
    fe, se, fp, sp, e2, e3 = (_zeros(n) for n in (ne * ne, ne * ne, npb * npb, npb * npb, 2, 1))
    if kind == "fock":
        sfx = "_f32_dev" if case["dtype"] else "_dev"
        neorx.call_dev("neorx_eg2ic1" + sfx, ne, npb, de, dp, state["g2"].data_ptr(), state["g2s"].data_ptr(),
                       fe.data_ptr(), se.data_ptr(), fp.data_ptr(), sp.data_ptr(), e2.data_ptr(), e2.data_ptr() + 8, 0)
        neorx.call_dev("neorx_eg3ic1" + sfx, ne, npb, de, dp, state["g3"].data_ptr(), fe.data_ptr(), fp.data_ptr(),
                       e3.data_ptr(), 0)
    else:
        h = state["S"].handle
        neorx.call_dev("neorx_gam2_dscf_dev", h, de, dp, fe.data_ptr(), fp.data_ptr(), se.data_ptr(), sp.data_ptr(),
                       e2.data_ptr(), e2.data_ptr() + 8, 0)
        neorx.call_dev("neorx_gam3_dscf_dev", h, de, dp, fe.data_ptr(), fp.data_ptr(), e3.data_ptr(), 0)
    return fe, se, fp, sp, e2, e3


# Operations of one primitive tuple at the benchmark system's angular momenta
# and four geminal terms (the host build's count), scaled by the geminal pairs.
_FLOPS = {1: 56734.0, 2: 113053.0, 3: 33681.0, 4: 40000.0}


def _tuple_flops(cls, ngtg):
    return _FLOPS[cls] * (ngtg * (ngtg + 1)) / 20.0


def work(case):
    """Bytes and operations of one pass.  Integrals over real functions do not
    change when a particle's bra and ket primitive are exchanged (for e-e-p
    after the average over the electrons), so a builder cannot do without one
    evaluation per distinct set of primitive pairs, and no more."""
    kind = case["kind"]
    ne, pe, npb = _sizes(case)
    ng = {"c1": 3}.get(case.get("system"), case.get("ngtg", 3))
    tri = lambda n: n * (n + 1) // 2  # noqa: E731
    n2, n3 = ne ** 4 * npb ** 2, ne ** 6 * npb ** 2
    if kind == "prim":
        c = case["cls"]
        return dict(bytes=case["n"] * (8 * (2 if c < 3 else 1) + (16 * (c + 1) if c > 1 else 0)),
                    flops=case["n"] * _tuple_flops(c, 4))
    if kind in ("gam2", "ne2"):
        return dict(bytes=16 * n2, flops=tri(pe) ** 2 * tri(npb) * _tuple_flops(2 if kind == "gam2" else 4, ng))
    if kind == "gam3":
        return dict(bytes=8 * n3, flops=tri(pe) ** 3 * tri(npb) * _tuple_flops(3, ng))
    if kind == "dscf":
        return dict(bytes=8 * (4 * ne * ne + 4 * npb * npb),
                    flops=tri(pe) ** 2 * tri(npb) * _tuple_flops(2, ng) + tri(pe) ** 3 * tri(npb) * _tuple_flops(3, ng))
    if kind == "fock":
        return dict(bytes=(8, 4)[case["dtype"]] * (2 * n2 + n3), flops=8 * n2 + 6 * n3)
    if kind == "rxne":
        return dict(bytes=(8, 4, 2)[case["dtype"]] * n2, flops=4 * n2)
    if kind == "xfock":  # the tensors of the context are symmetric in every index pair
        return dict(bytes={"f64": 8, "f32": 4, "bf16": 2}[case["prec"]] * tri(ne) ** 3 * tri(npb) +
                    16 * tri(ne) ** 2 * tri(npb), flops=6 * tri(ne) ** 3 * tri(npb) + 4 * ne ** 5 * 6)
    return dict(bytes=8 * (tri(ne) ** 3 * tri(npb) + 2 * tri(ne) ** 2 * tri(npb)),
                flops=tri(ne) ** 3 * tri(npb) * _tuple_flops(3, 3) + tri(ne) ** 2 * tri(npb) * _tuple_flops(2, 3))


def tolerance(case):
    """Integrals and FP64 contractions differ from the 64-bit values of
    ``exact`` by up to 3e-14 over the listed cases; combinations that cancel
    (E1 of RXCHF-ne, energies over random tensors) reach further in others.
    FP32 sums over BF16 storage differ by 1e-7."""
    kind = case["kind"]
    if kind == "rxne":
        return {"rel": 1e-12 if case["dtype"] < 2 else 1e-6}
    if kind == "xfock":
        return {"rel": 1e-6 if case["prec"] == "bf16" else 1e-11}
    if kind == "inst":  # rounding travels through the iterations; in "inc", up to the convergence thresholds
        return {"rel": 1e-8 if case["mode"] == "f64" else 1e-5}
    return {"rel": 1e-12}


# ----------------------------------------------------------------------
# reference values in plain torch, 64 bits
# ----------------------------------------------------------------------
# Every integral is one Gaussian average.  The bra-ket products and geminals
# of a star of particles (all linked to the last one) are a Gaussian in all
# coordinates; 1/r = 2/sqrt(pi) int exp(-t^2 r^2) dt keeps it one at each node
# u of the quadrature of the Boys integral, and the polynomials are averaged
# over it by the recursion <x_i P> = m_i <P> + sum_j C_ij <dP/dx_j>.  For an
# argument T > 20 the Boys integral runs to infinity, as the reference
# program's asymptotic formula does.
_GL = np.polynomial.legendre.leggauss(24)
_GH = np.polynomial.hermite.hermgauss(40)
_PI_G2 = 3.141592650  # the reference's pi in the e-p kinetic integrals


def _pairs(ex, cen, am, coef):
    """every (bra, ket) pair of a primitive set, flattened"""
    a, A, l = _dev(ex), _dev(np.asarray(cen)), _dev(np.asarray(am))
    n = a.numel()
    i, j = (x.reshape(-1) for x in torch.meshgrid(torch.arange(n).cuda(), torch.arange(n).cuda(), indexing="ij"))
    p = a[i] + a[j]
    P = (a[i, None] * A[i] + a[j, None] * A[j]) / p[:, None]
    return dict(p=p, P=P, K=torch.exp(-a[i] * a[j] / p * ((A[i] - A[j]) ** 2).sum(1)), beta=a[j], B=A[j], sA=P - A[i],
                sB=P - A[j], la=l[i], lb=l[j], deg=(l[i] + l[j]).max(1).values, c=_dev(coef)[i] * _dev(coef)[j], n=n)


def _take(q, k):
    return {x: v[k] for x, v in q.items() if x != "n"}


def _mul(a, b):
    out = a.new_zeros(torch.broadcast_shapes(a.shape[:-1], b.shape[:-1]) + (a.shape[-1] + b.shape[-1] - 1,))
    for i in range(a.shape[-1]):
        out[..., i:i + b.shape[-1]] += a[..., i:i + 1] * b
    return out


def _padd(a, b):
    n = max(a.shape[-1], b.shape[-1])
    return torch.nn.functional.pad(a, (0, n - a.shape[-1])) + torch.nn.functional.pad(b, (0, n - b.shape[-1]))


def _power(s, l, lmax):
    """(y + s)^l, coefficients [3, B, lmax + 1]; s, l are [B, 3]"""
    s, l = s.T[..., None], l.T[..., None]
    out = torch.cat([torch.ones_like(s), torch.zeros_like(s).expand(*s.shape[:2], lmax)], -1)
    for i in range(lmax):
        up = s * out
        up[..., 1:] += out[..., :-1]
        out = torch.where(l > i, up, out)
    return out


def _poly(q):
    la, lb = int(q["la"].max()), int(q["lb"].max())
    return _mul(_power(q["sA"], q["la"], la), _power(q["sB"], q["lb"], lb))[..., :int(q["deg"].max()) + 1]


def _moment(f, mean, cov):
    """average of prod_i f_i(y_i): f_i [3, B, K_i] against mean [3, B, L, U],
    cov [B, L, U]"""
    n = len(f)
    M, total = {}, 0.0
    for k in itertools.product(*[range(x.shape[-1]) for x in f]):
        i = next((i for i in range(n) if k[i]), None)
        if i is None:
            M[k] = torch.ones_like(mean[0])
        else:
            low = k[:i] + (k[i] - 1,) + k[i + 1:]
            v = mean[i] * M[low]
            for j in range(n):
                if low[j]:
                    v = v + low[j] * cov[i][j] * M[low[:j] + (low[j] - 1,) + low[j + 1:]]
            M[k] = v
        w = f[0][..., k[0]]
        for i in range(1, n):
            w = w * f[i][..., k[i]]
        total = total + w[..., None, None] * M[k]
    return total


class _Star:
    """particles q (the last one the hub), leaf i linked by exponents g[i] [L]"""

    def __init__(self, q, g):
        self.q, n = q, len(q)
        hub = q[-1]
        d = [(x["P"] - hub["P"]).T[..., None] for x in q]
        w, c, E0, W, beta = hub["p"][:, None], torch.zeros_like(d[0]), 0.0, [], []
        for i in range(n - 1):
            p = q[i]["p"][:, None]
            Wi = p + g[i]
            kap = p * g[i] / Wi
            E0 = E0 + w * kap / (w + kap) * ((c - d[i]) ** 2).sum(0)
            c = (w * c + kap * d[i]) / (w + kap)
            w = w + kap
            W.append(Wi)
            beta.append(g[i] / Wi)
        self.pre = torch.exp(-E0 + torch.zeros_like(w)) * (math.pi ** n / (math.prod(W, start=w))) ** 1.5
        for x in q:
            self.pre = self.pre * x["K"][:, None]
        beta.append(torch.ones_like(w))
        self.mean = [beta[i] * (c - d[i]) for i in range(n)]
        self.cov = [[beta[i] * beta[j] / (2 * w) + (1 / (2 * W[i]) if i == j < n - 1 else 0.0) for j in range(n)]
                    for i in range(n)]
        self.f = [_poly(x) for x in q]

    def _avg(self, f):
        return _moment(f, [m[..., None] for m in self.mean], [[c[..., None] for c in r] for r in self.cov])[..., 0]

    def ovl(self):
        return self.pre * self._avg(self.f).prod(0)

    def _boys(self, Cv, s2, D):
        T = (D ** 2).sum(0) / (2 * s2)
        far = (T > 20.0)[..., None]
        t = T[..., None]
        xl, wl = _dev(0.5 * (_GL[0] + 1)), _dev(0.5 * _GL[1])
        keep = _GH[0] > 0
        xh, wh = _dev(_GH[0][keep]), _dev(_GH[1][keep])
        pad = xl.numel() - xh.numel()
        xh, wh = (torch.nn.functional.pad(v, (0, pad)) for v in (xh, wh))
        rt = torch.sqrt(torch.where(far, t, torch.ones_like(t)))
        u2 = torch.where(far, xh / rt, xl) ** 2
        wt = torch.where(far, wh / rt, wl * torch.exp(-torch.where(far, torch.zeros_like(t), t) * xl * xl))
        n = len(self.q)
        mean = [self.mean[i][..., None] - u2 * (Cv[i] / s2 * D)[..., None] for i in range(n)]
        cov = [[self.cov[i][j][..., None] - u2 * (Cv[i] * Cv[j] / s2)[..., None] for j in range(n)] for i in range(n)]
        return self.pre * torch.sqrt(2 / (math.pi * s2)) * (wt * _moment(self.f, mean, cov).prod(0)).sum(-1)

    def coul(self, a, b):
        Cv = [r[a] - r[b] for r in self.cov]
        D = (self.q[a]["P"] - self.q[b]["P"]).T[..., None] + self.mean[a] - self.mean[b]
        return self._boys(Cv, Cv[a] - Cv[b], D)

    def nuc(self, a, s):
        Cv = [r[a] for r in self.cov]
        tot = 0.0
        for z, x in zip(s["zan"], np.asarray(s["cat"]).reshape(-1, 3)):
            D = self.q[a]["P"].T[..., None] + self.mean[a] - _dev(x)[:, None, None]
            tot = tot + float(z) * self._boys(Cv, Cv[a], D)
        return tot

    def kin(self, a, c, g, mass):
        """-1/(2 mass) <bra| d^2/dx_a^2 |ket exp(-g r_ac^2)>, g [L] or None"""
        A = self.q[a]
        out = 0.0
        S = self._avg(self.f)
        L = A["lb"].T[..., None].to(F64)
        lmax = int(A["lb"].max())
        be = A["beta"][:, None]
        bra = _power(A["sA"], A["la"], int(A["la"].max()))
        X = _power(A["sB"], A["lb"], lmax)
        X1 = _power(A["sB"], (A["lb"] - 1).clamp(min=0), lmax)
        X2 = _power(A["sB"], (A["lb"] - 2).clamp(min=0), lmax)
        one = torch.stack([A["sB"].T, torch.ones_like(A["sB"].T)], -1)  # X
        Ls = self.mean[a].shape[-1]
        for l in range(Ls):  # the polynomials depend on the geminal exponent
            gl = 0.0 if g is None else float(g[l])
            star = [[c_[:, l:l + 1, None] for c_ in r] for r in self.cov]
            mean = [m[..., l:l + 1, None] for m in self.mean]
            avg = lambda f: _moment(f, mean, star)[..., 0, 0]  # noqa: E731
            P0 = _padd(_padd(L * (L - 1) * X2, (-4 * be * L - 2 * (be + gl)) * X), 4 * be * be * _mul(X, _mul(one, one)))
            f = list(self.f)
            f[a] = _mul(bra, P0)
            T = avg(f)
            if gl:
                P1 = _mul(bra, _padd(-4 * gl * L * X1, 8 * be * gl * _mul(X, one)))
                P2 = _mul(bra, 4 * gl * gl * X)
                dl = (A["P"] - self.q[c]["P"]).T
                shift = torch.stack([dl, torch.ones_like(dl)], -1)
                fc = self.f[c]
                y = torch.nn.functional.pad(fc, (1, 0))
                for pa, pc in ((_padd(_mul(P1, shift), _mul(P2, _mul(shift, shift))), fc),
                               (-_padd(P1, 2 * _mul(P2, shift)), y), (P2, torch.nn.functional.pad(y, (1, 0)))):
                    f[a], f[c] = pa, pc
                    T = T + avg(f)
            s = S[..., l]
            v = T[0] * s[1] * s[2] + s[0] * T[1] * s[2] + s[0] * s[1] * T[2]
            col = (-0.5 / mass * self.pre[:, l] * v)[:, None]
            out = col if l == 0 else torch.cat([out, col], 1)
        return out


def _values(cls, s, q):
    """(E, S) of tuples with pairs q = electrons..., proton"""
    b, g = _dev(s["bcoef"]), _dev(s["gamma"])
    n = b.numel()
    k, l = (x.reshape(-1) for x in torch.meshgrid(torch.arange(n).cuda(), torch.arange(n).cuda(), indexing="ij"))
    bb, gk, gl, z1, z2 = b[k] * b[l], g[k], g[l], torch.zeros_like(g), torch.zeros(n * n, dtype=F64, device="cuda")
    none = torch.zeros(1, dtype=F64, device="cuda")
    if cls == 1:
        fac = (_PI_G2 / math.pi) ** 3
        x, xx = _Star(q, [g]), _Star(q, [gk + gl])
        m = s["pmass"]
        t = (x.kin(0, 1, None, 1.0) + x.kin(0, 1, g, 1.0) + x.kin(1, 0, None, m) + x.kin(1, 0, g, m)) @ b
        t = fac * (t + (xx.kin(0, 1, gl, 1.0) + xx.kin(1, 0, gl, m)) @ bb)
        v = lambda y, w: (y.nuc(1, s) - y.nuc(0, s) - y.coul(0, 1)) @ w  # noqa: E731
        return t + 2 * v(x, b) + v(xx, bb), 2 * (x.ovl() @ b) + xx.ovl() @ bb
    if cls == 2:
        one = _Star(q[:1], [])
        h1 = one.kin(0, -1, None, 1.0)[:, 0] - one.nuc(0, s)[:, 0]
        ov = lambda gg, w: _Star(q[1:], [gg]).ovl() @ w  # noqa: E731
        x, x2, xs = _Star(q, [z1, g]), _Star(q, [z2, gk + gl]), _Star(q, [gk, gl])
        E = 2 * (h1 * ov(g, b) + (x.coul(0, 1) - x.coul(0, 2)) @ b) + h1 * ov(gk + gl, bb) - x2.coul(0, 2) @ bb
        x1 = _Star(q, [gk + gl, z2])
        E = E + (xs.kin(2, 1, gl, s["pmass"]) + xs.nuc(2, s) + xs.kin(0, 2, None, 1.0) + xs.kin(0, 2, gk, 1.0) -
                 2 * (xs.nuc(0, s) + xs.coul(0, 2)) + xs.coul(0, 1) + x1.coul(0, 1)) @ bb
        return E, xs.ovl() @ bb
    if cls == 4:
        x, xs = _Star(q, [gk + gl, z2]), _Star(q, [gk, gl])
        return (x.coul(0, 1) - x.coul(1, 2)) @ bb, xs.coul(0, 1) @ bb
    e3 = _Star(q[2:3], [])
    h3 = e3.kin(0, -1, None, 1.0)[:, 0] - e3.nuc(0, s)[:, 0]
    v23 = _Star(q[1:3], [none]).coul(0, 1)[:, 0]
    ep = [q[0], q[3]]
    E = v23 * (_Star(ep, [g]).ovl() @ b + 0.5 * (_Star(ep, [gk + gl]).ovl() @ bb))
    E = E + h3 * (_Star([q[0], q[1], q[3]], [gk, gl]).ovl() @ bb)
    return E - _Star(q, [gk, gl, z2]).coul(2, 3) @ bb + 2 * (_Star(q, [gk, z2, gl]).coul(0, 1) @ bb), None


def _evaluate(cls, s, ep, pp, ie, ip):
    """tuples of electron pairs ie (list of index tensors) and proton pairs ip,
    grouped by the degrees of their polynomials"""
    ng = len(s["gamma"]) ** 2
    E, S = torch.empty(ip.numel(), dtype=F64, device="cuda"), torch.empty(ip.numel(), dtype=F64, device="cuda")
    key = pp["deg"][ip]
    for i in ie:
        key = key * 8 + ep["deg"][i]
    for v in torch.unique(key).tolist():
        sel = torch.nonzero(key == v)[:, 0]
        dims, r = 1, v
        for _ in range(len(ie) + 1):
            dims, r = dims * (r % 8 + 1), r // 8
        step = max(1, int(1.5e8 / (72 * ng * (dims + 4))))
        for o in range(0, sel.numel(), step):
            t = sel[o:o + step]
            e, x = _values(cls, s, [_take(ep, i[t]) for i in ie] + [_take(pp, ip[t])])
            E[t] = e
            if x is not None:
                S[t] = x
    return E, S


def _tables(s):
    return (_pairs(s["elcex"], s["elcbfc"], s["elcam"], s["agebfcc"]),
            _pairs(s["nucex"], s["nucbfc"], s["nucam"], s["agnbfcc"]))


def _contracted(cls, s):
    """unsymmetrised contracted tensors [pp][pair]..[pair]"""
    ep, pp = _tables(s)
    nel = 3 if cls == 3 else 2
    ne2, np2, pe2 = s["nebf"] ** 2, s["npbf"] ** 2, s["npebf"] ** 2
    a = _dev(s["ampeb2c"]) - 1
    cpair = (a[:, None] * s["nebf"] + a[None, :]).reshape(-1)
    outs = [torch.zeros(np2 * ne2 ** nel, dtype=F64, device="cuda") for _ in range(2)]
    total, step = np2 * pe2 ** nel, 1 << 20
    for o in range(0, total, step):
        t = torch.arange(o, min(total, o + step), device="cuda")
        ie = []
        for _ in range(nel):
            ie.insert(0, t % pe2)
            t = t // pe2
        E, S = _evaluate(cls, s, ep, pp, ie, t)
        cf, at = pp["c"][t], t
        for i in ie:
            cf, at = cf * ep["c"][i], at * ne2 + cpair[i]
        outs[0].index_add_(0, at, E * cf)
        if cls != 3:
            outs[1].index_add_(0, at, S * cf)
    return [o.view(np2, *[ne2] * nel) for o in outs]


def _gm2(s):
    return [0.5 * (x + x.transpose(1, 2)) for x in _contracted(2, s)]


def _gm3(s):
    x = _contracted(3, s)[0]
    return sum(x.permute(0, *[i + 1 for i in p]) for p in itertools.permutations(range(3))) / 6.0


def _fock(ne, npb, de, dp, g2, g2s, g3):
    """EG2IC1 + EG3IC1; the tensors may be given one (ip,jp) block at a time"""
    D, ne2 = de.view(ne, ne).T, ne * ne
    FE, SE = torch.zeros_like(D), torch.zeros_like(D)
    FP, SP = _zeros(npb * npb), _zeros(npb * npb)
    E2, E3 = _zeros(2), _zeros(1)
    out = lambda x, y, u, v: torch.einsum(x + "," + y + "->" + u, *v)  # noqa: E731
    wb = out("cd", "ef", "cdef", (D, D)) - 0.5 * out("cf", "ed", "cdef", (D, D))
    wd = -0.5 * out("cb", "ef", "bcef", (D, D)) + 0.25 * out("cf", "eb", "bcef", (D, D))
    wf = 0.25 * out("cb", "ed", "bcde", (D, D)) - 0.5 * out("cd", "eb", "bcde", (D, D))
    for ip, jp in itertools.product(range(npb), range(npb)):
        pp, w = ip * npb + jp, dp[jp * npb + ip]
        for k, t in enumerate((g2, g2s)):
            g = t[pp * ne2 * ne2:(pp + 1) * ne2 * ne2].to(F64).view(ne, ne, ne, ne)
            f = (g.reshape(ne2, ne2) @ D.reshape(-1)).view(ne, ne)
            f = f - 0.5 * (g.permute(0, 3, 1, 2).reshape(ne2, ne2) @ D.T.reshape(-1)).view(ne, ne)
            e = (D * f).sum()
            if k == 0:
                FE += 2 * w * f
                FP[jp * npb + ip] += e
            else:
                SE += w * f
                SP[jp * npb + ip] += e
            E2[k] += w * e
        n6 = ne2 ** 3
        g = g3[pp * n6:(pp + 1) * n6].to(F64).view(*[ne] * 6)
        f = (g.reshape(ne2, -1) @ wb.reshape(-1)).view(ne, ne)
        f = f + (g.permute(0, 3, 1, 2, 4, 5).reshape(ne2, -1) @ wd.reshape(-1)).view(ne, ne)
        f = 3 * (f + (g.permute(0, 5, 1, 2, 3, 4).reshape(ne2, -1) @ wf.reshape(-1)).view(ne, ne))
        e = (D * f).sum() / 3
        FE += w * f
        FP[jp * npb + ip] += e
        E3 += w * e
    return FE.T.reshape(-1), SE.T.reshape(-1), FP, SP, E2, E3


def exact(case, seed):
    kind = case["kind"]
    ne, pe, npb = _sizes(case)
    if kind in ("xfock", "inst"):
        return None
    if kind == "rxne":
        st = prepare(case, seed)
        A, B = (st[k].view(ne, ne).T.reshape(-1) for k in ("dae", "dbe"))
        P = st["dp"].view(npb, npb)
        fa, fb, fp = _zeros(ne * ne), _zeros(ne * ne), torch.zeros_like(P)
        for ip, jp in itertools.product(range(npb), range(npb)):
            o = (ip * npb + jp) * ne ** 4
            g = st["g2"][o:o + ne ** 4].to(F64).view(ne * ne, ne * ne)
            r = g @ A
            fa += P[jp, ip] * (B @ g)
            fb += P[jp, ip] * r
            fp[jp, ip] = (B * r).sum()
        t = lambda f: f.view(ne, ne).T.reshape(-1)  # noqa: E731
        return [t(fa), fp.reshape(-1), t(fb), (P * fp).sum().reshape(1)]
    if kind == "fock":
        st = prepare(case, seed)
        return _fock(ne, npb, st["de"], st["dp"], st["g2"], st["g2s"], st["g3"])
    s = _system(case, seed)
    d = 1.0 + ("d" in case.get("shells", ""))
    n2, n3 = pe ** 4 * npb ** 2, pe ** 6 * npb ** 2
    if kind == "prim":
        ep, pp = _tables(s)
        c, n = case["cls"], case["n"]
        if n > (900000, 130000, 800000)[c - 1]:
            return None
        if c == 1:  # sorted order: the order of neorx_prim_range_dev's enumeration
            h = neorx.System(s)
            eo, po = (_dev(x) for x in h.order())
            h.close()
            r = torch.arange(n, device="cuda")
            i, j = eo[(r // 60) % 60], eo[r % 60]
            ie, ip = [i * 60 + j], po[r // (3600 * 16)] * 16 + po[(r // 3600) % 16]
        else:
            x = _dev(_index_list(case, seed))
            ie, ip = [x[:, k] * 60 + x[:, c + 1 + k] for k in range(c)], x[:, c] * 16 + x[:, 2 * c + 1]
        e, o = _evaluate(c, s, ep, pp, ie, ip)
        return (e, o) if c < 3 else (e,)
    if kind == "gam2":
        return None if d * n2 > 3e6 else tuple(x.reshape(-1) for x in _gm2(s))
    if kind == "ne2":
        if d * n2 > 2e7:
            return None
        a, b = _contracted(4, s)
        return a.reshape(-1), (0.5 * (b + b.transpose(1, 2))).reshape(-1)
    if d * n3 > 2e7:
        return None
    if kind == "gam3":
        return (_gm3(s).reshape(-1),)
    g2, g2s = (x.reshape(-1) for x in _gm2(s))
    return _fock(ne, npb, _dens(ne, float(min(4, ne)), seed + 1), _dens(npb, 1.0, seed + 2), g2, g2s,
                 _gm3(s).reshape(-1))
