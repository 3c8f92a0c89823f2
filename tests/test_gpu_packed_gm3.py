"""The GM3 pass of a device-resident NEO-XCHF context, which holds GAM_3 over
distinct nuclear pairs and distinct third-electron pairs: against EG3IC1 over
the full tensor of the same system, for basis sizes with an odd and an even
number of packed columns (two BF16 columns per load where it is even), with
one block per slab and with slabs split over columns and over the second
index, and with more columns than a block has lanes."""
import numpy as np
import pytest

import neorx
from neorx import synth, xchf

pytestmark = pytest.mark.gpu

CASES = [dict(n_e_centres=1, e_shells=(0, 0), p_shells=(0,)),       # 2 functions, 3 columns
         dict(n_e_centres=1, e_shells=(0, 1), p_shells=(0, 1, 2)),  # 4, 10 columns, 55 nuclear pairs
         dict(n_e_centres=1, e_shells=(0, 0, 1), p_shells=(0, 1)),  # 5, 15
         dict(n_e_centres=2, e_shells=(0, 1), p_shells=(0, 1)),     # 8, 36
         dict(n_e_centres=1, e_shells=(0, 0, 0, 2), p_shells=(0,)),  # 9, 45
         dict(n_e_centres=3, e_shells=(0, 0, 1), p_shells=(0,))]    # 15, 120: several wavefronts a block


@pytest.mark.parametrize("kw", CASES, ids=["2", "4", "5", "8", "9", "15"])
def test_packed_gm3(kw):
    import torch

    torch.cuda.init()
    neorx.init(0)
    s = synth.small(seed=91, contract=(1, 1), ngtg=2, **kw)
    s["nelec"] = 4
    ne, npb = s["nebf"], s["npbf"]
    print(f"case packed gm3 nebf={ne} npbf={npb}", flush=True)
    S = neorx.System(s)
    G = torch.zeros(ne ** 6 * npb ** 2, dtype=torch.float64, device="cuda")
    neorx.call_dev("neorx_gam3_ic1_dev", S.handle, G.data_ptr(), 0)
    fe = torch.zeros(ne * ne, dtype=torch.float64, device="cuda")
    fp = torch.zeros(npb * npb, dtype=torch.float64, device="cuda")
    c = torch.zeros(14, dtype=torch.float64, device="cuda")
    o = [torch.zeros(n, dtype=torch.float64, device="cuda") for n in (ne * ne, npb * npb, 1)]
    g32 = G.float()
    ref = {"f64": G, "f32": g32.double(), "bf16": g32.bfloat16().double()}
    rng = np.random.default_rng(ne)
    # the energy over densities without symmetry fixes the weight and the place
    # of every row of F, which it is the trace of
    D = []
    for k in range(3):
        DE = synth.density(ne, 3.0, 5 + k) + 0.2 * rng.standard_normal((ne, ne))
        DP = synth.density(npb, 1.0, 6 + k) + 0.2 * rng.standard_normal((npb, npb))
        D.append((DE, DP, *(torch.from_numpy(np.ascontiguousarray(m.ravel(order="F"))).cuda() for m in (DE, DP))))
    for tuned in (False, True):
        X = xchf.XCHF(S, 4, store=("f64", "f32", "bf16"), autotune=tuned)
        for prec in ("f64", "f32", "bf16"):
            for DE, DP, de, dp in D:
                X.fock_dev(de.data_ptr(), dp.data_ptr(), prec, fe.data_ptr(), fp.data_ptr(), c.data_ptr())
                neorx.call_dev("neorx_eg3ic1_dev", ne, npb, de.data_ptr(), dp.data_ptr(), ref[prec].data_ptr(),
                               *[x.data_ptr() for x in o], 0)
                torch.cuda.synchronize()
                got, want = float(c[8]), float(o[2][0])
                # the energy's terms add weights 1 + 3/2 + 2/4 times an entry and three
                # densities: FP64 sums to 1e-13 of that; BF16 entries are summed in FP32
                # over nebf products with an FP32 density, to (nebf + 2) 2^-24
                mag = 3.0 * float(G.abs().max()) * np.abs(DE).sum() ** 3 * np.abs(DP).sum()
                bar = mag * (1e-13 if prec != "bf16" else (ne + 2) * 2.0 ** -24)
                assert abs(got - want) <= bar, (prec, tuned, got, want, bar)
        X.close()
    S.close()


def absolute_rows(torch, g, DE, DP):
    """sum of the absolute terms of every element of EG3IC1's FE (column-major)"""
    ne, npb = DE.shape[0], DP.shape[0]
    a = (g.abs().reshape(npb * npb, -1) * DP.abs().reshape(-1, 1)).sum(0).reshape([ne] * 6)
    d = DE.abs()
    t = lambda spec: torch.einsum(spec, a, d, d)  # noqa: E731
    rows = 3.0 * (t("abcdef,cd,ef->ab") + 0.5 * t("abcdef,cf,ed->ab") + 0.5 * t("abcdef,cb,ef->ad") +
                  0.25 * t("abcdef,cf,eb->ad") + 0.25 * t("abcdef,cb,ed->af") + 0.5 * t("abcdef,cd,eb->af"))
    return rows.T.reshape(-1)


@pytest.mark.parametrize("kw", CASES, ids=["2", "4", "5", "8", "9", "15"])
def test_packed_gm3_matrices(kw):
    """The rows of the pass in FE and FP: builds of one context that differ in
    the GM3 pass only (storage, full or increment) have F = f / S - H SE with
    the same S and SE, so S dF + S dH SE is the difference of their EG3 parts,
    which EG3IC1 gives over the full tensors."""
    import torch

    torch.cuda.init()
    neorx.init(0)
    s = synth.small(seed=91, contract=(1, 1), ngtg=2, **kw)
    s["nelec"] = 4
    ne, npb = s["nebf"], s["npbf"]
    print(f"case packed gm3 matrices nebf={ne} npbf={npb}", flush=True)
    zeros = lambda *n: [torch.zeros(k, dtype=torch.float64, device="cuda") for k in n]  # noqa: E731
    col = lambda m: torch.from_numpy(np.ascontiguousarray(m.ravel(order="F"))).cuda()  # noqa: E731
    S = neorx.System(s)
    G = torch.zeros(ne ** 6 * npb ** 2, dtype=torch.float64, device="cuda")
    neorx.call_dev("neorx_gam3_ic1_dev", S.handle, G.data_ptr(), 0)
    g32 = G.float()
    ref = {"f64": G, "f32": g32.double(), "bf16": g32.bfloat16().double()}
    rng = np.random.default_rng(ne + 40)
    D0, D1 = (synth.density(ne, 3.0, k) + 0.2 * rng.standard_normal((ne, ne)) for k in (5, 6))
    DP = synth.density(npb, 1.0, 7) + 0.2 * rng.standard_normal((npb, npb))
    d0, d1, dp = col(D0), col(D1), col(DP)

    def eg3(de, t):
        o = zeros(ne * ne, npb * npb, 1)
        neorx.call_dev("neorx_eg3ic1_dev", ne, npb, de.data_ptr(), dp.data_ptr(), t.data_ptr(),
                       *[x.data_ptr() for x in o], 0)
        torch.cuda.synchronize()
        return o

    # SE and SP of the overlap: se1 + 2 se2 and sp1 + sp2
    n2 = ne ** 4 * npb ** 2
    g2, g2s = zeros(n2, n2)
    neorx.call_dev("neorx_gam2_ic1_dev", S.handle, g2.data_ptr(), g2s.data_ptr(), 0)
    o = zeros(ne * ne, ne * ne, npb * npb, npb * npb, 1, 1)
    neorx.call_dev("neorx_eg2ic1_dev", ne, npb, d1.data_ptr(), dp.data_ptr(), g2.data_ptr(), g2s.data_ptr(),
                   *[x.data_ptr() for x in o], 0)
    torch.cuda.synchronize()
    g1s = np.asarray(S.GAM1()[1]).reshape(npb, npb, ne, ne)
    SE = col(np.einsum("pq,pqab->ab", DP, g1s)) + 2.0 * o[1]
    SP = col(np.einsum("ab,pqab->pq", D1, g1s)) + o[3]
    mag = absolute_rows(torch, G, torch.from_numpy(np.abs(D0) + np.abs(D1)).cuda(), torch.from_numpy(DP).cuda())
    full = eg3(d1, G)
    X = xchf.XCHF(S, 4, store=("f64", "f32", "bf16"))

    def fock(de, prec, g3pass=0):
        o = zeros(ne * ne, npb * npb, 14)
        X.fock_dev(de.data_ptr(), dp.data_ptr(), prec, *[x.data_ptr() for x in o], g3pass=g3pass)
        torch.cuda.synchronize()
        return o

    base = fock(d1, "f64")
    for prec in ("f32", "bf16"):
        got = fock(d1, prec)
        w = eg3(d1, ref[prec])
        Sov, dH = float(got[2][10]), float(got[2][13] - base[2][13])
        # the sums of the pass (FP64 to 1e-13 of their absolute terms, BF16 in
        # FP32) and the rounding of the matrices that are subtracted
        bar = mag * (1e-13 if prec == "f32" else (ne + 2) * 2.0 ** -24) + 1e-14 * abs(Sov) * base[0].abs().max()
        want = w[0] - full[0]
        err = (Sov * (got[0] - base[0]) + Sov * dH * SE - want).abs()
        assert (err <= bar).all(), (prec, "FE", float((err / bar).max()))
        assert float(bar.max()) < 0.5 * float(want.abs().max()), (prec, "bar")
        want = w[1] - full[1]
        err = (Sov * (got[1] - base[1]) + Sov * dH * SP - want).abs()
        # FP(p) = sum D F / 3, its nuclear weight left out
        barp = float((bar * (d1.abs() + d0.abs())).sum()) / 3.0 / np.abs(DP).min() + 1e-14 * abs(Sov) * base[1].abs().max()
        assert (err <= barp).all(), (prec, "FP")
    for prec in ("f64", "f32", "bf16"):
        fock(d0, "f64", 1)
        got = fock(d1, prec, 2)
        Sov, dH = float(got[2][10]), float(got[2][13] - base[2][13])
        # the reference rows and T(D1 - D0, D1 + D0) = Q(D1) - Q(D0)
        part = eg3(d0, G)[0] + eg3(d1, ref[prec])[0] - eg3(d0, ref[prec])[0]
        bar = 2.0 * mag * (1e-13 if prec != "bf16" else (ne + 2) * 2.0 ** -24) + 1e-14 * abs(Sov) * base[0].abs().max()
        err = (Sov * (got[0] - base[0]) + Sov * dH * SE - (part - full[0])).abs()
        assert (err <= bar).all(), (prec, "increment FE", float((err / bar).max()))
        assert float(bar.max()) < 0.05 * float(part.abs().max()), (prec, "bar")
        e = float((part * d1).sum()) / 3.0
        assert abs(float(got[2][8]) - e) <= float((bar * d1.abs()).sum()) / 3.0, (prec, "increment energy")
    X.close()
    S.close()
