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
