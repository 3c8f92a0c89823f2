"""EG3IC1 at basis sizes whose rows end in every kind of load batch (one batch
shorter than the depth, whole batches and a rest) and whose slab counts are
split over the second index, against the oracle; the allocation-free form
bit for bit."""
import numpy as np
import pytest

import neorx
import oracle
from neorx import synth
from _util import check_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ne,npb", [(1, 1), (2, 3), (7, 1), (9, 2), (13, 1), (17, 1), (21, 1),
                                    # 2400, 7938 and 8192 slabs: split into four, two and one
                                    (6, 20), (2, 63), (2, 64)])
def test_eg3_batches(ne, npb):
    import torch

    torch.cuda.init()
    neorx.init(0)
    print(f"case eg3 batches ne={ne} np={npb}", flush=True)
    rng = np.random.default_rng(ne * 10 + npb)
    DE, DP = synth.density(ne, 1.0 + ne // 2, ne), synth.density(npb, 1.0, 3)
    g = torch.from_numpy(rng.standard_normal(ne ** 6 * npb * npb)).cuda()
    de, dp = (torch.from_numpy(np.ascontiguousarray(m.ravel(order="F"))).cuda() for m in (DE, DP))

    def run(name, t):
        o = [torch.zeros(n, dtype=torch.float64, device="cuda") for n in (ne * ne, npb * npb, 1)]
        neorx.call_dev(name, ne, npb, de.data_ptr(), dp.data_ptr(), t.data_ptr(), *[x.data_ptr() for x in o], 0)
        torch.cuda.synchronize()
        return [x.cpu().numpy() for x in o]

    for name, t in (("neorx_eg3ic1_dev", g), ("neorx_eg3ic1_f32_dev", g.float())):
        got = run(name, t)
        FE, FP = np.zeros((ne, ne), order="F"), np.zeros((npb, npb), order="F")
        E = oracle.eg3ic1(ne, npb, DE, DP, t.double().cpu().numpy(), FE, FP)
        check_close(got[0], FE.ravel(order="F"), what=f"{name} FE")
        check_close(got[1], FP.ravel(order="F"), what=f"{name} FP")
        assert got[2][0] == pytest.approx(E, rel=1e-11)
    for a, b in zip(run("neorx_eg3ic1_dev", g), run("neorx_eg3ic1_noalloc_dev", g)):
        assert np.array_equal(a, b)
