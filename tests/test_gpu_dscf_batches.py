"""GAM2_DSCF and GAM3_DSCF where the distinct nuclear pairs do not fit one
batch of blocks (2^27 contracted values), the last batch a short one: against
EG2IC1 and EG3IC1 over the in-core tensors of the same handle, and with the
scratch of one batch, however many there are."""
import numpy as np
import pytest

import neorx
from neorx import synth
from _util import check_close

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev():
    import torch

    torch.cuda.init()
    neorx.init(0)
    return torch


def outputs(torch, sizes):
    return [torch.zeros(n, dtype=torch.float64, device="cuda") for n in sizes]


def densities(torch, ne, npb):
    # without symmetry, as the entry points accept
    rng = np.random.default_rng(ne)
    m = (synth.density(ne, 4.0, 5) + 0.1 * rng.standard_normal((ne, ne)),
         synth.density(npb, 1.0, 6) + 0.1 * rng.standard_normal((npb, npb)))
    return [torch.from_numpy(np.ascontiguousarray(x.ravel(order="F"))).cuda() for x in m]


def kept_bytes(torch, call):
    """bytes of scratch that the library keeps after the call"""
    neorx.release_resident()
    call()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    neorx.release_resident()
    return torch.cuda.mem_get_info()[0] - before


def test_gam3_dscf_batches(torch_dev):
    torch = torch_dev
    s = synth.small(seed=61, n_e_centres=3, e_shells=(0, 0, 0, 1), contract=(1,), p_shells=(0, 1), ngtg=1)
    ne, npb = s["nebf"], s["npbf"]
    nb, nq, npair = 2 ** 27 // ne ** 6, npb * (npb + 1) // 2, ne * (ne + 1) // 2
    assert 1 < nb < nq and nq % nb  # several batches, the last one short
    print(f"case gam3 dscf batches nebf={ne} npbf={npb}: {nq} nuclear pairs, {nb} a batch", flush=True)
    S = neorx.System(s)
    de, dp = densities(torch, ne, npb)
    got, want = (outputs(torch, (ne * ne, npb * npb, 1)) for _ in range(2))
    kept = kept_bytes(torch, lambda: neorx.call_dev("neorx_gam3_dscf_dev", S.handle, de.data_ptr(), dp.data_ptr(),
                                                    *[x.data_ptr() for x in got], 0))
    # star values of one batch, records of its primitive stars (three densities
    # of 27 doubles); the pair data, rows and allocation granularity are small
    one = 8 * nb * (npair * (npair + 1) // 2) * (npair + 3 * 27)
    assert kept < 1.25 * one, (kept, one)
    G = torch.empty(ne ** 6 * npb ** 2, dtype=torch.float64, device="cuda")
    neorx.call_dev("neorx_gam3_ic1_dev", S.handle, G.data_ptr(), 0)
    neorx.call_dev("neorx_eg3ic1_dev", ne, npb, de.data_ptr(), dp.data_ptr(), G.data_ptr(),
                   *[x.data_ptr() for x in want], 0)
    torch.cuda.synchronize()
    for a, b, nm in zip(got, want, ("FE", "FP", "E")):
        check_close(a.cpu().numpy(), b.cpu().numpy(), what=nm)
    S.close()


def test_gam2_dscf_batches(torch_dev):
    torch = torch_dev
    s = synth.small(seed=62, n_e_centres=6, e_shells=(0, 0, 0, 1), contract=(1,), p_shells=(0,) * 10 + (1,), ngtg=1)
    ne, npb = s["nebf"], s["npbf"]
    nb, nq = 2 ** 27 // ne ** 4, npb * (npb + 1) // 2
    assert 1 < nb < nq and nq % nb
    print(f"case gam2 dscf batches nebf={ne} npbf={npb}: {nq} nuclear pairs, {nb} a batch", flush=True)
    S = neorx.System(s)
    de, dp = densities(torch, ne, npb)
    sizes = (ne * ne, ne * ne, npb * npb, npb * npb, 1, 1)
    got, want = outputs(torch, sizes), outputs(torch, sizes)
    p = [x.data_ptr() for x in got]
    kept = kept_bytes(torch, lambda: neorx.call_dev("neorx_gam2_dscf_dev", S.handle, de.data_ptr(), dp.data_ptr(), p[0],
                                                    p[2], p[1], p[3], p[4], p[5], 0))
    # values of one launch's primitive stars (192 MiB); the values of a batch
    # are a larger block, which is not kept
    assert kept < 1.25 * (192 << 20), kept
    G, Gs = (torch.empty(ne ** 4 * npb ** 2, dtype=torch.float64, device="cuda") for _ in range(2))
    neorx.call_dev("neorx_gam2_ic1_dev", S.handle, G.data_ptr(), Gs.data_ptr(), 0)
    neorx.call_dev("neorx_eg2ic1_dev", ne, npb, de.data_ptr(), dp.data_ptr(), G.data_ptr(), Gs.data_ptr(),
                   *[x.data_ptr() for x in want], 0)
    torch.cuda.synchronize()
    for a, b, nm in zip(got, want, ("FE", "SE", "FP", "SP", "E", "S")):
        check_close(a.cpu().numpy(), b.cpu().numpy(), what=nm)
    S.close()


def test_refused_allocation_gives_scratch_back(torch_dev):
    """The scratch kept between calls does not stand in the way of another
    allocation: one that fails (here for terabytes) has emptied the list
    first."""
    torch = torch_dev
    s = synth.small(seed=61, n_e_centres=3, e_shells=(0, 0, 0, 1), contract=(1,), p_shells=(0, 1), ngtg=1)
    ne, npb = s["nebf"], s["npbf"]
    print(f"case refused allocation nebf={ne} npbf={npb}", flush=True)
    S = neorx.System(s)
    de, dp = densities(torch, ne, npb)
    out = outputs(torch, (ne * ne, npb * npb, 1))
    call = lambda: neorx.call_dev("neorx_gam3_dscf_dev", S.handle, de.data_ptr(), dp.data_ptr(),  # noqa: E731
                                  *[x.data_ptr() for x in out], 0)
    call()
    torch.cuda.synchronize()
    want = [x.clone() for x in out]
    free = torch.cuda.mem_get_info()[0]
    with pytest.raises(neorx.NeorxError, match="hipMalloc"):
        neorx.autotune_eg3_dev(2, 200000, 0, de.data_ptr(), de.data_ptr(), reps=1)
    assert torch.cuda.mem_get_info()[0] - free > 64 << 20  # 89 MB were kept
    for x in out:
        x.zero_()
    call()
    torch.cuda.synchronize()
    for a, b in zip(out, want):
        assert torch.equal(a, b)
    S.close()
