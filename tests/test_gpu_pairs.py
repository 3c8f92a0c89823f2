"""The tensor builders that evaluate distinct primitive pairs, against sums of
the primitive tuples (neorx_prim_list3_dev) over every permutation, bra/ket
order and contraction, at sampled entries of the full tensors."""
from itertools import permutations, product

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


# Angular momenta at the edges of the kernels' capacities (l of the electrons
# 0, 1, 2 with l of the nuclear functions 0 .. 2), and 1, 63..65 and more
# primitive pairs (lone-pair groups of 64: one partly filled, one full, more).
SYSTEMS = {
    "one-s": dict(seed=1, n_e_centres=1, e_shells=(0,), contract=(1,), p_shells=(0,), ngtg=1),
    "s-10prims-d": dict(seed=2, n_e_centres=2, e_shells=(0, 0, 0), contract=(1, 2), p_shells=(0, 2), ngtg=2),
    "sp-contracted": dict(seed=3, n_e_centres=2, e_shells=(0, 1), contract=(1, 2, 3), p_shells=(0, 1), ngtg=2),
    "sp-d-nucleus": dict(seed=4, n_e_centres=2, e_shells=(0, 1), contract=(1,), p_shells=(2,), ngtg=2),
    "p-66pairs": dict(seed=5, n_e_centres=1, e_shells=(0, 0, 1, 1, 1), contract=(1,), p_shells=(0,), ngtg=3),
    "d": dict(seed=6, n_e_centres=1, e_shells=(2,), contract=(2,), p_shells=(0,), ngtg=2),
    "spd-spd": dict(seed=7, n_e_centres=1, e_shells=(0, 1, 2), contract=(1,), p_shells=(0, 1, 2), ngtg=2),
}


def tuple_values(torch, S, cls, idx):
    """(n, 3) outputs of class cls for the index rows"""
    n = len(idx)
    d = torch.from_numpy(np.ascontiguousarray(idx)).cuda()
    out = torch.zeros((3, n), dtype=torch.float64, device="cuda")
    S.prim_list3_dev(cls, n, d.data_ptr(), *[out[k].data_ptr() for k in range(3)])
    torch.cuda.synchronize()
    return out.cpu().numpy().T


def contracted(torch, S, s, cls, nel, entries, perms):
    """sum over primitives and the given electron permutations (mean) of the
    tuples of contracted entries (ip, jp, i1, j1, ...)"""
    rows, coef, at = [], [], []
    kp = [list(range(a - 1, b)) for a, b in zip(s["kpestr"], s["kpeend"])]
    for n, en in enumerate(entries):
        ip, jp, br, kt = en[0], en[1], en[2::2], en[3::2]
        for p in perms:
            for prim in product(*[kp[br[k]] for k in p], *[kp[kt[k]] for k in p]):
                rows.append(list(prim[:nel]) + [ip] + list(prim[nel:]) + [jp])
                coef.append(np.prod(s["agebfcc"][list(prim)]) * s["agnbfcc"][ip] * s["agnbfcc"][jp] / len(perms))
                at.append(n)
    v = tuple_values(torch, S, cls, np.array(rows, dtype=np.int64)) * np.array(coef)[:, None]
    out = np.zeros((len(entries), 3))
    np.add.at(out, at, v)
    return out


def sample(s, nel, n, seed):
    rng = np.random.default_rng(seed)
    return [[int(rng.integers(s["npbf"])) for _ in range(2)] + [int(rng.integers(s["nebf"])) for _ in range(2 * nel)]
            for _ in range(n)]


def flat_index(s, entries):
    dims = [s["npbf"]] * 2 + [s["nebf"]] * (len(entries[0]) - 2)
    return np.ravel_multi_index(np.array(entries).T, dims)


@pytest.mark.parametrize("name", SYSTEMS)
def test_gam3_from_pairs(torch_dev, name):
    """GAM3_IC1 and RXCHFmult_GAM3_XCHF (classes 3 and 7)."""
    s = synth.small(**SYSTEMS[name])
    S = neorx.System(s)
    en = sample(s, 3, 40, 11)
    print(f"case gam3 pairs {name} nebf={s['nebf']} npebf={s['npebf']} npbf={s['npbf']}", flush=True)
    perms = list(permutations(range(3)))
    for cls, g in ((3, S.GAM3_IC1()), (7, S.RXCHFmult_GAM3_XCHF())):
        ref = contracted(torch_dev, S, s, cls, 3, en, perms)[:, 0]
        got = g[flat_index(s, en)]
        assert np.isfinite(g).all()
        check_close(np.append(got, np.abs(g).max()), np.append(ref, np.abs(g).max()), what=f"class {cls}")
    S.close()


@pytest.mark.parametrize("name", SYSTEMS)
def test_gam2_from_pairs(torch_dev, name):
    """GAM2_IC1 (class 2, averaged over the electrons) and RXCHFne_GAM2_IC1
    (class 4: the first output as it is, the second averaged)."""
    s = synth.small(**SYSTEMS[name])
    S = neorx.System(s)
    en = sample(s, 2, 60, 12)
    at = flat_index(s, en)
    print(f"case gam2 pairs {name} nebf={s['nebf']} npebf={s['npebf']} npbf={s['npbf']}", flush=True)
    both = list(permutations(range(2)))
    sym2, sym4 = (contracted(torch_dev, S, s, c, 2, en, both) for c in (2, 4))
    one4 = contracted(torch_dev, S, s, 4, 2, en, both[:1])
    g, gs = S.GAM2_IC1()
    n, nx = S.RXCHFne_GAM2_IC1()
    for got, ref, what in ((g, sym2[:, 0], "GM2ICR"), (gs, sym2[:, 1], "GM2sICR"), (n, one4[:, 0], "RXCHF-ne GM2ICR"),
                           (nx, sym4[:, 1], "GM2exICR")):
        assert np.isfinite(got).all()
        check_close(np.append(got[at], np.abs(got).max()), np.append(ref, np.abs(got).max()), what=what)
    S.close()


def test_build_reports_progress(torch_dev, monkeypatch, capfd):
    """NEORX_VERBOSE: a long e-e-e-p build says on stderr how far it is."""
    s = synth.small(**SYSTEMS["sp-contracted"])
    S = neorx.System(s)
    nc, nq = s["nebf"] * (s["nebf"] + 1) // 2, s["npbf"] * (s["npbf"] + 1) // 2
    try:
        monkeypatch.setenv("NEORX_VERBOSE", "1")
        neorx.init(0)
        S.GAM3_IC1()
        assert f"row {nc} of {nc}, nuclear pair {nq} of {nq}" in capfd.readouterr().err
    finally:
        monkeypatch.delenv("NEORX_VERBOSE")
        neorx.init(0)
    S.GAM3_IC1()
    assert "e-e-e-p" not in capfd.readouterr().err
    S.close()


def test_gam3_more_nuclear_pairs_than_a_launch(torch_dev):
    """32896 distinct nuclear pairs, of which the values of 32768 are held at
    once: entries of the second batch, in both nuclear orders."""
    s = synth.small(seed=8, n_e_centres=1, e_shells=(0,), contract=(1,), p_shells=(0,) * 256, ngtg=1)
    assert s["nebf"] == 1 and s["npbf"] == 256
    S = neorx.System(s)
    # pair i <= j is number j (j + 1) / 2 + i: 32768 is (128, 255)
    en = [[i, 255, 0, 0, 0, 0, 0, 0] for i in (0, 127, 128, 129, 200, 255)]
    en += [[e[1], e[0]] + e[2:] for e in en] + [[254, 254, 0, 0, 0, 0, 0, 0], [0, 0, 0, 0, 0, 0, 0, 0]]
    print("case gam3 pairs, 256 nuclear functions", flush=True)
    g = S.GAM3_IC1()
    ref = contracted(torch_dev, S, s, 3, 3, en, list(permutations(range(3))))[:, 0]
    assert np.isfinite(g).all()
    check_close(g[flat_index(s, en)], ref)
    S.close()
