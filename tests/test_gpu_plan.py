"""The pair plan of a System is formed by the first builder that needs it:
the results of a handle do not depend on which builder that is, nor on how
many threads call builders on a new handle at once."""
from concurrent.futures import ThreadPoolExecutor
from threading import Barrier

import numpy as np
import pytest

import neorx
from neorx import synth

pytestmark = pytest.mark.gpu


def test_first_builder():
    import torch

    torch.cuda.init()
    neorx.init(0)
    s = synth.small(seed=71, n_e_centres=2, e_shells=(0, 1), contract=(1, 2, 3), p_shells=(0, 1), ngtg=2)
    print(f"case pair plan nebf={s['nebf']} npebf={s['npebf']} npbf={s['npbf']}", flush=True)
    build = {"gam2": lambda S: S.GAM2_IC1(), "gam3": lambda S: (S.GAM3_IC1(),), "ne": lambda S: S.RXCHFne_GAM2_IC1()}
    want = {}
    for k, f in build.items():
        S = neorx.System(s)
        want[k] = f(S)
        S.close()
    S = neorx.System(s)
    names = [*build, *build]
    start = Barrier(len(names))

    def call(k):
        start.wait()
        return build[k](S)

    with ThreadPoolExecutor(len(names)) as ex:
        got = list(ex.map(call, names))
    for k, g in zip(names, got):
        for a, b in zip(g, want[k]):
            assert np.array_equal(a, b), k
    S.close()
