"""The several-determinant sweep with its inverses resident in LDS and, for expansions that do not
fit, in device memory: trajectories against the CPU oracle for 3, 64, 65, 100 and 160 determinants
of N2 (lanes over determinants: below, at and above a wavefront)."""
import itertools
import os
import shutil

import numpy as np
import pytest

from mainline_amd import engine as E
from oracle import oracle as O
from tests._util import golden

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ndet", [3, 64, 65, 100, 160])
@pytest.mark.parametrize("method", ["VMC", "DMC"])
def test_many_determinants_follow_the_oracle(ndet, method, tmp_path):
    g, deck = golden("n2_cij")
    src = os.path.dirname(deck)
    for f in os.listdir(src):
        shutil.copy(os.path.join(src, f), str(tmp_path))
    rng = np.random.default_rng(ndet)
    occ = list(itertools.combinations(range(1, 9), 5))
    pairs = [(occ[0], occ[0])] + [(occ[rng.integers(len(occ))], occ[rng.integers(len(occ))]) for _ in range(ndet - 1)]
    wt = np.concatenate([[1.0], 0.05 * rng.standard_normal(ndet - 1)])
    with open(os.path.join(str(tmp_path), "cidet"), "w") as f:
        f.write("DETWT { %s }\nSTATES {\n" % " ".join("%.8f" % x for x in wt))
        for u, d in pairs:
            f.write(" ".join(map(str, u)) + "\n" + " ".join(map(str, d)) + "\n")
        f.write("}\n")
    deck = os.path.join(str(tmp_path), os.path.basename(deck))
    nw = 7
    pos = g["pos"][:nw]
    tau = 0.05 if method == "VMC" else 0.01
    eng = E.Engine(deck, "fp64", seed=4711)
    eng.set_walkers(pos)
    eng.run(E.method(method, nw, nblock=1, nstep=2, timestep=tau))
    p, w = eng.get_walkers(nw)
    o = O.Oracle(deck).run(pos, method, nblock=1, nstep=2, timestep=tau, seed=4711, step0=0)
    # one FP64 trajectory evaluated twice (rounding 1e-16 over at most 40 short moves)
    assert np.max(np.abs(p - o["pos"])) < 1e-8
    assert np.max(np.abs(w - o["weights"])) < 1e-8
    eng.close()
