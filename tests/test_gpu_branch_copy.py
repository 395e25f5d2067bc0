"""Branching copies of a walker's state by several blocks per pair: a DMC block from uneven weights
against the CPU oracle, and the copied inverses and MO rows against a fresh evaluation, for walkers
of one to seven slices."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O
from test_gpu_panel import _molecule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nup,ndn", [(2, 1), (17, 16), (40, 39), (41, 41), (65, 31), (101, 99)])
def test_branching_copies_follow_the_oracle(nup, ndn, tmp_path):
    mol = _molecule(nup, ndn, 4)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    nw = 8
    eng, orc = E.Engine(deck, "fp64", seed=31), O.Oracle(deck)
    pos = synth.nonsingular_configs(mol, nw, lambda p: eng.eval(p)["logpsi"], seed=23)
    wt = np.array([3.0, 0.05, 1.0, 2.5, 0.1, 1.0, 0.02, 1.0])
    eng.set_walkers(pos, wt)
    eng.run(E.method("DMC", nw, nblock=1, nstep=5, timestep=0.002))
    p, w = eng.get_walkers(nw)
    o = orc.run(pos, "DMC", nblock=1, nstep=5, timestep=0.002, seed=31, weights=wt, nthreads=8)
    # the oracle's walkers after its own branching (rounding 1e-16 through five steps); which pairs
    # form depends on the drawn uniforms
    assert np.max(np.abs(p - o["pos"])) < 1e-8
    assert np.max(np.abs(w - o["weights"])) < 1e-8 * np.max(np.abs(o["weights"]))
    print(mol.name, "distinct walkers", len(np.unique(np.round(p[:, 0, 0], 9))), "of", nw, flush=True)
    st = eng.walker_state(nw)
    fresh = eng.clone(seed=31)
    fresh.set_walkers(p)
    f = fresh.walker_state(nw)
    assert np.max(np.abs(st["logdet"] - f["logdet"])) < 1e-8
    eng.close()
    fresh.close()
