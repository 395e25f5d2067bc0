"""FP64 VMC steps, all sweeps of both spins in one launch, against the CPU oracle: one, two and three
sweeps a step, a spin without electrons, and the edges of the register tiles."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O
from test_gpu_panel import _molecule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nup,ndn,ndecorr", [(1, 0, 2), (3, 0, 1), (2, 3, 3), (4, 5, 1), (16, 17, 2), (33, 20, 3), (64, 64, 1)])
def test_vmc_steps_follow_the_oracle(nup, ndn, ndecorr, tmp_path):
    mol = _molecule(nup, ndn, 4)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    nw = 6
    eng, orc = E.Engine(deck, "fp64", seed=53), O.Oracle(deck)
    pos = synth.nonsingular_configs(mol, nw, lambda p: eng.eval(p)["logpsi"], seed=19)
    eng.set_walkers(pos)
    r = eng.run(E.method("VMC", nw, nblock=1, nstep=1, timestep=0.02, ndecorr=ndecorr))
    p, _ = eng.get_walkers(nw)
    o = orc.run(pos, "VMC", nblock=1, nstep=1, timestep=0.02, seed=53, ndecorr=ndecorr)
    # one trajectory in FP64 twice: rounding (1e-16) through at most three short sweeps
    assert np.max(np.abs(p - o["pos"])) < 1e-8
    assert abs(r["eblock"][0, 0] - o["eblock"][0, 0]) < 1e-7 * abs(o["eblock"][0, 0])
    eng.close()
