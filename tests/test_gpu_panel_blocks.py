"""Populations that put one, two, three or four walkers into a block of the sweeps up to 64 electrons
of a spin (and leave the last block partly empty): a walker's moves are the same bits in each."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from test_gpu_panel import _molecule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,method", [("fp64", "DMC"), ("mixed_fp32", "DMC"), ("mixed_fp32", "VMC")])
@pytest.mark.parametrize("nup,ndn,nfunc", [(3, 2, 4), (9, 8, 5), (20, 17, 4), (40, 33, 4)])
def test_a_walker_does_not_see_its_block(prec, method, nup, ndn, nfunc, tmp_path):
    mol = _molecule(nup, ndn, nfunc)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    base = E.Engine(deck, prec, seed=43)
    sizes = (1030, 769, 768, 513, 512, 257, 256, 3)
    pos = synth.random_configs(mol, 64, seed=47)
    pos = pos[base.eval(pos)["logpsi"] > -1e200][:16]
    pos = np.tile(pos, (sizes[0] // len(pos) + 1, 1, 1))[:sizes[0]]
    ref = None
    for nw in sizes:
        eng = base.clone(seed=43)
        eng.set_walkers(pos[:nw])
        # no weight of DMC grows (those of low energies are cut off), so branching copies no walker
        eng.run(E.method(method, nw, nblock=1, nstep=1, timestep=0.01, ndecorr=1, branch_start_cutoff=1e-9))
        p, _ = eng.get_walkers(nw)
        if ref is None:
            ref = p
            assert np.all(np.isfinite(p)) and np.any(p != pos)
        else:
            assert np.array_equal(p, ref[:nw]), nw
        eng.close()
    base.close()
