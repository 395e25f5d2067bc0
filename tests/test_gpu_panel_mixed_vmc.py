"""Mixed-precision VMC sweeps (delayed rejection) with 65 to 256 electrons of a spin, two and four
wavefronts per walker, against the FP64 oracle with common random numbers: at this timestep one move
in twenty is rejected at both stages and more are decided by the second, whose shell lists take the
place in LDS of the first stage's orbital values, so a wavefront that still read them would decide
for itself."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O
from test_gpu_panel import _molecule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nup,ndn,nfunc,refresh,ndecorr", [
    (65, 64, 4, 0, 1), (66, 97, 4, 32, 1), (97, 65, 5, 64, 1), (128, 127, 4, 0, 1), (70, 66, 4, 0, 2), (129, 113, 4, 0, 1),
    (131, 40, 5, 96, 1), (256, 255, 4, 0, 1),
])
def test_mixed_panel_vmc_follows_the_oracle(nup, ndn, nfunc, refresh, ndecorr, tmp_path):
    mol = _molecule(nup, ndn, nfunc)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    nw, tau = 6, 0.1
    eng = E.Engine(deck, "mixed_fp32", seed=97, refresh_interval=refresh)
    orc = O.Oracle(deck)
    pos = synth.nonsingular_configs(mol, nw, lambda p: eng.eval(p)["logpsi"], seed=13)
    eng.set_walkers(pos)
    eng.run(E.method("VMC", nw, nblock=1, nstep=1, timestep=tau, ndecorr=ndecorr))
    p, _ = eng.get_walkers(nw)
    st = eng.walker_state(nw)
    o = orc.run(pos, "VMC", nblock=1, nstep=1, timestep=tau, seed=97, ndecorr=ndecorr, nthreads=8)
    assert 0.8 < o["acceptance"] < 0.99  # second stages ran
    # FP32 drifts displace a proposal by at most 1e-4 of its length (4e-5 bohr); a sweep multiplies a
    # displacement of the electrons moved before by up to 300 (the oracle's own spread from starts
    # 1e-6 apart).  A decision within FP32 rounding of its threshold (1e-4 a move) takes a walker
    # elsewhere: a tenth of the walkers of 512 electrons
    d = np.abs(p - o["pos"]).max(axis=(1, 2))
    print(mol.name, o["acceptance"], np.sort(d), flush=True)
    assert np.median(np.abs(p - o["pos"])) < 1e-4
    assert np.count_nonzero(d > 5e-2) <= 2
    # the carried state against a fresh evaluation at the same positions
    fresh = eng.clone(seed=97)
    fresh.set_walkers(p)
    f = fresh.walker_state(nw)
    assert np.array_equal(st["sign"], f["sign"])
    assert np.max(np.abs(st["logdet"] - f["logdet"])) < 1e-2
    kin = fresh.eval(p)["eparts"][:, 0]
    assert np.median(np.abs(st["elast"][:, 0] - kin) / np.abs(kin)) < 1e-2
    eng.close()
    fresh.close()
