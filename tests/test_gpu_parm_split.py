"""Linear-parameter derivatives against the CPU oracle at the edges of the split of an electron's
partners over neighbouring lanes (1, 2, 4 and 8 lanes per electron, one to eight wavefronts per
configuration), with like-spin, unlike-spin and single-spin partner ranges."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O
from test_gpu_panel import _molecule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nup,ndn,nfunc", [(1, 0, 4), (4, 3, 4), (4, 4, 4), (8, 8, 5), (32, 31, 4), (32, 32, 4), (33, 32, 5),
                                           (64, 64, 4), (65, 64, 4), (128, 128, 4), (129, 128, 4), (17, 2, 4)])
def test_parm_deriv_at_the_split_edges(nup, ndn, nfunc, tmp_path):
    mol = _molecule(nup, ndn, nfunc)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    eng, orc = E.Engine(deck, "fp64"), O.Oracle(deck)
    pos = synth.nonsingular_configs(mol, 3, lambda p: eng.eval(p)["logpsi"], seed=37)
    a, b = eng.parm_deriv(pos), orc.parm_deriv(pos)
    for k in ("gradient", "gradderiv", "val_gradient"):
        # sums of at most 512 terms in another order, and the determinant's gradient at the
        # conditioning of these Slater matrices (1e5)
        assert a[k].shape == b[k].shape
        assert np.max(np.abs(a[k] - b[k])) < 1e-9 * np.max(np.abs(b[k])), k
    eng.close()
