"""The nonlocal pseudopotential in systems of more functions than it forms coefficients for at once,
where only shells that reach a quadrature point take part, against the CPU oracle: basis sizes around
that limit, one and several chunks of functions, steep shells (few reach), rules of 4, 6 and 12 points, and
a caller's rotation that is not orthonormal (points off the electron's sphere)."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O
from tests._util import scaled_err

pytestmark = pytest.mark.gpu


def _molecule(natoms, nup, ndn, aip, steep):
    m = synth.z4_molecule(natoms, 20267000 + natoms, name="ppr%d_%d_%d_%d" % (natoms, nup, aip, steep), pseudo=True)
    m.pseudo["aip"] = aip
    if steep:
        m.shells = [(s, [(a * 4.0, c) for a, c in p]) for s, p in m.shells]
    m.mo_up, m.mo_dn, m.nup, m.ndn = m.mo_up[:, :nup], m.mo_dn[:, :ndn], nup, ndn
    return m


@pytest.mark.parametrize("natoms,nup,ndn,aip,steep", [
    (19, 30, 29, 12, 0), (20, 30, 28, 6, 0), (20, 8, 9, 4, 1), (32, 64, 64, 4, 1), (40, 25, 24, 6, 1), (60, 20, 22, 4, 0),
])
@pytest.mark.parametrize("prec", ["fp64", "mixed_fp32"])
def test_shells_that_reach_a_point(natoms, nup, ndn, aip, steep, prec, tmp_path):
    mol = _molecule(natoms, nup, ndn, aip, steep)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    eng, orc = E.Engine(deck, prec), O.Oracle(deck)
    K, rng = 4, np.random.default_rng(6)
    pos = synth.nonsingular_configs(mol, K, lambda p: eng.eval(p, rot=np.eye(3))["logpsi"], seed=59, spread=0.6)
    q, _ = np.linalg.qr(rng.standard_normal((3, 3)))
    for rot in (q, 1.4 * q, q @ np.diag([0.6, 1.0, 1.9])):
        for mode, rand in ((0, None), (1, rng.random((K, natoms, mol.nelec)))):
            a = eng.eval(pos, rot=rot, pp_mode=mode, pp_rand=rand)
            b = orc.eval(pos, rot=rot, pp_mode=mode, pp_rand=rand)
            print(mol.name, prec, mode, a["eparts"][:, 2], b["eparts"][:, 2], flush=True)
            # FP64 sums of at most a few thousand terms; mixed: FP32 inverse rows (relative 1e-6 per
            # well-conditioned row, ratios summed with both signs)
            assert scaled_err(a["eparts"][:, 2], b["eparts"][:, 2]) < (1e-10 if prec == "fp64" else 1e-2)
    eng.close()
