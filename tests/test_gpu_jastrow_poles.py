"""Electron pairs beyond the cutoff of a POLYPADE function with a negative BETA0 (its denominator
1 + beta z has a zero there) and inside the cutoff of the cusp function, against the CPU oracle: at
separations in steps of one unit in the last place around that zero, and in short runs."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


class ShortRange(synth.Molecule):
    """BETA0 -1/8 and cutoff 3 for the electron-electron POLYPADE, 7.5 for the cusp function."""

    def jast_text(self):
        return synth.Molecule.jast_text(self).replace("EE POLYPADE BETA0 0.5 NFUNC 4 RCUT 7.5",
                                                      "EE POLYPADE BETA0 -0.125 NFUNC 4 RCUT 3.0")


def _deck(n, tmp_path):
    m = synth.z4_molecule(2, 20264000 + n, name="pole%d" % n)
    m.__class__ = ShortRange
    m.coords = np.array([[0.0, 0.0, 0.7], [6.0, 0.0, -0.7]])
    m.mo_up, m.mo_dn, m.nup, m.ndn = m.mo_up[:, :n], m.mo_dn[:, :n], n, n
    return m, m.write(os.path.join(str(tmp_path), m.name))


@pytest.mark.parametrize("prec", ["fp64", "mixed_fp32"])
def test_pairs_at_a_zero_of_the_denominator(prec, tmp_path):
    mol, deck = _deck(1, tmp_path)
    # z(s) = s^2 (6 - 8 s + 3 s^2), s = r / 3, is 8 at twice the cutoff
    r0, K = 6.0, 8192
    r = r0 + (np.arange(K) - K // 2) * np.spacing(r0)
    pos = np.zeros((K, 2, 3))
    pos[:, 1, 0] = r  # from the origin: the separation is r itself
    eng, orc = E.Engine(deck, prec), O.Oracle(deck)
    a, b = eng.eval(pos), orc.eval(pos[::K - 1])
    for k in ("logpsi", "grad", "lap", "eparts"):
        x = a[k].reshape(K, -1)
        assert np.all(np.isfinite(x)), (k, np.count_nonzero(~np.isfinite(x).all(axis=1)))
        # the separations differ by 1e-12: one value, the oracle's
        tol = (1e-9 if prec == "fp64" else 1e-4) * np.max(np.abs(b[k]))
        assert np.max(np.abs(x - b[k].reshape(2, -1)[:1])) < tol, k
    eng.close()


@pytest.mark.parametrize("method", ["DMC", "VMC"])
def test_short_range_function_follows_the_oracle(method, tmp_path):
    mol, deck = _deck(4, tmp_path)
    nw = 6
    eng, orc = E.Engine(deck, "fp64", seed=61), O.Oracle(deck)
    pos = synth.nonsingular_configs(mol, nw, lambda p: eng.eval(p)["logpsi"], seed=37)
    eng.set_walkers(pos)
    eng.run(E.method(method, nw, nblock=1, nstep=2, timestep=0.02, ndecorr=1))
    p, _ = eng.get_walkers(nw)
    o = orc.run(pos, method, nblock=1, nstep=2, timestep=0.02, seed=61, ndecorr=1)
    # two FP64 evaluations of one trajectory of eight electrons
    assert np.max(np.abs(p - o["pos"])) < 1e-8
    eng.close()
