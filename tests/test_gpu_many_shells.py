"""Molecules of thousands of shells, whose shell records four walkers of a block cannot share in LDS:
DMC in FP64, both methods in mixed precision, and two determinants with the system tables left in
device memory, against the CPU oracle."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


class TwoDeterminants(synth.Molecule):
    def slater_text(self):
        up, dn = list(range(1, self.nup + 1)), list(range(self.nup + 1, self.nup + self.ndn + 1))
        rows = [up, dn, dn[-1:] + up[1:], dn]  # the second takes a down orbital in the first place
        return ("SLATER\nORBITALS {\n  CUTOFF_MO\n  MAGNIFY 1\n  NMO %d\n  ORBFILE %s.orb\n  INCLUDE %s.basis\n"
                "  CENTERS { USEATOMS }\n}\nDETWT { 0.9 0.4 }\nSTATES {\n%s\n}\n"
                % (self.nup + self.ndn, self.name, self.name, "\n".join(" ".join(map(str, r)) for r in rows)))


def _molecule(natoms, per_atom, nup, ndn, cls=synth.Molecule):
    """natoms Z=4 atoms of per_atom shells each, the electrons on the first atoms."""
    rng = np.random.default_rng(20265000 + natoms + per_atom)
    m = synth.z4_molecule(natoms, 20265000 + natoms, name="many%d_%d_%d" % (natoms, per_atom, nup))
    m.__class__ = cls
    m.shells = [(("S", "P")[i % 4 == 3], [(float(a), 1.0)]) for i, a in
                enumerate(np.exp(rng.uniform(np.log(0.1), np.log(10.0), per_atom)))]
    m.mo_up = synth._lowdin(rng.standard_normal((m.nbasis, nup)))
    m.mo_dn = synth._lowdin(rng.standard_normal((m.nbasis, ndn)))
    m.nup, m.ndn = nup, ndn
    return m


CASES = [("fp64", "DMC", 100, 26, 5, 4, synth.Molecule), ("fp64", "DMC", 60, 50, 40, 33, synth.Molecule),
         ("mixed_fp32", "DMC", 100, 30, 5, 4, synth.Molecule), ("mixed_fp32", "DMC", 60, 50, 40, 33, synth.Molecule),
         ("mixed_fp32", "VMC", 100, 30, 5, 4, synth.Molecule), ("mixed_fp32", "VMC", 60, 50, 40, 33, synth.Molecule),
         ("fp64", "DMC", 100, 72, 3, 2, TwoDeterminants), ("fp64", "VMC", 100, 72, 3, 2, TwoDeterminants)]


@pytest.mark.parametrize("prec,method,natoms,per_atom,nup,ndn,cls", CASES)
def test_many_shells_follow_the_oracle(prec, method, natoms, per_atom, nup, ndn, cls, tmp_path):
    mol = _molecule(natoms, per_atom, nup, ndn, cls)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    nw = 5
    eng, orc = E.Engine(deck, prec, seed=71), O.Oracle(deck)
    pos = synth.nonsingular_configs(mol, nw, lambda p: eng.eval(p)["logpsi"], seed=41)
    eng.set_walkers(pos)
    eng.run(E.method(method, nw, nblock=1, nstep=1, timestep=0.01, ndecorr=1))
    p, _ = eng.get_walkers(nw)
    o = orc.run(pos, method, nblock=1, nstep=1, timestep=0.01, seed=71, ndecorr=1, nthreads=8)
    d = np.abs(p - o["pos"]).max(axis=(1, 2))
    print(mol.name, prec, method, np.sort(d), flush=True)
    if prec == "fp64":  # one trajectory evaluated twice in FP64
        assert np.max(d) < 1e-8
    else:  # FP32 drifts; an acceptance within FP32 rounding of its threshold moves one walker elsewhere
        assert np.median(np.abs(p - o["pos"])) < 1e-5
        assert np.count_nonzero(d > 1e-2) <= 1
    fresh = eng.clone(seed=71)
    fresh.set_walkers(p)
    f, st = fresh.walker_state(nw), eng.walker_state(nw)
    if cls is synth.Molecule:
        assert np.array_equal(st["sign"], f["sign"])
        assert np.max(np.abs(st["logdet"] - f["logdet"])) < (1e-8 if prec == "fp64" else 1e-2)
    kin = fresh.eval(p)["eparts"][:, 0]
    assert np.median(np.abs(st["elast"][:, 0] - kin) / np.abs(kin)) < (1e-8 if prec == "fp64" else 1e-2)
    eng.close()
    fresh.close()
