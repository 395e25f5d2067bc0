"""The nonlocal pseudopotential energy, whose quadrature points are spread over the lanes of a
wavefront (several pairs together), against the CPU oracle: rules of 4, 6 and 12 points (9, 9 and 4
pairs at a time, capped at 8), two species with different pseudopotentials and rules in one
molecule, more basis functions than one LDS chunk, a Jastrow outside the usual form, deterministic
and stochastic selection."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O
from tests._util import scaled_err

pytestmark = pytest.mark.gpu


class TwoSpecies(synth.Molecule):
    """Atoms alternate between two labels with pseudopotentials of their own."""
    aips = (12, 6)

    def sys_text(self):
        lines, n = [], 0
        for ln in synth.Molecule.sys_text(self).split("\n"):
            if "ATOM {" in ln:
                if self.two and n % 2:
                    ln = ln.replace("ATOM { %s" % self.label, "ATOM { N")
                n += 1
            lines.append(ln)
        text = "\n".join(lines)
        head, pseudo = text.split("PSEUDO {", 1)
        first = "PSEUDO {" + pseudo.replace("AIP 12", "AIP %d" % self.aips[0])
        if not self.two:
            return head + first
        # the second species: same form, steeper and of the other sign
        second = first.replace("  %s\n" % self.label, "  N\n").replace("BASIS { %s" % self.label, "BASIS { N")
        return head + first + second.replace("AIP %d" % self.aips[0], "AIP %d" % self.aips[1])

    def basis_text(self):
        t = synth.Molecule.basis_text(self)
        return t + (t.replace("\n%s\n" % self.label, "\nN\n") if self.two else "")

    def jast_text(self):
        t = synth.Molecule.jast_text(self)
        if not self.two:
            return t
        t = t.replace("  ONEBODY {", "  EIBASIS { N POLYPADE BETA0 0.3 NFUNC %d RCUT 6.5 }\n  ONEBODY {" % self.jast_nfunc)
        n = " COEFFICIENTS { N %s } }\n" % " ".join("%.17g" % (-c) for c in self.jast_ei)
        return t.replace(" } }\n  EEBASIS { EE POLYPADE", " }%s  EEBASIS { EE POLYPADE" % n)


def _molecule(natoms, nup, ndn, aips, nfunc):
    m = synth.z4_molecule(natoms, 20263000 + natoms, name="ppl%d_%d_%d_%d" % (natoms, nup, aips[0], nfunc), pseudo=True)
    m.__class__ = TwoSpecies
    rng = np.random.default_rng(8)
    m.two, m.aips = len(aips) == 2, aips
    m.mo_up, m.mo_dn, m.nup, m.ndn = m.mo_up[:, :nup], m.mo_dn[:, :ndn], nup, ndn
    m.jast_ei, m.jast_ee, m.jast_nfunc = rng.uniform(-0.1, 0.1, nfunc), rng.uniform(-0.1, 0.1, nfunc), nfunc
    return m


@pytest.mark.parametrize("natoms,nup,ndn,aips,nfunc", [
    (2, 4, 3, (12,), 4), (5, 10, 9, (6,), 4), (3, 6, 5, (4,), 3), (8, 16, 15, (12, 6), 4), (17, 34, 33, (12,), 4),
    (32, 64, 64, (6, 12), 4), (52, 20, 18, (12,), 4), (6, 12, 11, (12, 4), 5),
])
@pytest.mark.parametrize("prec", ["fp64", "mixed_fp32"])
def test_nonlocal_energy_matches_the_oracle(natoms, nup, ndn, aips, nfunc, prec, tmp_path):
    mol = _molecule(natoms, nup, ndn, aips, nfunc)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    eng, orc = E.Engine(deck, prec), O.Oracle(deck)
    K, rng = 3, np.random.default_rng(4)
    pos = synth.random_configs(mol, K, seed=31)
    rot, _ = np.linalg.qr(rng.standard_normal((3, 3)))
    for mode, rand in ((0, None), (1, rng.random((K, natoms, mol.nelec)))):
        a = eng.eval(pos, rot=rot, pp_mode=mode, pp_rand=rand)
        b = orc.eval(pos, rot=rot, pp_mode=mode, pp_rand=rand)
        print(mol.name, prec, mode, a["eparts"][:, 2], b["eparts"][:, 2], flush=True)
        # FP64 sums of at most a few thousand terms; mixed: FP32 inverse rows (relative 1e-6 per
        # well-conditioned row, ratios summed with both signs)
        assert scaled_err(a["eparts"][:, 2], b["eparts"][:, 2]) < (1e-10 if prec == "fp64" else 1e-2)
    eng.close()
