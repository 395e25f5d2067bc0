"""The nonlocal pseudopotential with several determinants, whose inverse rows are gathered onto the
orbital list a half-wave per (atom, electron) pair, against the CPU oracle: determinant counts around the
eight in flight, 1 to 32 electrons of a spin, odd numbers of pairs, rules of 4, 6 and 12 points."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O
from tests._util import scaled_err

pytestmark = pytest.mark.gpu


class Expansion(synth.Molecule):
    """ndet determinants over the same nmo orbitals for both spins, the first the lowest ones."""

    def slater_text(self):
        rng, nmo, rows = np.random.default_rng(14), self.mo_up.shape[1], []
        for d in range(self.ndet):
            for n in (self.nup, self.ndn):
                occ = range(n) if d == 0 else np.sort(rng.choice(nmo, n, replace=False))
                rows.append(" ".join(str(i + 1) for i in occ))
        wt = " ".join("%.3f" % ((-1) ** d / (d + 1.0)) for d in range(self.ndet))
        return ("SLATER\nORBITALS {\n  CUTOFF_MO\n  MAGNIFY 1\n  NMO %d\n  ORBFILE %s.orb\n  INCLUDE %s.basis\n"
                "  CENTERS { USEATOMS }\n}\nDETWT { %s }\nSTATES {\n%s\n}\n" % (nmo, self.name, self.name, wt, "\n".join(rows)))


def _molecule(natoms, nup, ndn, ndet, nmo, aip):
    m = synth.z4_molecule(natoms, 20268000 + natoms, name="mdp%d_%d_%d" % (natoms, nup, ndet), pseudo=True)
    m.__class__ = Expansion
    m.pseudo["aip"], m.nup, m.ndn, m.ndet = aip, nup, ndn, ndet
    m.mo_up = synth._lowdin(np.random.default_rng(15).standard_normal((m.nbasis, nmo)))
    m.mo_dn = m.mo_up[:, :0]
    return m


@pytest.mark.parametrize("natoms,nup,ndn,ndet,nmo,aip", [
    (2, 1, 2, 2, 4, 12), (2, 3, 4, 7, 7, 6), (3, 5, 3, 8, 9, 4), (5, 9, 10, 9, 20, 12), (5, 10, 9, 65, 20, 6),
    (16, 32, 31, 17, 50, 4), (20, 17, 32, 5, 64, 12),
])
def test_nonlocal_energy_of_an_expansion(natoms, nup, ndn, ndet, nmo, aip, tmp_path):
    mol = _molecule(natoms, nup, ndn, ndet, nmo, aip)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    eng, orc = E.Engine(deck, "fp64"), O.Oracle(deck)
    K, rng = 5, np.random.default_rng(16)
    pos = synth.random_configs(mol, K, seed=61, spread=0.7)
    rot, _ = np.linalg.qr(rng.standard_normal((3, 3)))
    for mode, rand in ((0, None), (1, rng.random((K, natoms, mol.nelec)))):
        a = eng.eval(pos, rot=rot, pp_mode=mode, pp_rand=rand)
        b = orc.eval(pos, rot=rot, pp_mode=mode, pp_rand=rand)
        print(mol.name, mode, a["eparts"][:, 2], b["eparts"][:, 2], flush=True)
        # FP64 sums of at most a few thousand terms with both signs over well-conditioned inverses
        assert scaled_err(a["eparts"][:, 2], b["eparts"][:, 2]) < 1e-10
    eng.close()
