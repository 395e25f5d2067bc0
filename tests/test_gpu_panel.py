"""The FP64 DMC sweep that updates the inverse panel by panel (16 rows) against the CPU oracle:
trajectories, log|det| and determinant parts at the edges of its size classes (whole matrix in
registers up to 32 electrons of a spin, one wavefront up to 64, two up to 128, four up to 256),
with odd and unequal electron counts, rows that do not start 16-byte aligned and a partial last
panel, for the usual trial function and for one that takes the general path."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _molecule(nup, ndn, nfunc):
    """Z=4 atoms (enough for the electrons) with the given electrons of each spin and Jastrow
    polynomial functions (4: the usual form; 5: the general one)."""
    natoms = max(2, (max(nup, ndn) + 1) // 2)
    m = synth.z4_molecule(natoms, 20262000 + 300 * nup + ndn, name="pnl%d_%d_%d" % (nup, ndn, nfunc))
    rng = np.random.default_rng(5)
    m.mo_up, m.mo_dn = m.mo_up[:, :nup], m.mo_dn[:, :ndn]
    m.nup, m.ndn = nup, ndn
    m.jast_ei, m.jast_ee = rng.uniform(-0.1, 0.1, nfunc), rng.uniform(-0.1, 0.1, nfunc)
    m.jast_nfunc = nfunc
    return m


@pytest.mark.parametrize("nup,ndn,nfunc", [
    (1, 1, 4), (4, 3, 4), (5, 8, 4), (16, 9, 4), (17, 32, 4), (33, 31, 4), (48, 47, 4), (64, 64, 4), (65, 64, 4),
    (97, 80, 4), (128, 127, 4), (129, 113, 4), (255, 130, 4), (256, 256, 4),
    (7, 6, 5), (34, 33, 5), (66, 65, 5),
])
def test_panel_dmc_follows_the_oracle(nup, ndn, nfunc, tmp_path):
    mol = _molecule(nup, ndn, nfunc)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    nw, nstep = 5, 2  # not a multiple of the walkers per block
    eng = E.Engine(deck, "fp64", seed=97)
    orc = O.Oracle(deck)
    pos = synth.nonsingular_configs(mol, nw, lambda p: eng.eval(p)["logpsi"], seed=13)
    eng.set_walkers(pos)
    r = eng.run(E.method("DMC", nw, nblock=1, nstep=nstep, timestep=0.01))
    p, w = eng.get_walkers(nw)
    st = eng.walker_state(nw)
    o = orc.run(pos, "DMC", nblock=1, nstep=nstep, timestep=0.01, seed=97, nthreads=8)
    print(mol.name, r["eblock"][0, 0], o["eblock"][0, 0], flush=True)
    # two FP64 evaluations of one trajectory: a move's rounding (1e-16 of bohr-sized terms, times
    # the conditioning of ratios and drifts) stays far below 1e-8 over two steps
    assert np.max(np.abs(p - o["pos"])) < 1e-8
    # the carried inverse and log|det| against a fresh evaluation at the final positions
    fresh = eng.clone(seed=97)
    fresh.set_walkers(p)
    f = fresh.walker_state(nw)
    assert np.array_equal(st["sign"], f["sign"])
    assert np.max(np.abs(st["logdet"] - f["logdet"])) < 1e-8
    ev = fresh.eval(p)
    assert np.max(np.abs(st["elast"][:, 0] - ev["eparts"][:, 0]) / np.abs(ev["eparts"][:, 0])) < 1e-8
    eng.close()
    fresh.close()


def test_panel_batch_equals_the_engines_alone(tmp_path):
    """Systems of every size class in one batch: bitwise each engine's own run."""
    mols = [_molecule(a, b, c) for a, b, c in [(3, 4, 4), (20, 21, 5), (50, 33, 4), (70, 66, 4), (140, 129, 4)]]
    m = E.method("DMC", 0, nblock=1, nstep=2, timestep=0.01)
    engs, refs = [], []
    for i, mol in enumerate(mols):
        deck = mol.write(os.path.join(str(tmp_path), mol.name))
        nw = 5 + i
        a, b = E.Engine(deck, "fp64", seed=41 + i), E.Engine(deck, "fp64", seed=41 + i)
        pos = synth.nonsingular_configs(mol, nw, lambda p: a.eval(p)["logpsi"], seed=17)
        a.set_walkers(pos)
        b.set_walkers(pos)
        refs.append((b.run(m)["eblock"], b.get_walkers(nw)))
        engs.append((a, nw))
        b.close()
    B = E.Batch([a for a, _ in engs])
    r = B.run(m)
    for i, (a, nw) in enumerate(engs):
        p, w = a.get_walkers(nw)
        print(mols[i].name, r["eblock"][i, 0, 0], flush=True)
        assert np.array_equal(r["eblock"][i], refs[i][0])
        assert np.array_equal(p, refs[i][1][0]) and np.array_equal(w, refs[i][1][1])
    B.close()
