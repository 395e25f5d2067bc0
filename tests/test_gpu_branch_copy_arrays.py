"""Branching copies of the mixed path's FP32 inverses and MO rows and of several determinants' inverses:
walkers are copied from uneven weights, and the trajectories after the copies follow the CPU oracle."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O
from test_gpu_multidet_pseudo import Expansion
from test_gpu_panel import _molecule

pytestmark = pytest.mark.gpu
WEIGHTS = np.array([3.0, 0.05, 1.0, 2.5, 0.1, 1.0, 0.02, 1.0])


def _run(deck, prec, pos, nstep, tau):
    eng = E.Engine(deck, prec, seed=31)
    eng.set_walkers(pos, WEIGHTS)
    eng.run(E.method("DMC", len(pos), nblock=1, nstep=nstep, timestep=tau))
    return eng


def _check(deck, prec, pos, tau):
    nw = len(pos)
    # branching follows the fifth step: copied walkers are in the same place, as many as the oracle's
    eng = _run(deck, prec, pos, 5, tau)
    p = eng.get_walkers(nw)[0]
    o = O.Oracle(deck).run(pos, "DMC", nblock=1, nstep=5, timestep=tau, seed=31, weights=WEIGHTS, nthreads=8)
    copies = [nw - len(np.unique(x.reshape(nw, -1), axis=0)) for x in (p, o["pos"])]
    print(prec, "copies", copies, flush=True)
    assert copies[0] == copies[1]
    eng.close()
    # two steps on, the copies have moved on from the copied inverses and rows
    eng = _run(deck, prec, pos, 7, tau)
    p = eng.get_walkers(nw)[0]
    o = O.Oracle(deck).run(pos, "DMC", nblock=1, nstep=7, timestep=tau, seed=31, weights=WEIGHTS, nthreads=8)
    d = np.abs(p - o["pos"])
    print(prec, np.sort(d.max(axis=(1, 2))), flush=True)
    if prec == "fp64":
        assert np.max(d) < 1e-8
    else:  # FP32 drifts; an acceptance within FP32 rounding of its threshold moves one walker elsewhere
        assert np.median(d) < 1e-5
        assert np.count_nonzero(d.max(axis=(1, 2)) > 1e-2) <= 1
    fresh = eng.clone(seed=31)
    fresh.set_walkers(p)
    kin = fresh.eval(p)["eparts"][:, 0]
    e = np.abs(eng.walker_state(nw)["elast"][:, 0] - kin) / np.abs(kin)
    assert np.median(e) < (1e-8 if prec == "fp64" else 1e-2)
    eng.close()
    fresh.close()
    return copies[0]


# (with 17 + 16 electrons the weights fall below the pairing threshold before the fifth step)
@pytest.mark.parametrize("nup,ndn,copied", [(2, 1, True), (17, 16, False), (40, 39, True), (65, 31, True), (101, 99, True)])
def test_mixed_copies(nup, ndn, copied, tmp_path):
    mol = _molecule(nup, ndn, 4)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    eng = E.Engine(deck, "mixed_fp32")
    pos = synth.nonsingular_configs(mol, 8, lambda p: eng.eval(p)["logpsi"], seed=23)
    assert (_check(deck, "mixed_fp32", pos, 0.002) > 0) == copied
    eng.close()


@pytest.mark.parametrize("natoms,nup,ndn,ndet,nmo", [(2, 3, 4, 7, 7), (5, 10, 9, 33, 20)])
def test_copies_of_an_expansion(natoms, nup, ndn, ndet, nmo, tmp_path):
    m = synth.z4_molecule(natoms, 20268100 + natoms, name="mdc%d_%d" % (natoms, ndet))
    m.__class__ = Expansion
    m.nup, m.ndn, m.ndet = nup, ndn, ndet
    m.mo_up = synth._lowdin(np.random.default_rng(15).standard_normal((m.nbasis, nmo)))
    m.mo_dn = m.mo_up[:, :0]
    deck = m.write(os.path.join(str(tmp_path), m.name))
    assert _check(deck, "fp64", synth.random_configs(m, 8, seed=73, spread=0.7), 0.002) > 0
