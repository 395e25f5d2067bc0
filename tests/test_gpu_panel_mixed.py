"""The mixed-precision sweeps that hold only the rows of the electrons about to move: up to 64
electrons of a spin (registers, updated 16 rows at a time) and 65 to 256 (two or four wavefronts
per walker, the other rows updated by a launch of their own), against the FP64 oracle with common
random numbers and against a fresh evaluation, at the edges of the size classes, with odd and
unequal electron counts and rows that do not start 16-byte aligned, for recompute intervals of one
panel, of several, and longer than the sweep."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O
from test_gpu_panel import _molecule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nup,ndn,nfunc,refresh", [
    (1, 1, 4, 0), (4, 3, 4, 0), (5, 8, 4, 0), (17, 16, 4, 32), (32, 33, 4, 0), (47, 64, 4, 0), (64, 63, 4, 64),
    (65, 64, 4, 0), (66, 97, 4, 32), (97, 80, 4, 128), (128, 127, 4, 64), (129, 113, 4, 256), (255, 130, 4, 0),
    (256, 256, 4, 32), (7, 6, 5, 0), (34, 33, 5, 0), (66, 65, 5, 96), (131, 40, 5, 0),
])
def test_mixed_panel_dmc_follows_the_oracle(nup, ndn, nfunc, refresh, tmp_path):
    mol = _molecule(nup, ndn, nfunc)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    nw = 5  # not a multiple of the walkers per block
    eng = E.Engine(deck, "mixed_fp32", seed=97, refresh_interval=refresh)
    orc = O.Oracle(deck)
    pos = synth.nonsingular_configs(mol, nw, lambda p: eng.eval(p)["logpsi"], seed=13)
    eng.set_walkers(pos)
    eng.run(E.method("DMC", nw, nblock=1, nstep=1, timestep=0.01))
    p, _ = eng.get_walkers(nw)
    st = eng.walker_state(nw)
    o = orc.run(pos, "DMC", nblock=1, nstep=1, timestep=0.01, seed=97, nthreads=8)
    # FP32 drifts (relative 1e-4 of at most a few hundred 1/bohr, times the timestep): below 1e-2
    # bohr and far less for nearly every electron; an acceptance decided within FP32 rounding of its
    # threshold (1e-4 per move of at most 5 x 512) takes its walker to another point
    d = np.abs(p - o["pos"]).max(axis=(1, 2))
    print(mol.name, np.sort(d), flush=True)
    assert np.median(np.abs(p - o["pos"])) < 1e-5
    assert np.count_nonzero(d > 1e-2) <= 1
    # the carried log|det| and determinant parts (FP32 updates of the rows) against a fresh
    # evaluation at the same positions: every row was brought up to date
    fresh = eng.clone(seed=97)
    fresh.set_walkers(p)
    f = fresh.walker_state(nw)
    assert np.array_equal(st["sign"], f["sign"])
    assert np.max(np.abs(st["logdet"] - f["logdet"])) < 1e-2
    kin = fresh.eval(p)["eparts"][:, 0]
    assert np.median(np.abs(st["elast"][:, 0] - kin) / np.abs(kin)) < 1e-2
    eng.close()
    fresh.close()


@pytest.mark.parametrize("method", ["DMC", "VMC"])
def test_mixed_panel_batch_equals_the_engines_alone(method, tmp_path):
    """Systems of every size class with their own recompute intervals in one batch, its launches 32
    and 64 moves apart: bitwise each engine's own run."""
    for lo in (32, 64):
        mols = [(_molecule(3, 4, 4), 0), (_molecule(20, 21, 5), lo), (_molecule(50, 64, 4), 2 * lo),
                (_molecule(70, 66, 4), lo), (_molecule(128, 101, 4), 2 * lo), (_molecule(97, 65, 5), 128)]
        m = E.method(method, 0, nblock=1, nstep=2, timestep=0.01, ndecorr=1)
        engs, refs = [], []
        for i, (mol, rf) in enumerate(mols):
            deck = mol.write(os.path.join(str(tmp_path), "%s_%d" % (mol.name, lo)))
            nw = 5 + i
            a = E.Engine(deck, "mixed_fp32", seed=41 + i, refresh_interval=rf or lo)
            b = E.Engine(deck, "mixed_fp32", seed=41 + i, refresh_interval=rf or lo)
            pos = synth.nonsingular_configs(mol, nw, lambda p: a.eval(p)["logpsi"], seed=17)
            a.set_walkers(pos)
            b.set_walkers(pos)
            refs.append((b.run(m)["eblock"], b.get_walkers(nw)))
            engs.append((a, nw))
            b.close()
        if method == "DMC":
            B = E.Batch([a for a, _ in engs])
            eb = list(B.run(m)["eblock"])
        else:  # VMC members advance step by step
            B = E.Batch(precision="mixed_fp32", refresh_interval=lo)
            ids = [B.join(a, [m]) for a, _ in engs]
            done = {}
            while len(done) < len(ids):
                for mid in B.step():
                    done[mid] = B.leave(mid)["eblock"]
            eb = [done[i] for i in ids]
        for i, (a, nw) in enumerate(engs):
            p, w = a.get_walkers(nw)
            print(lo, mols[i][0].name, eb[i][0, 0], flush=True)
            assert np.array_equal(eb[i], refs[i][0])
            assert np.array_equal(p, refs[i][1][0]) and np.array_equal(w, refs[i][1][1])
        B.close()
        for a, _ in engs:
            a.close()
