"""MO rows with F and G shells, whose kernels take one electron per wavefront and a larger tile: bases
smaller and larger than the tile, populations at which other shells' electrons would share a
wavefront, one, two and four orbitals per lane, against the CPU oracle; and mixed-precision sweeps of
such molecules below and above 64 electrons of a spin."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _molecule(natoms, syms, nup, ndn):
    m = synth.z4_molecule(natoms, 20266000 + natoms, name="fgr%d_%d_%d" % (natoms, nup, len(syms)))
    rng = np.random.default_rng(12)
    m.shells = m.shells + [(s, [(float(a), 1.0)]) for s, a in zip(syms, rng.uniform(0.4, 1.2, len(syms)))]
    m.mo_up = synth._lowdin(rng.standard_normal((m.nbasis, nup)))
    m.mo_dn = synth._lowdin(rng.standard_normal((m.nbasis, ndn)))
    m.nup, m.ndn = nup, ndn
    return m


@pytest.mark.parametrize("natoms,syms,nup,ndn", [
    (2, ("7F",), 4, 3), (3, ("7F_crystal", "15G", "9G"), 6, 5), (12, ("9G_pyscf", "7F"), 17, 16), (30, ("9G",), 60, 57),
    (36, ("7F",), 70, 66), (66, ("9G", "7F"), 130, 60),
])
def test_fg_rows_against_the_oracle(natoms, syms, nup, ndn, tmp_path):
    mol = _molecule(natoms, syms, nup, ndn)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    eng, orc = E.Engine(deck, "fp64"), O.Oracle(deck)
    pos = synth.nonsingular_configs(mol, 3, lambda p: eng.eval(p)["logpsi"], seed=29)
    a, b = eng.eval(pos), orc.eval(pos)
    assert np.array_equal(a["sign"], b["sign"])
    # FP64 sums of the same terms: 1e-16 of each, times the conditioning of the Slater matrix (at
    # most 1e5 for these configurations)
    for k in ("grad", "lap"):
        assert np.max(np.abs(a[k] - b[k])) < 1e-9 * np.max(np.abs(b[k])), k
    assert np.max(np.abs(a["logpsi"] - b["logpsi"])) < 1e-9 * max(1.0, np.max(np.abs(b["logpsi"])))
    mx = E.Engine(deck, "mixed_fp32")
    m = mx.eval(pos)
    # FP32 rows: 1e-7 relative per term, the same conditioning
    assert np.array_equal(m["sign"], b["sign"])
    assert np.max(np.abs(m["logpsi"] - b["logpsi"])) < 1e-1
    assert np.quantile(np.abs(m["grad"] - b["grad"]), 0.9) < 1e-2 * np.quantile(np.abs(b["grad"]), 0.9)
    if nup <= 32:
        r = 16384 // (3 * (nup + ndn)) + 2
        for e, x in ((eng, a), (mx, m)):
            g = e.eval(np.tile(pos, (r, 1, 1)))
            for k in ("logpsi", "grad", "lap"):
                assert np.array_equal(g[k], np.tile(x[k], (r,) + (1,) * (x[k].ndim - 1))), k
    eng.close()
    mx.close()


@pytest.mark.parametrize("method", ["DMC", "VMC"])
@pytest.mark.parametrize("natoms,nup,ndn", [(3, 6, 5), (12, 20, 24), (36, 70, 66)])
def test_mixed_sweeps_with_fg_shells(natoms, nup, ndn, method, tmp_path):
    mol = _molecule(natoms, ("7F", "15G", "9G"), nup, ndn)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    nw, tau = 5, 0.01
    eng, orc = E.Engine(deck, "mixed_fp32", seed=83), O.Oracle(deck)
    pos = synth.nonsingular_configs(mol, nw, lambda p: eng.eval(p)["logpsi"], seed=53)
    eng.set_walkers(pos)
    eng.run(E.method(method, nw, nblock=1, nstep=1, timestep=tau, ndecorr=1))
    p, _ = eng.get_walkers(nw)
    o = orc.run(pos, method, nblock=1, nstep=1, timestep=tau, seed=83, ndecorr=1, nthreads=8)
    # FP32 drifts; an acceptance within FP32 rounding of its threshold moves one walker elsewhere
    d = np.abs(p - o["pos"]).max(axis=(1, 2))
    print(mol.name, method, np.sort(d), flush=True)
    assert np.median(np.abs(p - o["pos"])) < 1e-5
    assert np.count_nonzero(d > 1e-2) <= 1
    eng.close()
