"""MO rows (value, gradient, laplacian of every orbital at every electron) at the edges of their
size classes against the CPU oracle's evaluation: four, two and one electrons per wavefront (up to
16, 32 and 64 orbitals), two and four orbitals per lane (up to 128 and 256), spins of unequal size
sharing a wavefront, walker counts that leave the last group partly empty, more shells than one
window takes, and the general shells' kernels."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O
from test_gpu_panel import _molecule

pytestmark = pytest.mark.gpu

SIZES = [(1, 0, 4), (2, 1, 4), (16, 15, 4), (17, 3, 4), (32, 31, 4), (33, 1, 4), (64, 64, 4), (65, 2, 4), (128, 127, 4),
         (129, 128, 4), (256, 255, 4), (15, 16, 5), (31, 30, 5), (50, 49, 5), (70, 69, 5)]


@pytest.mark.parametrize("nup,ndn,nfunc", SIZES)
def test_rows_against_the_oracle(nup, ndn, nfunc, tmp_path):
    mol = _molecule(nup, ndn, nfunc)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    eng, orc = E.Engine(deck, "fp64"), O.Oracle(deck)
    pos = synth.nonsingular_configs(mol, 3, lambda p: eng.eval(p)["logpsi"], seed=29)
    a, b = eng.eval(pos), orc.eval(pos)
    assert np.array_equal(a["sign"], b["sign"])
    # FP64 sums of the same terms: 1e-16 of each, times the conditioning of the Slater matrix
    # (at most 1e5 for these configurations)
    for k in ("grad", "lap"):
        assert np.max(np.abs(a[k] - b[k])) < 1e-9 * np.max(np.abs(b[k])), k
    assert np.max(np.abs(a["logpsi"] - b["logpsi"])) < 1e-9 * max(1.0, np.max(np.abs(b["logpsi"])))
    m = E.Engine(deck, "mixed_fp32").eval(pos)
    # FP32 rows: 1e-7 relative per term, the same conditioning
    assert np.array_equal(m["sign"], b["sign"])
    assert np.median(np.abs(m["logpsi"] - b["logpsi"])) < 1e-2
    assert np.median(np.abs(m["grad"] - b["grad"])) < 1e-3 * np.median(np.abs(b["grad"]))
    if nup <= 32:  # the groups form only where there are electrons enough: the same rows, repeated
        r = 16384 // (3 * (nup + ndn)) + 2
        g = eng.eval(np.tile(pos, (r, 1, 1)))
        for k in ("logpsi", "grad", "lap"):
            assert np.array_equal(g[k], np.tile(a[k], (r,) + (1,) * (a[k].ndim - 1))), k
    eng.close()
