"""The mixed path's MO rows: four, two and one electrons per wavefront give the same bits, and nearly every
gradient component and laplacian lies within FP32 rounding of the CPU oracle's."""
import os

import numpy as np
import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from oracle import oracle as O
from test_gpu_panel import _molecule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nup,ndn,nfunc", [(1, 0, 4), (2, 1, 4), (16, 15, 4), (17, 3, 4), (32, 31, 4), (15, 16, 5),
                                           (31, 30, 5), (64, 63, 4), (70, 69, 4), (130, 128, 4)])
def test_mixed_rows(nup, ndn, nfunc, tmp_path):
    mol = _molecule(nup, ndn, nfunc)
    deck = mol.write(os.path.join(str(tmp_path), mol.name))
    eng, orc = E.Engine(deck, "mixed_fp32"), O.Oracle(deck)
    pos = synth.nonsingular_configs(mol, 3, lambda p: eng.eval(p)["logpsi"], seed=29)
    a, b = eng.eval(pos), orc.eval(pos)
    assert np.array_equal(a["sign"], b["sign"])
    # FP32 rows: 1e-7 relative per term, times the conditioning of the Slater matrix (at most 1e5); one
    # orbital or electron left out would change every electron of its spin by order one
    assert np.max(np.abs(a["logpsi"] - b["logpsi"])) < 1e-1
    for k in ("grad", "lap"):
        err = np.abs(a[k] - b[k]) / (np.abs(b[k]) + np.median(np.abs(b[k])))
        assert np.quantile(err, 0.95) < 1e-2, k
    if nup <= 32:
        r = 16384 // (3 * (nup + ndn)) + 2
        g = eng.eval(np.tile(pos, (r, 1, 1)))
        for k in ("logpsi", "grad", "lap"):
            assert np.array_equal(g[k], np.tile(a[k], (r,) + (1,) * (a[k].ndim - 1))), k
    eng.close()
