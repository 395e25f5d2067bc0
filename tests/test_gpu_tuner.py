"""The online tuner's choice of a sweep launch is of the kernel that it timed: FP64 VMC above 64
electrons of a spin has none, and a choice made on FP64 VMC steps is not taken for the DMC sweep."""
import os

import pytest

from mainline_amd import engine as E
from mainline_amd import synth
from test_gpu_panel import _molecule

pytestmark = pytest.mark.gpu


def _engine(nup, ndn, nw, monkeypatch, tmp_path):
    monkeypatch.setenv("QW_GRAPHS", "0")  # every step launched, so that each can be timed
    mol = _molecule(nup, ndn, 4)
    eng = E.Engine(mol.write(os.path.join(str(tmp_path), mol.name)), "fp64", seed=67)
    eng.set_walkers(synth.nonsingular_configs(mol, nw, lambda p: eng.eval(p)["logpsi"], seed=71))
    return eng


def test_vmc_above_64_electrons_makes_no_choice(monkeypatch, tmp_path):
    nw = 4
    eng = _engine(66, 65, nw, monkeypatch, tmp_path)
    eng.run(E.method("VMC", nw, nblock=1, nstep=3, timestep=0.05))  # 12 sweep launches
    assert eng.tuning()["sweep"] == 0
    eng.run(E.method("DMC", nw, nblock=1, nstep=3, timestep=0.005))  # 6: each of 3 candidates twice
    assert eng.tuning()["sweep"] in (2, 4, 8)
    eng.close()


def test_dmc_is_measured_after_vmc(monkeypatch, tmp_path):
    nw = 8
    eng = _engine(5, 4, nw, monkeypatch, tmp_path)
    eng.run(E.method("VMC", nw, nblock=1, nstep=6, timestep=0.1))  # 6 launches
    vmc = eng.tuning()["sweep"]
    assert vmc in (2, 4, 8)
    eng.run(E.method("DMC", nw, nblock=1, nstep=2, timestep=0.01))  # 4: measuring
    assert eng.tuning()["sweep"] == 0
    eng.run(E.method("DMC", nw, nblock=1, nstep=1, timestep=0.01))
    assert eng.tuning()["sweep"] in (2, 4, 8)
    eng.run(E.method("VMC", nw, nblock=1, nstep=1, timestep=0.1))
    assert eng.tuning()["sweep"] == vmc
    eng.close()
