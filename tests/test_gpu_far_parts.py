"""Tile expansions whose roots go to two or four work-groups (lt_far.hip), against the extended oracle with the
FP64 criterion of parity.py as test_gpu_far.py has it: grids of 385 to 705 pixels a side, ragged, with an offset
that cuts the first root so that a half or a quarter of it lies past the grid, every halo type."""
import numpy as np
import pytest

import ltmodel as M
import test_gpu_far as far
from test_gpu_far import hip  # noqa: F401

pytestmark = pytest.mark.gpu

PARTS = {
    "quarters": lambda: (far._mixed(160, n14=2), far._grid(110.0, 449, 385), 0, 0),
    "quarters_cut": lambda: (far._mixed(160, n14=2), far._grid(110.0, 449, 385), 37, 35),
    "halves": lambda: (far._mixed(160, n14=2), far._grid(110.0, 673, 577), 0, 0),
    "halves_cut": lambda: (M.cluster_lens(seed=8, ngal=255), far._grid(110.0, 705, 577), 5, 35),
}


@pytest.mark.parametrize("name", PARTS)
@pytest.mark.parametrize("kmap", [False, True])
def test_hessian(hip, oracle, monkeypatch, name, kmap):  # noqa: F811
    monkeypatch.setitem(far.CASES, name, PARTS[name])
    far.test_hessian(hip, oracle, name, kmap)


@pytest.mark.parametrize("name", PARTS)
def test_gradient_and_potential(hip, oracle, monkeypatch, name):  # noqa: F811
    monkeypatch.setitem(far.CASES, name, PARTS[name])
    far.test_gradient_and_potential(hip, oracle, name)
