"""Edges of single kernels: sizes at which a tile, a chunk or a buffer is full,
just short of full or nearly empty, against the oracle or plain FP64 numpy."""
import numpy as np
import pytest

from helios_amd import capi, molecules as M
from oracle import ccsd
from tests._molprep import prepare

pytestmark = pytest.mark.gpu


def test_diis_two_vectors_step_by_step():
    """The smallest bordered system (a history of two vectors alone does not
    converge on this molecule): the first six iterations against the oracle's,
    with the tolerance of test_iterate_mirrors_iterationCC."""
    p = prepare(M.random_fragment(14, seed=5))
    cc = ccsd.CCSD(p["C"], p["F"], p["G"], p["nocc"], p["eref"], diis_scale=True, diis_steps=2)
    ctx = capi.Context(0, capi.HCC_FP64, 2)
    ctx.set_molecule(p["C"], p["F"], p["G"], p["nocc"], p["eref"])
    ctx.guess(capi.GUESS_REFERENCE)
    for it in range(1, 7):
        acc, ref = ctx.iterate(it, 1e-12), cc.iterate(it, 1e-12)
        assert abs(acc[0] - ref[0]) < 1e-9 * max(1, ref[0])
        assert abs(acc[1] - ref[1]) < 1e-9 * max(1, ref[1])
    ctx.close()


@pytest.mark.parametrize("steps", [3, 31, 32])
def test_diis_system_sizes(steps):
    """Solves with small and the largest DIIS histories (bordered systems of up
    to 33 unknowns; a solve to 1e-12 fills a history of 32 vectors) reach
    the oracle's fixed point: energy 1e-8 eV and T2 1e-7 (the solver's parity
    tolerances)."""
    p = prepare(M.random_fragment(14, seed=5))
    eps = 1e-12 if steps > 3 else 1e-9
    ref = ccsd.solve(p["C"], p["F"], p["G"], p["nocc"], p["eref"], eps=eps, diis_scale=True, diis_steps=steps)
    assert ref["status"] == 1
    ctx = capi.Context(0, capi.HCC_FP64, steps)
    ctx.set_molecule(p["C"], p["F"], p["G"], p["nocc"], p["eref"])
    e, it, st = ctx.solve(capi.GUESS_REFERENCE, 2000, eps)
    _, t2 = ctx.amplitudes()
    ctx.close()
    print(steps, it, ref["iterations"], e[0] - ref["energy"][0])
    assert st == 1
    assert abs(e[0] - ref["energy"][0]) < 1e-8
    assert np.abs(t2 - ref["t2"]).max() < 1e-7
