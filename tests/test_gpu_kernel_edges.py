"""Edges of single kernels: sizes at which a tile, a chunk or a buffer is full,
just short of full or nearly empty, against the oracle or plain FP64 numpy."""
import numpy as np
import pytest

from helios_amd import capi, molecules as M
from oracle import ccsd, triples as T
from tests._molprep import prepare, random_amplitudes

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


@pytest.mark.parametrize("o,v", [(3, 2), (5, 15), (2, 16), (9, 17), (17, 9), (4, 23), (3, 24), (5, 25), (25, 26),
                                 (6, 31), (31, 32)])
def test_triples_size_classes(o, v):
    """(T) at given amplitudes on both sides of the size classes' limits (v = 16,
    24, 32; ragged row tiles, a second virtual block of 9 to 16), with the
    tolerance of the kernel parity test: 1e-11 of |E[T]|."""
    p = prepare(M.random_fragment(o + v + (o + v) % 2, seed=11))
    n = o + v
    C, F, G = p["C"][:, :n], p["F"][:n, :n], p["G"]
    if n < p["n"]:   # an odd count: leave the last site and orbital out
        C, G = C[:n], G[:n, :n]
    t1, t2 = random_amplitudes(o, v, 100 * o + v, 0.05, 0.05)
    ctx = capi.Context(0, capi.HCC_FP64, 20)
    ctx.set_molecule(C, F, G, o, p["eref"])
    ctx.set_amplitudes(t1, t2)
    _, et = ctx.batch_triples()
    ctx.close()
    ref = T.closed_shell_sliced(C, F, G, o, t1, t2)
    print(o, v, et[0], ref, et[0] - ref)
    assert abs(et[0, 0] - ref[0]) < 1e-11 * abs(ref[0])
    assert abs(et[0, 1] - ref[1]) < 1e-11 * abs(ref[0])
