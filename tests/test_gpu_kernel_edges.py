"""Edges of single kernels: sizes at which a tile, a chunk or a buffer is full,
just short of full or nearly empty, against the oracle or plain FP64 numpy."""
import numpy as np
import pytest

from helios_amd import capi, molecules as M, ppp
from oracle import ccsd, mlp, triples as T
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


def _rows(count, seed):
    rng = np.random.default_rng(seed)
    rows = np.zeros((count, mlp.NF + 2), dtype=np.float32)
    rows[:, :mlp.NF] = rng.normal(0, 1, (count, mlp.NF))
    rows[:, mlp.NF] = rng.normal(0, 0.5, count)
    rows[:, mlp.NF + 1] = rng.uniform(0.2, 1.0, count)
    p = mlp.init(7).astype(np.float64)
    p[mlp.OFF_W3:mlp.OFF_B3] *= 20.0
    p[mlp.OFF_B1:mlp.OFF_W2] = rng.normal(0, 0.3, 64)
    p[mlp.OFF_B2:mlp.OFF_W3] = rng.normal(0, 0.3, 64)
    return rows, p.astype(np.float32)


@pytest.mark.parametrize("count", [1, 17, 64, 65, 16384, 16385])
def test_mlp_gradient_sizes(count):
    """Loss and gradient where a wave's 16 samples, a workgroup's 64 and the
    switch to 256 samples per workgroup begin and end, against the oracle with
    the tolerances of test_gradient_matches_oracle, parameter block by block."""
    rows, p = _rows(count, count)
    tr = capi.Trainer(count)
    tr.set_params(p)
    tr.write_samples(rows)
    loss, g = tr.gradient()
    tr.close()
    lo, go = mlp.backward(p, rows[:, :mlp.NF], rows[:, mlp.NF].astype(np.float64),
                          rows[:, mlp.NF + 1].astype(np.float64))
    assert abs(loss - lo) <= 1e-4 * lo
    for a, b in [(mlp.OFF_W1, mlp.OFF_B1), (mlp.OFF_B1, mlp.OFF_W2), (mlp.OFF_W2, mlp.OFF_B2),
                 (mlp.OFF_B2, mlp.OFF_W3), (mlp.OFF_W3, mlp.OFF_B3), (mlp.OFF_B3, mlp.NPARAM)]:
        assert np.abs(g[a:b] - go[a:b]).max() <= 1e-2 * np.abs(go[a:b]).max() + 1e-7


def test_epoch_loss_with_a_short_last_batch():
    """The last mini-batch of an epoch (44 of 300 rows in batches of 128) fills
    fewer workgroups than the others; with steps of 1e-30 the epoch's mean loss
    is the plain loss, up to FP32 rounding of each row's."""
    rows, p = _rows(300, 5)
    tr = capi.Trainer(300)
    tr.set_params(p)
    tr.write_samples(rows)
    loss, _ = tr.gradient()
    hist = tr.train(epochs=2, batch=128, lr=1e-30, lr_final=1e-30)
    moved = np.abs(tr.params().astype(np.float64) - p).max()   # six Adam steps of at most about 1e-30
    tr.close()
    assert moved < 1e-29
    assert np.abs(hist - loss).max() <= 1e-6 * loss


@pytest.mark.parametrize("o,v", [(1, 1), (1, 4), (3, 4), (4, 3), (5, 9), (8, 8), (7, 17), (16, 17), (33, 5), (5, 33)])
def test_residual_at_ragged_sizes(o, v):
    """Residuals at random amplitudes where n_occ and n_virt differ in parity and
    size (runs of odd radix along K, single rows and columns, tiles of 16, 32,
    33 and 64), with the tolerance of the residual parity test: 1e-11."""
    m = M.polyene(o + v)
    G, _, hk = ppp.model(m.coords, m.bonds)
    e, C = np.linalg.eigh(hk)   # any orthonormal orbitals with a diagonal Fock matrix will do
    F = np.diag(e)
    t1, t2 = random_amplitudes(o, v, 10 * o + v)
    B = ccsd.Blocks(ccsd.rint(C, G), o)
    r1, r2 = ccsd.singles(F, B, t1, t2), ccsd.doubles(F, B, t1, t2)
    ctx = capi.Context(0, capi.HCC_FP64, 20)
    ctx.set_molecule(C, F, G, o, 0.0)
    ctx.set_amplitudes(t1, t2)
    d1, d2 = ctx.residual()
    ctx.close()
    print(o, v, np.abs(d1 - r1).max(), np.abs(d2 - r2).max())
    assert np.abs(d1 - r1).max() < 1e-11 * max(1.0, np.abs(r1).max())
    assert np.abs(d2 - r2).max() < 1e-11 * max(1.0, np.abs(r2).max())


@pytest.mark.parametrize("m,n,k", [(12 * 64, 64, 17), (12 * 64 + 1, 129, 20), (25 * 64 - 3, 3 * 64, 33), (700, 13 * 64, 16)])
def test_tile_bands_fp64(m, n, k):
    """Products whose tile rows fill one band of 12, start the next one and end
    inside the third: k roundings of a sum of k products, each 2^-53 of the sum
    of magnitudes."""
    rng = np.random.default_rng(m + n)
    A, B, C0 = rng.standard_normal((m, k)), rng.standard_normal((k, n)), rng.standard_normal((m, n))
    C = capi.selftest_gemm(A, B, C0, alpha=0.5, beta=2.0)
    bound = 2.0 ** -53 * (k + 4) * (np.abs(A) @ np.abs(B) + 2 * np.abs(C0))
    assert (np.abs(C - (0.5 * A @ B + 2.0 * C0)) <= bound).all()


@pytest.mark.parametrize("tile,m,n,k", [(128, 8 * 128, 130, 40), (128, 8 * 128 + 1, 257, 64), (128, 17 * 128 - 5, 128, 33),
                                        (64, 12 * 64 + 1, 65, 40), (64, 12 * 64 + 1, 65, 70), (32, 12 * 32 + 1, 33, 40),
                                        (32, 25 * 32 + 7, 70, 100)])
@pytest.mark.parametrize("kinds", [(True, True), (True, False), (False, True)])
@pytest.mark.parametrize("a_kfast,b_nfast", [(True, True), (True, False), (False, True), (False, False)])
def test_tile_bands_correction(tile, m, n, k, kinds, a_kfast, b_nfast):
    """The correction GEMM over every layout, either operand constant, at the
    edges of its bands and on both sides of the short-K rule.  Each of the two
    products rounds both factors to BF16 (2^-8 relative each, with B0's copy
    rounded before dB is added: 2^-9 more) and accumulates in FP32."""
    rng = np.random.default_rng(m * 7 + n)
    A0, B0 = rng.standard_normal((m, k)), rng.standard_normal((k, n))
    dA = (1e-3 * rng.standard_normal((m, k))).astype(np.float32) if kinds[0] else None
    dB = (1e-3 * rng.standard_normal((k, n))).astype(np.float32) if kinds[1] else None
    C0 = rng.standard_normal((m, n)).astype(np.float32)
    C, _ = capi.selftest_gemm_correction(A0, dA, B0, dB, C0, alpha=0.5, beta=1.0, a_kfast=a_kfast, b_nfast=b_nfast, tile=tile)
    a, b = (np.zeros((m, k)) if dA is None else dA.astype(float)), (np.zeros((k, n)) if dB is None else dB.astype(float))
    ref = 0.5 * (A0 @ b + a @ (B0 + b)) + C0
    mag = 0.5 * (np.abs(A0) @ np.abs(b) + np.abs(a) @ (np.abs(B0) + np.abs(b)))
    assert (np.abs(C - ref) <= 2.0 ** -7 * mag + 2.0 ** -23 * (np.abs(C0) + mag)).all()


def test_correction_residual_at_every_run_length():
    """BF16 corrections over composite K of every run length modulo 4 (n_occ =
    n_virt = 5 .. 23) against the FP64 corrections.  Each outer step of the
    exact form contracts the residual by kappa = 0.05; BF16 rounding (2^-8 per
    factor, a few factors deep) adds about 0.02, so from 1 to 1e-8 the
    ln(1e8) / ln(1/0.05) = 6.1 outer steps become ln(1e8) / ln(1/0.07) = 6.9: at
    most two more in whole steps.  A product missing or repeating elements is
    off by an order of its own size and needs several times as many."""
    mols = [ppp.prepare(M.random_fragment(2 * o, seed=o)) for o in (5, 6, 7, 8, 9, 10, 11, 14, 17, 23)]
    outer = {}
    for bf16 in (False, True):
        ctx = capi.Context(0, capi.HCC_MIXED, 8)
        ctx.set_mixed(bf16=bf16, kappa=0.05, max_inner=60, max_outer=40)
        ctx.batch_load(mols)
        ctx.batch_solve(capi.GUESS_MP2, 4000, 1e-8)
        _, _, st = ctx.batch_results()
        outer[bf16], inner = ctx.batch_statistics()
        ctx.close()
        print("bf16", bf16, "outer", outer[bf16], "inner", inner)
        assert (st == 1).all()
    assert (outer[True] <= outer[False] + 2).all()
