"""One context that loads batches of other sizes one after another gives what
fresh contexts give: nothing of a replaced batch's memory is read."""
import numpy as np
import pytest

from helios_amd import capi, molecules as M, ppp

pytestmark = pytest.mark.gpu


def _results(ctx, mols):
    ctx.batch_load(mols)
    ctx.batch_solve(capi.GUESS_MP2, 400, 1e-8)
    e, it, st = ctx.batch_results()
    assert (st == 1).all()
    last = mols[-1]
    t1, t2 = ctx.batch_amplitudes(len(mols) - 1, last["nocc"], last["C"].shape[0] - last["nocc"])
    ov = [m["nocc"] * (m["C"].shape[0] - m["nocc"]) for m in mols]
    s1, s2 = ctx.batch_lr_sigma(np.full(sum(ov), 0.1), np.full(sum(x * x for x in ov), 0.01))
    return e, it, t1, t2, s1, s2, ctx.batch_triples()[1]


@pytest.mark.parametrize("precision", [capi.HCC_FP64, capi.HCC_MIXED])
def test_loads_of_other_sizes_in_one_context(precision):
    """Larger, smaller, larger again, of equal total size, one molecule: each
    equal bit by bit to the same load in a context of its own (sums have a fixed
    order)."""
    sizes = [(24, 30, 36), (10, 14), (24, 30, 36), (30,) * 5, (40, 8, 22), (12,), (24, 30, 36)]
    made = {n: ppp.prepare(M.random_fragment(n, seed=n)) for s in sizes for n in s}
    ctx = capi.Context(0, precision, 8)
    for s in sizes:
        mols = [made[n] for n in s]
        fresh = capi.Context(0, precision, 8)
        want = _results(fresh, mols)
        fresh.close()
        got = _results(ctx, mols)
        print(s, [float(np.abs(g - w).max()) for g, w in zip(got, want)], flush=True)
        assert all(np.array_equal(g, w) for g, w in zip(got, want))
    ctx.close()
