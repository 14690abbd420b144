"""What the library's host code does when device memory runs out, and how much
of it a load holds: run on the CPU with the HIP runtime replaced (_hoststub)."""
import numpy as np
import pytest

from helios_amd import capi
from tests import _hoststub
from tests._hoststub import molecule


@pytest.fixture(scope="module")
def stub_lib(tmp_path_factory):
    return _hoststub.build(tmp_path_factory.mktemp("hoststub"))


def _batch(precision, mols):
    ctx = capi.Context(0, precision, 8)
    ctx.set_graphs(False)
    ctx.batch_load(mols)
    return ctx


# enough molecules that the tables of all contractions outgrow the block the load left
MANY = [molecule(6, 3)] * 700


def _profiled_solve(ctx):
    ctx.profile(True)
    ctx.batch_solve(capi.GUESS_MP2, 8, 1e-8)


def profiled_solve(stub):
    stub.each_failure(lambda: _batch(capi.HCC_FP64, MANY), _profiled_solve)


def tune_correction_tables(stub):
    stub.each_failure(lambda: _batch(capi.HCC_MIXED, MANY), lambda ctx: [ctx.tune_gemm(100 + q, 0, 0, 1) for q in range(25)])


def tune_own_tables(stub):
    stub.each_failure(lambda: _batch(capi.HCC_FP64, MANY), lambda ctx: [ctx.tune_gemm(q, 0, 0, 1) for q in range(25)])


@pytest.mark.parametrize("function", [profiled_solve, tune_own_tables, tune_correction_tables], ids=lambda f: f.__name__)
def test_tables_per_contraction_after_a_failed_build(stub_lib, function):
    """A profiled solve and a tuning call build tables of their own; when that
    fails half-way, the next one builds them again."""
    _hoststub.check(stub_lib, function)


def _exact(ctx):
    ctx.set_mixed(bf16=False, max_inner=3, max_outer=1)


def switch_corrections(stub):
    def make():
        ctx = _batch(capi.HCC_MIXED, MANY)
        ctx.set_mixed(bf16=True, max_inner=3, max_outer=1)
        return ctx

    def solve(ctx):
        ctx.batch_solve(capi.GUESS_MP2, 8, 1e-8)

    def again(ctx):
        _exact(ctx)
        solve(ctx)

    stub.lib.stub_running(len(MANY))
    assert stub.launches(lambda: again(make())) != stub.launches(lambda: solve(make()))
    stub.each_failure(make, _exact, solve)
    stub.each_failure(make, _exact, again)


def test_correction_form_after_a_failed_switch(stub_lib):
    """When the tables of the other correction form cannot be built, the solves
    that follow run the form that was set before, and the switch can be repeated."""
    _hoststub.check(stub_lib, switch_corrections)


def _trainer(rows):
    tr = capi.Trainer(rows)
    tr.write_samples(np.zeros((rows, capi.MLP_ROW), dtype=np.float32))
    return tr


def trainer_buffers(stub):
    """Calls on all samples that need larger buffers than the trainer has, and
    after a failed one a call on a few, which needs no more than it has."""
    few = lambda tr: tr.gradient(0, 100)
    stub.each_failure(lambda: _trainer(100000), lambda tr: tr.gradient(), few)
    stub.each_failure(lambda: _trainer(100000), lambda tr: tr.evaluate(), few)
    stub.each_failure(lambda: _trainer(100000), lambda tr: tr.train(epochs=1, batch=90000), few)
    stub.each_failure(lambda: _trainer(100000), lambda tr: tr.gradient())


def test_trainer_buffers_after_a_failed_growth(stub_lib):
    _hoststub.check(stub_lib, trainer_buffers)


def _solved(mols):
    ctx = _batch(capi.HCC_FP64, mols)
    ctx.batch_solve(capi.GUESS_MP2, 4, 1e-8)
    return ctx


def triples_setup(stub):
    # 12 x 5984 work items: their partial sums are an allocation of their own
    stub.each_failure(lambda: _solved([molecule(34, 32)] * 12), lambda ctx: ctx.batch_triples())


def response_setup(stub):
    # 33000 molecules: each of the pointer lists is an allocation of its own
    mols = [molecule(2, 1)] * 33000
    r1, r2 = np.zeros(len(mols)), np.zeros(len(mols))
    stub.each_failure(lambda: _solved(mols), lambda ctx: ctx.batch_lr_sigma(r1, r2))


def response_staging(stub):
    def make():
        ctx = _solved([molecule(8, 4)] * 4)
        ctx.lr_space(4)
        ctx.lr_gram([[0, 1, 1, 0, 0]], [0])
        return ctx

    jobs = [[m, 4, 4, 0, 0] for m in range(4)] * 8
    few = lambda ctx: ctx.lr_gram([[0, 1, 1, 0, 0]], [0])
    stub.each_failure(make, lambda ctx: ctx.lr_gram(jobs, range(4)), few)


def residual_outputs(stub):
    def make():
        ctx = capi.Context(0, capi.HCC_FP64, 8)
        m = molecule(80, 40)
        ctx.set_molecule(m["C"], m["F"], m["G"], m["nocc"], 0.0)
        ctx.guess()
        return ctx

    stub.each_failure(make, lambda ctx: ctx.residual())


def compaction(stub):
    stub.lib.stub_running(100)
    for precision in (capi.HCC_FP64, capi.HCC_MIXED):
        def make():
            ctx = _batch(precision, MANY)
            ctx.set_mixed(max_inner=3, max_outer=1)
            return ctx
        stub.each_failure(make, lambda ctx: ctx.batch_solve(capi.GUESS_MP2, 8, 1e-8))


@pytest.mark.parametrize("function", [triples_setup, response_setup, response_staging, residual_outputs, compaction],
                         ids=lambda f: f.__name__)
def test_set_up_on_first_use_after_a_failure(stub_lib, function):
    """What a batch allocates when a call first needs it counts as there only
    when all of it is."""
    _hoststub.check(stub_lib, function)


def load_peak(stub):
    """Memory held while a batch replaces another: never more than the larger of the two."""
    def mols(sizes):
        return [molecule(n, n // 2) for n in sizes]

    shapes = [mols([20] * 40), mols([26] * 25), mols([8] * 300), mols(range(10, 40, 2)), mols([40])]
    alone = []
    for m in shapes:
        ctx = _batch(capi.HCC_FP64, m)
        alone.append(stub.lib.stub_held())
        ctx.close()
        assert stub.lib.stub_held() == 0
    ctx = capi.Context(0, capi.HCC_FP64, 8)
    for first in range(len(shapes)):
        for second in range(len(shapes)):
            ctx.batch_load(shapes[first])
            stub.lib.stub_peak(1)
            ctx.batch_load(shapes[second])
            peak, held = stub.lib.stub_peak(0), stub.lib.stub_held()
            # a block taken again may exceed the request by an eighth and 64 KiB
            assert held <= 1.125 * alone[second] + (64 << 16), (first, second, held, alone[second])
            assert peak <= 1.125 * max(alone[first], alone[second]) + (64 << 16), (first, second, peak, alone)


def test_load_holds_no_more_than_the_larger_batch(stub_lib):
    _hoststub.check(stub_lib, load_peak)


def scf_load(stub):
    n = 48   # the three matrices of the molecules are allocations of their own
    mols = [dict(core=np.eye(n), G=np.eye(n), huckel=np.eye(n), nocc=n // 2)] * 60

    def load(ctx):
        ctx.batch_load_scf(mols)

    ctx = capi.Context(0, capi.HCC_FP64, 8)
    first = stub.lib.stub_allocations()
    load(ctx)
    count = stub.lib.stub_allocations() - first
    for k in range(1, count + 1):
        ctx = capi.Context(0, capi.HCC_FP64, 8)
        assert stub.fails(lambda: load(ctx), k), k
        assert stub.fails(lambda: ctx.batch_solve(), 0), f"allocation {k} of {count} failed, yet there is a batch"


def test_no_batch_after_a_failed_scf_load(stub_lib):
    _hoststub.check(stub_lib, scf_load)
