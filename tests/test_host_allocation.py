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
