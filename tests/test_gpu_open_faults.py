"""An allocation that fails anywhere inside the whole Pcs::open or the quotient: the
call returns PG_E_OOM, the challenger is as before, no device memory stays behind,
and the next call gives the undisturbed result."""
import numpy as np
import pytest

import pico_amd
from pico_amd import KOALABEAR, air
from pico_amd._lib import PG_E_OOM
from pico_amd.air import RESIDENT, WINDOWED

pytestmark = pytest.mark.gpu
F = KOALABEAR


def sweep(ctx, call):
    """call() under a failure at each of its allocations in turn; returns how many failed"""
    want = call()
    base = ctx.bytes_in_use
    for k in range(200):
        ctx.debug_fail_alloc(k)
        try:
            got = call()
        except pico_amd.PgError as e:
            assert e.code == PG_E_OOM, (k, str(e))
            assert ctx.bytes_in_use == base, k
            continue
        finally:
            ctx.debug_fail_alloc(-1)
        assert got == want and ctx.bytes_in_use == base
        return k
    raise AssertionError("every call failed")


@pytest.fixture()
def fctx():
    c = pico_amd.Context(0)
    yield c
    c.close()


def test_open(fctx):
    ctx = fctx
    pcs = pico_amd.TwoAdicFriPcs(ctx, F, 1)
    shapes = [(6, 9), (9, 30), (4, 3), (9, 41)]
    mats = [ctx.random_matrix(F, k, 1 << L, w) for k, (L, w) in enumerate(shapes)]
    root, data = pcs.commit([(pcs.natural_domain_for_degree(m.rows), m) for m in mats])
    points = np.array([[3, 1, 4, 1], [2, 7, 1, 8]], np.uint64)

    def call():
        ch = pico_amd.DuplexChallenger(F)
        ch.observe(root)
        before = bytes(ch.c)
        try:
            return pcs.open([(data, [points] * len(shapes))], ch, 5, 3)[1]["bincode"]
        except pico_amd.PgError:
            held.append(bytes(ch.c) == before)
            raise

    held = []
    try:
        assert sweep(ctx, call) > 10
        assert held[0]  # the first failure is before anything was observed
    finally:
        data.free()
        for m in mats:
            m.free()


@pytest.mark.parametrize("form", [WINDOWED, RESIDENT])
def test_quotient(fctx, form):
    ctx = fctx
    pcs = pico_amd.TwoAdicFriPcs(ctx, F, 1)
    m = ctx.random_matrix(F, 1, 1 << 7, 30)
    _, data = pcs.commit([(pcs.natural_domain_for_degree(1 << 7), m)])
    b = air.AirBuilder(F)
    for c in range(30):
        b.when_transition().assert_zero(b.main(c) * b.main((c + 1) % 30) - b.main(c, next=True))
    prog = b.compile()
    prog.debug_form(form)

    def call():
        q = air.quotient_values(ctx, prog, data, 0, 1, 1, [1, 2, 3, 4])
        try:
            return q.to_host(F).tobytes()
        finally:
            q.free()

    try:
        assert sweep(ctx, call) >= 2
    finally:
        data.free()
        m.free()
