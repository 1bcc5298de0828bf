"""Inputs of the FRI commit phase as callers may hold them: vectors that join on
the way in memory of the caller's own, at addresses that are multiples of 4 bytes
only, and challengers in a state that no sequence of calls makes (refused)."""
import numpy as np
import pytest

import pico_amd
from pico_amd import BABYBEAR, KOALABEAR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f", [KOALABEAR, BABYBEAR])
@pytest.mark.parametrize("log_n,log_in", [(5, 3), (17, 16), (17, 12)])  # folded in the tree's launch and before it
@pytest.mark.parametrize("offset", [1, 2, 3])
def test_joining_vector_at_any_word(ctx, oracle, f, log_n, log_in, offset):
    v, extra = oracle.random_matrix(f, 1, 1 << log_n, 4), oracle.random_matrix(f, 2, 1 << log_in, 4)
    flat = np.zeros((4 << log_in) + 4, np.uint32)
    flat[offset:offset + extra.size] = extra.ravel()
    held, top = ctx.upload(flat.reshape(-1, 4), field=f), ctx.upload(v, field=f)
    joined = ctx.wrap(held.device_ptr + 4 * offset, 1 << log_in, 4)
    fd = pico_amd.fri_commit_phase(ctx, f, pico_amd.DuplexChallenger(f), {log_n: top, log_in: joined}, 1, final_mode=1)
    roots, _, final, betas = oracle.fri_commit_phase(oracle.Challenger(f), v, 1, inputs={log_in: extra})
    assert np.array_equal(fd.commits, roots) and np.array_equal(fd.betas, betas) and np.array_equal(fd.final_poly, final)
    for x in (fd, joined, held, top):
        x.free()


@pytest.mark.parametrize("pending", [-1, 8, 9, 1 << 20])
def test_impossible_challenger_is_refused(ctx, pending):
    f = KOALABEAR
    ch, v = pico_amd.DuplexChallenger(f), ctx.random_matrix(f, 3, 1 << 4, 4)
    ch.c.n_input = pending
    before = bytes(ch.c)
    with pytest.raises(pico_amd.PgError):
        pico_amd.fri_commit_phase(ctx, f, ch, {4: v}, 1, final_mode=1)
    assert bytes(ch.c) == before
    v.free()
