"""Query answers of a FRI commit phase where the budget leaves little: they take
no more memory than answering round by round does, down to single queries at a
time, and are the same answers."""
import numpy as np
import pytest

import pico_amd
from pico_amd import BABYBEAR, KOALABEAR

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f", [KOALABEAR, BABYBEAR])
@pytest.mark.parametrize("log_n,queries", [(14, 300), (6, 40), (9, 1)])
def test_answers_within_budget(f, log_n, queries):
    budget = 64 << 20
    idx = np.random.default_rng(queries).integers(0, 1 << log_n, queries)
    # one round's answers: per query an index, a row and log_n - 1 digests (each part
    # rounded to the pool's 512 bytes); at least one query's answers of all rounds
    room = max(queries * (8 + 32 + 32 * (log_n - 1)) + 1536, 256 + 512 * log_n + 32 * log_n * log_n)
    got = []
    with pico_amd.Context(0, budget) as ctx:
        held = [ctx.random_matrix(f, 1, 1 << log_n, 4)]  # nothing may outlive the context
        try:
            held.append(pico_amd.fri_commit_phase(ctx, f, pico_amd.DuplexChallenger(f), {log_n: held[0]}, 0))
            for limited in (False, True):
                if limited:
                    held.append(ctx.matrix((budget - ctx.bytes_in_use - room) // 512, 128))
                got.append(pico_amd.fri_answer_queries(held[1], idx, log_n))
        finally:
            for x in held[::-1]:
                x.free()
    (s0, p0), (s1, p1) = got
    assert np.array_equal(s0, s1) and s0.any()
    assert all(np.array_equal(a, b) for q0, q1 in zip(p0, p1) for a, b in zip(q0, q1))
