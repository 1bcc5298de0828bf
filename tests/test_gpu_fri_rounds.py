"""The FRI commit phase with the challenger on the device: every number of
pending challenger inputs, vectors from one round to several launches per
round, inputs that join on the way, and the answers of all rounds at once.
Everything equals the oracle's, bit for bit."""
import numpy as np
import pytest

import pico_amd
from pico_amd import BABYBEAR, KOALABEAR

pytestmark = pytest.mark.gpu
FIELDS = [KOALABEAR, BABYBEAR]


def check(ctx, oracle, f, log_n, log_stop, extra_logs=(), observed=0):
    v = oracle.random_matrix(f, 80 + log_n, 1 << log_n, 4)
    extra = {k: oracle.random_matrix(f, 81 + k, 1 << k, 4) for k in extra_logs}
    ch, och = pico_amd.DuplexChallenger(f), oracle.Challenger(f)
    for c in (ch, och):
        c.observe([17 + i for i in range(observed)])
    inputs = {log_n: ctx.upload(v, field=f)}
    inputs.update({k: ctx.upload(a, field=f) for k, a in extra.items()})
    fd = pico_amd.fri_commit_phase(ctx, f, ch, inputs, log_stop, final_mode=1)
    roots, layers, final, betas = oracle.fri_commit_phase(och, v, log_stop, inputs=extra)
    assert np.array_equal(fd.commits, roots)
    assert np.array_equal(fd.betas, betas)
    assert np.array_equal(fd.final_poly, final)
    och.observe(final.ravel())
    assert [ch.sample() for _ in range(11)] == [och.sample() for _ in range(11)]
    rng = np.random.default_rng(log_n)
    idx = [0, (1 << log_n) - 1] + [int(x) for x in rng.integers(0, 1 << log_n, 5)]
    sib, paths = pico_amd.fri_answer_queries(fd, idx, log_n)
    for q, i in enumerate(idx):
        for r in range(log_n - log_stop):
            assert np.array_equal(sib[q, r], layers[r][(i >> r) ^ 1])
    # the rounds' trees serve openings as any tree does
    for r in range(log_n - log_stop):
        td = fd.round_data(r)
        leaf = layers[r].reshape(-1, 8)
        ot = oracle.MerkleTree(f, [leaf]) if log_n <= 10 else None
        at = sorted({(i >> r) >> 1 for i in idx})
        rows, rpaths = pico_amd.MerkleTreeMmcs(ctx, f).open_many(at, td)
        for k, j in enumerate(at):
            assert np.array_equal(rows[k], leaf[j])
            if ot is not None:
                assert np.array_equal(rpaths[k], ot.open(j)[1])
        for q, i in enumerate(idx):
            assert np.array_equal(paths[q][r], rpaths[at.index((i >> r) >> 1)])
        assert np.array_equal(td.root(), roots[r])


@pytest.mark.parametrize("f", FIELDS)
@pytest.mark.parametrize("observed", range(9))
def test_pending_inputs(ctx, oracle, f, observed):
    check(ctx, oracle, f, 6, 1, observed=observed)


@pytest.mark.parametrize("f", FIELDS)
@pytest.mark.parametrize("log_n,log_stop,extra", [(0, 0, ()), (1, 0, (0,)), (1, 1, ()), (2, 0, (1,)), (7, 0, ()), (8, 2, (7, 2)),
                                                  (9, 1, (3,)), (14, 3, (13, 3)), (16, 12, ()), (17, 13, (16,)), (18, 15, ())],
                         ids=str)
def test_rounds(ctx, oracle, f, log_n, log_stop, extra):
    check(ctx, oracle, f, log_n, log_stop, extra, observed=5)
