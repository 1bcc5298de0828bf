"""Batched jobs of fewer than 64 extended rows, whose leaves share waves: rows of
equal and of unequal widths in one wave, whole and partial chunks mixed, packs
that end at 64 rows or before, single rows, and long jobs between them.  Every
digest layer equals the oracle's."""
import numpy as np
import pytest

import pico_amd
from pico_amd import BABYBEAR, KOALABEAR

pytestmark = pytest.mark.gpu

# (log height, width, log blowup) of each job
CASES = {
    "equal widths": [(2, 16, 1)] * 30,
    "one chunk, every width": [(1, w, 1) for w in range(1, 9)] * 3,
    "two chunks, one whole": [(3, 9 + k % 8, 1) for k in range(20)],
    "single rows": [(0, 1 + k, 0) for k in range(70)],
    "exactly 64 rows": [(4, 24, 1), (4, 24, 1), (0, 24, 0)],
    "around long jobs": [(4, 11, 1), (5, 11, 1), (7, 24, 1), (6, 15, 0), (0, 300, 1), (2, 14, 3)],
    "no two alike": [(k % 5, 8 * k + 5, 1) for k in range(12)],
}


@pytest.mark.parametrize("f", [KOALABEAR, BABYBEAR])
@pytest.mark.parametrize("name", list(CASES))
def test_short_jobs_match_oracle(ctx, oracle, f, name):
    jobs, g = CASES[name], pico_amd.GENERATORS[f]
    hosts = [oracle.random_matrix(f, 70 + k, 1 << L, w) for k, (L, w, _) in enumerate(jobs)]
    mats = [ctx.upload(a, field=f) for a in hosts]
    batch = pico_amd.CommitBatch(ctx, f, [(m, b) for m, (_, _, b) in zip(mats, jobs)])
    for _ in range(2):
        roots = batch.run()
    for k, (a, (_, _, b)) in enumerate(zip(hosts, jobs)):
        ot = oracle.MerkleTree(f, [oracle.coset_lde(f, a, b, g)])
        assert np.array_equal(roots[k], ot.root), (name, k)
        tree = batch.take(k)
        for j in range(tree.log_height + 1):
            assert np.array_equal(tree.digest_layer(j), ot.layer(j)), (name, k, j)
        tree.free()
    batch.free()
    for m in mats:
        m.free()


def test_many_jobs(ctx, oracle):
    f, rng = KOALABEAR, np.random.default_rng(8)
    jobs = [(int(rng.integers(0, 6)), int(rng.integers(1, 40)), int(rng.integers(0, 2))) for _ in range(600)]
    hosts = [oracle.random_matrix(f, k, 1 << L, w) for k, (L, w, _) in enumerate(jobs)]
    mats = [ctx.upload(a, field=f) for a in hosts]
    batch = pico_amd.CommitBatch(ctx, f, [(m, b) for m, (_, _, b) in zip(mats, jobs)], use_graph=False)
    roots = batch.run()
    g = pico_amd.GENERATORS[f]
    for k, (a, (_, _, b)) in enumerate(zip(hosts, jobs)):
        assert np.array_equal(roots[k], oracle.MerkleTree(f, [oracle.coset_lde(f, a, b, g)]).root), k
    batch.free()
    for m in mats:
        m.free()


@pytest.mark.parametrize("f", [KOALABEAR, BABYBEAR])
@pytest.mark.parametrize("jobs", [
    [(L, 5, 1) for L in (14, 9, 7, 6, 5, 1, 0)],    # first layers of 2^14 .. 1 nodes, trees that end early
    [(6, 3, 0), (7, 3, 0), (8, 3, 0), (0, 3, 0)],   # 64, 128 and 256 leaves, and one
    [(5, 9, 1)] * 40,                               # one workgroup per tree
    [(4, 9, 1)] * 1100 + [(8, 2, 1)],               # more trees than run side by side, then one
], ids=["tall to short", "around a workgroup", "equal", "many"])
def test_levels_match_oracle(ctx, oracle, f, jobs):
    g = pico_amd.GENERATORS[f]
    hosts = [oracle.random_matrix(f, 900 + k, 1 << L, w) for k, (L, w, _) in enumerate(jobs)]
    mats = [ctx.upload(a, field=f) for a in hosts]
    batch = pico_amd.CommitBatch(ctx, f, [(m, b) for m, (_, _, b) in zip(mats, jobs)])
    for _ in range(2):
        roots = batch.run()
    for k, (a, (_, _, b)) in enumerate(zip(hosts, jobs)):
        ot = oracle.MerkleTree(f, [oracle.coset_lde(f, a, b, g)])
        assert np.array_equal(roots[k], ot.root), k
        if k % 100 < 8:
            tree = batch.take(k)
            for j in range(tree.log_height + 1):
                assert np.array_equal(tree.digest_layer(j), ot.layer(j)), (k, j)
            tree.free()
    batch.free()
    for m in mats:
        m.free()
