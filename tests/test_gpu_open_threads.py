"""Pcs::open on one context beside other opens and commits: every proof is the
one the call gives alone, every root the one the commit gives alone."""
import threading

import numpy as np
import pytest

import pico_amd
from pico_amd import BABYBEAR, KOALABEAR

pytestmark = pytest.mark.gpu


def test_concurrent_opens_and_commits(ctx, oracle):
    opens = []  # (pcs, data, root, points per matrix)
    for k, f in enumerate((KOALABEAR, BABYBEAR, KOALABEAR)):
        pcs = pico_amd.TwoAdicFriPcs(ctx, f, 1)
        shapes = [(6 + (3 * k + j) % 6, 3 + 17 * j + k) for j in range(9 + k)]
        mats = [ctx.random_matrix(f, 100 * k + j, 1 << L, w) for j, (L, w) in enumerate(shapes)]
        root, data = pcs.commit([(pcs.natural_domain_for_degree(1 << L), m) for (L, _), m in zip(shapes, mats)])
        for m in mats:
            m.free()
        pts = [np.array([[3 + j, 1, 4, k], [1, 5, 9, 2 + j % 2]][:1 + j % 2], np.uint64) for j in range(len(shapes))]
        opens.append((f, pcs, data, root, pts))
    big = ctx.random_matrix(KOALABEAR, 999, 1 << 15, 60)
    cpcs = pico_amd.TwoAdicFriPcs(ctx, KOALABEAR, 1)
    domain = cpcs.natural_domain_for_degree(1 << 15)

    def open_one(k):
        f, pcs, data, root, pts = opens[k]
        ch = pico_amd.DuplexChallenger(f)
        ch.observe(root)
        opened, proof = pcs.open([(data, pts)], ch, 11, 6)
        return proof["bincode"], [v.tolist() for per_round in opened for v in per_round], [int(x) for x in ch.sample_ext()]

    def commit_one():
        root, data = cpcs.commit([(domain, big)])
        data.free()
        return [int(x) for x in root]

    want, want_root = [open_one(k) for k in range(len(opens))], commit_one()
    wrong = []

    def opener(k):
        for _ in range(6):
            if open_one(k) != want[k]:
                wrong.append(("open", k))

    def committer():
        for _ in range(12):
            if commit_one() != want_root:
                wrong.append("commit")

    threads = [threading.Thread(target=opener, args=(k,)) for k in (0, 1, 2, 0, 1)]
    threads += [threading.Thread(target=committer) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    for _, _, data, _, _ in opens:
        data.free()
    big.free()
