"""Poseidon2 on the matrix cores (16 or 64 states per wave) at the sizes where
it can go wrong: heights below, at and above one wave's rows, rows whose 8-word
chunks are partial or cross matrices, leaf layers and compress layers on both
sides of the limit between the two forms (2^15) with and without injected
rows, several layers per launch, and words at the ends of the field's range.  Every digest layer equals the oracle's, bit for bit."""
import numpy as np
import pytest

import pico_amd
from pico_amd import BABYBEAR, KOALABEAR

pytestmark = pytest.mark.gpu
FIELDS = [KOALABEAR, BABYBEAR]


def check_tree(ctx, oracle, f, hosts):
    root, pd = pico_amd.MerkleTreeMmcs(ctx, f).commit([ctx.upload(a, field=f) for a in hosts])
    ot = oracle.MerkleTree(f, hosts)
    for j in range(pd.log_height + 1):
        assert np.array_equal(pd.digest_layer(j), ot.layer(j)), j
    assert np.array_equal(root, ot.root)


# (widths of the tallest matrices): whole chunks, tails of every length,
# chunks that cross one or several matrices, an empty matrix in between
WIDTHS = [(8,), (16,), (24, 8)] + [(w,) for w in (1, 2, 3, 4, 5, 6, 7, 9, 15, 17, 20, 31)] + [
    (5, 11), (3, 3, 3), (1, 1, 1, 1, 1, 1, 1, 1, 1), (12, 0, 13), (8, 4, 4), (4, 8, 7)]


@pytest.mark.parametrize("f", FIELDS)
@pytest.mark.parametrize("widths", WIDTHS, ids=lambda w: "+".join(map(str, w)))
def test_leaf_rows(ctx, oracle, f, widths):
    for h in (1, 2, 32, 64, 128, 512):
        check_tree(ctx, oracle, f, [oracle.random_matrix(f, 7 * h + i, h, w) for i, w in enumerate(widths)])


@pytest.mark.parametrize("f", FIELDS)
@pytest.mark.parametrize("inj", [(), (8,), (5,), (3, 14)], ids=str)
def test_tall_layers(ctx, oracle, f, inj):
    # 2^17 leaves: layers of 2^16 and 2^15 nodes are above and at the limit
    hosts = [oracle.random_matrix(f, 1, 1 << 17, 8)]
    for log_h in (16, 15, 6):
        hosts += [oracle.random_matrix(f, 10 * log_h + k, 1 << log_h, w) for k, w in enumerate(inj)]
    check_tree(ctx, oracle, f, hosts)


@pytest.mark.parametrize("f", FIELDS)
@pytest.mark.parametrize("widths", [(16,), (7, 6)], ids=str)
@pytest.mark.parametrize("log_h", [15, 16])
def test_leaf_limit(ctx, oracle, f, widths, log_h):
    check_tree(ctx, oracle, f, [oracle.random_matrix(f, 3 + i, 1 << log_h, w) for i, w in enumerate(widths)])


@pytest.mark.parametrize("f", FIELDS)
def test_layers_per_launch(ctx, oracle, f):
    # every first-layer size: partial waves, one and two passes of a
    # workgroup, a second launch after seven layers, from 8-word rows and from
    # digests
    for log_h in range(0, 11):
        for w in (8, 9):
            check_tree(ctx, oracle, f, [oracle.random_matrix(f, log_h, 1 << log_h, w)])


@pytest.mark.parametrize("f", FIELDS)
def test_extreme_words(ctx, oracle, f):
    # Montgomery words 0, 1, p-1 and bytes 0x00, 0x7f, 0x80, 0xff, as they
    # reach the signed byte planes
    p = pico_amd.PRIMES[f]
    words = np.array([0, 1, p - 1, p - 2, 0x7F7F7F7F % p, 0x00808080, 0x00FFFFFF, 0x7F000000 % p, 0x0080FF7F, 0x007F7F80,
                      0x80, 0xFF, 0xFF00, 0x8000, 0x40404040, 0x3FFFFFFF], np.uint32)
    mont = words[np.random.default_rng(3).integers(0, words.size, (256, 19))]
    mont[0], mont[1] = 0, p - 1
    check_tree(ctx, oracle, f, [pico_amd.from_monty(f, mont)])


@pytest.mark.parametrize("f", FIELDS)
def test_batched_leaf_groups(ctx, oracle, f):
    # jobs of fewer than 64 rows, of exactly one group and of several
    jobs = [(0, 9, 1), (3, 8, 1), (5, 21, 1), (7, 16, 2), (9, 3, 1)]
    hosts = [oracle.random_matrix(f, 40 + k, 1 << L, w) for k, (L, w, _) in enumerate(jobs)]
    batch = pico_amd.CommitBatch(ctx, f, [(ctx.upload(a, field=f), b) for a, (_, _, b) in zip(hosts, jobs)])
    roots = batch.run()
    g = pico_amd.GENERATORS[f]
    for k, (a, (_, _, b)) in enumerate(zip(hosts, jobs)):
        ot = oracle.MerkleTree(f, [oracle.coset_lde(f, a, b, g)])
        assert np.array_equal(roots[k], ot.root), k
    batch.free()


@pytest.mark.parametrize("f", FIELDS)
@pytest.mark.parametrize("width", [3, 13, 24, 61])
def test_leaves_and_layers_in_one_launch(ctx, oracle, f, width):
    # one tallest matrix of one or several chunks, then injected rows: leaves and
    # the layers down to them share a launch (64 rows per workgroup, then more)
    for log_h, log_inj in ((4, 2), (6, 0), (7, 3), (9, 1), (13, 5)):
        check_tree(ctx, oracle, f, [oracle.random_matrix(f, log_h, 1 << log_h, width),
                                    oracle.random_matrix(f, 99, 1 << log_inj, 10)])
