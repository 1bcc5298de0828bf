"""Leaf and injected rows of layers taller than the 16-state kernels take (2^16
rows: 64 states per wave): tails of every length, chunks that cross one or
several matrices, empty matrices, in the leaf layer and injected.  Every digest
layer equals the oracle's, bit for bit."""
import numpy as np
import pytest

import pico_amd
from pico_amd import BABYBEAR, KOALABEAR

pytestmark = pytest.mark.gpu
FIELDS = [KOALABEAR, BABYBEAR]
WIDTHS = [(8,), (24, 8), (1,), (2,), (3,), (4,), (5,), (6,), (7,), (9,), (15,), (17,), (20,), (31,), (5, 11), (3, 3, 3),
          (1, 1, 1, 1, 1, 1, 1, 1, 1), (12, 0, 13), (0, 8), (8, 4, 4), (4, 8, 7)]


def check_tree(ctx, oracle, f, hosts):
    mats = [ctx.upload(a, field=f) for a in hosts]
    root, pd = pico_amd.MerkleTreeMmcs(ctx, f).commit(mats)
    ot = oracle.MerkleTree(f, hosts)
    for j in range(pd.log_height + 1):
        assert np.array_equal(pd.digest_layer(j), ot.layer(j)), j
    assert np.array_equal(root, ot.root)
    pd.free()
    for m in mats:
        m.free()


@pytest.mark.parametrize("f", FIELDS)
@pytest.mark.parametrize("widths", WIDTHS, ids=lambda w: "+".join(map(str, w)))
def test_leaf_rows(ctx, oracle, f, widths):
    check_tree(ctx, oracle, f, [oracle.random_matrix(f, 50 + i, 1 << 16, w) for i, w in enumerate(widths)])


@pytest.mark.parametrize("f", FIELDS)
@pytest.mark.parametrize("widths", [(6,), (9,), (12, 0, 13), (0, 5), (1,) * 9, (4, 8, 7)], ids=lambda w: "+".join(map(str, w)))
def test_injected_rows(ctx, oracle, f, widths):
    check_tree(ctx, oracle, f, [oracle.random_matrix(f, 3, 1 << 17, 8)] +
               [oracle.random_matrix(f, 60 + i, 1 << 16, w) for i, w in enumerate(widths)])
