"""Pcs::open under a budget that holds what opening one matrix after the other
takes, whatever the order of the matrices' sizes: the proof is the one an
unlimited context gives."""
import numpy as np
import pytest

import pico_amd
from pico_amd import BABYBEAR, KOALABEAR

pytestmark = pytest.mark.gpu

# (log height, width): the largest opening's partial sums are 8 MiB; all of them
# together 50 and more
WIDTHS = [40 + 40 * k for k in range(12)]
SHAPES = {"ascending": [(13, w) for w in WIDTHS], "descending": [(13, w) for w in WIDTHS[::-1]],
          "many columns, few rows": [(4, 3000 + 100 * k) for k in range(30)]}


@pytest.mark.parametrize("f", [KOALABEAR, BABYBEAR])
@pytest.mark.parametrize("order", list(SHAPES))
def test_open_within_budget(f, order):
    shapes, budget = SHAPES[order], 1 << 30
    points = np.array([[3, 1, 4, 1], [2, 7, 1, 8]], np.uint64)
    # 2^13 rows: 256 KiB of weights and 8 MiB of partial sums; 2^4 rows: all values
    # take 3 MiB, one matrix's partial sums and values 0.4
    room = {"many columns, few rows": 5 << 20}.get(order, (8 << 20) + (256 << 10))
    proofs = []
    with pico_amd.Context(0, budget) as ctx:
        pcs = pico_amd.TwoAdicFriPcs(ctx, f, 1)
        mats = [ctx.random_matrix(f, k, 1 << L, w) for k, (L, w) in enumerate(shapes)]
        root, data = pcs.commit([(pcs.natural_domain_for_degree(m.rows), m) for m in mats])
        held = [data]  # nothing may outlive the context
        for m in mats:
            m.free()
        try:
            for limited in (False, True):  # the first makes the tables that the context keeps
                if limited:
                    held.append(ctx.matrix((budget - ctx.bytes_in_use - room) // 512, 128))
                ch = pico_amd.DuplexChallenger(f)
                ch.observe(root)
                proofs.append(pcs.open([(data, [points] * len(shapes))], ch, 5, 3)[1]["bincode"])
        finally:
            for x in held:
                x.free()
    assert proofs[0] == proofs[1]
