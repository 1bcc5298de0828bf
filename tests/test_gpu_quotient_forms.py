"""Each program through both quotient kernels, whichever the rule would choose:
equal to the oracle's constraint evaluation and so to each other.  Minimal
programs, 4, 8 and 16 waves with even and uneven slices, slices of more than 64
and 128 instructions, more column pieces than are prefetched, every operand kind
(constants, public values, selectors, preprocessed columns, both rows), from 1
row to several blocks per workgroup."""
import numpy as np
import pytest

import pico_amd
from pico_amd import BABYBEAR, KOALABEAR, air
from pico_amd.air import RESIDENT, WINDOWED

pytestmark = pytest.mark.gpu


def _program(f, shape):
    """(builder, main columns, preprocessed columns, public values)"""
    b = air.AirBuilder(f)
    if shape == "one leaf":
        b.assert_zero(b.main(0))
        return b, 1, 0, 0
    if shape == "one column":
        b.when_transition().assert_zero(b.main(0, next=True) - b.main(0) * b.main(0))
        b.when_first_row().assert_zero(b.main(0))
        return b, 1, 0, 0
    if shape == "every operand":
        for c in range(24):
            x = b.main(c) * b.preprocessed(c % 5) - b.main((c + 1) % 24, next=True) + b.preprocessed(c % 3, next=True)
            y = x * b.public(c % 4) + (c * 7 + 1)
            [b, b.when_first_row(), b.when_last_row(), b.when_transition()][c % 4].assert_zero(-y if c % 2 else y * x)
        return b, 24, 5, 4
    if shape == "uneven":  # one constraint longer than the others together
        x = b.main(0)
        for k in range(300):
            x = x * b.main(k % 9) + b.main((k + 4) % 9, next=k % 3 == 0)
        b.assert_zero(x)
        for c in range(9):
            b.when_last_row().assert_zero(b.main(c) * b.main(c) - 1)
        return b, 9, 0, 0
    if shape == "pieces":  # runs too far apart to join, both rows: twelve pieces
        cols = [40 * k for k in range(5)] + [200 + j for j in range(70)]
        for i, c in enumerate(cols):
            b.when_transition().assert_zero(b.main(c) * b.main(cols[i - 1]) - b.main(c, next=i % 2 == 0))
        return b, cols[-1] + 1, 0, 0
    width = {"chain of 4 waves": 6, "8 waves": 44, "16 waves": 100, "long slices": 150}[shape]
    for c in range(width):
        x = b.main(c) * b.main((c + 1) % width) * b.main((c + 2) % width) - b.main(c, next=True)
        for k in range(12 if shape == "long slices" else 0):
            x = x * b.main((c + k) % width) + k
        b.when_transition().assert_zero(x)
    return b, width, 0, 0


SHAPES = ["one leaf", "one column", "every operand", "uneven", "pieces", "chain of 4 waves", "8 waves", "16 waves",
          "long slices"]


@pytest.mark.parametrize("f", [KOALABEAR, BABYBEAR])
@pytest.mark.parametrize("shape", SHAPES)
def test_both_forms_match_oracle(ctx, oracle, f, shape):
    rng = np.random.default_rng(31 + f)
    p, g = pico_amd.PRIMES[f], pico_amd.GENERATORS[f]
    builder, width, pre_width, npublic = _program(f, shape)
    prog = builder.compile()
    nodes, asserts = builder.node_array(), builder.asserts
    publics = [int(x) for x in rng.integers(0, p, npublic)]
    for log_n, qdb, lb in ((0, 0, 1), (2, 1, 1), (5, 1, 1), (6, 0, 1), (7, 2, 2), (11, 1, 1)):
        print(f"quotient forms {shape} field {f} 2^{log_n} qdb={qdb}", flush=True)
        pcs = pico_amd.TwoAdicFriPcs(ctx, f, lb)
        dom = pcs.natural_domain_for_degree(1 << log_n)
        datas, ldes = [], []
        for w in (width, pre_width):
            if not w:
                datas.append(None)
                ldes.append(None)
                continue
            host = rng.integers(0, p, (1 << log_n, w)).astype(np.uint32)
            m = ctx.upload(host, field=f)
            datas.append(pcs.commit([(dom, m)])[1])
            ldes.append(oracle.coset_lde(f, host, qdb, g, bit_reverse=False))
            m.free()
        alpha = [int(x) for x in rng.integers(0, p, 4)]
        want = oracle.quotient_values(f, nodes, asserts, ldes[0], log_n, qdb, alpha, publics=publics, pre_q=ldes[1])
        for form in (WINDOWED, RESIDENT):
            prog.debug_form(form)
            assert prog.form(1 << (log_n + qdb)) == form
            q = air.quotient_values(ctx, prog, datas[0], 0, lb, qdb, alpha, publics=publics, pre_data=datas[1])
            assert np.array_equal(q.to_host(f), want), (shape, log_n, qdb, form)
            q.free()
        for d in datas:
            if d:
                d.free()
