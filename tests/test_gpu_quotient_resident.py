"""The quotient's two kernels at the edges of their shapes, against the oracle's
constraint evaluation: column runs of one column, of a piece (64 columns) and
one more, more pieces than are prefetched, scattered columns, programs that
share all their work or read more columns than a compute unit's memory holds
(the windowed kernel takes those), few and many constraints (4, 8 and 16
waves), fewer rows than a wave has lanes, and steps to the next row that carry
into a later block."""
import numpy as np
import pytest

import pico_amd
from pico_amd import BABYBEAR, KOALABEAR, air

pytestmark = pytest.mark.gpu


def _program(f, shape):
    """(builder, columns)"""
    b = air.AirBuilder(f)
    if shape == "one column":
        b.when_transition().assert_zero(b.main(0, next=True) - b.main(0) * b.main(0))
        b.when_first_row().assert_zero(b.main(0))
        return b, 1
    if shape == "shared":  # every constraint reads one long chain
        s = [b.main(c) for c in range(6)]
        for _ in range(5):
            t = s[0]
            for x in s[1:]:
                t = t + x
            s = [x * x * x + t for x in s]
        for c in range(6):
            b.assert_zero(s[c] - b.main(c, next=True))
        b.when_last_row().assert_zero(b.main(0))
        return b, 6
    if shape == "scattered":  # runs too far apart to join
        cols = [0, 1, 40, 90, 91, 150, 299]
        for i, c in enumerate(cols):
            b.when_last_row().assert_zero(b.main(c) * b.main(cols[i - 1]) - b.main(c, next=True))
        return b, 300
    width = {"64 columns": 64, "65 columns": 65, "20 columns": 20, "512 slots": 256, "700 columns": 700}[shape]
    for c in range(width):
        x = b.main(c) * b.main((c + 1) % width) - b.main((c + 7) % width, next=shape != "700 columns")
        if c % 5 == 0:
            b.assert_zero(-x)
        elif c % 5 == 1:
            b.when_first_row().assert_zero(x)
        else:
            b.when_transition().assert_zero(x * b.main(c) + 3)
    return b, width


@pytest.mark.parametrize("f", [KOALABEAR, BABYBEAR])
@pytest.mark.parametrize("shape", ["one column", "20 columns", "64 columns", "65 columns", "scattered", "512 slots",
                                   "700 columns", "shared"])
def test_quotient_shapes_match_oracle(ctx, oracle, f, shape):
    rng = np.random.default_rng(11 + f)
    p, g = pico_amd.PRIMES[f], pico_amd.GENERATORS[f]
    builder, width = _program(f, shape)
    prog = builder.compile()
    nodes, asserts = builder.node_array(), builder.asserts
    for log_n, qdb, lb in ((0, 0, 1), (1, 2, 2), (5, 1, 1), (6, 0, 1), (6, 2, 2), (10, 1, 1)):
        print(f"quotient {shape} field {f} 2^{log_n} qdb={qdb}", flush=True)
        pcs = pico_amd.TwoAdicFriPcs(ctx, f, lb)
        main = rng.integers(0, p, (1 << log_n, width)).astype(np.uint32)
        m = ctx.upload(main, field=f)
        _, data = pcs.commit([(pcs.natural_domain_for_degree(1 << log_n), m)])
        m.free()
        alpha = [int(x) for x in rng.integers(0, p, 4)]
        q = air.quotient_values(ctx, prog, data, 0, lb, qdb, alpha)
        got = q.to_host(f)
        q.free()
        data.free()
        want = oracle.quotient_values(f, nodes, asserts, oracle.coset_lde(f, main, qdb, g, bit_reverse=False),
                                      log_n, qdb, alpha)
        assert np.array_equal(got, want), (log_n, qdb, lb)
