"""Kernel families of the event timing: a launch that hashes leaves and layers
above them is a family of its own, and the leaf and layer families hold nothing
else."""
import pytest

import pico_amd
from pico_amd import KOALABEAR

pytestmark = pytest.mark.gpu
HASHING = ("leaf_hash", "leaf_hash_w8", "compress", "compress_inject", "tree_layers", "fri_fold")


def launches(ctx, call):
    ctx.profile(True)
    ctx.profile_reset()
    try:
        call()
    finally:
        ctx.profile(False)
    return {k: n for k in HASHING if (n := ctx.profile_get(k)[1])}


@pytest.mark.parametrize("log_h,width,want", [
    (5, 8, {"tree_layers"}),
    (5, 13, {"tree_layers"}),
    (14, 8, {"tree_layers"}),                # 2^15 leaves
    (15, 8, {"leaf_hash_w8", "compress"}),   # more than a launch of layers takes
    (15, 13, {"leaf_hash", "compress"}),
])
def test_commit(ctx, log_h, width, want):
    pcs = pico_amd.TwoAdicFriPcs(ctx, KOALABEAR, 1)
    m = ctx.random_matrix(KOALABEAR, 5, 1 << log_h, width)

    def call():
        _, data = pcs.commit([(pcs.natural_domain_for_degree(1 << log_h), m)])
        data.free()

    assert set(launches(ctx, call)) == want
    m.free()


def test_fri_commit_phase(ctx):
    v = ctx.random_matrix(KOALABEAR, 5, 1 << 18, 4)

    def call():
        pico_amd.fri_commit_phase(ctx, KOALABEAR, pico_amd.DuplexChallenger(KOALABEAR), {18: v}, 2, final_mode=1).free()

    got = launches(ctx, call)
    # 16 rounds: trees of 2^17 and 2^16 leaves hash them apart, fourteen lower ones do not
    assert got["leaf_hash_w8"] == 2 and got["tree_layers"] == 14 and got["compress"] >= 2
    assert got["fri_fold"] == 2  # the second round's vector and the final one; the others in the tree launches
    v.free()
