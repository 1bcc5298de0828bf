"""Performance cases of the commitment path: the calls a prover makes, through
the package's public interface, over the sizes it makes them at.

Every output is a whole number (field elements, Merkle digests, proof bytes),
so a result is either the right one or wrong; there are no rounding errors to
measure.  `work` counts bytes as each input read once and each output written
once, and operations as the field additions and multiplications of the
textbook form (radix-2 butterflies, the Poseidon2 permutation as defined).
"""
import math

import numpy as np
import torch

from pico_amd import air, core, workloads

FIELDS = {"koalabear": core.KOALABEAR, "babybear": core.BABYBEAR}

_context = None


def context():
    """The one device context a prover process keeps."""
    global _context
    if _context is None:
        _context = core.Context(0)
    return _context


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # A small chip's table (byte lookups, program memory): launches and
        # host work are all there is.
        {"name": "commit_small", "kind": "commit", "field": "koalabear", "log_h": 8, "width": 13, "log_blowup": 1},
        # The main trace of one large chip: the benchmark's shape.
        {"name": "commit_large", "kind": "commit", "field": "koalabear", "log_h": 20, "width": 256, "log_blowup": 1},
        # A recursion-style commit: BabyBear, ragged width, blowup 8.
        {"name": "commit_blowup8", "kind": "commit", "field": "babybear", "log_h": 17, "width": 203, "log_blowup": 3},
        # One shard's 40 chip tables in one mixed-height commit.
        {"name": "commit_tables", "kind": "tables", "field": "koalabear", "tables": 40, "min_log": 10, "max_log": 22,
         "shape_seed": 6 << 32, "log_blowup": 1},
        # A trace that the emulator left in ordinary host memory.
        {"name": "commit_host", "kind": "host", "field": "koalabear", "log_h": 18, "width": 150, "log_blowup": 1},
        # The bare DFT trait: a tall, narrow extension in natural row order.
        {"name": "lde_tall", "kind": "lde", "field": "babybear", "log_h": 21, "width": 45, "log_blowup": 1},
        # Mmcs over matrices that are already extended, then a verifier's queries.
        {"name": "mmcs_queries", "kind": "mmcs", "field": "koalabear", "log_h": 18, "width": 100, "width2": 37,
         "width3": 19, "queries": 50},
        # Pcs::open of a main and a quotient round: values, reduced openings,
        # FRI, proof of work and every query opening.
        {"name": "open", "kind": "open", "field": "koalabear", "tables": 10, "min_log": 10, "max_log": 19,
         "shape_seed": 11, "log_blowup": 1, "queries": 100, "pow_bits": 16},
        # The FRI commit phase alone: many short rounds, each a tree.
        {"name": "fri_commit", "kind": "fri", "field": "babybear", "log_n": 18, "log_second": 15, "log_stop": 4},
        # The constraint quotient of a wide chip.
        {"name": "quotient_wide", "kind": "quotient", "field": "koalabear", "log_n": 20, "width": 256},
        # The permutation (LogUp) side of a lookup-heavy chip.
        {"name": "quotient_lookups", "kind": "lookups", "field": "koalabear", "log_n": 17, "width": 90,
         "interactions": 24},
        # Many independent jobs of a proving service as one captured sequence.
        {"name": "batch", "kind": "batch", "field": "koalabear", "jobs": 64, "min_log": 10, "max_log": 18,
         "max_width": 512, "shape_seed": 4 << 32},
    ]


def _ragged(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["commit", "commit", "commit", "tables", "host", "lde", "mmcs", "open", "fri", "quotient",
                       "lookups", "batch"])
    field = rng.choice(["koalabear", "babybear"])
    if kind in ("commit", "host", "lde"):
        lb = rng.choice([1, 1, 2, 3])
        log_h = rng.randint(4, 21)
        top = max(4, min(512, 1 << max(2, 28 - log_h - lb)))
        return {"kind": kind, "field": field, "log_h": log_h, "width": _ragged(rng, 3, top), "log_blowup": lb}
    if kind == "tables":
        return {"kind": kind, "field": field, "tables": rng.randint(5, 40), "min_log": rng.randint(4, 10),
                "max_log": rng.randint(14, 20), "shape_seed": rng.randrange(1 << 30), "log_blowup": 1}
    if kind == "mmcs":
        return {"kind": kind, "field": field, "log_h": rng.randint(6, 20), "width": _ragged(rng, 3, 200),
                "width2": _ragged(rng, 3, 100), "width3": _ragged(rng, 1, 60), "queries": rng.randint(1, 120)}
    if kind == "open":
        return {"kind": kind, "field": field, "tables": rng.randint(2, 14), "min_log": rng.randint(5, 10),
                "max_log": rng.randint(12, 19), "shape_seed": rng.randrange(1 << 30), "log_blowup": rng.choice([1, 1, 3]),
                "queries": rng.randint(20, 100), "pow_bits": rng.choice([8, 16])}
    if kind == "fri":
        log_n = rng.randint(8, 22)
        return {"kind": kind, "field": field, "log_n": log_n, "log_second": rng.randint(6, log_n - 1),
                "log_stop": rng.randint(1, 5)}
    if kind == "quotient":
        return {"kind": kind, "field": field, "log_n": rng.randint(8, 20), "width": _ragged(rng, 4, 256)}
    if kind == "lookups":
        return {"kind": kind, "field": "koalabear", "log_n": rng.randint(8, 18), "width": _ragged(rng, 12, 200),
                "interactions": rng.randint(2, 32)}
    return {"kind": kind, "field": field, "jobs": rng.randint(4, 64), "min_log": rng.randint(6, 10),
            "max_log": rng.randint(12, 17), "max_width": _ragged(rng, 16, 512), "shape_seed": rng.randrange(1 << 30)}


def _batch_shapes(case):
    r = workloads.SplitMix64(case["shape_seed"])
    return [(r.uniform_int(case["min_log"], case["max_log"]), r.uniform_int(8, case["max_width"]), r.uniform_int(1, 3))
            for _ in range(case["jobs"])]


def _table_shapes(case):
    return workloads.chip_table_shapes(case["shape_seed"], case["tables"], case["min_log"], case["max_log"])


def _wide_air(field, width):
    """One degree-3 transition constraint per column."""
    b = air.AirBuilder(field)
    for c in range(width):
        x, y, z = b.main(c), b.main((c + 1) % width), b.main((c + 2) % width)
        b.when_transition().assert_zero(x * y * z - b.main(c, next=True))
    return b


# ---------------------------------------------------------------- prepare --
def prepare(case, seed):
    ctx, f, kind = context(), FIELDS[case["field"]], case["kind"]
    p = core.PRIMES[f]
    rng = np.random.default_rng(seed)
    stream = (seed & 0xFFFFFFFF) << 16
    s = {"kind": kind, "ctx": ctx, "field": f}

    def matrix(k, log_h, width):
        return ctx.random_matrix(f, stream | k, 1 << log_h, width)

    def ext(n):
        return rng.integers(1, p, (n, 4)).astype(np.uint64)

    if kind in ("commit", "host", "lde"):
        m = matrix(0, case["log_h"], case["width"])
        s["added_bits"] = case["log_blowup"]
        s["dft"], s["shift"] = core.Radix2DitParallel(ctx, f), core.GENERATORS[f]
        s["pcs"] = core.TwoAdicFriPcs(ctx, f, case["log_blowup"])
        s["domain"] = s["pcs"].natural_domain_for_degree(m.rows)
        s["trace"] = m.to_host() if kind == "host" else m
    elif kind == "tables":
        s["pcs"] = core.TwoAdicFriPcs(ctx, f, case["log_blowup"])
        mats = [matrix(k, h, w) for k, (h, w) in enumerate(_table_shapes(case))]
        s["evaluations"] = [(s["pcs"].natural_domain_for_degree(m.rows), m) for m in mats]
    elif kind == "mmcs":
        s["mmcs"] = core.MerkleTreeMmcs(ctx, f)
        h = case["log_h"]
        s["mats"] = [matrix(0, h, case["width"]), matrix(1, h, case["width2"]), matrix(2, h - 3, case["width3"])]
        s["indices"] = rng.integers(0, 1 << h, case["queries"])
    elif kind == "open":
        s["pcs"] = core.TwoAdicFriPcs(ctx, f, case["log_blowup"])
        dom = s["pcs"].natural_domain_for_degree
        shapes = _table_shapes(case)
        mats = [matrix(k, h, w) for k, (h, w) in enumerate(shapes)]
        root, main = s["pcs"].commit([(dom(m.rows), m) for m in mats])
        top = max(h for h, _ in shapes)
        qroot, quot = s["pcs"].commit([(dom(1 << top), matrix(200, top, 8))])
        s["challenger"] = core.DuplexChallenger(f)
        s["challenger"].observe(root)
        s["challenger"].observe(qroot)
        zeta = ext(1)
        pair = np.concatenate([zeta, zeta * core.two_adic_generator(f, top) % p])
        s["rounds"] = [(main, [pair] * len(shapes)), (quot, [zeta])]
        s["queries"], s["pow_bits"] = case["queries"], case["pow_bits"]
    elif kind == "fri":
        s["inputs"] = {case["log_n"]: matrix(0, case["log_n"], 4), case["log_second"]: matrix(1, case["log_second"], 4)}
        s["challenger"], s["log_stop"] = core.DuplexChallenger(f), case["log_stop"]
    elif kind in ("quotient", "lookups"):
        n, w = case["log_n"], case["width"]
        pcs = core.TwoAdicFriPcs(ctx, f, 1)
        dom = pcs.natural_domain_for_degree(1 << n)
        _, s["main"] = pcs.commit([(dom, matrix(0, n, w))])
        s["alpha"] = [int(x) for x in ext(1)[0]]
        if kind == "quotient":
            builder, s["extra"] = _wide_air(f, w), {}
        else:
            builder, cols = workloads.lookup_air(w, case["interactions"], 2)
            _, perm = pcs.commit([(dom, matrix(1, n, 4 * cols))])
            s["extra"] = {"perm_data": perm, "challenges": ext(2).tolist(), "regional_sum": ext(1)[0].tolist()}
        s["program"] = builder.compile()
    else:
        jobs = [(matrix(k, h, w), lb) for k, (h, w, lb) in enumerate(_batch_shapes(case))]
        s["batch"] = core.CommitBatch(ctx, f, jobs)
    return s


class _DeviceArray:
    """A device matrix as an array-interface object; it keeps its owner alive
    for as long as a tensor made from it exists."""

    def __init__(self, matrix, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (matrix.rows, matrix.cols), "typestr": "<i4", "version": 2,
                                         "data": (matrix.device_ptr, False)}


def _tensor(matrix, owner):
    return torch.as_tensor(_DeviceArray(matrix, owner), device="cuda")


# -------------------------------------------------------------------- run --
def run(state):
    kind, ctx, f = state["kind"], state["ctx"], state["field"]
    if kind == "commit":
        root, data = state["pcs"].commit([(state["domain"], state["trace"])])
        return {"root": root, "lde": _tensor(_matrices(data)[0], data)}
    if kind == "host":
        root, data = state["pcs"].commit_host([(state["domain"], state["trace"])], canonical=False)
        return {"root": root, "lde": _tensor(_matrices(data)[0], data)}
    if kind == "lde":
        lde = state["dft"].coset_lde_batch(state["trace"], state["added_bits"], state["shift"], bit_reversed=False)
        return _tensor(lde, lde)
    if kind == "tables":
        root, data = state["pcs"].commit(state["evaluations"])
        return {"root": root, "ldes": [_tensor(m, data) for m in _matrices(data)]}
    if kind == "mmcs":
        root, data = state["mmcs"].commit(state["mats"])
        rows, paths = state["mmcs"].open_many(state["indices"], data)
        return {"root": root, "rows": rows, "paths": paths}
    if kind == "open":
        opened, proof = state["pcs"].open(state["rounds"], state["challenger"].clone(), state["queries"],
                                          state["pow_bits"])
        return {"values": np.concatenate([v.reshape(-1) for per_round in opened for v in per_round]),
                "alpha": proof["alpha"], "betas": proof["betas"], "witness": proof["pow_witness"],
                "indices": np.array(proof["query_indices"], np.int64),
                "proof": np.frombuffer(proof["bincode"], np.uint8)}
    if kind == "fri":
        fri = core.fri_commit_phase(ctx, f, state["challenger"].clone(), state["inputs"], state["log_stop"],
                                    final_mode=1)
        return {"commits": fri.commits, "betas": fri.betas, "final": fri.final_poly}
    if kind in ("quotient", "lookups"):
        q = air.quotient_values(ctx, state["program"], state["main"], 0, 1, 1, state["alpha"], **state["extra"])
        return _tensor(q, q)
    return state["batch"].run()


def _matrices(data):
    return core.MerkleTreeMmcs(data.ctx, data.field).get_matrices(data)


# ------------------------------------------------------------------- work --
def _permutation_ops(field):
    full, partial, cube = (8, 20, 2) if field == "koalabear" else (8, 13, 4)
    external = 4 * 11 + 12 + 16  # additions of one external layer
    internal = 15 + 2 * 16
    return (full + 1) * external + full * 16 * (1 + cube) + partial * (1 + cube + internal)


def _lde_work(log_h, w, lb):
    h, n = 1 << log_h, 1 << (log_h + lb)
    return 4 * (h + n) * w, 3 * w * (h // 2 * log_h + n // 2 * log_h) + 2 * n * w


def _tree_perms(shapes):
    """Permutations of a Merkle tree over matrices of (log height, width)."""
    by = {}
    for h, w in shapes:
        by[h] = by.get(h, 0) + w
    top = max(by)
    perms = sum((1 << h) * (-(-w // 8) + (h < top)) for h, w in by.items())
    return perms + (1 << top) - 1, 32 * ((2 << top) - 1)


def _commit_work(field, shapes):
    b = o = 0
    for h, w, lb in shapes:
        x, y = _lde_work(h, w, lb)
        b, o = b + x, o + y
    perms, digests = _tree_perms([(h + lb, w) for h, w, lb in shapes])
    return b + digests, o + perms * _permutation_ops(field)


def work(case):
    kind, field = case["kind"], case["field"]
    if kind in ("commit", "host"):
        b, o = _commit_work(field, [(case["log_h"], case["width"], case["log_blowup"])])
    elif kind == "lde":
        b, o = _lde_work(case["log_h"], case["width"], case["log_blowup"])
    elif kind == "tables":
        b, o = _commit_work(field, [(h, w, case["log_blowup"]) for h, w in _table_shapes(case)])
    elif kind == "mmcs":
        h = case["log_h"]
        shapes = [(h, case["width"]), (h, case["width2"]), (h - 3, case["width3"])]
        perms, digests = _tree_perms(shapes)
        b = digests + sum(4 * w << k for k, w in shapes)
        b += case["queries"] * (4 * sum(w for _, w in shapes) + 32 * h)
        o = perms * _permutation_ops(field)
    elif kind == "open":
        lb = case["log_blowup"]
        shapes = [(h, w, 2) for h, w in _table_shapes(case)]
        top = max(h for h, _, _ in shapes)
        shapes.append((top, 8, 1))
        b = o = 0
        for h, w, npts in shapes:  # values: the trace-sized part; reduced openings: the whole LDE
            b += 4 * w << (h + lb)
            o += 8 * w * npts << h
            o += 8 * w << (h + lb)
        perms, digests = _tree_perms([(top + lb - 1, 8)])  # FRI: trees of halving size
        b += 2 * digests + (4 * 16 << (top + lb))
        o += (2 * perms + (1 << case["pow_bits"])) * _permutation_ops(field)
    elif kind == "fri":
        perms, digests = _tree_perms([(case["log_n"] - 1, 8)])
        b = 2 * digests + 3 * (16 << case["log_n"]) + (16 << case["log_second"])
        o = 2 * perms * _permutation_ops(field) + (60 << case["log_n"])
    elif kind == "quotient":
        q = 1 << (case["log_n"] + 1)
        b = q * (4 * case["width"] + 16)
        o = q * case["width"] * 12  # three products, a difference, the fold into ext4
    elif kind == "lookups":
        q, i = 1 << (case["log_n"] + 1), case["interactions"]
        read = min(case["width"], 2 * i + 2) + 4 * (i // 2 + 1)
        b = q * (4 * read + 16)
        o = q * i * 110  # two ext4 products and a fold per interaction, running sum
    else:
        b = o = 0
        for h, w, lb in _batch_shapes(case):
            x, y = _commit_work(field, [(h, w, lb)])
            b, o = b + x, o + y
    return {"bytes": int(b), "flops": int(o)}
