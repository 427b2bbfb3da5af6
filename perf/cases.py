"""Performance cases: the work a program gives this library, through its Python entry points.

Six kinds of work, each over the range of sizes the benchmark, the tests and the configurations
use:

* ``host``    one chain join on host columns, results fetched to the host (exec-AMHJ's whole
              path for a small query: upload, hash builds, probe, download);
* ``chain``   a chain join over relations resident in HBM, with the hash builds (``step``) or over
              tables built before (``resident``), materialised or counted, through the engines the
              switches choose: the defaults (count pass + write pass), ``fib=1 ws=1 dro=1`` (the
              benchmark's switches; the frequent-item writer), or ``ws=1`` (work sharing);
* ``batch``   several small chain queries and a triangle query over resident tables as one batch;
* ``lftj``    a leapfrog triejoin over a graph's edges: the trie build and the triangles written
              (``step``), or triangles / 4-cliques counted over a resident trie;
* ``amhj``    TRI or FOUR over the hash table of a graph's edges, table build included.

A pass returns the result columns (device memory of the library, wrapped without a copy and
released with the last tensor), the count and, where the options compute it, the checksum. The
passes that place rows by atomic reservation (dro without fib) are not listed on their own: their
row order is not reproducible.
"""
import math

import numpy as np
import torch

from accmultiwayjoins_amd import Context
from accmultiwayjoins_amd import generators as G
from accmultiwayjoins_amd.serving import Batch, device_rmat

TRI = [(0, 1), (1, 2), (0, 2)]
FOUR = [(0, 1), (1, 2), (2, 3), (0, 3), (0, 2), (1, 3)]
ENGINES = {"plain": {}, "fib": {"ws": 1, "dro": 1, "fib": 1}, "ws": {"ws": 1}}
EDGE_FACTOR = 16


def listed():
    return [
        # the smallest whole call: 4,096 rows per relation from host memory and back (the size of
        # the recorded 3-way chain fixture); launches, allocations and copies are all there is
        {"name": "host_chain3_4k", "kind": "host", "n0": 4096, "n1": 4096, "n2": 4096, "n3": 0,
         "n4": 0, "keys": 1024, "zipf": 0.0, "engine": "plain"},
        # the first configuration at full size: 1 M tuples per relation, default switches
        {"name": "chain3_1m", "kind": "chain", "n0": 1_000_000, "n1": 1_000_000, "n2": 1_000_000,
         "n3": 0, "n4": 0, "keys": 1_000_000, "zipf": 0.0, "engine": "plain", "resident": False,
         "mat": True},
        # an ordinary served query: five relations of odd sizes, skewed, tables resident
        {"name": "chain5_ragged", "kind": "chain", "n0": 300_007, "n1": 65_537, "n2": 50_021,
         "n3": 40_009, "n4": 70_001, "keys": 50_021, "zipf": 0.8, "engine": "plain",
         "resident": True, "mat": True},
        # the benchmark's 4-way chain at a quarter of its size: 1.07 G result rows, 21 GB
        {"name": "chain4_16m_fib", "kind": "chain", "n0": 1 << 24, "n1": 1 << 22, "n2": 1 << 22,
         "n3": 1 << 22, "n4": 0, "keys": 1 << 20, "zipf": 0.0, "engine": "fib",
         "resident": False, "mat": True},
        # the same shape at odd sizes with the benchmark's strongest skew
        {"name": "chain4_4m_zipf1_fib", "kind": "chain", "n0": 4_000_037, "n1": 1_000_003,
         "n2": 999_983, "n3": 1_048_583, "n4": 0, "keys": 262_147, "zipf": 1.0, "engine": "fib",
         "resident": False, "mat": True},
        # counting only (count + checksum) with work sharing over resident tables
        {"name": "chain3_20m_ws_count", "kind": "chain", "n0": 20_000_000, "n1": 10_000_000,
         "n2": 10_000_000, "n3": 0, "n4": 0, "keys": 10_000_000, "zipf": 0.5, "engine": "ws",
         "resident": True, "mat": False},
        # a serving batch: nine small chains and one triangle query in one run
        {"name": "batch_10", "kind": "batch", "queries": 10, "lo": 1_000, "hi": 100_000,
         "scale": 11},
        # triangles of a small graph, trie build included: launch-bound
        {"name": "tri_12", "kind": "lftj", "scale": 12, "query": "TRI", "resident": False,
         "mat": True, "ws": 0},
        # the benchmark's graph: trie build + 2.1 G triangles written (25 GB)
        {"name": "tri_22", "kind": "lftj", "scale": 22, "query": "TRI", "resident": False,
         "mat": True, "ws": 0},
        # triangles of an ordinary graph counted over a resident trie
        {"name": "tri_20_count", "kind": "lftj", "scale": 20, "query": "TRI", "resident": True,
         "mat": False, "ws": 0},
        # 4-cliques counted with work sharing over a resident trie (the served FOUR request)
        {"name": "four_18_ws", "kind": "lftj", "scale": 18, "query": "FOUR", "resident": True,
         "mat": False, "ws": 1},
        # TRI through the hash-join engine, table build included
        {"name": "amhj_tri_17", "kind": "amhj", "scale": 17, "query": "TRI", "mat": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["host", "chain_plain", "chain_plain", "chain_fib", "chain_fib",
                       "chain_count", "batch", "tri", "tri", "tri_count", "four", "amhj"])
    if kind == "batch":
        return {"kind": "batch", "queries": rng.randint(4, 10), "lo": 1_000,
                "hi": _log_int(rng, 20_000, 200_000), "scale": rng.randint(9, 12)}
    if kind == "tri":
        return {"kind": "lftj", "scale": rng.randint(10, 21), "query": "TRI",
                "resident": rng.random() < 0.3, "mat": True, "ws": 0}
    if kind == "tri_count":
        return {"kind": "lftj", "scale": rng.randint(12, 21), "query": "TRI",
                "resident": rng.random() < 0.7, "mat": False, "ws": rng.randint(0, 1)}
    if kind == "four":
        return {"kind": "lftj", "scale": rng.randint(10, 18), "query": "FOUR",
                "resident": rng.random() < 0.7, "mat": False, "ws": rng.randint(0, 1)}
    if kind == "amhj":
        if rng.random() < 0.3:
            return {"kind": "amhj", "scale": rng.randint(10, 14), "query": "FOUR", "mat": False}
        return {"kind": "amhj", "scale": rng.randint(10, 18), "query": "TRI",
                "mat": rng.random() < 0.7}
    k = rng.randint(3, 5)
    lo, hi = {"host": (500, 20_000), "chain_plain": (5_000, 3_000_000),
              "chain_fib": (1 << 18, 1 << 24), "chain_count": (100_000, 20_000_000)}[kind]
    n0 = _log_int(rng, lo, hi)
    # build tables between a quarter of the probe relation and its size, the keys such that a
    # probe row has one match on average, or up to four in the benchmark's shape
    build = [max(64, int(n0 * rng.uniform(0.25, 1.0))) for _ in range(k - 1)]
    if kind == "chain_fib":
        build = [max(64, n0 // 4 + rng.randint(0, n0 // 16)) for _ in range(k - 1)]
        # at most 20 GB of result rows
        fan = min(rng.uniform(1.5, 4.0), (20e9 / (4 * (k + 1) * n0)) ** (1 / (k - 1)))
        keys = max(16, int(max(build) / fan))
    else:
        keys = max(16, max(build))
    case = {"kind": "host" if kind == "host" else "chain", "n0": n0}
    for i in range(4):
        case["n%d" % (i + 1)] = build[i] if i < k - 1 else 0
    case.update(keys=keys, zipf=round(rng.choice([0.0, rng.uniform(0.2, 1.2)]), 2),
                engine={"chain_fib": "fib", "chain_count": rng.choice(["ws", "plain"])}.get(
                    kind, "plain"))
    if kind != "host":
        case.update(resident=rng.random() < 0.4, mat=kind != "chain_count")
    return case


def _sizes(case):
    return [case["n%d" % i] for i in range(5) if case["n%d" % i]]


_contexts = {}


def _context():
    """One context per process, as a program keeps one per GPU."""
    if not _contexts:
        _contexts["ctx"] = Context(0)
    return _contexts["ctx"]


# A case's sizes say how many rows go in; its results have a size of their own, which a program
# that repeats a query of one shape sees change little. The structure of the inputs is drawn with
# one fixed seed, and the seed of a state gives every join key and vertex another value, the
# payload columns other values and the relations another row order: other inputs, results of the
# same size.
_STRUCTURE = 42


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _edges(ctx, scale, seed):
    """Edges of an R-MAT graph, symmetrised, deduplicated and oriented from the lower to the higher
    degree, stored as sorted CSR, vertices numbered by the seed."""
    cols = device_rmat(ctx, scale, EDGE_FACTOR, seed=_STRUCTURE)
    src, dst = (torch.from_numpy(cols.to_host(c)).cuda().long() for c in (0, 1))
    cols.close()
    number = torch.randperm(1 << scale, device="cuda", generator=_generator(seed))
    pairs = torch.sort((number[src] << 32) | number[dst]).values
    return ctx.relation([(pairs >> 32).int().cpu().numpy(), pairs.int().cpu().numpy()], [0, 1])


def _chain(sizes, keys, zipf, seed):
    rels = G.chain_relations(sizes, keys, seed=_STRUCTURE, zipf_s=zipf, payload_range=1 << 31)
    gen = _generator(seed)
    number = {}
    out = []
    for i, (cols, ids) in enumerate(rels):
        order = torch.randperm(sizes[i], device="cuda", generator=gen)
        new = []
        for col, attr in zip(cols, ids):
            if attr in (0, len(sizes)):  # the outer columns join with nothing
                v = torch.randint(1 << 31, (sizes[i],), device="cuda", generator=gen)
            else:
                if attr not in number:
                    number[attr] = torch.randperm(keys, device="cuda", generator=gen)
                v = number[attr][torch.from_numpy(col).cuda().long()][order]
            new.append(v.int().cpu().numpy())
        out.append((new, ids))
    return out


def _batch_sizes(case, q):
    """Relation sizes of chain query q, spread over the batch's range."""
    k = 3 + q % 3
    span = math.log(case["hi"] / case["lo"])
    return [int(case["lo"] * math.exp(span * ((q * 7 + i * 5) % 11) / 10)) | 1 for i in range(k)]


def prepare(case, seed):
    ctx = _context()
    state = {"ctx": ctx, "case": case}
    if case["kind"] == "host":
        state["rels"] = _chain(_sizes(case), case["keys"], case["zipf"], seed)
    elif case["kind"] == "chain":
        rels = _chain(_sizes(case), case["keys"], case["zipf"], seed)
        state["rels"] = [ctx.relation(c, ids) for c, ids in rels]
        if case["resident"]:
            state["tables"] = [ctx.hash_table(r) for r in state["rels"][1:]]
    elif case["kind"] == "batch":
        state["queries"] = []
        for q in range(case["queries"] - 1):
            sizes = _batch_sizes(case, q)
            rels = _chain(sizes, max(sizes[1:]), 0.1 * q, seed + q)
            rels = [ctx.relation(c, ids) for c, ids in rels]
            state["queries"].append((rels, [ctx.hash_table(r) for r in rels[1:]]))
        edges = _edges(ctx, case["scale"], seed)
        state["edges"] = (edges, ctx.hash_table(edges, 0, sort_vals=True))
    else:
        state["edges"] = _edges(ctx, case["scale"], seed)
        if case["kind"] == "lftj" and case["resident"]:
            state["trie"] = ctx.trie_from_relation(state["edges"])
    return state


class _Rows:
    """The device columns of one result; released when the last view is dropped."""

    def __init__(self, ctx, result):
        self.ctx, self.result = ctx, result

    def __del__(self):
        self.ctx.free(self.result)


class _Column:
    def __init__(self, rows, pointer, n):
        self.rows = rows
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<i4", "version": 2,
                                         "data": (pointer, False), "strides": None}


def _signed(checksum):
    return checksum - (1 << 64) if checksum >= 1 << 63 else checksum


def _outputs(ctx, r):
    out = [r.count, _signed(r.checksum)]
    if r.rows_written:
        rows = _Rows(ctx, r)
        out += [torch.as_tensor(_Column(rows, r._res.cols[a], r.rows_written), device="cuda")
                for a in range(len(r.attr_ids))]
    else:
        ctx.free(r)
    return out


def run(state):
    ctx, case = state["ctx"], state["case"]
    if case["kind"] == "host":
        r = ctx.chain_join(state["rels"], fetch=True, **ENGINES[case["engine"]])
        return [r.count, _signed(r.checksum)] + r.cols
    if case["kind"] == "chain":
        rels = state["rels"]
        tables = state["tables"] if case["resident"] else [ctx.hash_table(r) for r in rels[1:]]
        r = ctx.execute(rels[0], tables, materialize=case["mat"], **ENGINES[case["engine"]])
        if not case["resident"]:
            for t in tables:
                t.close()
        return _outputs(ctx, r)
    if case["kind"] == "batch":
        batch = Batch(ctx)
        ids = [batch.add(rels[0], tables) for rels, tables in state["queries"]]
        ids.append(batch.add_pattern(*state["edges"], "TRI"))
        batch.run()
        out = [_outputs(ctx, batch.result(i)) for i in ids]
        batch.close()
        # counts and checksums of the queries as one array, then every result column
        return [np.array([o[:2] for o in out], dtype=np.int64)] + [c for o in out for c in o[2:]]
    if case["kind"] == "lftj":
        trie = state["trie"] if case["resident"] else ctx.trie_from_relation(state["edges"])
        pairs = TRI if case["query"] == "TRI" else FOUR
        order = list(range(3 if case["query"] == "TRI" else 4))
        r = ctx.lftj([trie] * len(pairs), order, "DFS", trie_attrs=pairs,
                     materialize=case["mat"], ws=case["ws"])
        if not case["resident"]:
            trie.close()
        return _outputs(ctx, r)
    table = ctx.hash_table(state["edges"], 0, sort_vals=True)
    r = ctx.execute_pattern(state["edges"], table, case["query"], materialize=case["mat"])
    table.close()
    return _outputs(ctx, r)


def _chain_bytes(sizes, keys, mat):
    """Columns in once, result rows out once. Probe-side keys are uniform over `keys`, so every
    join multiplies the expected rows by (build rows / keys) whatever the build side's skew."""
    rows = float(sizes[0])
    for n in sizes[1:]:
        rows *= n / keys
    return 8 * sum(sizes) + (4 * (len(sizes) + 1) * rows if mat else 0)


def work(case):
    if case["kind"] in ("host", "chain"):
        return {"bytes": _chain_bytes(_sizes(case), case["keys"], case.get("mat", True)),
                "flops": 0}
    # R-MAT, edge factor 16: edges kept after deduplication, and triangles, by scale (powers
    # fitted to the generator's counts at scales 10 and 22)
    edges = 15.3 * 2 ** case["scale"]
    triangles = 75564 * 2.347 ** (case["scale"] - 10)
    if case["kind"] == "batch":
        total = 8 * edges + 12 * triangles
        for q in range(case["queries"] - 1):
            sizes = _batch_sizes(case, q)
            total += _chain_bytes(sizes, max(sizes[1:]), True)
        return {"bytes": total, "flops": 0}
    return {"bytes": 8 * edges + (12 * triangles if case["mat"] else 0), "flops": 0}


def exact(case, seed):
    """Every output is a whole number (keys, counts, checksums): there is nothing to round."""
    return None
