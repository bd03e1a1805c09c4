"""The work a user of the engine has it do, as timed cases.

Every case is one pass through the public entry points of the `hvm64`
package: a net made, booted, reduced to normal form and read back, the
batched and serving forms of the same, or one evaluation of an expression
from its text.  Programs come from `hvm64.configs` (the two programs shipped
with the package and the Church numerals); the seed decides the numbers in
them: sort keys, leaves, offsets, operands.

A case's `kind` names the flow (the functions below), its sizes and heap
are the caller's choices.  Heap sizes matter: a net that allocates more nodes
than its heap holds reuses freed ones.
"""
import math
import os
import random
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "hvm-64_amd"))

import hvm64  # noqa: E402
from hvm64 import configs, serve  # noqa: E402

VARIANTS = [("tree_sum", d) for d in range(8, 17)] + [("bitonic", k) for k in range(6, 13)]
MIB = 1 << 20


def listed():
    return [
        # `hvm64 reduce`: one arithmetic expression typed against a small
        # book, numbers of all three types; a call's fixed cost is all there is
        {"name": "expression", "kind": "expression", "terms": 3, "heap_mib": 1024},
        # the smallest whole program: boot, normal form, text
        {"name": "sum depth 4", "kind": "sum", "size": 4, "heap_mib": 1024},
        # a short program with some parallel work: the smallest sort of the
        # batched mix
        {"name": "sort 2^6", "kind": "sort", "size": 6, "heap_mib": 1024},
        # an ordinary program: millions of rewrites, milliseconds
        {"name": "sort 2^11", "kind": "sort", "size": 11, "heap_mib": 4096},
        # a sequential program: one chain of applications, nothing parallel
        {"name": "church 2^9", "kind": "church", "size": 9, "labels": 16, "heap_mib": 1024},
        # a wide net with a short critical path, at its configured size
        {"name": "sum depth 18", "kind": "sum", "size": 18, "heap_mib": 4096},
        # the headline benchmark: one large net
        {"name": "sort 2^16", "kind": "sort", "size": 16, "heap_mib": 16384},
        # a program whose result is a data structure: the readback counts
        {"name": "sorted tree 2^10", "kind": "tree", "size": 10, "heap_mib": 2048},
        # a debugger, or a pre-reduction with a bound: Net::reduce(limit) until
        # nothing is left
        {"name": "stepped sort 2^8", "kind": "stepped", "size": 8, "limit": 20011, "heap_mib": 1024},
        # several tenants' programs in one book (each definition of each under
        # its own name, too many for on-chip memory), their nets in one launch
        {"name": "tenants 96", "kind": "tenants", "nets": 96, "mix": 3, "heap_mib": 16384},
        # a fixed batch of independent nets of uneven size, planned once and
        # run again and again
        {"name": "planned batch 512", "kind": "planned", "nets": 512, "mix": 7, "heap_mib": 36864},
        # a burst of requests to the serving launch, from start to stop
        {"name": "served burst 128", "kind": "served", "nets": 128, "mix": 5, "slots": 32, "heap_mib": 16384},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heap(rng, rewrites):
    """A heap from what the net needs with reuse up to 16 GiB."""
    lo = max(256, rewrites * 24 // MIB)
    return _log(rng, lo, max(lo + 1, 16384))


def draw(rng):
    kind = rng.choice(["expression", "sum", "sum", "sort", "sort", "sort", "church", "tree", "stepped", "tenants",
                       "planned", "served"])
    if kind == "expression":
        return {"kind": kind, "terms": rng.randint(1, 24), "heap_mib": _log(rng, 256, 4096)}
    if kind == "sum":
        d = rng.randint(2, 18)
        return {"kind": kind, "size": d, "heap_mib": _heap(rng, 46 << d)}
    if kind == "sort":
        k = rng.randint(3, 16)
        return {"kind": kind, "size": k, "heap_mib": _heap(rng, _sort_rewrites(k))}
    if kind == "church":
        return {"kind": kind, "size": rng.randint(3, 10), "labels": rng.randint(1, 40), "heap_mib": _log(rng, 256, 4096)}
    if kind == "tree":
        k = rng.randint(2, 11)
        return {"kind": kind, "size": k, "heap_mib": _heap(rng, _sort_rewrites(k))}
    if kind == "stepped":
        k = rng.randint(3, 9)
        return {"kind": kind, "size": k, "limit": _log(rng, 3000, 100000), "heap_mib": _log(rng, 512, 4096)}
    if kind == "tenants":
        return {"kind": kind, "nets": _log(rng, 3, 96), "mix": rng.randrange(1 << 20), "heap_mib": 16384}
    if kind == "planned":
        n = _log(rng, 5, 400)
        return {"kind": kind, "nets": n, "mix": rng.randrange(1 << 20), "heap_mib": 6144 + 72 * n}
    return {"kind": kind, "nets": _log(rng, 5, 128), "mix": rng.randrange(1 << 20), "slots": rng.randint(7, 32),
            "heap_mib": 16384}


# ---------------------------------------------------------------------------
# programs
# ---------------------------------------------------------------------------
def _offset(text, seed):
    """The program with a seeded number added to its result."""
    out = text.replace("& @sum ~ (b a)\n", f"& @sum ~ (b $([+{_small(seed)}] a))\n", 1)
    assert out != text
    return out


def _small(seed):
    return random.Random(seed).randrange(1, 1 << 23)


def _program(case, seed):
    kind, size = case["kind"], case["size"]
    if kind == "sum":
        return _offset(configs.tree_sum(size), seed)
    if kind == "church":
        text = configs.church(size, case["labels"])
        out = text.replace("(@inc (0 r))", f"(@inc ({_small(seed)} r))", 1)
        assert out != text
        return out
    return configs.bitonic(size, seed, result="tree" if kind == "tree" else "sum")


ARITHMETIC = """@add = ($([+] $(a b)) (a b))
@div = ($([/] $(a b)) (a b))
@mod = ($([%] $(a b)) (a b))
@mul = ($([*] $(a b)) (a b))
@sub = ($([-] $(a b)) (a b))
"""


def _expression(terms, seed):
    """A tuple of `terms` results, each two operations on numbers of one type
    in turn (u24, i24, f24), as net text."""
    rng = random.Random(seed)
    tree, redexes = "*", []
    for i in range(terms):
        f, g = rng.choice(["add", "sub", "mul"]), rng.choice(["add", "mul", "div", "mod"])
        if i % 3 == 0:
            x, y, z = (str(rng.randrange(1, 1 << 24)) for _ in range(3))
        elif i % 3 == 1:
            x, y, z = (f"{rng.choice([-1, 1]) * rng.randrange(1, 1 << 23):+d}" for _ in range(3))
        else:
            x, y, z = (f"{rng.uniform(0.5, 1e4):.3f}" for _ in range(3))
        tree = f"(r{i} {tree})"
        redexes += [f"@{f} ~ ({x} ({y} m{i}))", f"@{g} ~ (m{i} ({z} r{i}))"]
    return "\n& ".join([tree] + redexes)


def _nets(case):
    """The batch's (program, size) list: part of the case, not of the seed, so
    that every seed's batch is the same amount of work."""
    rng = random.Random(case["mix"])
    return [configs.mix_choice(rng) for _ in range(case["nets"])]


def _tenants_book(seed):
    parts, table = [], {}
    for v in VARIANTS:
        pre = configs.variant_prefix(*v)
        parts.append(configs.prefixed(configs.variant(*v, seed=seed)[0], pre))
        table[v] = pre + "main"
    return "\n".join(parts), table


# ---------------------------------------------------------------------------
# what a program has in hand, and one pass
# ---------------------------------------------------------------------------
class State:
    pass


def prepare(case, seed):
    s = State()
    s.case = case
    s.kind = kind = case["kind"]
    if kind == "served":
        # every request arrives at once
        s.server = serve.Server(slots=case["slots"], heap_bytes=case["heap_mib"] * MIB, book_seed=seed % configs.U24,
                                timeout_s=60, queue=1024)
        s.requests = [serve.Request(i, 0.0, *v) for i, v in enumerate(_nets(case))]
        return s
    s.heap = hvm64.Heap(case["heap_mib"] * MIB)
    s.heap.set_timeout(60)
    if kind == "expression":
        s.host = hvm64.Host(ARITHMETIC, s.heap)
        s.text = _expression(case["terms"], seed)
    elif kind == "planned":
        book, table = configs.mix_book(VARIANTS, seed % configs.U24)
        s.host = hvm64.Host(book, s.heap)
        defs = [s.host.defs[table[v][0]] for v in _nets(case)]
        s.plan = hvm64.PlannedBatch(s.heap, defs, hvm64.arena_sizes(s.heap, defs, margin=1.3))
    elif kind == "tenants":
        book, table = _tenants_book(seed % configs.U24)
        s.host = hvm64.Host(book, s.heap)
        s.defs = [s.host.defs[table[v]] for v in _nets(case)]
    else:
        s.host = hvm64.Host(_program(case, seed), s.heap)
        s.main = s.host.defs["main"]
        s.limit = case.get("limit")
    return s


def _text(case, text):
    """The text in a buffer of the size a caller of this case sets aside."""
    kind = case["kind"]
    cap = 64 * case["terms"] if kind == "expression" else 48 << case["size"] if kind == "tree" else 16
    buf = np.zeros(cap, dtype=np.uint8)
    buf[:len(text)] = np.frombuffer(text.encode(), dtype=np.uint8)
    return buf


def _counts(r):
    return np.array([r.anni, r.comm, r.eras, r.dref, r.oper], dtype=np.int64)


def run(s):
    if s.kind == "planned":
        ports = s.plan.run()
        return {"ports": np.array(ports, dtype=np.int64), "rewrites": _counts(s.plan.rwts)}
    if s.kind == "served":
        return _serve(s)
    if s.kind == "tenants":
        batch = hvm64.Batch(s.heap)
        batch.boot(s.defs)
        batch.normal()
        return {"ports": np.array(batch.ports(), dtype=np.int64), "rewrites": _counts(batch.rwts)}
    net = hvm64.Net(s.heap)
    if s.kind == "expression":
        s.host.encode_net(net, s.text)
    else:
        net.boot(s.main)
    if s.kind == "stepped":
        while net.reduce(s.limit) is None:
            pass
    net.normal()
    return {"normal_form": _text(s.case, s.host.readback(net)), "rewrites": _counts(net.rwts)}


def _serve(s):
    stats = s.server.run(s.requests)
    return {"ports": np.array([r.port for r in s.requests], dtype=np.int64), "rewrites": stats.rewrites}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _sort_rewrites(k):
    return 21 * k * (k + 1) << k


def _net_rewrites(v):
    return 46 << v[1] if v[0] == "tree_sum" else _sort_rewrites(v[1])


def work(case):
    """A rewrite reads the two nodes of its pair (32 bytes) and writes, on
    average, the two that replace them; `flops` counts rewrites."""
    kind = case["kind"]
    if kind == "expression":
        n = 12 * case["terms"]
    elif kind == "sum":
        n = 46 << case["size"]
    elif kind == "church":
        n = (3 << case["size"]) + 6 * case["size"]
    elif kind in ("sort", "tree", "stepped"):
        n = _sort_rewrites(case["size"])
    else:
        n = sum(_net_rewrites(v) for v in _nets(case))
    return {"bytes": 64.0 * n, "flops": float(n)}


def exact(case, seed):
    """The number a net reduces to, as its normal form's text; the sorted
    tree, the expressions and the counts have no such value."""
    kind = case["kind"]
    if kind == "sum":
        value = ((1 << case["size"]) + _small(seed)) % configs.U24
    elif kind == "church":
        value = ((1 << case["size"]) + _small(seed)) % configs.U24
    elif kind in ("sort", "stepped"):
        # the u24 hash of every leaf position, summed
        t = (np.arange(1 << case["size"], dtype=np.int64) * configs.HASH_M1 + seed) % configs.U24
        v = ((t ^ (t >> 11)) * configs.HASH_M2) % configs.U24
        value = int((v ^ (v >> 13)).sum() % configs.U24)
    else:
        return None
    return {"normal_form": _text(case, str(value)), "rewrites": None}
