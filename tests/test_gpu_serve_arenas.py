"""Serving with slots that hold little more than their net allocates: the
lanes of a wave take their nodes from a slot's sub-arenas with one add, and
pass over a sub-arena that is full, so nearly the whole slot is used.  Every
request's result is the net's value (configs.*_expected), and the summed
counts are the oracle's."""
import time

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,size,slots,requests", [("tree_sum", 10, 3, 40), ("tree_sum", 13, 64, 200),
                                                      ("bitonic", 6, 1, 7), ("bitonic", 8, 17, 60)])
def test_tight_slots(gpu_heap, oracle, kind, size, slots, requests):
    import hvm64
    from hvm64 import configs
    print("case tight slots", kind, size, slots, requests, flush=True)
    book, table = configs.mix_book([(kind, size)], seed=9)
    main, expected = table[(kind, size)]
    ref = oracle.run(book, entry=main, heap_words=1 << 26)
    host = hvm64.Host(book, gpu_heap)
    d = host.defs[main]
    nodes = hvm64.arena_sizes(gpu_heap, [d], margin=1.0, extra=0)[0]
    s = hvm64.Serving(gpu_heap, slots, nodes + nodes // 4 + 8192, queue=256)
    got, t0 = [], time.time()
    try:
        s.submit([d] * requests, list(range(requests)))
        while len(got) < requests and time.time() - t0 < 30:
            got += s.poll()
    finally:
        s.stop()
    assert sorted(t for t, _ in got) == list(range(requests))
    assert all(p == hvm64.u24_port(int(expected)) for _, p in got)
    assert ref["nf"] == expected
    counts = hvm64.Net.rwts.fget(s).as_dict()
    assert counts == {k: v * requests for k, v in ref["rwts"].items()}


def wide_calls(depth, width):
    """The tree-sum program, whose generator's every call writes a list of
    `width` numbers and takes its head for the leaf: as many nodes in one
    block, and 2**depth such calls at once."""
    from hvm64 import configs
    tree = "*"
    for i in range(width, 0, -1):
        tree = f"({i} {tree})"
    text = configs.tree_sum(depth)
    out = text.replace("& @Leaf ~ (1 c)\n", f"& @Leaf ~ (h c)\n& @first ~ ({tree} h)\n")
    assert out != text
    return out + "@first = ((n *) n)\n"


@pytest.mark.parametrize("depth,width,slots,requests", [(6, 17, 1, 20), (6, 24, 4, 60), (5, 60, 2, 40), (4, 110, 1, 20)])
def test_a_wave_asks_for_more_than_a_sub_arena(gpu_heap, oracle, depth, width, slots, requests):
    """The smallest slot (eight sub-arenas of 1,024 nodes) holds a net whose
    calls ask, the lanes of a wave together, for more nodes than one sub-arena
    has."""
    import hvm64
    print("case wide calls", depth, width, slots, requests, flush=True)
    book = wide_calls(depth, width)
    ref = oracle.run(book, heap_words=1 << 20)
    assert ref["nf"] == str(1 << depth)
    host = hvm64.Host(book, gpu_heap)
    d = host.defs["main"]
    nodes = hvm64.arena_sizes(gpu_heap, [d], margin=1.0, extra=0)[0]
    print("nodes", nodes, flush=True)
    assert nodes < 7000 and width << depth > 1024
    s = hvm64.Serving(gpu_heap, slots, 8192, queue=256)
    got, t0 = [], time.time()
    try:
        s.submit([d] * requests, list(range(requests)))
        while len(got) < requests and time.time() - t0 < 30:
            got += s.poll()
    finally:
        s.stop()
    assert sorted(t for t, _ in got) == list(range(requests))
    assert all(p == hvm64.u24_port(1 << depth) for _, p in got)
    counts = hvm64.Net.rwts.fget(s).as_dict()
    assert counts == {k: v * requests for k, v in ref["rwts"].items()}
