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
