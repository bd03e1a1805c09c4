"""Handles come and go: an open that fails for want of memory says so and
leaves nothing behind that the next handle would report, and a dropped book
frees its heap at once."""
import gc
import weakref

import pytest

pytestmark = pytest.mark.gpu


def test_an_open_that_fails_is_not_the_next_handles_error():
    import hvm64
    with pytest.raises(hvm64.HvmError):
        hvm64.Heap(1 << 46)  # 64 TiB
    with hvm64_heap() as heap:
        assert hvm64.Host("@main = 7", heap).defs["main"].idx == 0


def test_a_dropped_book_frees_its_heap():
    import hvm64
    heap = hvm64.Heap(1 << 28)
    seen = weakref.ref(heap)
    gc.disable()
    try:
        host = hvm64.Host("@main = 7", heap)
        assert host.defs["main"].idx == 0
        del host, heap
        assert seen() is None
    finally:
        gc.enable()


@pytest.mark.parametrize("before", ["unfinished", "failed"])
def test_a_planned_run_after_a_net_that_did_not_end(gpu_heap, before):
    """Redexes that an unfinished or failed net left in the global ring reach
    neither the planned nets nor the next net."""
    import hvm64
    from hvm64 import configs
    print("case", before, flush=True)
    book, table = configs.mix_book([("tree_sum", 8), ("bitonic", 6), ("bitonic", 8)], 3)
    book += "\n@bad = a & 1 ~ $([/] $(0 a))"
    host = hvm64.Host(book, gpu_heap)
    defs = [host.defs[name] for name, _ in table.values()] * 20
    want = [hvm64.u24_port(int(nf)) for _, nf in table.values()] * 20
    plan = hvm64.PlannedBatch(gpu_heap, defs, hvm64.arena_sizes(gpu_heap, defs))
    main, normal_form = table[("bitonic", 8)]
    net = hvm64.Net(gpu_heap)
    if before == "unfinished":
        net.boot(host.defs[main])
        assert net.reduce(20000) is None
    else:
        with pytest.raises(hvm64.HvmError):
            net.boot(host.defs["bad"])
            net.normal()
    assert plan.run() == want
    net = hvm64.Net(gpu_heap)
    net.boot(host.defs[main])
    net.normal()
    assert host.readback(net) == normal_form


def hvm64_heap():
    import contextlib
    import hvm64
    return contextlib.closing(hvm64.Heap(1 << 28))
