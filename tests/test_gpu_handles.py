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


def hvm64_heap():
    import contextlib
    import hvm64
    return contextlib.closing(hvm64.Heap(1 << 28))
