"""Books on either side of the sizes at which a reduction keeps all of the
book in LDS, all but its instructions, or nothing: n copies of the sort
program, each under names of its own (1,892 words each, 572 without the
instructions; LDS holds 6,144).  Every net's normal form and counts are the
oracle's, for a net alone, an unplanned batch and a planned one."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("copies", [3, 4, 10, 11])
def test_books_around_the_lds_sizes(gpu_heap, oracle, copies):
    import hvm64
    from hvm64 import configs
    print("case book copies", copies, flush=True)
    book = "\n".join(configs.prefixed(configs.bitonic(5, i), f"p{i}_") for i in range(copies))
    host = hvm64.Host(book, gpu_heap)
    ref = [oracle.run(configs.bitonic(5, i), heap_words=1 << 22) for i in range(copies)]
    defs = [host.defs[f"p{i}_main"] for i in range(copies)]
    for i in (0, copies - 1):
        net = hvm64.Net(gpu_heap)
        net.boot(defs[i])
        net.normal()
        assert host.readback(net) == ref[i]["nf"] == configs.bitonic_expected(5, i)
        assert net.rwts.as_dict() == ref[i]["rwts"]
    total = {k: sum(r["rwts"][k] for r in ref) for k in ref[0]["rwts"]}
    ports = [hvm64.u24_port(int(r["nf"])) for r in ref]
    batch = hvm64.Batch(gpu_heap)
    batch.boot(defs)
    batch.normal()
    assert batch.ports() == ports and batch.rwts.as_dict() == total
    plan = hvm64.PlannedBatch(gpu_heap, defs, hvm64.arena_sizes(gpu_heap, defs))
    assert plan.run() == ports and plan.rwts.as_dict() == total
