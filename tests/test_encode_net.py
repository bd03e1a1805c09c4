"""Host::encode_net of nets wider than the book on either side of the ten
registers that the kernels keep on chip, with and without compiled
definitions.  On the CPU through the engine's own host code and a one-lane
device (tests/fake_device.cpp), which sees a register written outside its
area; on the GPU through the package.  Rewrite counts (and on the GPU normal
forms) are the oracle's, and the same handle boots a definition afterwards."""
import random
import subprocess

import pytest

import fake_device

BOOK = """@add = ($([+] $(a b)) (a b))
@mul = ($([*] $(a b)) (a b))
@sub = ($([-] $(a b)) (a b))
@main = a & @mul ~ (3 (4 a))
"""


def terms(n):
    """A tuple of n results of two operations each."""
    rng = random.Random(n)
    tree, redexes = "*", []
    for i in range(n):
        x, y, z = (rng.randrange(1, 1 << 24) for _ in range(3))
        tree = f"(r{i} {tree})"
        redexes += [f"@{rng.choice(['add', 'sub', 'mul'])} ~ ({x} ({y} m{i}))", f"@add ~ (m{i} ({z} r{i}))"]
    return "\n& ".join([tree] + redexes)


def nest(n):
    """A left comb of n numbers: n registers."""
    tree = "1"
    for i in range(2, n + 1):
        tree = f"({tree} {i})"
    return tree


NETS = {f"terms {n}": terms(n) for n in (1, 7, 8, 9, 10, 11, 12, 24)}
NETS.update({f"nest {n}": nest(n) for n in (9, 10, 11, 14, 16, 17, 30)})


@pytest.fixture(scope="module")
def encode_check(tmp_path_factory):
    return fake_device.build("encode_check", tmp_path_factory.mktemp("encode"))


@pytest.mark.parametrize("compiled", [1, 0])
@pytest.mark.parametrize("net", NETS)
def test_registers_stay_in_their_area(encode_check, oracle, net, compiled):
    r = subprocess.run([encode_check, BOOK, NETS[net], str(compiled)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    got = [[int(x) for x in line.split()] for line in r.stdout.splitlines()]
    ran = oracle.run(BOOK, heap_words=1 << 16)["rwts"]
    assert got == [oracle.reduce_expr(BOOK, NETS[net])[1], [ran[k] for k in ("anni", "comm", "eras", "dref", "oper")]]


@pytest.mark.gpu
@pytest.mark.parametrize("compiled", [True, False])
@pytest.mark.parametrize("book", ["", BOOK])
def test_wide_nets_on_the_gpu(gpu_heap, oracle, book, compiled):
    import hvm64
    gpu_heap.set_compiled(compiled)
    try:
        host = hvm64.Host(book, gpu_heap)
        for name, text in NETS.items():
            if not book and "@" in text:
                continue
            print("case", name, "compiled", compiled, flush=True)
            net = hvm64.Net(gpu_heap)
            host.encode_net(net, text)
            net.normal()
            nf, counts = oracle.reduce_expr(book, text)
            r = net.rwts
            assert host.readback(net) == nf
            assert [r.anni, r.comm, r.eras, r.dref, r.oper] == counts
        if book:
            net = hvm64.Net(gpu_heap)
            net.boot(host.defs["main"])
            net.normal()
            assert host.readback(net) == "12"
    finally:
        gpu_heap.set_compiled(True)
