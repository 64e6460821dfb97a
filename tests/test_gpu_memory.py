"""Device memory of batches on the matrix-core and the double-precision steps: what is held is what a
server counts, nothing of the transform kernels' is held beside it, and a budget that was enough for
the transform plan is enough."""

import random

import pytest

import common
import montmul_amd as mm
from montmul_amd import Hip, ModBatch
from oracle_backends import Gmp

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def default():
    h = Hip()
    yield h
    h.close()


# Bytes a slot in units of L, all of the exponent's k words included: 18 at most on the matrix cores, 38 in double
# precision, 48 at L = 32,768 (its parts).
@pytest.mark.parametrize("length,held", [(512, 18), (1024, 18), (2048, 38), (8192, 38), (16384, 38), (32768, 48)])
def test_step_kernels_hold_their_own_state_only(default, length, held):
    """34 L or more of the transform kernels' state a slot would be 256 MiB here; allocations are rounded
    up by less than 2 MiB each, and there are at most 12."""
    n = common.rand_odd(random.Random(length), 16 * length - 4)
    ModBatch(default, [n], 3).free()  # tables and code
    slots = (256 << 20) // (34 * length)
    before = default.free_memory()
    b = ModBatch(default, [n] * slots, 3)
    assert b.params().len == length
    used = before - default.free_memory()
    b.free()
    assert used <= slots * (held * length + 24) + (24 << 20), (length, used / slots / length)
    assert held * length + 24 <= mm.Server.slot_bytes(length)


def test_double_step_product_keeps_its_scratch(default):
    """mul's scratch comes with the first product, at L = 32,768 too, and serves the next ones."""
    rng = random.Random(5)
    for bits in (20_000, 400_000):
        n = common.rand_odd(rng, bits)
        b = ModBatch(default, [n] * 3, 3)
        xs = [rng.randrange(n) for _ in range(3)]
        for i, x in enumerate(xs):
            b.load(i, x)
        b.mul(2, 0, 1)
        first = default.free_memory()
        b.mul(0, 2, 1)
        b.mul(0, 0, 0)
        assert default.free_memory() == first
        assert b.read(2) == xs[0] * xs[1] % n and b.read(0) == pow(xs[0] * xs[1] * xs[1], 2, n)
        b.free()


def test_step_memory_limit_at_65536():
    """The step over several workgroups is taken where its constants and scratch fit the limit, to the byte,
    else the transform plan's kernel; both give the closed form's raw limbs."""
    length, slots = 65536, 3
    own = slots * (50 * length + 42 * length + 8)
    rng = random.Random(9)
    moduli = [common.rand_odd(rng, 600_000) for _ in range(slots)]
    h = Hip()
    try:
        want = ModBatch(Gmp(full_k=True), moduli, 3)
        xs = [rng.randrange(n) for n in moduli]
        for i, x in enumerate(xs):
            want.load_raw(i, x)
            want.set_exponent(i, 0b10)
        want.run(2)
        for limit, kernel in ((0, 4), (own - 1, 4), (own, 64)):
            h.limit_step_memory(limit)
            b = ModBatch(h, moduli, 3)
            assert Hip.step_kernel(b) == kernel, limit
            for i, x in enumerate(xs):
                b.load_raw(i, x)
                b.set_exponent(i, 0b10)
            b.run(2)
            assert [b.read_raw(i) for i in range(slots)] == [want.read_raw(i) for i in range(slots)], limit
            b.free()
    finally:
        h.close()


@pytest.mark.parametrize("bits,length", [(20_000, 2048), (500_000, 32768), (600_000, 65536)])
def test_server_budget_of_one_transform_slot_serves(bits, length):
    """A budget of one slot as the transform plan holds it (50 L + 24, and 12 L at L = 32,768) serves that
    length, one request after the other."""
    rng = random.Random(bits)
    budget = 50 * length + 24 + (12 * length if length == 32768 else 0)
    srv = mm.Server(base=3, pool_slots=4, target_ms=20, hbm_bytes=budget)
    try:
        ids = [srv.submit(common.rand_odd(rng, bits), 5 + j) for j in range(2)]
        got = []
        for _ in range(60):
            got += srv.poll(8, 1.0)
            if len(got) == 2:
                break
        assert sorted(r["id"] for r in got) == ids and all(r["prp"] == 0 and r["len"] == length for r in got), got
        assert srv.stats()["failed"] == 0 and srv.stats()["hbm_used"] <= budget
    finally:
        srv.close()
