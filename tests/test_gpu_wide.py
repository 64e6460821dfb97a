"""The double-precision step at L = 65,536, several workgroups to a slot, against the oracle, bit for
bit."""

import ctypes
import random

import pytest

import common
import montmul_amd as mm
from montmul_amd import CarryError, Hip, MixBatch, ModBatch
from oracle_backends import Gmp

pytestmark = pytest.mark.gpu

K = 32768
R = 1 << (32 * K)


@pytest.fixture(scope="module")
def default():
    h = Hip()
    yield h
    h.close()


def pattern(digits):
    b = bytes(digits)
    return int.from_bytes((b * (4 * K // len(b) + 1))[: 4 * K], "little")


@pytest.mark.parametrize("bits", [524285, 800001, 32 * K - 4])
def test_wide_step_chain(default, bits):
    """A chain of steps, in two runs and with exponents of different lengths."""
    rng = random.Random(bits)
    moduli = [common.rand_odd(rng, bits) for _ in range(3)]
    exps = [0b101101, 0b11, 0b1000]
    xs = [rng.randrange(2 * n) for n in moduli]
    b, want = ModBatch(default, moduli, 3), ModBatch(Gmp(full_k=True), moduli, 3)
    assert b.params().len == 2 * K and Hip.step_kernel(b) == 64
    for i in range(3):
        for t in (b, want):
            t.load_raw(i, xs[i])
            t.set_exponent(i, exps[i])
    for bits_run in (3, 4):
        for t in (b, want):
            t.run(bits_run)
        for i in range(3):
            assert b.read_raw(i) == want.read_raw(i) and b.remaining(i) == want.remaining(i)
    b.free()


@pytest.mark.parametrize("base", [1, 3])
def test_wide_step_edges(default, base):
    """One step at the ends of the range, on digits of the largest size, and for raw values in the
    upper half of [0, R)."""
    bits = 32 * K - 4
    top, low = 1 << (bits - 1), (1 << (bits - 1)) - 1
    rng = random.Random(base)
    moduli = [2**bits - 1, pattern([0x7F]) & low | top | 1, pattern([0x80]) & low | top | 1, pattern([0x7F, 0x80]) & low | top | 1]
    picks = [lambda n: 0, lambda n: 1, lambda n: 2 * n - 1, lambda n: pattern([0x7F]) % (2 * n), lambda n: pattern([0x80]) % (2 * n),
             lambda n: pattern([0x80, 0x7F, 0x7F]) % (2 * n), lambda n: rng.randrange(2 * n)]
    if base == 1:
        picks += [lambda n: rng.randrange(R // 2, R // 4 * 3), lambda n: pattern([0x80]), lambda n: pattern([0x7F])]
    gmp = Gmp(full_k=True)
    b, want = ModBatch(default, moduli, base), ModBatch(gmp, moduli, base)
    for j, pick in enumerate(picks):
        xs = [pick(n) for n in moduli]
        for i, x in enumerate(xs):
            for t, be in ((b, default), (want, gmp)):
                assert be.table.load(ctypes.c_void_p(t.state), i, mm.to_limbs(x, K)) == 0
                t.set_exponent(i, 1)
        print("edges", base, j, flush=True)
        b.run(1)
        want.run(1)
        for i in range(len(moduli)):
            assert b.read_raw(i) == want.read_raw(i), (base, j, i)
    b.free()


def test_wide_step_groups_carry_out_and_readmission(default):
    """More slots than run together; a carry out names its slots; a replaced modulus is used; the same
    slots in a mixed run."""
    rng = random.Random(7)
    moduli = [common.rand_odd(rng, 700000 + i) for i in range(66)]
    b = ModBatch(default, moduli, 3)
    for i in range(66):
        b.load(i, 2 + i)
        b.set_exponent(i, 2)
    for i in (1, 65):
        assert default.table.load(ctypes.c_void_p(b.state), i, (ctypes.c_uint32 * K)(*([0xFFFFFFFF] * K))) == 0
    with pytest.raises(CarryError) as ei:
        b.run(1)
    assert ei.value.slots == [1, 65]
    b.run(1)
    for i in (0, 2, 63, 64):
        assert b.read(i) == pow(2 + i, 4, moduli[i]) * 9 % moduli[i]
    n = common.rand_odd(rng, 900001)
    b.set_modulus(64, n)
    b.load(64, 7)
    b.set_exponent(64, 0b1011)
    b.run(4)
    assert b.read(64) == pow(7, 16, n) * pow(3, 11, n) % n
    Hip.run_bare(b, 1)
    b.free()
    sizes = [3000, 20000, 700000, 100000]
    ns = [common.rand_odd(rng, s) for s in sizes]
    m = MixBatch(default, ns, 3)
    for i in range(4):
        m.load(i, 5 + i)
        m.set_exponent(i, 6)
    m.run(3)
    assert [m.read(i) for i in range(4)] == [pow(5 + i, 8, n) * pow(3, 6, n) % n for i, n in enumerate(ns)]
    m.free()


def test_wide_groups_of_slots_end_at_different_steps(default):
    """Slots run together 64 at a time; each such group takes its own count of steps: the second group's
    one slot, then the first group's, outlasts the other, one has none at all, and a run goes on where the one before ended."""
    rng = random.Random(17)
    n = common.rand_odd(rng, 530000)
    for nbits in ([2] * 64 + [5], [5] + [2] * 63 + [1], [0] * 64 + [3], [3] + [1] * 63 + [0]):
        b = ModBatch(default, [n] * 65, 3)
        exps = [(1 << c) - 1 for c in nbits]
        for i, e in enumerate(exps):
            b.load(i, 2 + i)
            b.set_exponent(i, e)
        for run in (1, 8):
            b.run(run)
            for i in (0, 1, 63, 64):
                done = min(nbits[i], 1 if run == 1 else 8)
                e = exps[i] >> (nbits[i] - done)
                assert b.remaining(i) == nbits[i] - done
                assert b.read(i) == pow(2 + i, 1 << done, n) * pow(3, e, n) % n, (nbits[i], i, run)
        b.free()


def test_wide_batch_that_ends_early_in_a_mixed_run(default):
    """A batch of L = 65,536 with no steps, or few, beside one with 20,000: right, and without the nine
    launches a step that the other's length would make of it (180,000 of them took 0.69 s, the other batch's steps
    take 0.031)."""
    import time

    rng = random.Random(19)
    wide, short = common.rand_odd(rng, 600000), common.rand_odd(rng, 1000)
    e = rng.getrandbits(20000) | 1 << 19999

    def timed(t, i):
        t.load(i, 7)
        t.set_exponent(i, e)
        a = time.perf_counter()
        t.run(20000)
        return time.perf_counter() - a

    alone = ModBatch(default, [short], 3)
    base = min(timed(alone, 0) for _ in range(3))
    want = pow(7, 1 << 20000, short) * pow(3, e, short) % short
    assert alone.read(0) == want
    alone.free()
    m = MixBatch(default, [wide, short], 3)
    for few in (0, 3):
        times = []
        for _ in range(2):
            m.load(0, 5)
            m.set_exponent(0, (1 << few) - 1)
            times.append(timed(m, 1))
            assert m.read(1) == want and m.remaining(0) == 0
            assert m.read(0) == pow(5, 1 << few, wide) * pow(3, (1 << few) - 1, wide) % wide
        print("mixed beside", few, "wide steps:", times, "alone", base, flush=True)
        assert min(times) < 3 * base + 0.05
    m.free()


def powers(x, e, n):
    """x after e's bits as steps from x, base 3."""
    return common.powmod(x, 1 << e.bit_length(), n) * common.powmod(3, e, n) % n


def test_wide_chunks_replayed_as_a_graph():
    """max_launch_ms: the nine launches a step are captured once and replayed, alone and in a mixed run, with
    reads and another backend's work between the runs; equal to the single run's raw limbs after each."""
    rng = random.Random(23)
    split, eager = Hip(max_launch_ms=2), Hip()
    try:
        moduli = [common.rand_odd(rng, 560000) for _ in range(3)]
        exps = [rng.getrandbits(c) | 1 << (c - 1) for c in (90, 41, 90)]
        a, b = ModBatch(split, moduli, 3), ModBatch(eager, moduli, 3)
        for t in (a, b):
            for i, e in enumerate(exps):
                t.load(i, 3 + i)
                t.set_exponent(i, e)
        for chunk in (30, 25, 40):
            a.run(chunk)
            launches = Hip.last_run_kernel_ms(a)[1]
            b.run(chunk)
            assert [a.read_raw(i) for i in range(3)] == [b.read_raw(i) for i in range(3)], chunk
            assert launches > 1
        for i, (n, e) in enumerate(zip(moduli, exps)):
            assert a.remaining(i) == 0 and a.read(i) == powers(3 + i, e, n)
        a.free()
        b.free()
        ns = moduli[:2] + [common.rand_odd(rng, c) for c in (900, 5000, 100000)]
        es = [rng.getrandbits(c) | 1 << (c - 1) for c in (20, 60, 200, 150, 200)]
        m = MixBatch(split, ns, 3)
        for _ in range(2):
            for i, e in enumerate(es):
                m.load(i, 5 + i)
                m.set_exponent(i, e)
            m.run(50)
            m.run(200)
            for i, (n, e) in enumerate(zip(ns, es)):
                assert m.remaining(i) == 0 and m.read(i) == powers(5 + i, e, n), i
        m.free()
    finally:
        split.close()
        eager.close()
