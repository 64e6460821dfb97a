"""The double-precision step (L = 2,048 .. 32,768) against the closed form and the oracle, bit for
bit, with digits at the ends of their range, where rounding has the least room."""

import ctypes
import random

import pytest

import common
import montmul_amd as mm
from montmul_amd import CarryError, Hip, ModBatch
from oracle_backends import Gmp

pytestmark = pytest.mark.gpu

SIZES = [(16381, 2048), (20000, 2048), (32764, 2048), (32765, 4096), (50001, 4096), (65532, 4096), (65533, 8192),
         (100000, 8192), (131068, 8192), (131069, 16384), (200003, 16384), (262140, 16384), (262141, 32768), (400000, 32768), (524284, 32768)]


@pytest.fixture(scope="module")
def default():
    h = Hip()
    yield h
    h.close()


def closed_form(x, c, n, nprime, k):
    r = 1 << (32 * k)
    t = x * x * c
    return (t + (t % r * nprime) % r * n) >> (32 * k)


@pytest.mark.parametrize("bits,length", SIZES)
def test_double_step_matches_closed_form(default, bits, length):
    b = ModBatch(default, [common.rand_odd(random.Random(bits), bits)], 3)
    assert b.params().len == length and Hip.step_kernel(b) == 64
    b.free()
    print("double step", bits, length, flush=True)
    common.assert_same_raw(lambda: default, lambda: Gmp(full_k=True), bits, 3, 12, seed=bits)


def pattern(words, k):
    """k limbs repeating the given 16-bit digits, lowest first."""
    b = b"".join(w.to_bytes(2, "little") for w in words)
    return int.from_bytes((b * (4 * k // len(b) + 1))[: 4 * k], "little")


@pytest.mark.parametrize("length", [2048, 4096, 8192, 16384, 32768])
def test_double_step_edges(default, length):
    """One step at the ends of the range and on digits of the largest size (0x7fff, 0x8000 and
    alternating signs), and for raw values in the upper half of [0, R) (x = x' + R)."""
    k = length // 2
    bits = 32 * k - 4
    r = 1 << (32 * k)
    rng = random.Random(length)
    top = 1 << (bits - 1)
    low = (1 << (bits - 1)) - 1
    moduli = [2**bits - 1, 2**bits - 2 ** (bits // 2) + 1, pattern([0x7FFF], k) & low | top | 1,
              pattern([0x8000], k) & low | top | 1, pattern([0x7FFF, 0x8000], k) & low | top | 1, common.rand_odd(rng, bits)]
    primes = [-pow(n, -1, r) % r for n in moduli]
    for base in (1, 4 if length < 32768 else 3):  # the largest base that each length takes
        picks = [lambda n: 0, lambda n: 1, lambda n: 2 * n - 1, lambda n: pattern([0x7FFF], k) % (2 * n),
                 lambda n: pattern([0x8000], k) % (2 * n), lambda n: pattern([0x7FFF, 0x8000], k) % (2 * n),
                 lambda n: pattern([0x8000, 0x7FFF, 0x7FFF], k) % (2 * n), lambda n: rng.randrange(2 * n)]
        if base == 1:
            picks += [lambda n: rng.randrange(r // 2, r // 4 * 3), lambda n: pattern([0x8000], k), lambda n: pattern([0x7FFF], k)]
        for j, pick in enumerate(picks):
            b = ModBatch(default, moduli, base)
            assert Hip.step_kernel(b) == 64
            xs = [pick(n) for n in moduli]
            for i, x in enumerate(xs):
                assert default.table.load(ctypes.c_void_p(b.state), i, mm.to_limbs(x, k)) == 0
                b.set_exponent(i, 1)
            print("edges", length, base, j, flush=True)
            b.run(1)
            for i, (x, n) in enumerate(zip(xs, moduli)):
                assert b.read_raw(i) == closed_form(x, base, n, primes[i], k), (length, base, j, i)
            b.free()


@pytest.mark.parametrize("length", [2048, 4096, 8192, 16384, 32768])
def test_double_step_carry_out_bare_and_readmission(default, length):
    """A carry out names its slots; run_bare leaves x and T = c x^2; a replaced modulus is used."""
    k = length // 2
    rng = random.Random(length)
    moduli = [common.rand_odd(rng, 32 * k - 10) for _ in range(4)]
    c = 4 if length < 32768 else 3
    b = ModBatch(default, moduli, c)
    for i in range(4):
        b.load(i, 1)
        b.set_exponent(i, 1)
    for i in (1, 3):
        assert default.table.load(ctypes.c_void_p(b.state), i, (ctypes.c_uint32 * k)(*([0xFFFFFFFF] * k))) == 0
    with pytest.raises(CarryError) as ei:
        b.run(1)
    assert ei.value.slots == [1, 3]
    assert b.read(0) == c % moduli[0] and b.read(2) == c % moduli[2]
    xs = [rng.randrange(n) for n in moduli]
    for i in range(4):
        b.load_raw(i, xs[i])
        b.set_exponent(i, 1)
    Hip.run_bare(b, 1)
    for i in range(4):
        assert b.read_raw(i) == xs[i] and Hip.read_product(b, i) == c * xs[i] * xs[i]
    n = common.rand_odd(rng, 32 * k - 5)
    b.set_modulus(2, n)
    b.load(2, 7)
    b.set_exponent(2, 0b1011)
    b.run(4)
    assert b.read(2) == pow(7, 16, n) * pow(c, 11, n) % n
    b.free()
