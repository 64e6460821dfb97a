"""The matrix-core step (L = 16 .. 1,024) against the closed form and the oracle, bit for bit."""

import ctypes
import random

import pytest

import common
import montmul_amd as mm
from montmul_amd import CarryError, Hip, ModBatch
from oracle_backends import Gmp

pytestmark = pytest.mark.gpu

# Bits at the bottom, inside and at the top of each length's bucket (32 k - 4 bits is the most).
SIZES = [(125, 16), (252, 16), (253, 32), (700, 64), (1020, 64), (1021, 128), (2044, 128), (2045, 256), (4092, 256),
         (4093, 512), (8188, 512), (8189, 1024), (12345, 1024), (16380, 1024)]


@pytest.fixture(scope="module")
def default():
    h = Hip()
    yield h
    h.close()


def closed_form(x, c, n, k):
    r = 1 << (32 * k)
    t = x * x * c
    return (t + (t * -pow(n, -1, r)) % r * n) // r


@pytest.mark.parametrize("bits,length", SIZES)
def test_matrix_step_matches_closed_form(default, bits, length):
    """Chains on random moduli (one slot and many) against the Gmp closed form, both bases."""
    for slots, base in ((1, 3), (9, 4)):
        b = ModBatch(default, [common.rand_odd(random.Random(bits + i), bits) for i in range(slots)], base)
        assert b.params().len == length and Hip.step_kernel(b) == 32
        b.free()
    print("matrix step", bits, length, flush=True)
    common.assert_same_raw(lambda: default, lambda: Gmp(full_k=True), bits, 5, 40, seed=bits)


@pytest.mark.parametrize("length", [16, 32, 64, 128, 256, 512, 1024])
def test_matrix_step_edges(default, length):
    """One step at the ends of the range, for moduli with extreme digit patterns, and for raw values
    in the upper half of [0, R), whose signed digits overflow (x = x' + R)."""
    k = length // 2
    bits = 32 * k - 4
    r = 1 << (32 * k)
    rng = random.Random(length)
    half = bits // 2
    moduli = [2**bits - 1, 2**bits - 2**half + 1, 2 ** (bits - 1) + 1, (0x7F << (bits - 7)) | 1,
              int("80" * (bits // 8), 16) | 1, int("7f" * (bits // 8), 16) | 1, common.rand_odd(rng, bits)]
    moduli = [n if n.bit_length() + 4 > 16 * k else n | 1 << (bits - 1) for n in moduli]
    for base in (1, 3):
        for pick in range(8):
            b = ModBatch(default, moduli, base)
            xs = []
            for n in moduli:
                x = [0, 1, n - 1, n, 2 * n - 1, rng.randrange(2 * n), rng.randrange(r // 2, r // 4 * 3),
                     int("80" * (4 * k - 1), 16) if base == 1 else 2 * n - 2][pick]
                if base != 1 and pick == 6:
                    x = rng.randrange(2 * n)
                xs.append(x)
            for i, x in enumerate(xs):
                buf = mm.to_limbs(x, k)
                assert default.table.load(ctypes.c_void_p(b.state), i, buf) == 0
                b.set_exponent(i, 1)
            print("edges", length, base, pick, flush=True)
            b.run(1)
            for i, (x, n) in enumerate(zip(xs, moduli)):
                assert b.read_raw(i) == closed_form(x, base, n, k), (length, base, pick, i)
            b.free()


@pytest.mark.parametrize("length", [16, 256, 512, 1024])
def test_matrix_step_carry_out_and_bare(default, length):
    """A carry out names its slots; run_bare leaves x and, on a global plan, T = c x^2."""
    k = length // 2
    rng = random.Random(length)
    moduli = [common.rand_odd(rng, 32 * k - 10) for _ in range(4)]
    b = ModBatch(default, moduli, 4)
    for i in range(4):
        b.load(i, 1)
        b.set_exponent(i, 1)
    for i in (1, 3):
        assert default.table.load(ctypes.c_void_p(b.state), i, (ctypes.c_uint32 * k)(*([0xFFFFFFFF] * k))) == 0
    with pytest.raises(CarryError) as ei:
        b.run(1)
    assert ei.value.slots == [1, 3]
    assert b.read(0) == 4 % moduli[0] and b.read(2) == 4 % moduli[2]
    x = rng.randrange(moduli[0])
    b.load_raw(0, x)
    for i in range(4):
        b.load_raw(i, x % moduli[i])
        b.set_exponent(i, 1)
    Hip.run_bare(b, 1)
    assert b.read_raw(0) == x
    if Hip.plan_of(b)["global"]:
        assert Hip.read_product(b, 0) == 4 * x * x
    b.free()


@pytest.mark.parametrize("bits", [200, 1000, 2044, 8000, 20000, 32764, 40000, 100000, 200000, 300000])
def test_mul_by_the_step_kernels(default, bits):
    """mul on the matrix-core and double-precision kernels: random factors, values at the ends of the
    range, factors in the upper half of [0, R) (each, and both), the output a factor, and a carry out."""
    rng = random.Random(bits)
    n = common.rand_odd(rng, bits)
    b = ModBatch(default, [n] * 3, 2)
    assert Hip.step_kernel(b) in (32, 64)
    k = b.params().k
    r = 1 << (32 * k)
    nprime = -pow(n, -1, r) % r

    def load(i, x):
        assert default.table.load(ctypes.c_void_p(b.state), i, mm.to_limbs(x, k)) == 0

    big = [rng.randrange(r // 2, r // 4 * 3) for _ in range(2)]
    small = rng.randrange(2 * n)
    for x, y in ((small, rng.randrange(2 * n)), (0, small), (2 * n - 1, 2 * n - 1), (1, n), (big[0], small), (small, big[1]), big):
        for out in (0, 1, 2):
            load(0, x)
            load(1, y)
            b.mul(out, 0, 1)
            t = x * y
            assert b.read_raw(out) == (t + (t % r * nprime) % r * n) >> (32 * k), (bits, out)
    load(0, r - 1)
    load(1, r - 1)
    with pytest.raises(CarryError) as ei:
        b.mul(2, 0, 1)
    assert ei.value.slot == 2
    b.free()
