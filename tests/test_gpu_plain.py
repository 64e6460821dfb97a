"""read() of many slots, converted out of Montgomery form on the device (the matrix-core and the
double-precision kernels), against Python integers."""

import random

import pytest

import montmul_amd as mm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    h = mm.Hip()
    yield h
    h.close()


def _bits(length):
    return 16 * length - 4  # the longest that the length takes


@pytest.mark.parametrize("length", [16, 32, 64, 128, 256, 512, 1024, 2048, 4096, 8192, 16384, 32768])
def test_reads_are_canonical(be, length):
    rng = random.Random(length)
    top, low = _bits(length), _bits(length) // 2 + 1
    count = 45 if length <= 4096 else 21
    mods = [(1 << top) - 1, (1 << (top - 1)) + 1, (1 << low) + 1] + [rng.getrandbits(top) | (1 << (top - 1)) | 1 for _ in range(count - 3)]
    b = mm.ModBatch(be, mods, 3)
    k = b.params().k
    assert 2 * k == length
    vals = [rng.randrange(n) for n in mods]
    vals[1], vals[2], vals[3] = mods[1] - 1, 1, 0
    for i, v in enumerate(vals):
        b.load(i, v)
        b.set_exponent(i, 1)
    zeros = [0, 11, count - 1]
    for i in zeros:  # N stands for 0, and stays N through steps
        b.load_raw(i, mods[i])
        vals[i] = 0
    b.run(1)
    want = [3 * v * v % n for v, n in zip(vals, mods)]
    got = [b.read(i) for i in range(count)]
    assert got == want
    # Every way a row changes is seen: a load, a product, another run, another modulus.
    b.load(8, 7)
    b.load(9, 11)
    assert [b.read(8), b.read(9)] == [7, 11]
    b.mul(10, 10, 10)
    want = [7 if j == 8 else 11 if j == 9 else g for j, g in enumerate(got)]
    want[10] = got[10] * got[10] % mods[10]
    assert [b.read(i) for i in range(count)] == want
    for i in range(count):
        b.set_exponent(i, 2)
    b.run(2)
    want = [pow(v * v * 3, 2, n) for v, n in zip(want, mods)]
    assert [b.read(i) for i in range(count)] == want
    raw = b.read_raw(12)
    n = rng.getrandbits(top) | (1 << (top - 1)) | 1
    b.set_modulus(12, n)
    assert b.read(12) == raw * pow(1 << (32 * k), -1, n) % n
    b.free()
