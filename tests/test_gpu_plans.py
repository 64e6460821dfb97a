"""The transform plans beside the step kernels that are the default: which kernel a batch gets by its
options, and each plan's raw limbs against the oracle's closed form."""

import ctypes
import random

import pytest

import common
import montmul_amd as mm
from montmul_amd import CarryError, Hip, MixBatch, ModBatch
from oracle_backends import Gmp

pytestmark = pytest.mark.gpu


def test_autotuner_knows_the_step_kernels():
    """The autotuner times the matrix-core or the double-precision step too, keeps it where a batch can have it
    (1.7 to 20 times as fast as the fastest transform plan at these lengths), and goes on reporting the
    fastest transform plan. A base that the step does not take (4 at L = 32,768) has a choice of its own, before
    and after; `prefer_lds` still names the transform kernels; a batch's slots are as new after the timing."""
    tuned, lds = Hip(autotune=True), Hip(autotune=True, prefer_lds=True)
    try:
        for bits, length, base, kernels in ((200, 16, 3, (32,)), (3000, 256, 3, (32,)), (9000, 1024, 4, (32,)), (20_000, 2048, 3, (64,)),
                                            (100_000, 8192, 4, (64,)), (300_000, 32768, 4, (4, 8)), (300_000, 32768, 3, (64,)),
                                            (400_000, 32768, 4, (4, 8)), (600_000, 65536, 3, (64,))):
            moduli = [common.rand_odd(random.Random(bits + i), bits) for i in range(3)]
            plans = []
            for _ in range(2):  # timed, then from the cache
                b = ModBatch(tuned, moduli, base)
                assert b.params().len == length and Hip.step_kernel(b) in kernels, (bits, base, Hip.step_kernel(b))
                plans.append(Hip.plan_of(b))
                assert plans[-1]["tuned"] and plans[-1]["kernel"] in (4, 8)
                assert all(b.read_raw(i) == 0 and b.remaining(i) == 0 for i in range(3))
                b.run(5)
                assert all(b.read_raw(i) == 0 for i in range(3))
                b.free()
            assert plans[0] == plans[1]
            common.assert_same_raw(lambda: tuned, lambda: Gmp(full_k=True), bits, 3, 6, seed=bits)
        b = ModBatch(lds, [common.rand_odd(random.Random(1), 20_000)], 3)
        assert Hip.step_kernel(b) in (4, 8) and Hip.plan_of(b)["tuned"]
        b.free()
    finally:
        tuned.close()
        lds.close()


def test_autotuner_leaves_a_step_kernel_without_memory():
    """At L = 65,536 with no memory allowed for the step's own state, the tuned transform plan runs; with
    it allowed again, the step does."""
    h = Hip(autotune=True)
    try:
        moduli = [common.rand_odd(random.Random(3), 600_000)]
        for limit, kernel in ((0, 4), (1 << 40, 64), (0, 4)):
            h.limit_step_memory(limit)
            b = ModBatch(h, moduli, 3)
            assert Hip.step_kernel(b) == kernel and Hip.plan_of(b)["tuned"]
            b.load(0, 9)
            b.set_exponent(0, 0b11)
            b.run(2)
            assert b.read(0) == common.powmod(9, 4, moduli[0]) * 27 % moduli[0]
            b.free()
    finally:
        h.close()


# The register kernel's default exchange tile in global mode, asked for by its size, by length.
TILES = {1024: 256, 2048: 512, 4096: 1024, 8192: 2048, 16384: 4096, 32768: 4096}


@pytest.mark.parametrize("length", sorted(TILES))
def test_register_kernel_global_plan(length):
    """The register kernel in global mode with its default tile (which the options name here; the step kernels
    would run otherwise), against the closed form: chains, the ends of the range, a carry out, run_bare's T,
    a replaced modulus, and chunks replayed as a graph."""
    h, split = Hip(tile=TILES[length]), Hip(tile=TILES[length], max_launch_ms=1)
    try:
        k, bits = length // 2, 16 * length - 4
        rng = random.Random(length)
        moduli = [(1 << bits) - 1, common.rand_odd(rng, bits), common.rand_odd(rng, bits // 2 + 1)]
        b = ModBatch(h, moduli, 4)
        plan = Hip.plan_of(b)
        assert b.params().len == length and Hip.step_kernel(b) == 8 and plan["kernel"] == 8 and plan["global"], plan
        print("register kernel", length, plan, flush=True)
        for be in (h, split):
            common.assert_same_raw(lambda: be, lambda: Gmp(full_k=True), bits - 7, 9, 40, seed=length)
        want = ModBatch(Gmp(full_k=True), moduli, 4)
        xs = [2 * moduli[0] - 1, 2 * moduli[1] - 1, 0]
        for t in (b, want):
            for i, x in enumerate(xs):
                t.load_raw(i, x)
                t.set_exponent(i, 0b1011)
            t.run(4)
        assert [b.read_raw(i) for i in range(3)] == [want.read_raw(i) for i in range(3)]
        xs = [b.read_raw(i) for i in range(3)]
        for i in range(3):
            b.set_exponent(i, 0b10)
        for c in (4, 1):
            Hip.run_bare(b, 1)
            assert [b.read_raw(i) for i in range(3)] == xs
            assert [Hip.read_product(b, i) for i in range(3)] == [c * x * x for x in xs]
        b.load(0, 1)
        b.load(2, 1)
        common.load_all_ones(b, 1)
        for i in range(3):
            b.set_exponent(i, 1)
        with pytest.raises(CarryError) as ei:
            b.run(1)
        assert ei.value.slots == [1] and b.read(0) == 4 and b.read(2) == 4
        n = common.rand_odd(rng, bits)
        b.set_modulus(1, n)
        b.load(1, 7)
        b.set_exponent(1, 0b11)
        b.run(2)
        assert b.read(1) == pow(7, 4, n) * 64 % n
        b.free()
    finally:
        h.close()
        split.close()


@pytest.mark.parametrize("length", [1024, 2048, 4096])
def test_register_kernel_tiles_agree(length):
    """The half-vector tile (T kept in registers) and the whole-vector tile, both named: the same raw limbs."""
    half, whole = Hip(tile=length // 4), Hip(tile=length // 2)
    try:
        for be, tile in ((half, length // 4), (whole, length // 2)):
            b = ModBatch(be, [common.rand_odd(random.Random(length), 12 * length)], 3)
            plan = Hip.plan_of(b)
            assert Hip.step_kernel(b) == 8 and plan["global"] and plan["tile"] == tile, plan
            b.free()
        common.assert_same_raw(lambda: half, lambda: whole, 12 * length, 64, 96, seed=length)
    finally:
        half.close()
        whole.close()


def group_kernels(mix):
    return [mm.lib.mm_step_kernel(ctypes.c_void_p(mm.lib.mm_mixbatch_group_state(mix._h, g))) for g in range(mix.groups())]


# Moduli sizes, by transform length 8 .. 32,768.
SIZES = {8: 64, 16: 200, 64: 1000, 128: 2000, 256: 3000, 512: 6000, 1024: 12000, 2048: 20000, 4096: 40000, 8192: 100000, 16384: 200000,
         32768: 300000}


@pytest.mark.parametrize("lengths,copies", [
    ([8, 16, 64, 128, 256, 512, 1024, 2048, 4096, 8192, 16384], 2),  # 1,024 threads: slot groups, wide and full workgroups
    ([512, 1024, 2048, 4096, 8192, 16384, 32768], 3),                # and the radix-4 step in global mode over 1,024
    ([16384], 5),                                                    # full workgroups alone
    ([8, 64, 256, 512, 16384, 32768], 2),
    ([512, 1024, 2048, 4096, 8192, 32768], 9),                       # 512 threads: whole slot groups and partial ones
])
@pytest.mark.parametrize("ms", [0, 1])
def test_mixed_launch_of_transform_kernels(lengths, copies, ms):
    """The mixed-length launch itself (`prefer_lds` names the transform kernels at every length), in one
    launch or in chunks, against the closed form's raw limbs."""
    h = Hip(prefer_lds=True, max_launch_ms=ms)
    try:
        sizes = [SIZES[length] + 7 * c for length in lengths for c in range(copies)]
        probe = MixBatch(h, [common.rand_odd(random.Random(b), b) for b in sizes], 3)
        assert all(kernel in (4, 8) for kernel in group_kernels(probe)) and probe.groups() == len(lengths)
        probe.free()
        print("mixed launch", lengths, copies, ms, flush=True)
        got = common.mixed_lengths(lambda: h, sizes, 24, 9, seed=copies + len(lengths), ref=lambda: Gmp(full_k=True))
        assert got == lengths
    finally:
        h.close()


@pytest.mark.parametrize("ms", [0, 1])
def test_base_4_at_32768_alone_and_among_step_kernels(ms):
    """Base 4 at L = 32,768 is beyond the double-precision step: the register kernel alone, and the radix-4
    step in the mixed-length launch beside the other lengths' step kernels on their streams."""
    h = Hip(max_launch_ms=ms)
    try:
        rng = random.Random(44)
        sizes = [64, 1000, 9000, 20_000, 100_000, 200_000, 300_000, 520_000]
        moduli = [common.rand_odd(rng, b) for b in sizes]
        exps = [rng.getrandbits(c) | 1 << (c - 1) for c in (60, 30, 60, 5, 40, 12, 12, 9)]
        xs = [rng.randrange(n) for n in moduli]
        alone, mix = ModBatch(h, moduli[6:], 4), MixBatch(h, moduli, 4)
        assert Hip.step_kernel(alone) == 8
        assert [mix.params(i).len for i in range(len(moduli))] == [8, 64, 1024, 2048, 8192, 16384, 32768, 32768]
        assert group_kernels(mix) == [4, 32, 32, 64, 64, 64, 8]
        for t, first in ((alone, 6), (mix, 0)):
            for i in range(len(moduli) - first):
                t.load(i, xs[first + i])
                t.set_exponent(i, exps[first + i])
            t.run(7)
            t.run(60)
            for i in range(len(moduli) - first):
                x, n, e = xs[first + i], moduli[first + i], exps[first + i]
                assert t.remaining(i) == 0
                assert t.read(i) == common.powmod(x, 1 << e.bit_length(), n) * common.powmod(4, e, n) % n, (ms, i)
            t.free()
    finally:
        h.close()


@pytest.mark.parametrize("bits,options", [(5000, {"prefer_lds": True}), (100_000, {"prefer_lds": True}), (300_000, {"tile": 4096}), (600_000, {})])
def test_radix4_product_with_and_without_allocation(bits, options):
    """mul and mul_noalloc by the radix-4 kernel (at L = 65,536 by default), in its kept and in the fixed scratch."""
    h = Hip(**options)
    try:
        rng = random.Random(bits)
        n = common.rand_odd(rng, bits)
        xs = [rng.randrange(n) for _ in range(3)]
        pair = []
        for _ in range(2):
            b = ModBatch(h, [n] * 3, 3)
            assert Hip.step_kernel(b) in (4, 8) or b.params().len == 65536
            for i, x in enumerate(xs):
                b.load(i, x)
            pair.append(b)
        a, b = pair
        for out, p, q in ((0, 1, 2), (2, 0, 1), (1, 1, 1)):
            a.mul(out, p, q)
            assert mm.lib.mm_mul_noalloc(ctypes.c_void_p(b.state), out, p, q) == mm.MM_OK
            assert a.read_raw(out) == b.read_raw(out)
        assert a.read(2) == xs[1] * xs[2] * xs[1] % n and a.read(1) == xs[1] * xs[1] % n
        a.free()
        b.free()
    finally:
        h.close()
