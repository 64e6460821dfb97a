"""The transform plans beside the step kernels that are the default: which kernel a batch gets by its
options, and each plan's raw limbs against the oracle's closed form."""

import random

import pytest

import common
from montmul_amd import Hip, ModBatch
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
