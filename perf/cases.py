"""The work that users of montmul_amd have it do, as cases to be timed and compared.

Every case goes through the public Python API on one `Hip` backend with its default options, as a
program that tests or exponentiates many moduli at once does. The ranges: moduli of 1,000 to
1,000,000 bits (L = 64 to 65,536), 1 to 2,048 slots, one batch length or several, single products,
short exponents and full Fermat exponents.

Kinds:
    mul     Montgomery products of two slots of one modulus: load two values, mul, read one
    powm    base^e mod N in every slot: load, set_exponent, run, read
    prp     the same from base 3, read as is_one flags and raw limbs (PRP residues)
    fermat  fermat(): batch creation, N - 1 as exponent, run in chunks, is_one
    mixed   moduli of several lengths stepped together (MixBatch)
"""

import functools
import math
import random

import numpy as np

import montmul_amd as mm

# Exponents p of Mersenne primes 2^p - 1 that need L = 256, for Fermat tests that pass.
_PRIME_EXPONENTS = (2203, 2281, 3217)


def listed():
    return [
        # One modular product: the smallest call, all launch and host latency.
        {"name": "mul_1k", "kind": "mul", "bits": 1024, "slots": 8, "ebits": 1},
        # RSA-sized exponentiations with a short exponent, a few at a time.
        {"name": "powm_2k_few", "kind": "powm", "bits": 2048, "slots": 16, "ebits": 256},
        # The 4,096-bit CPU comparison workload: 64 slots, 512 steps.
        {"name": "powm_4k", "kind": "powm", "bits": 4096, "slots": 64, "ebits": 512},
        # Sieving: whole Fermat tests of small candidates, setup included, primes among them.
        {"name": "fermat_3k", "kind": "fermat", "bits": 3000, "slots": 256, "ebits": 3000},
        # An odd number of odd-sized moduli at L = 1,024.
        {"name": "powm_9k_ragged", "kind": "powm", "bits": 9001, "slots": 777, "ebits": 300},
        # The batched Fermat workload's shape (2,048 moduli of 20,000 bits), part of its steps.
        {"name": "prp_20k", "kind": "prp", "bits": 20000, "slots": 2048, "ebits": 400},
        # The headline workload's moduli, a part of its slots and steps.
        {"name": "prp_100k", "kind": "prp", "bits": 100000, "slots": 1024, "ebits": 400},
        # A single large number under test: one chain, nothing beside it.
        {"name": "prp_88k_single", "kind": "prp", "bits": 87914, "slots": 1, "ebits": 1000},
        # Large candidates, about one per CU.
        {"name": "prp_200k", "kind": "prp", "bits": 200003, "slots": 250, "ebits": 100},
        {"name": "prp_300k", "kind": "prp", "bits": 300000, "slots": 200, "ebits": 40},
        # The largest numbers that are tested in batches.
        {"name": "prp_1m", "kind": "prp", "bits": 1000000, "slots": 64, "ebits": 8},
        # Uneven sizes in one batch, log-uniform over the mixed workload's range.
        {"name": "mixed_2k_200k", "kind": "mixed", "bits": 200000, "slots": 300, "ebits": 200},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    """Rough work of a pass: steps times n log n of the modulus size."""
    return case["slots"] * case["ebits"] * case["bits"] * math.log2(case["bits"])


def draw(rng):
    kind = rng.choice(["mul", "powm", "powm", "prp", "prp", "prp", "fermat", "mixed"])
    if kind == "mul":
        return {"kind": kind, "bits": _log_uniform(rng, 1000, 100000), "slots": rng.randint(2, 16), "ebits": 1}
    if kind == "fermat":
        return {"kind": kind, "bits": rng.randint(2050, 4000), "slots": _log_uniform(rng, 16, 256), "ebits": 4000}
    if kind == "mixed":
        case = {"kind": kind, "bits": _log_uniform(rng, 10000, 200000), "slots": rng.randint(40, 300),
                "ebits": rng.randint(20, 150)}
        return case
    lo, hi = (1000, 12000) if kind == "powm" else (12000, 500000)
    bits = _log_uniform(rng, lo, hi)
    slots = _log_uniform(rng, 1, 2048)
    ebits = _log_uniform(rng, 16, 600)
    case = {"kind": kind, "bits": bits, "slots": slots, "ebits": ebits}
    # No dearer than half the 100,000-bit case, in steps and in bytes held.
    limit = 0.5 * 1024 * 400 * 100000 * math.log2(100000)
    case["slots"] = max(1, min(slots, int(limit / (ebits * bits * math.log2(bits))), 150000000 // bits))
    return case


@functools.lru_cache(maxsize=None)
def _hip():
    """The one backend of the process, as a user's program opens it."""
    return mm.Hip()


def _odd(rng, bits):
    return rng.getrandbits(bits) | (1 << (bits - 1)) | 1


def _inputs(case, seed):
    """(moduli, values, exponents), from the seed alone."""
    rng = random.Random(seed)
    kind, bits, slots, ebits = case["kind"], case["bits"], case["slots"], case["ebits"]
    if kind == "mul":
        n = _odd(rng, bits)
        moduli = [n] * slots
    elif kind == "mixed":
        sizes = [_log_uniform(rng, 2048, bits) for _ in range(slots - 1)] + [bits]
        moduli = [_odd(rng, b) for b in sizes]
    elif kind == "fermat":
        moduli = [_odd(rng, bits) for _ in range(slots)]
        for p in _PRIME_EXPONENTS:
            moduli[rng.randrange(slots)] = 2**p - 1
    else:
        moduli = [_odd(rng, bits) for _ in range(slots)]
    values = [rng.randrange(n) if kind in ("mul", "powm") else 1 for n in moduli]
    # Exponents: the top bits of N - 1 (PRP chains), random ones (powers).
    exps = []
    for n in moduli:
        if kind == "powm":
            exps.append(_odd(rng, ebits))
        else:
            exps.append((n - 1) >> max(0, n.bit_length() - ebits))
    return moduli, values, exps


def prepare(case, seed):
    moduli, values, exps = _inputs(case, seed)
    state = {"case": case, "moduli": moduli, "values": values, "exps": exps}
    kind = case["kind"]
    if kind == "mixed":
        state["batch"] = mm.MixBatch(_hip(), moduli, 3)
    elif kind != "fermat":
        state["batch"] = mm.ModBatch(_hip(), moduli, 3)
    else:
        _hip()
    return state


def _limbs(value, k):
    return np.frombuffer(value.to_bytes(4 * k, "little"), dtype=np.uint32)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "fermat":
        return np.array(mm.fermat(_hip(), state["moduli"], 3, 4096), dtype=np.uint8)
    b = state["batch"]
    values, exps = state["values"], state["exps"]
    if kind == "mul":
        k = b.params().k
        b.load(0, values[0])
        b.load(1, values[1])
        b.mul(0, 0, 1)
        return _limbs(b.read(0), k)
    slots = range(len(values))
    for i in slots:
        b.load(i, values[i])
        b.set_exponent(i, exps[i])
    b.run(case["ebits"])
    if kind == "powm":
        k = b.params().k
        return np.stack([_limbs(b.read(i), k) for i in slots])
    flags = np.array(b.is_one_many(slots), dtype=np.uint8)
    if kind == "prp":
        k = b.params().k
        return flags, np.stack([_limbs(b.read_raw(i), k) for i in slots])
    k = max(b.params(i).k for i in slots)  # rows as wide as the longest modulus
    return flags, np.stack([_limbs(b.read_raw(i), k) for i in slots])


def work(case):
    """Bytes: modulus, loaded value, exponent and result of each slot once. Operations: the
    multiplications and additions of five real transforms of 16-bit digits per step (the square's
    two and the reduction's three), or of schoolbook byte products where that is fewer."""
    kind, bits, slots, ebits = case["kind"], case["bits"], case["slots"], case["ebits"]
    if kind == "mixed":
        sizes = [2048 * (bits / 2048) ** ((i + 0.5) / slots) for i in range(slots)]
    else:
        sizes = [bits] * (1 if kind == "mul" else slots)
    total_bytes, flops = 0.0, 0.0
    for b in sizes:
        steps = b if kind == "fermat" else min(b, ebits)
        length = 2 * b / 16
        per_step = min(5 * 2.5 * length * math.log2(max(2.0, length)), 3 * (b / 8) ** 2)
        total_bytes += 3 * b / 8 + steps / 8
        flops += steps * per_step
    return {"bytes": total_bytes, "flops": flops}


def exact(case, seed):
    kind, bits, slots = case["kind"], case["bits"], case["slots"]
    if kind in ("prp", "mixed"):
        return None  # raw limbs of long chains: too many big-integer steps
    ebits = bits if kind == "fermat" else case["ebits"]
    # Python's pow: about 0.15 us per squaring at 1,000 bits, growing as bits^1.7.
    if slots * ebits * 4e-7 * (bits / 1000.0) ** 1.7 > 12.0:
        return None
    moduli, values, exps = _inputs(case, seed)
    if kind == "fermat":
        return np.array([pow(3, n - 1, n) == 1 for n in moduli], dtype=np.uint8)
    k = 4  # limbs per residue: the power of two that holds the modulus and four spare bits
    while 32 * k < bits + 4:
        k *= 2
    if kind == "mul":
        return _limbs(values[0] * values[1] % moduli[0], k)
    out = []
    for n, v, e in zip(moduli, values, exps):
        # Left-to-right from v: the exponent's bits square x and multiply in base 3.
        nb = max(1, (e.bit_length()))
        out.append(_limbs(pow(v, 1 << nb, n) * pow(3, e, n) % n, k))
    return np.stack(out)
