"""CPU model of the reduction that ends the int8 basis conversion (bconv_ntt.hip mf_reduce, constants as ops.cpp mf_add
forms them): V = sum_s 256^s D_s + e of up to 16 source limbs must come out in [0, 2q), congruent to V mod q, for primes of
35 to 60 bits (the form is taken for primes above 2^34) and |e| up to 2^59 + 16.  The eight D_s are those of real digits --
source digits at their extremes -128 and 127, constants at 0, 1, q - 1 and the balanced digits' edges -- and e brings V to
the multiples of q and their neighbours, where a wrong quotient would show first."""
import random

import pytest

BIAS = 0x8080808080808080
M64 = (1 << 64) - 1


def i32(x):
    x &= 0xFFFFFFFF
    return x - (1 << 32) if x >> 31 else x


def i64(x):
    x &= M64
    return x - (1 << 64) if x >> 63 else x


def digits(v):
    """the eight signed base-256 digits of a word below 2^60"""
    w = ((v + BIAS) & M64) ^ BIAS
    return [((w >> (8 * s)) & 0xFF) - (0x100 if (w >> (8 * s + 7)) & 1 else 0) for s in range(8)]


def constants(q):
    bits = q.bit_length()
    sh = bits - 47 if bits > 47 else 0
    nq = (-q) & M64
    nq_lo = i32(nq)
    return {"sh": sh, "M": i32((1 << (64 + sh)) // q), "nq_lo": nq_lo, "nq_hi": i32((nq - nq_lo) >> 32)}


def reduce_model(D, e, c, quarter=1 << 30, sh_off=0):
    """mf_reduce in the widths of the kernel's variables"""
    E = [i32(D[2 * k] + (D[2 * k + 1] << 8)) for k in range(4)]
    F = i64(E[1] * 65536 + E[0] + (e & 0xFFFFFFFF))
    W = i64(E[3] * 65536 + i32(i32(F >> 32) + E[2] + i32((e & M64) >> 32)))
    G = i32((W & M64) >> (c["sh"] + sh_off))
    k = i32((G * c["M"] - quarter) >> 32)
    v = ((W & 0xFFFFFFFF) << 32) | (F & 0xFFFFFFFF)
    r = v + k * c["nq_lo"]
    return (r + (((k * c["nq_hi"]) & 0xFFFFFFFF) << 32)) & M64


def samples(q, n_in, rng):
    """(D_0..D_7, V without e)"""
    half = sum(127 << (8 * p) for p in range(8))
    edges = [0, 1, q - 1, q // 2, half % q, 0x8080808080808080 % q]
    for kind in range(14):
        D, V = [0] * 8, 0
        for i in range(n_in):
            for p in range(8):
                d = (-128, 127, -128 if i & 1 else 127, rng.randint(-128, 127))[kind % 4]
                C = edges[kind % len(edges)] if kind < 12 else rng.randrange(q)
                if kind % 4 < 2 and kind >= 4:  # the constant that pushes V furthest in the digits' direction
                    C = q - 1
                V += d * C
                for s, t in enumerate(digits(C)):
                    D[s] += d * t
        assert V == sum(D[s] << (8 * s) for s in range(8))
        assert abs(V) < (q << 10) * n_in
        yield D, V


def extras(V, q, rng):
    """e of at most 2^59 + 16 that put V + e at multiples of q, their neighbours and mid-way; and the extremes"""
    big = (1 << 59) + 16
    out = [0, big, -big]
    for t in (0, 1, q - 1, q // 2):
        r = (t - V) % q
        out += [x for x in (r, r - q) if abs(x) <= big]
        j = (big - r) // q
        out += [r + j * q, r - ((big + r) // q) * q]
    return [x for x in out if abs(x) <= big] + [rng.randint(-big, big)]


def primes(bits):
    """the smallest and the largest odd values of a size stand for its primes (the bound uses q's size alone)"""
    lo = (1 << 34) + (1 << 17) + 1 if bits == 35 else (1 << (bits - 1)) + (1 << 17) + 1
    return [lo, (1 << bits) - (1 << 17) + 1]


@pytest.mark.parametrize("bits", [35, 36, 40, 47, 48, 50, 54, 59, 60])
def test_reduction_stays_in_its_range(bits):
    rng = random.Random(bits)
    for q in primes(bits):
        c = constants(q)
        assert 0 < c["M"] < 1 << 31 and (c["nq_hi"] << 32) + c["nq_lo"] == -q
        for n_in in (1, 8, 9, 16):
            for D, V in samples(q, n_in, rng):
                for e in extras(V, q, rng):
                    r = reduce_model(D, e, c)
                    assert r < 2 * q and (r - V - e) % q == 0, (q, n_in, e, r / q)


@pytest.mark.parametrize("mistake", ["no quarter", "one bit less of the shift", "no borrow in -q's high word"])
def test_planted_mistakes_leave_the_range(mistake):
    bad = 0
    for bits in (35, 48, 60):
        rng = random.Random(bits)
        for q in primes(bits):
            c = constants(q)
            if mistake == "no borrow in -q's high word":
                c["nq_hi"] = i32(((-q) & M64) >> 32)
            for D, V in samples(q, 16, rng):
                for e in extras(V, q, rng):
                    r = reduce_model(D, e, c, quarter=0 if mistake == "no quarter" else 1 << 30,
                                     sh_off=-1 if mistake == "one bit less of the shift" and c["sh"] else 0)
                    bad += r >= 2 * q
    assert bad
