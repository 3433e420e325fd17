"""Basis conversions at the extremes of what they convert.  The conversion reads y_i = x_i qhat_i^-1 mod q_i of an inverse
NTT's output, so the inputs are made backwards: y is chosen -- 0, 1, q - 1, words whose signed base-256 digits are all -128
or all 127, sums sum_i y_i / p_i at a half (the exact rounding's tie) and beside it -- x_i = y_i qhat_i mod q_i, and the
oracle's forward NTT gives the words that the call takes.  Primes of 35 bits (just above the 2^34 below which the other form
is taken) to 60 bits.  Every value is an integer residue: the words must equal the CPU oracle's."""
from fractions import Fraction

import numpy as np
import pytest

from engine_loader import load_ckks

pytestmark = pytest.mark.gpu

N = 1 << 16


@pytest.fixture(scope="module")
def ckks():
    return load_ckks()


def prime(n):
    if n % 2 == 0:
        return False
    d, r = n - 1, 0
    while d % 2 == 0:
        d, r = d // 2, r + 1
    for a in (2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31, 37):
        x = pow(a, d, n)
        if x in (1, n - 1):
            continue
        for _ in range(r - 1):
            x = x * x % n
            if x == n - 1:
                break
        else:
            return False
    return True


def smallest_primes(above, count):
    """the first NTT primes past a bound"""
    out, c = [], (above // (2 * N) + 1) * 2 * N + 1
    while len(out) < count:
        if prime(c):
            out.append(c)
        c += 2 * N
    return out


def high_digits(q):
    """the largest word below q whose low digits are all 127"""
    return max(v for v in (127 * (256**m - 1) // 255 for m in range(1, 9)) if v < q)


def low_digits(q):
    """the largest word below q whose digits under the top one are all -128"""
    best = 0
    for m in range(1, 8):
        low = 128 * (256**m - 1) // 255
        t = min(127, (q - 1 + low) // 256**m)
        if t >= 1:
            best = max(best, t * 256**m - low)
    return best


def sources(qs, rng):
    """y [len(qs)][N]: the patterns in turn over the coefficients"""
    n = len(qs)
    pats = [[0] * n, [1] * n, [q - 1 for q in qs], [high_digits(q) for q in qs], [low_digits(q) for q in qs],
            [low_digits(q) if i & 1 else high_digits(q) for i, q in enumerate(qs)],
            [q - 1 if i & 1 else 0 for i, q in enumerate(qs)], [q // 2 for q in qs]]
    for k in range(24):  # the last limb brings sum y_i / q_i to a half, from below or above
        y = [int(rng.integers(0, q)) for q in qs[:-1]] if k & 1 else [(q - 1, 0, low_digits(q))[k % 3] for q in qs[:-1]]
        want = (Fraction(1, 2) - sum(Fraction(a, q) for a, q in zip(y, qs))) % 1
        pats.append(y + [(int(want * qs[-1]) + (k >> 1) % 2) % qs[-1]])
    y = np.array([[p[i] for p in pats] for i in range(n)], dtype=np.uint64)
    out = np.take(y, np.arange(N) % (len(pats) + 1) % len(pats), axis=1)
    fresh = np.arange(N) % (len(pats) + 1) == len(pats)  # and uniform words among them
    for i, q in enumerate(qs):
        out[i, fresh] = rng.integers(0, q, int(fresh.sum()), dtype=np.uint64)
    return out


def to_eval(oc, y, idx):
    """evaluation-form words whose conversion input is y"""
    qs = [oc.q[i] for i in idx]
    x = np.empty_like(y)
    for i, q in enumerate(qs):
        qhat = 1
        for j, p in enumerate(qs):
            if j != i:
                qhat = qhat * p % q
        x[i] = np.array([v * qhat % q for v in y[i].tolist()], dtype=np.uint64)
    return oc.ntt_fwd(x, idx)


# name: (Q primes, P primes, dnum)
def chain(name, ckks):
    if name == "35 bits, 16 sources":
        p = smallest_primes(1 << 34, 28)
        return p[:16], p[16:], 1
    if name == "35 bits under 60":
        p, big = smallest_primes(1 << 34, 12), ckks.gen_primes(60, 10)
        return p + big[:1], big[1:], 2
    if name == "54 and 60 bits, 16 sources":
        return ckks.gen_primes(54, 16), ckks.gen_primes(60, 16), 1
    return ckks.gen_primes(40, 13), ckks.gen_primes(60, 7), 4


NAMES = ["35 bits, 16 sources", "35 bits under 60", "54 and 60 bits, 16 sources", "40 and 60 bits"]


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("name", NAMES)
def test_conversion_inputs_at_their_extremes(ckks, oracle, name, exact):
    q, p, dnum = chain(name, ckks)
    L, K, moduli = len(q), len(p), q + p
    rng = np.random.default_rng(len(name))
    ctx = ckks.Context(num_q=L, num_p=K, dnum=dnum, moduli=moduli)
    ctx.set_moddown_exact(exact)
    oc = oracle.Ctx(16, moduli, L, K, dnum, moddown_exact=exact)
    print(f"{name}: L {L}, K {K}, digits {ctx.num_digits(L)}", flush=True)
    if not exact:  # ModUp has one form
        D, E, al = ctx.num_digits(L), L + K, -(-L // dnum)
        x = np.empty((L, N), dtype=np.uint64)
        for d in range(D):
            idx = list(range(d * al, min((d + 1) * al, L)))
            x[idx] = to_eval(oc, sources([moduli[i] for i in idx], rng), idx)
        dx, dext = ckks.DeviceBuffer.from_array(x), ckks.DeviceBuffer(D * E * N * 8)
        ctx.modup(dx.ptr, 1, L, dext.ptr)
        assert np.array_equal(dext.download((D, E, N)), oc.modup(x, L)), "ModUp"
    x = np.empty((2, L + K, N), dtype=np.uint64)
    for b in range(2):
        for i, m in enumerate(moduli[:L]):
            x[b, i] = rng.integers(0, m, N, dtype=np.uint64)
        idx = list(range(L, L + K))
        x[b, L:] = to_eval(oc, sources(moduli[L:], rng), idx)
    dx, dout = ckks.DeviceBuffer.from_array(x), ckks.DeviceBuffer(2 * L * N * 8)
    ctx.moddown(dx.ptr, 2, L, dout.ptr)
    got = dout.download((2, L, N))
    for b in range(2):
        assert np.array_equal(got[b], oc.moddown(x[b], L)), (b, "ModDown")
    # a product with its rescale: the dropped limb's lifted value (up to 2^59 under a 60-bit prime) joins the sums
    a, b = (rng.integers(0, 2**63, (2, L, N), dtype=np.uint64) % np.array(q, dtype=np.uint64)[:, None] for _ in "ab")
    evk = rng.integers(0, 2**63, (dnum, 2, L + K, N), dtype=np.uint64) % np.array(moduli, dtype=np.uint64)[:, None]
    da, db, dk = (ckks.DeviceBuffer.from_array(v) for v in (a, b, evk))
    dm = ckks.DeviceBuffer(2 * (L - 1) * N * 8)
    ctx.eval_mult_rescale(da.ptr, db.ptr, 1, L, dk.ptr, dm.ptr)
    assert np.array_equal(dm.download((2, L - 1, N)), oc.hmult_relin_rescale(a, b, L, evk)), "product"
    ctx.close()
