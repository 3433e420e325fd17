"""Basis conversions on both sides of the lines between their two forms (the int8 matrix product fused with the next
forward NTT, and the VALU conversion before a whole NTT): numbers of outputs and polys where the choice changes, both
roundings, one and many polys.  Which form ran is read off the launch records: the matrix-core form of an exact or a
rescaling ModDown has a launch of its own for what all source limbs enter (bconv_head), which a few output limbs cannot
pay for.  Every value is an integer residue: the words must equal the CPU oracle's."""
import numpy as np
import pytest

from engine_loader import load_ckks

pytestmark = pytest.mark.gpu

N = 1 << 16


@pytest.fixture(scope="module")
def ckks():
    return load_ckks()


def residues(moduli, shape_prefix, prime_idx, seed):
    rng = np.random.default_rng(seed)
    q = np.array([moduli[i] for i in prime_idx], dtype=np.uint64)
    x = rng.integers(0, 2**63, tuple(shape_prefix) + (len(prime_idx), N), dtype=np.uint64)
    return x % q.reshape((1,) * len(shape_prefix) + (-1, 1))


# name: (Q limbs, special primes, dnum)
CHAINS = {"one special prime": (4, 1, 4), "two special primes": (12, 2, 4), "eight special primes": (13, 8, 2)}
# level -> polys of a lone exact ModDown, items of a key-switch list, pairs of a product that take the matrix cores
LEVELS = (1, 2, 3, 4, 5, 6, 7, 8, 12)


def head_expected(what, l, n, K):
    if what == "moddown":
        return l >= 12 or (l >= 8 and n * K >= 48)
    if what == "list":
        return l >= (4 if n <= 12 else 6 if n <= 24 else 7)
    return l >= (3 if n <= 4 else 5 if n <= 16 else 7)  # a product with its rescale


@pytest.mark.parametrize("n", [1, 5, 13, 25])
@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("chain", sorted(CHAINS))
def test_both_forms_bit_exact_at_the_lines(ckks, oracle, chain, exact, n):
    L, K, dnum = CHAINS[chain]
    ctx = ckks.Context(num_q=L, num_p=K, dnum=dnum, q_bits=54, p_bits=60)
    ctx.set_moddown_exact(exact)
    oc = oracle.Ctx(16, ctx.moduli, L, K, dnum, moddown_exact=exact)
    evk = residues(ctx.moduli, (dnum, 2), list(range(L + K)), 3)
    devk = ckks.DeviceBuffer.from_array(evk)

    def heads(call):
        ctx.profile(True)
        ctx.profile_reset()
        call()
        names = ctx.profile_report()
        ctx.profile(False)
        return "bconv_head" in names

    for l in [v for v in LEVELS if v <= L]:
        print(f"{chain}, {'exact' if exact else 'approximate'}, level {l}, {n} items", flush=True)
        D, E = ctx.num_digits(l), l + K
        x = np.repeat(residues(ctx.moduli, (1,), list(range(l)), 10 + l), n, axis=0)
        dx, dext = ckks.DeviceBuffer.from_array(x), ckks.DeviceBuffer(n * D * E * N * 8)
        ctx.modup(dx.ptr, n, l, dext.ptr)
        want = oc.modup(x[0], l)
        assert all(np.array_equal(g, want) for g in dext.download((n, D, E, N))), (l, "ModUp")
        y = np.repeat(residues(ctx.moduli, (1,), list(range(l)) + [L + k for k in range(K)], 20 + l), 2 * n, axis=0)
        dy, dout = ckks.DeviceBuffer.from_array(y), ckks.DeviceBuffer(2 * n * l * N * 8)
        head = heads(lambda: ctx.moddown(dy.ptr, 2 * n, l, dout.ptr))
        want = oc.moddown(y[0], l)
        assert all(np.array_equal(g, want) for g in dout.download((2 * n, l, N))), (l, "ModDown")
        assert head == (exact and head_expected("moddown", l, 2 * n, K)), (l, "ModDown's form")
        dks = ckks.DeviceBuffer(n * 2 * l * N * 8)
        head = heads(lambda: ctx.keyswitch(dx.ptr, n, l, devk.ptr, dks.ptr))
        want = oc.keyswitch(x[0], l, evk)
        assert all(np.array_equal(g, want) for g in dks.download((n, 2, l, N))), (l, "key switch")
        assert head == (exact and head_expected("list", l, n, K)), (l, "key switch's form")
        if l > 1:
            a, b = (np.repeat(residues(ctx.moduli, (1, 2), list(range(l)), 30 + l + s), n, axis=0) for s in (0, 1))
            da, db = ckks.DeviceBuffer.from_array(a), ckks.DeviceBuffer.from_array(b)
            dm = ckks.DeviceBuffer(n * 2 * (l - 1) * N * 8)
            head = heads(lambda: ctx.eval_mult_rescale(da.ptr, db.ptr, n, l, devk.ptr, dm.ptr))
            want = oc.hmult_relin_rescale(a[0], b[0], l, evk)
            assert all(np.array_equal(g, want) for g in dm.download((n, 2, l - 1, N))), (l, "product")
            assert head == head_expected("product", l, n, K), (l, "product's form")
    ctx.close()


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("shape", [(16, 2, 8, (16, 13, 9)), (6, 2, 6, (6, 5))])
def test_five_to_eight_digits_bit_exact(ckks, oracle, shape, exact):
    """more than four digits: the inner products and the addend's dropped limb take launches of their own, in both forms
    (at the first chain's upper levels the matrix cores, whose limbs are column-major within 16 rows)"""
    L, K, dnum, levels = shape
    ctx = ckks.Context(num_q=L, num_p=K, dnum=dnum, q_bits=54, p_bits=60)
    ctx.set_moddown_exact(exact)
    oc = oracle.Ctx(16, ctx.moduli, L, K, dnum, moddown_exact=exact)
    evk = residues(ctx.moduli, (dnum, 2), list(range(L + K)), 3)
    devk = ckks.DeviceBuffer.from_array(evk)
    for l in levels:
        D, E, n = ctx.num_digits(l), l + K, 2
        print(f"{D} digits at level {l}, {'exact' if exact else 'approximate'}", flush=True)
        assert D > 4
        x = residues(ctx.moduli, (n,), list(range(l)), 10 + l)
        dx, dext = ckks.DeviceBuffer.from_array(x), ckks.DeviceBuffer(n * D * E * N * 8)
        ctx.modup(dx.ptr, n, l, dext.ptr)
        ext = dext.download((n, D, E, N))
        dks = ckks.DeviceBuffer(n * 2 * l * N * 8)
        ctx.keyswitch(dx.ptr, n, l, devk.ptr, dks.ptr)
        ks = dks.download((n, 2, l, N))
        for i in range(n):
            assert np.array_equal(ext[i], oc.modup(x[i], l)), (l, i, "ModUp")
            assert np.array_equal(ks[i], oc.keyswitch(x[i], l, evk)), (l, i, "key switch")
        a, b = (residues(ctx.moduli, (n, 2), list(range(l)), 30 + l + s) for s in (0, 1))
        da, db = ckks.DeviceBuffer.from_array(a), ckks.DeviceBuffer.from_array(b)
        steps, drot = [1, -3], ckks.DeviceBuffer(2 * 2 * l * N * 8)
        ctx.eval_rotate_hoisted(da.ptr, l, steps, [devk.ptr, devk.ptr], drot.ptr)
        rot = drot.download((2, 2, l, N))
        for i, s in enumerate(steps):
            assert np.array_equal(rot[i], oc.rotate(a[0], l, oc.rot_index(s), evk)), (l, s, "rotation")
        dm = ckks.DeviceBuffer(n * 2 * (l - 1) * N * 8)
        ctx.eval_mult_rescale(da.ptr, db.ptr, n, l, devk.ptr, dm.ptr)
        got = dm.download((n, 2, l - 1, N))
        want = [oc.hmult_relin_rescale(a[i], b[i], l, evk) for i in range(n)]
        assert all(np.array_equal(got[i], want[i]) for i in range(n)), (l, "product")
        ctx.eval_mult_sum([[(da.ptr, db.ptr)]], l, devk.ptr, dm.ptr)
        assert np.array_equal(dm.download((2, l - 1, N)), want[0]), (l, "sum of products")
        # in place: the combine may not read the inputs again
        ctx.eval_mult_rescale(da.ptr, db.ptr, n, l, devk.ptr, da.ptr)
        got = da.download((n, 2, l - 1, N))
        assert all(np.array_equal(got[i], want[i]) for i in range(n)), (l, "product in place")
    ctx.close()
