"""GPU parity of the basis conversions (ModUp, ModDown with and without the rescale, both roundings) over the shapes that
their matrix-core form splits by: source limbs in steps of 8 (with one left over, or more), outputs in groups of four (the
last one padded), primes of 36 to 60 bits mixed in a chain, and chains with smaller primes, which take the other form.
Every value is an integer residue: the words must equal the CPU oracle's."""
import numpy as np
import pytest

from engine_loader import load_ckks

pytestmark = pytest.mark.gpu

N = 1 << 16


@pytest.fixture(scope="module")
def ckks():
    return load_ckks()


def residues(moduli, shape_prefix, prime_idx, seed):
    """uniform residues; the first words of every limb are 0, 1, q - 1, 0x7f.. and 0x80.. (evaluation form: what the
    conversions read is an inverse NTT of these; test_gpu_conversion_extremes.py forms their own extremes)"""
    rng = np.random.default_rng(seed)
    q = np.array([moduli[i] for i in prime_idx], dtype=np.uint64)
    x = rng.integers(0, 2**63, tuple(shape_prefix) + (len(prime_idx), N), dtype=np.uint64)
    x = x % q.reshape((1,) * len(shape_prefix) + (-1, 1))
    for i, m in enumerate(q):
        for j, v in enumerate((0, 1, int(m) - 1, 0x7F7F7F7F7F7F7F7F % int(m), 0x8080808080808080 % int(m))):
            x[..., i, j] = v
    return x


# (Q sizes in bits, P sizes, dnum, levels): source limbs 1 to 16 a digit, special primes 1 to 16
SHAPES = {
    "one step, padded groups": ([54] * 5, [60] * 2, 2, (5, 4, 2)),
    "one source limb left over": ([50] * 18, [60] * 9, 2, (18, 10)),
    "two steps": ([54] * 11, [60] * 16, 1, (11, 3)),
    "sixteen of the largest": ([60] * 16, [60] * 3, 1, (16,)),
    "mixed sizes": ([50, 40, 41, 60, 36, 40, 60], [60, 58, 40], 2, (7, 5)),
    "smaller primes": ([36, 30, 36], [32, 36], 2, (3, 2)),
}


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("shape", sorted(SHAPES))
def test_conversions_bit_exact(ckks, oracle, shape, exact):
    q_bits, p_bits, dnum, levels = SHAPES[shape]
    moduli = []
    for b in q_bits + p_bits:
        moduli += ckks.gen_primes(b, 1, skip=moduli)
    L, K = len(q_bits), len(p_bits)
    ctx = ckks.Context(num_q=L, num_p=K, dnum=dnum, moduli=moduli)
    ctx.set_moddown_exact(exact)
    oc = oracle.Ctx(16, ctx.moduli, L, K, dnum, moddown_exact=exact)
    evk = residues(moduli, (dnum, 2), list(range(L + K)), 5)
    devk = ckks.DeviceBuffer.from_array(evk)
    for l in levels:
        D, E = ctx.num_digits(l), l + K
        x = residues(moduli, (2,), list(range(l)), 10 + l)
        dx, dext = ckks.DeviceBuffer.from_array(x), ckks.DeviceBuffer(2 * D * E * N * 8)
        ctx.modup(dx.ptr, 2, l, dext.ptr)
        ext = dext.download((2, D, E, N))
        assert np.array_equal(ext[1], oc.modup(x[1], l)), (l, "ModUp")
        # the same polynomial many times in one launch: a pass that wrote over another workgroup's input would show
        n = 17
        y = np.repeat(residues(moduli, (1,), list(range(l)) + [L + k for k in range(K)], 20 + l), n, axis=0)
        dy, dout = ckks.DeviceBuffer.from_array(y), ckks.DeviceBuffer(n * l * N * 8)
        ctx.moddown(dy.ptr, n, l, dout.ptr)
        got, want = dout.download((n, l, N)), oc.moddown(y[0], l)
        assert all(np.array_equal(g, want) for g in got), (l, "ModDown")
        dks = ckks.DeviceBuffer(2 * 2 * l * N * 8)
        ctx.keyswitch(dx.ptr, 2, l, devk.ptr, dks.ptr)
        assert np.array_equal(dks.download((2, 2, l, N))[0], oc.keyswitch(x[0], l, evk)), (l, "key switch")
        if l > 1:
            a, b = (residues(moduli, (1, 2), list(range(l)), 30 + l + s) for s in (0, 1))
            da, db = ckks.DeviceBuffer.from_array(a), ckks.DeviceBuffer.from_array(b)
            dm = ckks.DeviceBuffer(2 * (l - 1) * N * 8)
            ctx.eval_mult_rescale(da.ptr, db.ptr, 1, l, devk.ptr, dm.ptr)
            assert np.array_equal(dm.download((2, l - 1, N)), oc.hmult_relin_rescale(a[0], b[0], l, evk)), (l, "product")
            # the sum of products transforms its d2 in place
            ctx.eval_mult_sum([[(da.ptr, db.ptr)]], l, devk.ptr, dm.ptr)
            assert np.array_equal(dm.download((2, l - 1, N)), oc.hmult_relin_rescale(a[0], b[0], l, evk)), (l, "sum")
    ctx.close()
