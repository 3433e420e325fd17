"""The calls that a program of this framework spends its time in, through the public front end (ckks.py over the C ABI),
from one addition of two small ciphertexts to a batch of bootstraps.

Three sessions, as programs open them: "mult" (24 Q limbs of 54 bits, 8 special primes, dnum 3: transforms, products,
rotations and matrix products), "boot" (the full-slot bootstrap's chain: 60-bit q0, 22 x 50 bits, 3 x 60 bits) and
"decode" (the batched decode step's chain: 40-bit scaling primes, dnum 4, exact ModDown rounding).  A session is the
context with its keys and bootstrap plan, opened once and kept, as a server keeps them; what a case makes from its seed
is what changes from call to call: ciphertexts, plaintexts, matrix diagonals.  Ciphertext, key and diagonal words are
uniform residues, which is what encryption, key generation and encoding leave in evaluation form.

Every output is a tensor of residues: whole numbers that any correct implementation gives word for word, so the
tolerance is "exact" and there is no result in 64-bit floating point to compare with.
"""
import importlib
import math
import os
import sys

import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
N = 1 << 16
LIMB = N * 8  # bytes

# chain: (num_q, num_p, dnum)
CHAINS = {"mult": (24, 8, 3), "boot": (26, 8, 3), "decode": (32, 7, 4)}
DIGIT = {c: -(-q // d) for c, (q, p, d) in CHAINS.items()}  # Q limbs of a key-switching digit
BOOT_STEPS = 72  # about how many rotation keys a bootstrap plan reads
DECODE_PERIOD, DECODE_LOG_REP = 1024, 5  # the decode step's matrix diagonals repeat every 1,024 slots


def _module(name):
    """a module of the package (its folder's name is no Python identifier, its modules import each other by name)"""
    path = os.path.join(REPO, "fhe-ssm_amd")
    if path not in sys.path:
        sys.path.insert(0, path)
    return importlib.import_module(name)


class Session:
    """a context and what a program keeps with it: switching keys by name, the bootstrap plan"""

    def __init__(self, chain):
        self.ckks = ckks = _module("ckks")
        q, p, d = CHAINS[chain]
        if chain == "mult":
            self.ctx = ckks.Context(num_q=q, num_p=p, dnum=d, q_bits=54, p_bits=60, scale=2.0**50)
        elif chain == "boot":
            big = ckks.gen_primes(60, 12)
            self.ctx = ckks.Context(num_q=q, num_p=p, dnum=d, scale=2.0**50,
                                    moduli=big[:1] + ckks.gen_primes(50, 22) + big[1:4] + big[4:])
        else:
            self.ctx = ckks.Context(num_q=q, num_p=p, dnum=d, scale=2.0**40, moduli=_module("decode_step").config5_moduli(ckks))
            self.ctx.set_moddown_exact(True)
        self.chain, self.keys, self.gen = chain, {}, torch.Generator(device="cuda").manual_seed(1)
        self.plan = None

    def key(self, name):
        """a switching key [dnum][2][L + K][N], the same for the life of the session"""
        if name not in self.keys:
            q, p, d = CHAINS[self.chain]
            self.keys[name] = residues((d, 2), self.ctx.moduli, self.gen)
        return self.keys[name].data_ptr()

    def bootstrap(self):
        """the refresh plan, with sparse-secret encapsulation, and its rotation keys"""
        if self.plan is None:
            deg, top, ins = (59, 2.0**55, 2.0**55) if self.chain == "boot" else (39, 2.0**52, 2.0**53)
            self.plan = self.ckks.Bootstrap(self.ctx, K=14.0, cheb_degree=deg, double_angles=2, top_scale=top,
                                            in_scale=ins)
            self.plan.set_sparse_keys(self.key("to sparse"), self.key("from sparse"))
        return self.plan


_sessions = {}


def session(chain):
    if chain not in _sessions:
        _sessions[chain] = Session(chain)
    return _sessions[chain]


def residues(shape, moduli, gen):
    """uniform words [*shape][len(moduli)][N], limb i below moduli[i]"""
    out = torch.empty(tuple(shape) + (len(moduli), N), dtype=torch.int64, device="cuda")
    for i, q in enumerate(moduli):
        out[..., i, :] = torch.randint(0, q, tuple(shape) + (N,), generator=gen, dtype=torch.int64, device="cuda")
    return out


def empty(*shape):
    return torch.empty(shape, dtype=torch.int64, device="cuda")


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one addition of two ciphertexts near the end of the chain: the smallest call there is
        {"name": "add one", "op": "add", "chain": "mult", "batch": 1, "level": 4},
        # ciphertext times plaintext and the rescale after it, a few ciphertexts at a middle level
        {"name": "scale three", "op": "scale", "chain": "mult", "batch": 3, "level": 13},
        # forward and inverse transforms of one ciphertext's limbs, and of the batch of 64 that throughput is quoted on
        {"name": "ntt one", "op": "ntt", "chain": "mult", "polys": 2, "level": 24},
        {"name": "ntt batch", "op": "ntt", "chain": "mult", "polys": 128, "level": 24},
        # product, relinearization and rescale: a single pair, an odd few at a level that cuts a digit, the quoted batch
        {"name": "product one", "op": "product", "chain": "mult", "batch": 1, "level": 24},
        {"name": "product five", "op": "product", "chain": "mult", "batch": 5, "level": 13},
        {"name": "product batch", "op": "product", "chain": "mult", "batch": 64, "level": 24},
        # rotations of one ciphertext that share their ModUp, as a program's own sums and permutations use them
        {"name": "rotations", "op": "rotations", "chain": "mult", "n": 8, "level": 16},
        # the 768 x 768 plaintext matrix times one ciphertext by 28 x 28 baby and giant steps
        {"name": "matrix", "op": "matrix", "chain": "mult", "diagonals": 768, "babies": 28, "level": 16},
        # a decode step's matrix products: three outputs (as r, k, v) share an input's babies, diagonals expanded from
        # their stored coefficients
        {"name": "decode matrices", "op": "matrices", "chain": "decode", "outputs": 3, "babies": 64, "giants": 24,
         "level": 9},
        # one full-slot bootstrap, and the batch that the decode step refreshes its state by
        {"name": "bootstrap one", "op": "bootstrap", "chain": "boot", "batch": 1},
        {"name": "bootstrap batch", "op": "bootstrap", "chain": "decode", "batch": 6},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["add", "scale", "ntt", "product", "product", "rotations", "matrix", "matrices", "bootstrap"])
    chain = rng.choice(["mult", "mult", "boot", "decode"])
    top = CHAINS[chain][0]
    if op in ("add", "scale"):
        return {"op": op, "chain": chain, "batch": _log(rng, 1, 24), "level": rng.randint(2, top)}
    if op == "ntt":
        return {"op": op, "chain": chain, "polys": _log(rng, 1, 96), "level": rng.randint(1, top)}
    if op == "product":
        return {"op": op, "chain": chain, "batch": _log(rng, 1, 40), "level": rng.randint(2, top)}
    if op == "rotations":
        return {"op": op, "chain": chain, "n": _log(rng, 1, 40), "level": rng.randint(1, top)}
    if op == "matrix":
        babies = rng.randint(4, 28)
        return {"op": op, "chain": "mult", "diagonals": babies * rng.randint(3, 27) - rng.randint(0, 3),
                "babies": babies, "level": rng.randint(2, 16)}
    if op == "matrices":
        return {"op": op, "chain": "decode", "outputs": rng.randint(1, 3), "babies": rng.choice([16, 24, 32, 48, 64]),
                "giants": rng.randint(3, 24), "level": rng.randint(3, 12)}
    chain = rng.choice(["boot", "decode"])
    return {"op": op, "chain": chain, "batch": rng.randint(2 if chain == "boot" else 1, 5)}


# ------------------------------------------------------------------------------------------------ inputs
class State:
    pass


def prepare(case, seed):
    st = State()
    st.case, st.session = case, session(case["chain"])
    ctx, op = st.session.ctx, case["op"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    lvl = case.get("level", 1)
    q = ctx.moduli[:lvl]
    if op == "ntt":
        st.x, st.y = residues((case["polys"],), q, gen), residues((case["polys"],), q, gen)
        st.primes = list(range(lvl))
    elif op == "add":
        st.a, st.b = residues((case["batch"], 2), q, gen), residues((case["batch"], 2), q, gen)
        st.out = empty(case["batch"], 2, lvl, N)
    elif op == "scale":
        st.a, st.pt = residues((case["batch"], 2), q, gen), residues((), q, gen)
        st.prod, st.out = empty(case["batch"], 2, lvl, N), empty(case["batch"], 2, lvl - 1, N)
    elif op == "product":
        st.a, st.b = residues((case["batch"], 2), q, gen), residues((case["batch"], 2), q, gen)
        st.out = empty(case["batch"], 2, lvl - 1, N)
        st.key = st.session.key("relin")
    elif op == "rotations":
        st.a, st.out = residues((2,), q, gen), empty(case["n"], 2, lvl, N)
        st.steps = list(range(1, case["n"] + 1))
        st.keys = [st.session.key(s) for s in st.steps]
    elif op == "matrix":
        st.a, st.out = residues((2,), q, gen), empty(2, lvl - 1, N)
        st.diags = residues((case["diagonals"],), q, gen)
        b, g = case["babies"], -(-case["diagonals"] // case["babies"])
        st.babies = [st.session.key(s) for s in range(1, b)]
        st.giants = [st.session.key(b * s) for s in range(1, g)]
    elif op == "matrices":
        b, g, o = case["babies"], case["giants"], case["outputs"]
        st.a, st.out = residues((2,), q, gen), empty(o, 2, lvl - 1, N)
        n = o * b * g
        # a weight's coefficients at scale 2^40: about +-2^40 over sqrt(period)
        st.coef = torch.randint(-(1 << 36), 1 << 36, (n, 2 * DECODE_PERIOD), generator=gen, dtype=torch.int64,
                                device="cuda")
        st.approx = torch.zeros(n, dtype=torch.int32, device="cuda")
        st.diags = empty(n, lvl, 2 * DECODE_PERIOD)
        st.n = n
        st.baby_steps = list(range(b))
        st.giant_steps = [b * (s - g // 2) for s in range(g)]
        st.babies = [st.session.key(s) if s else 0 for s in st.baby_steps]
        st.giants = [st.session.key(s) if s else 0 for s in st.giant_steps]
    else:
        plan = st.session.bootstrap()
        st.a, st.out = residues((case["batch"], 2), ctx.moduli[:1], gen), empty(case["batch"], 2, plan.out_level, N)
        st.plan, st.relin, st.conj = plan, st.session.key("relin"), st.session.key("conjugation")
        st.keys = {s: st.session.key(s) for s in plan.steps}
    return st


# ------------------------------------------------------------------------------------------------ one pass
def run(st):
    case, ctx, op = st.case, st.session.ctx, st.case["op"]
    lvl = case.get("level", 1)
    if op == "ntt":  # in place, one buffer in each direction
        ctx.ntt_forward(st.x.data_ptr(), case["polys"], st.primes)
        ctx.ntt_inverse(st.y.data_ptr(), case["polys"], st.primes)
        return {"forward": st.x, "inverse": st.y}
    if op == "add":
        ctx.eval_add(st.a.data_ptr(), st.b.data_ptr(), 2 * case["batch"], lvl, st.out.data_ptr())
    elif op == "scale":
        ctx.eval_mult_plain(st.a.data_ptr(), case["batch"], lvl, st.pt.data_ptr(), st.prod.data_ptr())
        ctx.rescale(st.prod.data_ptr(), 2 * case["batch"], lvl, st.out.data_ptr())
    elif op == "product":
        ctx.eval_mult_rescale(st.a.data_ptr(), st.b.data_ptr(), case["batch"], lvl, st.key, st.out.data_ptr())
    elif op == "rotations":
        ctx.eval_rotate_hoisted(st.a.data_ptr(), lvl, st.steps, st.keys, st.out.data_ptr())
    elif op == "matrix":
        ctx.linear_transform_bsgs(st.a.data_ptr(), lvl, st.diags.data_ptr(), case["diagonals"], case["babies"],
                                  st.babies, st.giants, st.out.data_ptr())
    elif op == "matrices":
        ctx.expand_periodic(st.coef.data_ptr(), st.approx.data_ptr(), st.n, DECODE_PERIOD, lvl, st.diags.data_ptr())
        ctx.linear_transform_multi([st.a.data_ptr()], lvl, st.diags.data_ptr(), DECODE_LOG_REP, st.baby_steps,
                                   st.babies, st.giant_steps, st.giants, case["outputs"], True, st.out.data_ptr())
    else:
        st.plan.run_many(st.a.data_ptr(), case["batch"], st.relin, st.conj, st.keys, st.out.data_ptr())
    return st.out


# ------------------------------------------------------------------------------------------------ what it takes
def _switch(chain, lvl):
    """(key bytes, modular products) of one key switch at a level"""
    p, digit = CHAINS[chain][1], DIGIT[chain]
    digits, ext = -(-lvl // digit), lvl + p
    ntt = N * 8  # products of one limb's transform
    modup = lvl * ntt + digits * ext * ntt + sum(min(digit, lvl - d * digit) for d in range(digits)) * ext * N
    moddown = 2 * (p * ntt + p * lvl * N + lvl * ntt)
    return digits * 2 * ext * LIMB, modup + 2 * digits * ext * N + moddown


def work(case):
    """bytes: inputs, keys and diagonals read once, outputs written once; flops: two for each modular product"""
    op, chain, lvl, b = case["op"], case["chain"], case.get("level", 1), case.get("batch", 1)
    key, switch = _switch(chain, lvl)
    if op == "ntt":
        limbs = 2 * case["polys"] * lvl
        return {"bytes": 2 * limbs * LIMB, "flops": 2 * limbs * N * 8}
    if op == "add":
        return {"bytes": 6 * b * lvl * LIMB, "flops": 2 * b * lvl * N}
    if op == "scale":
        products = 2 * b * (lvl * N + N * 8 + (lvl - 1) * N * 9)
        return {"bytes": (2 * b * lvl * 2 + lvl + 2 * b * (lvl - 1)) * LIMB, "flops": 2 * products}
    if op == "product":
        return {"bytes": b * (4 * lvl + 2 * (lvl - 1)) * LIMB + key, "flops": 2 * b * (switch + 4 * lvl * N)}
    if op == "rotations":
        return {"bytes": (2 + 2 * case["n"]) * lvl * LIMB + case["n"] * key, "flops": 2 * case["n"] * switch}
    if op == "matrix":
        n, giants = case["diagonals"], -(-case["diagonals"] // case["babies"])
        keys = case["babies"] - 1 + giants - 1
        return {"bytes": (n * lvl + 4 * lvl) * LIMB + keys * key, "flops": 2 * (keys * switch + 2 * n * lvl * N)}
    if op == "matrices":
        n, keys = case["outputs"] * case["babies"] * case["giants"], case["babies"] - 1 + case["giants"] - 1
        switches = case["babies"] - 1 + case["outputs"] * (case["giants"] - 1)
        return {"bytes": n * 2 * DECODE_PERIOD * 8 + (2 + 2 * case["outputs"]) * lvl * LIMB + keys * key,
                "flops": 2 * (switches * switch + 2 * n * lvl * N)}
    # six double-hoisted levels of 64 diagonals over Q_l P and about 16 products of each half, from the top level down
    q, p, d = CHAINS[chain]
    key, switch = _switch(chain, 3 * q // 4)
    return {"bytes": 6 * 64 * (3 * q // 4 + p) * LIMB + BOOT_STEPS * key,
            "flops": 2 * b * ((6 * 8 + 2 * 16) * switch + 6 * 64 * 4 * (3 * q // 4 + p) * N)}


def tolerance(case):
    return "exact"
