"""Workloads of the CKKS evaluation core whose times are followed.

Each case is a plain dict: `op` names one path of the library, `log_n`,
`depth`, `scale_bits`, `first_bits` and `dnum` its parameter set (as
fhemamba_amd.gen_moduli takes them), `limbs` the level, and the rest its
shape.  The sizes are those of the encrypted Mamba-2 decode, the bootstrap,
the benchmark and the tests: rings 2^12 .. 2^17, 5 to 45 limbs, one to four
key-switching digits, single ciphertexts and batches.

Ciphertext inputs are uniform residues (what real ciphertexts are), made on
the GPU from the seed; keys come from the library's seeded family.  Every
output but a decoded vector is a whole residue word and must not change at
all.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "fhe-mamba_amd"))

import fhemamba_amd as F  # noqa: E402
from fhemamba_amd.ckks_probes import build_toy_context  # noqa: E402

# Parameter sets in use: the smallest test ring, the rotation benchmark, the
# decode at N = 2^16 and the classical-128 decode at N = 2^17.
TINY = {"log_n": 12, "depth": 4, "scale_bits": 40, "first_bits": 60, "dnum": 2}
BENCH = {"log_n": 16, "depth": 23, "scale_bits": 59, "first_bits": 60, "dnum": 3}
DECODE = {"log_n": 16, "depth": 44, "scale_bits": 59, "first_bits": 60, "dnum": 3}
CLASSICAL = {"log_n": 17, "depth": 44, "scale_bits": 59, "first_bits": 60, "dnum": 4}


def listed():
    return [
        # The smallest call: one rotation of a toy ring (smoke tests, probes);
        # launches and host work decide it.
        {"name": "rotate_n12", "op": "rotate", **TINY, "limbs": 5, "count": 1},
        # One rescale in the decode chain, about one per product: ~15,000 a token.
        {"name": "rescale_n16_l30", "op": "rescale", **DECODE, "limbs": 30, "count": 1},
        # One rotation at the benchmark's level: one ciphertext's key switch,
        # ~15,000 a token with the relinearizations.
        {"name": "rotate_n16_l24", "op": "rotate", **BENCH, "limbs": 24, "count": 1},
        # One product of the decode (tensor, relinearize, rescale) at a level
        # whose last digit is ragged (37 = 15 + 15 + 7).
        {"name": "mult_n16_l37", "op": "mult", **DECODE, "limbs": 37, "count": 1},
        # The same rotation of the six SSM state groups, deep in the chain.
        {"name": "rotate6_n16_l21", "op": "rotate", **DECODE, "limbs": 21, "count": 6},
        # The headline workload: 30 rotations of one ciphertext off one ModUp,
        # and a rescale.
        {"name": "hoisted30_n16_l24", "op": "hoisted", **BENCH, "limbs": 24, "count": 30},
        # One CoeffToSlot / projection group: 31 diagonals by baby steps of 8,
        # one key per giant step.
        {"name": "transform31_n16_l41", "op": "transform", **DECODE, "limbs": 41, "rows": 31,
         "bstep": 8, "count": 1},
        # Batch of 64 ciphertexts: forward NTT, inner product with 64
        # plaintexts, inverse NTT (24 primes of 60 bits).
        {"name": "ntt64_n16_l24", "op": "ntt", "log_n": 16, "limbs": 24, "count": 64},
        # Plaintexts of one projection's look-ahead batch: 16 diagonals.
        {"name": "encode16_n16_l34", "op": "encode", **DECODE, "limbs": 34, "count": 16,
         "log_slots": 15},
        # The client's side of a token: encode and encrypt the input, decrypt
        # and decode the result.
        {"name": "client_n16_l24", "op": "client", **BENCH, "limbs": 24, "log_slots": 15},
        # A product in the classical-128 chain (45 + 12 primes, four digits).
        {"name": "mult_n17_l41", "op": "mult", **CLASSICAL, "limbs": 41, "count": 1},
        # One whole refresh as the decode makes it: SlotToCoeff first, sparse
        # secret, one pass.
        {"name": "bootstrap_n16", "op": "bootstrap", **DECODE, "log_slots": 15, "passes": 1},
    ]


def _chain(rng):
    """A parameter set of the ranges above; at most 15 limbs a digit."""
    log_n = rng.choice([12, 13, 14, 15, 16, 16, 16, 17])
    lo, hi = {12: (2, 6), 13: (4, 11), 14: (6, 18), 15: (11, 30), 16: (20, 44), 17: (30, 44)}[log_n]
    depth = rng.randint(lo, hi)
    dnum = rng.choice([d for d in (2, 3, 4) if -(-(depth + 1) // d) <= 15])
    return {"log_n": log_n, "depth": depth, "scale_bits": rng.choice([45, 50, 59, 59]),
            "first_bits": 60, "dnum": dnum}


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    op = rng.choice(["rotate", "rotate", "rescale", "mult", "mult", "hoisted", "transform", "ntt",
                     "encode", "client", "bootstrap"])
    if op == "ntt":
        log_n = rng.randint(11, 17)
        return {"op": op, "log_n": log_n, "limbs": rng.randint(3, 40),
                "count": _log_uniform(rng, 1, max(1, min(96, 2 ** (21 - log_n))))}
    if op == "bootstrap":
        return {"op": op, **dict(DECODE, depth=rng.randint(36, 44), log_n=rng.choice([14, 15, 16])),
                "log_slots": 0, "passes": 1}
    c = {"op": op, **_chain(rng)}
    c["limbs"] = rng.randint(2 if op in ("rescale", "mult", "hoisted") else 1, c["depth"] + 1)
    if op in ("rotate", "rescale", "mult"):
        c["count"] = _log_uniform(rng, 1, 8 if c["log_n"] < 17 else 4)
    elif op == "hoisted":
        c["count"] = _log_uniform(rng, 1, 40 if c["log_n"] < 17 else 20)
    elif op == "transform":
        c["rows"] = rng.randint(3, 48)
        c["bstep"] = rng.choice([4, 8, 8, 16])
        c["count"] = rng.randint(1, 3 if c["log_n"] < 17 else 1)
    elif op == "encode":
        c["count"] = _log_uniform(rng, 1, 24)
        c["log_slots"] = c["log_n"] - rng.choice([1, 1, 2, 4])
    else:
        c["log_slots"] = c["log_n"] - rng.choice([1, 1, 2, 4])
    return c


# --------------------------------------------------------------- set-up

def _is_prime(n):
    d, s = n - 1, 0
    while d % 2 == 0:
        d, s = d // 2, s + 1
    for b in (2, 3, 5, 7, 11, 13, 17, 19, 23, 29, 31, 37):
        if n % b == 0:
            return n == b
        x = pow(b, d, n)
        if x in (1, n - 1):
            continue
        for _ in range(s - 1):
            x = x * x % n
            if x == n - 1:
                break
        else:
            return False
    return True


def _primes60(log_n, count):
    """The largest `count` primes below 2^60 that are 1 mod 2N."""
    out, c = [], (1 << 60) + 1
    while len(out) < count:
        c -= 2 << log_n
        if _is_prime(c):
            out.append(c)
    return out


@functools.lru_cache(maxsize=None)
def _context(log_n, depth, scale_bits, first_bits, dnum):
    """A program keeps one context per parameter set."""
    q, p = F.gen_moduli(log_n, depth, scale_bits, first_bits, dnum)
    return F.Context(log_n, q, p, dnum, sampling="seeded")


@functools.lru_cache(maxsize=None)
def _ntt_context(log_n, limbs):
    return F.Context(log_n, _primes60(log_n, limbs), [], 1, sampling="seeded")


@functools.lru_cache(maxsize=2)
def _boot_context(log_n, depth, scale_bits, first_bits, log_slots):
    """The server's bootstrapping context: keys and encoded transforms."""
    slots = 1 << (log_slots or log_n - 1)
    cc, keys = build_toy_context(ring_dimension=1 << log_n, batch=slots, depth=depth,
                                 scale_bits=scale_bits, first_mod_bits=first_bits, seed=21,
                                 secret_dist="SPARSE_TERNARY")
    cc.EvalBootstrapSetup([4, 4], [0, 0], slots, s2c_first=True, real_slots=True)
    cc.EvalBootstrapKeyGen(keys.secretKey, slots)
    return cc, keys, slots


class _Words:
    """A poly's device words as the array interface torch reads."""

    def __init__(self, poly):
        self.poly = poly
        npoly, nlimb = poly.shape
        self.__cuda_array_interface__ = {
            "shape": (npoly, nlimb, poly.ctx.n), "typestr": "<i8",
            "data": (poly.data_ptr(), False), "version": 2}


def _view(poly):
    """torch tensor over the poly's own words (kept alive by the tensor)."""
    return torch.as_tensor(_Words(poly), device="cuda")


def _residues(gen, mods, npoly, n):
    out = torch.empty((npoly, len(mods), n), dtype=torch.int64, device="cuda")
    for j, q in enumerate(mods):
        out[:, j] = torch.randint(0, q, (npoly, n), generator=gen, device="cuda")
    return out


def _uniform(ctx, gen, npoly, limbs):
    poly = ctx.poly(npoly, limbs)
    _view(poly).copy_(_residues(gen, ctx.q[:limbs], npoly, ctx.n))
    return poly


def _vector(case, seed, count=1):
    return np.random.default_rng(seed).uniform(-1, 1, (count, 1 << case["log_slots"]))


def prepare(case, seed):
    op = case["op"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    s = {"op": op, "case": case}
    if op == "ntt":
        ctx = s["ctx"] = _ntt_context(case["log_n"], case["limbs"])
        s["x"] = _residues(gen, ctx.q, 2 * case["count"], ctx.n)
        s["w"] = _residues(gen, ctx.q, case["count"], ctx.n)
        s["acc"] = torch.zeros((2, ctx.L, ctx.n), dtype=torch.int64, device="cuda")
    elif op == "bootstrap":
        cc, keys, slots = _boot_context(case["log_n"], case["depth"], case["scale_bits"],
                                        case["first_bits"], case["log_slots"])
        s["cc"] = cc
        x = np.random.default_rng(seed).uniform(-1, 1, slots)
        pt = cc.MakeCKKSPackedPlaintext(list(x))
        # the encryption's samples from the seed too, so that a state is the
        # same whatever was drawn from the context before
        poly = cc.device.encrypt(keys.publicKey.poly, pt.poly, 5000 + seed)
        ct = cc._wrap(poly, pt.level, pt.deg, pt.scale, pt.slots)
        ct.SetLevel(cc.GetBootstrapInputCeiling())
        s["ct"] = ct
        if not getattr(cc, "_perf_warm", False):
            cc.EvalBootstrap(ct, case["passes"])  # the encoded transforms are kept
            cc._perf_warm = True
    else:
        ctx = s["ctx"] = _context(case["log_n"], case["depth"], case["scale_bits"],
                                  case["first_bits"], case["dnum"])
        _prepare_core(s, ctx, case, seed, gen)
    torch.cuda.synchronize()
    return s


def _prepare_core(s, ctx, case, seed, gen):
    op, nl, n = case["op"], case["limbs"], ctx.n
    count = case.get("count", 1)
    sk = ctx.keygen_secret(seed)

    def galois(steps):
        g = [F.galois_element(r, n) for r in steps]
        return [ctx.keygen_galois(sk, x, 1000 + x) for x in g], g

    if op == "rotate":
        s["cts"] = [_uniform(ctx, gen, 2, nl) for _ in range(count)]
        keys, g = galois([1 + seed % 7])
        s["keys"], s["gal"] = keys * count, g * count
        s["outs"] = [ctx.poly(2, nl) for _ in range(count)]
    elif op == "rescale":
        s["cts"] = [_uniform(ctx, gen, 2, nl) for _ in range(count)]
        s["outs"] = [ctx.poly(2, nl - 1) for _ in range(count)]
    elif op == "mult":
        s["cts"] = [_uniform(ctx, gen, 2, nl) for _ in range(2 * count)]
        s["key"] = ctx.keygen_relin(sk, 7)
        s["prods"] = [ctx.poly(2, nl) for _ in range(count)]
        s["outs"] = [ctx.poly(2, nl - 1) for _ in range(count)]
    elif op == "hoisted":
        steps = [t * (1 << k) for k in range(case["log_n"] - 1) for t in (1, -1)]
        steps += list(range(3, 3 + 2 * case["count"], 2))
        s["ct"] = _uniform(ctx, gen, 2, nl)
        s["keys"], s["gal"] = galois(steps[:count])
        s["outs"] = [ctx.poly(2, nl) for _ in range(count)] + [ctx.poly(2, nl - 1)]
    elif op == "transform":
        rows, b = case["rows"], case["bstep"]
        s["cts"] = [_uniform(ctx, gen, 2, nl) for _ in range(count)]
        s["pts"] = [_uniform(ctx, gen, 1, nl) for _ in range(rows)]
        babies, s["baby_gal"] = galois(range(1, min(b, rows)))
        s["baby_keys"], s["baby_gal"] = [None] + babies, [1] + s["baby_gal"]
        s["giant_keys"], s["giant_gal"] = galois([b * i for i in range(1, -(-rows // b))])
        s["outs"] = [ctx.poly(2, nl) for _ in range(count)]
    elif op == "encode":
        s["rows"] = 0.02 * _vector(case, seed, count)
        s["scale"] = float(ctx.q[-1])
    else:
        s["x"] = _vector(case, seed)[0]
        s["scale"] = float(ctx.q[-1]) if nl > 1 else 2.0 ** 40
        s["sk"], s["pk"], s["seed"] = sk, ctx.keygen_public(sk, 3), seed
        s["ct"] = ctx.encrypt(s["pk"], ctx.encode(_vector(case, seed + 1)[0],
                                                  1 << case["log_slots"], s["scale"], nl), seed)
    s["views"] = [_view(p) for p in s.get("outs", [])]


def run(s):
    op, ctx = s["op"], s.get("ctx")
    if op == "rotate":
        if len(s["cts"]) == 1:
            ctx.rotate(s["cts"][0], s["keys"][0], s["gal"][0], out=s["outs"][0])
        else:
            ctx.rotate_many(s["cts"], s["keys"], s["gal"], outs=s["outs"])
        return s["views"]
    if op == "rescale":
        if len(s["cts"]) == 1:
            ctx.rescale(s["cts"][0], out=s["outs"][0])
        else:
            ctx.rescale_many(s["cts"], outs=s["outs"])
        return s["views"]
    if op == "mult":
        cts = s["cts"]
        tensors = [ctx.tensor(a, b) for a, b in zip(cts[::2], cts[1::2])]
        if len(tensors) == 1:
            ctx.relinearize(tensors[0], s["key"], out=s["prods"][0])
            ctx.rescale(s["prods"][0], out=s["outs"][0])
        else:
            ctx.relinearize_many(tensors, s["key"], outs=s["prods"])
            ctx.rescale_many(s["prods"], outs=s["outs"])
        return s["views"]
    if op == "hoisted":
        digits = ctx.rotation_precompute(s["ct"])
        ctx.rotate_hoisted(s["ct"], digits, s["keys"], s["gal"], s["outs"][:-1])
        ctx.rescale(s["ct"], out=s["outs"][-1])
        digits.close()
        return s["views"]
    if op == "transform":
        ctx.linear_transform_hoisted_many(s["cts"], s["pts"], s["case"]["bstep"], s["baby_keys"],
                                          s["baby_gal"], s["giant_keys"], s["giant_gal"],
                                          outs=s["outs"])
        return s["views"]
    if op == "ntt":
        x, n2, nl = s["x"].data_ptr(), s["x"].shape[0], s["x"].shape[1]
        ctx.ntt_forward_dev(x, n2, nl, 0)
        ctx.mac_dev(x, s["w"].data_ptr(), n2 // 2, nl, s["acc"].data_ptr())
        ctx.ntt_inverse_dev(x, n2, nl, 0)
        return [s["acc"], s["x"]]
    if op == "encode":
        polys = ctx.encode_many(s["rows"], 1 << s["case"]["log_slots"], s["scale"],
                                s["case"]["limbs"])
        return [_view(p) for p in polys]
    if op == "client":
        slots = 1 << s["case"]["log_slots"]
        ct = ctx.encrypt(s["pk"], ctx.encode(s["x"], slots, s["scale"], s["case"]["limbs"]),
                         s["seed"] + 1)
        values = ctx.decode(ctx.decrypt(s["ct"], s["sk"]), slots, s["scale"])
        return {"ct": _view(ct), "values": values}
    return _view(s["cc"].EvalBootstrap(s["ct"], s["case"]["passes"]).poly)


# ------------------------------------------------------------ what it takes

def _shape(case):
    nl, n = case.get("limbs", 0), 1 << case["log_n"]
    dnum = case.get("dnum", 1)
    alpha = -(-(case.get("depth", 0) + 1) // dnum)
    # special primes of 60 bits covering a digit
    k = -(-(60 + (alpha - 1) * case.get("scale_bits", 60)) // 60)
    return nl, n, alpha, k


def _keyswitch(case, nl, n, alpha, k):
    """(key bytes, modular products) of one key switch at nl limbs."""
    nd = -(-nl // alpha)
    return 8 * n * 2 * nd * (nl + k), n * 2 * nd * (nl + k)


def _modup(case, nl, n, alpha, k):
    nd = -(-nl // alpha)
    moved = sum(nl + k - min(alpha, nl - alpha * d) for d in range(nd))
    return n * (case["log_n"] / 2 * (nl + moved) + min(alpha, nl) * moved)


def _moddown(case, nl, n, alpha, k):
    return 2 * n * (case["log_n"] / 2 * (k + nl) + k * nl)


def work(case):
    """Bytes: every input and key word once, every output word once.  flops:
    two for each modular product of the transforms, conversions and inner
    products the definition of the operation asks for."""
    op, half = case["op"], case["log_n"] / 2
    nl, n, alpha, k = _shape(case)
    count = case.get("count", 1)
    limb = 8 * n
    if op == "ntt":
        c = 2 * count
        return {"bytes": limb * nl * (2 * c + count + 2),
                "flops": 2 * n * nl * (2 * c * half + c)}
    if op == "encode":
        slots = 1 << case["log_slots"]
        return {"bytes": count * (limb * nl + 8 * slots),
                "flops": count * (2 * n * nl * half + 10 * slots * case["log_slots"] / 2)}
    if op == "client":
        slots = 1 << case["log_slots"]
        return {"bytes": limb * nl * (2 + 2 + 2) + 32 * slots, "flops": 2 * n * nl * (4 * half + 3)}
    if op == "bootstrap":
        # 14 levels of EvalMod and the two transforms over about 3/4 of the
        # chain: 65 rotation keys, and 24 products of one relinearization key
        nl = 3 * (case["depth"] + 1) // 4
        kb, km = _keyswitch(case, nl, n, alpha, k)
        ops = 65 + 24
        return {"bytes": ops * kb + limb * 2 * (case["depth"] + 1),
                "flops": 2 * ops * (km + _modup(case, nl, n, alpha, k) / 2
                                    + _moddown(case, nl, n, alpha, k))}
    rs_bytes = limb * (2 * nl + 2 * (nl - 1))
    rs_ops = 2 * n * (half * nl + 2 * (nl - 1))
    if op == "rescale":
        return {"bytes": count * rs_bytes, "flops": 2 * count * rs_ops}
    kb, km = _keyswitch(case, nl, n, alpha, k)
    up, down = _modup(case, nl, n, alpha, k), _moddown(case, nl, n, alpha, k)
    if op == "rotate":
        return {"bytes": kb + count * 4 * limb * nl, "flops": 2 * count * (km + up + down)}
    if op == "mult":
        return {"bytes": kb + count * limb * (4 * nl + 2 * (nl - 1)),
                "flops": 2 * count * (km + up + down + rs_ops + 4 * n * nl)}
    if op == "hoisted":
        return {"bytes": count * (kb + 2 * limb * nl) + rs_bytes,
                "flops": 2 * (count * (km + down) + up + rs_ops)}
    rows, b = case["rows"], case["bstep"]
    babies, giants = min(b, rows) - 1, -(-rows // b) - 1
    return {"bytes": (babies + giants) * kb + rows * limb * nl + count * 4 * limb * nl,
            "flops": 2 * count * ((babies + giants) * (km + down) + (1 + giants) * up
                                  + 2 * rows * n * nl)}


def tolerance(case):
    # Residues are whole numbers with one right value.  The decoded vector is
    # a double-precision FFT over up to 2^16 slots: 2.4e-15 (2-norm) and
    # 7.3e-15 (largest) from the encoded values where no noise is added.
    if case["op"] == "client":
        return {"rel": 1e-14, "max": 3e-14}
    return "exact"


def exact(case, seed):
    """The decoded values of a client's round trip are the encoded ones (up
    to the encryption noise, which both sides share).  Everything else is
    whole residues, compared word for word."""
    if case["op"] != "client":
        return None
    return {"ct": None, "values": _vector(case, seed + 1)[0] + 0j}
