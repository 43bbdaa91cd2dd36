"""Workloads of the engine as a program uses it: each case is one pass through the public
Python entry points at sizes of the encrypted BERT layer, its tests and its benchmark.

A party (context, secret, public, relinearisation and Galois keys, bootstrapping plan) is
made once per parameter set and kept while cases of that set run, as a client or a server
keeps it; what a seed decides is the data: messages, ciphertexts, weights.
"""
from __future__ import annotations

import gc
import math

import numpy as np
import torch

import shmoai_amd as shm

# Prime chains by name: data primes first, then the special primes of key switching.
CHAINS = {
    # one rotation and product at N = 2^13: 8 x 50 bits, one 60-bit special prime
    "small50": ([50] * 8 + [60], 1),
    # the quarter-width projection: 24 x 50 bits
    "wide50": ([50] * 24 + [60], 1),
    # the reference layer (scale 2^46, 5 special primes, dnum 7)
    "layer": ([51] + [46] * 23 + [51] * 11 + [51] * 5, 5),
    # bootstrapping at N = 2^16 (51 + 20 x 46 + 14 x 51 bits, dnum 7)
    "boot": ([51] + [46] * 20 + [51] * 14 + [51] * 5, 5),
    # bootstrapping at N = 2^13, as a smaller ring uses it
    "boot_small": ([51] + [46] * 3 + [51] * 14 + [51] * 3, 3),
}
SCALE = {"small50": 2.0 ** 50, "wide50": 2.0 ** 40, "layer": 2.0 ** 46, "boot": 2.0 ** 46, "boot_small": 2.0 ** 46}
# Chebyshev series of GELU on [-19.5, 12.5], degree 24 (the non-linear layer's own)
GELU = (
    3.4550752799e+00, 5.7852067632e+00, 3.1727714170e+00, 7.0234932500e-01, -4.6200569546e-01,
    -3.7817535966e-01, 8.4136420694e-02, 2.2427456987e-01, 2.9451916291e-02, -1.2928072669e-01,
    -6.6659430283e-02, 6.4349502364e-02, 7.1733295078e-02, -1.9882581810e-02, -6.1145844240e-02,
    -8.4827295421e-03, 4.3597254356e-02, 2.3373027950e-02, -2.4790187963e-02, -2.7940100474e-02,
    8.8404026343e-03, 2.3776567058e-02, 8.8171887083e-03, -4.6290425955e-02, -9.7997267900e-03)


def listed():
    return [
        # one ciphertext of a small ring through transform, rotation, product, rescale and
        # back: a handful of launches, where latency counts
        {"name": "pipeline_n13", "kind": "pipeline", "log_n": 13, "chain": "small50", "limbs": 8},
        # a client's round trip on host data: encode, public-key encryption, decryption, decode
        {"name": "client_n16", "kind": "client", "log_n": 16, "chain": "layer", "limbs": 24, "slots": 32768},
        # the transform itself, both directions, over a layer's batch of polynomials
        {"name": "ntt_64x24_n16", "kind": "ntt", "log_n": 16, "chain": "wide50", "polys": 64, "limbs": 24},
        # one rotation at the top level of the bootstrapping chain (a whole hybrid key switch)
        {"name": "rotate_top_n16", "kind": "keyswitch", "op": "rotate", "log_n": 16, "chain": "boot", "limbs": 35,
         "steps": 1},
        # a ciphertext product with relinearisation and rescale in the middle of a layer
        {"name": "multiply_mid_n16", "kind": "keyswitch", "op": "multiply", "log_n": 16, "chain": "layer", "limbs": 22,
         "steps": 1},
        # projection of 192 columns onto one attention head's 64 (column packing, 24 x 50 bits)
        {"name": "matmul_192x64_n16", "kind": "matmul", "log_n": 16, "chain": "wide50", "limbs": 24, "rows": 192,
         "cols": 64},
        # an uneven projection on the layer's 46-bit primes, more rows than one launch takes
        {"name": "matmul_301x37_n15", "kind": "matmul", "log_n": 15, "chain": "layer", "limbs": 11, "rows": 301,
         "cols": 37},
        # masked projection (uneven token counts): every weight is its own plaintext
        {"name": "masked_40x24_n16", "kind": "masked", "log_n": 16, "chain": "wide50", "limbs": 24, "rows": 40,
         "cols": 24},
        # attention scores: ciphertext x ciphertext in column packing, a head's 64 columns
        {"name": "scores_64x3_n16", "kind": "scores", "log_n": 16, "chain": "layer", "limbs": 24, "cols": 64,
         "rows": 3},
        # GELU on a group of 8 ciphertexts
        {"name": "gelu_8_n16", "kind": "gelu", "log_n": 16, "chain": "layer", "limbs": 24, "members": 8},
        # one ciphertext refreshed by itself (the per-ciphertext bootstrap)
        {"name": "boot_1_n16", "kind": "boot", "log_n": 16, "chain": "boot", "members": 1, "shared": False},
        # one chunk of the layer's 768 ciphertexts: 8 members sharing their a part
        {"name": "boot_shared_8_n16", "kind": "boot", "log_n": 16, "chain": "boot", "members": 8, "shared": True},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["pipeline", "client", "ntt", "ntt", "rotate", "rotate", "multiply", "multiply", "sum", "matmul",
                       "matmul", "masked", "scores", "gelu", "boot", "boot"])
    if kind == "pipeline":
        return {"kind": "pipeline", "log_n": rng.randint(13, 16), "chain": "small50", "limbs": rng.randint(2, 8)}
    if kind == "client":
        log_n = rng.randint(13, 16)
        return {"kind": "client", "log_n": log_n, "chain": "layer", "limbs": rng.randint(2, 35),
                "slots": _log_int(rng, 1, 1 << (log_n - 1))}
    if kind == "ntt":
        return {"kind": "ntt", "log_n": rng.randint(13, 16), "chain": rng.choice(["wide50", "layer", "small50"]),
                "polys": _log_int(rng, 1, 64), "limbs": rng.randint(1, 8)}
    if kind in ("rotate", "multiply", "sum"):
        small = rng.random() < 0.3
        return {"kind": "keyswitch", "op": kind, "log_n": 13 if small else rng.randint(14, 16),
                "chain": "boot_small" if small else rng.choice(["layer", "boot"]),
                "limbs": rng.randint(3, 15) if small else rng.randint(4, 35),
                "steps": rng.randint(2, 7) if kind == "sum" else 1}
    if kind == "matmul":
        chain = rng.choice(["wide50", "layer"])
        log_n = rng.randint(13, 16)
        return {"kind": "matmul", "log_n": log_n, "chain": chain, "limbs": rng.randint(3, 24 if log_n < 16 else 12),
                "rows": _log_int(rng, 5, 400), "cols": _log_int(rng, 1, 64)}
    if kind == "masked":
        return {"kind": "masked", "log_n": rng.randint(13, 16), "chain": "wide50", "limbs": rng.randint(3, 24),
                "rows": _log_int(rng, 1, 48), "cols": _log_int(rng, 1, 32)}
    if kind == "scores":
        return {"kind": "scores", "log_n": rng.randint(13, 16), "chain": "layer", "limbs": rng.randint(4, 24),
                "cols": _log_int(rng, 2, 48), "rows": rng.randint(1, 4)}
    if kind == "gelu":
        return {"kind": "gelu", "log_n": rng.randint(14, 16), "chain": "layer", "limbs": rng.randint(9, 24),
                "members": rng.randint(1, 9)}
    if rng.random() < 0.3:
        return {"kind": "boot", "log_n": 16, "chain": "boot", "members": rng.randint(1, 3), "shared": False}
    return {"kind": "boot", "log_n": 13, "chain": "boot_small", "members": rng.randint(1, 8),
            "shared": rng.random() < 0.7}


class _Words:
    """Device words of a ciphertext as torch sees them (no copy)."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<i8", "data": (int(ptr), False),
                                         "version": 2, "strides": None}


def words(ct):
    size, _, limbs, _ = ct.info()
    return torch.as_tensor(_Words(ct, ct.data_ptr(), (size, limbs, ct.ctx.N)), device="cuda")


class Party:
    """Context and keys of one parameter set."""

    def __init__(self, log_n, chain):
        bits, n_special = CHAINS[chain]
        self.ctx = shm.Context(log_n, bits, n_special)
        self.scale = SCALE[chain]
        self.sk = shm.SecretKey(self.ctx, seed=1, hamming_weight=192 if log_n >= 15 else 64)
        self.enc, self.dec = shm.Encoder(self.ctx), shm.Decryptor(self.ctx, self.sk)
        self.ev = shm.Evaluator(self.ctx)
        self._made = {}

    def get(self, what, make):
        if what not in self._made:
            self._made[what] = make()
        return self._made[what]

    def relin(self):
        return self.get("relin", lambda: self.sk.gen_relinkey(seed=3))

    def public(self):
        return self.get("public", lambda: self.sk.gen_publickey(seed=4))

    def galois(self, steps):
        steps = tuple(sorted(set(steps)))
        return self.get(("galois", steps), lambda: self.sk.create_galois_keys_from_steps(list(steps), seed=2))

    def boot(self):
        def make():
            b = shm.Bootstrapper(self.ctx)
            b.prepare()
            return b
        return self.get("boot", make)

    def shared(self, n):
        def make():
            k = shm.SharedAKeys(self.ctx, self.sk, n, 192 if self.ctx.N >= 1 << 15 else 64, 12, self.ctx.chain(4))
            k.add_galois(self.boot().rotation_steps(), seed=13)
            return k
        return self.get(("shared", n), make)


_party = {}


def party(case):
    key = (case["log_n"], case["chain"], case.get("shared"), case["members"] if case.get("shared") else 0)
    if key not in _party:
        _party.clear()
        gc.collect()
        _party[key] = Party(case["log_n"], case["chain"])
    return _party[key]


def _uniform(p, limbs, gen, out):
    """Residues uniform below each prime: the limbs of a ciphertext."""
    for k in range(limbs):
        q = int(p.ctx.coeff_modulus[k])
        out[:, k] = torch.randint(0, q, (out.shape[0], out.shape[2]), generator=gen, device="cuda")


def _ciphertexts(p, limbs, count, gen):
    cts = []
    for _ in range(count):
        ct = shm.Ciphertext(p.ctx, 2, p.ctx.chain(limbs))
        ct.scale = p.scale
        _uniform(p, limbs, gen, words(ct))
        cts.append(ct)
    return cts


def _encrypted(p, zs, limbs, seed):
    return [p.sk.encrypt_symmetric(p.enc.encode(z, p.scale, p.ctx.chain(limbs)), seed=seed * 1000 + i)
            for i, z in enumerate(zs)]


def prepare(case, seed):
    p = party(case)
    kind, n = case["kind"], p.ctx.N
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    s = {"case": case, "party": p}
    if kind == "pipeline":
        s["x"] = _ciphertexts(p, case["limbs"], 1, gen)[0]
        s["gk"] = p.galois([1])
        s["pt"] = p.enc.encode(float(rng.uniform(0.1, 1.0)), p.scale, p.ctx.chain(case["limbs"]))
    elif kind == "client":
        s["z"] = rng.uniform(-1, 1, case["slots"])
        s["seed"] = seed
        s["encryptor"] = shm.Encryptor(p.ctx, p.public())
    elif kind == "ntt":
        limbs = case["limbs"]
        s["x"] = torch.empty((case["polys"], limbs, n), dtype=torch.int64, device="cuda")
        _uniform(p, limbs, gen, s["x"])
    elif kind == "keyswitch":
        count = 2 if case["op"] == "multiply" else 1
        s["x"] = _ciphertexts(p, case["limbs"], count, gen)
        if case["op"] == "multiply":
            s["rk"] = p.relin()
        else:
            s["steps"] = [1 << i for i in range(case["steps"])]
            s["gk"] = p.galois(s["steps"])
    elif kind in ("matmul", "masked"):
        s["x"] = _ciphertexts(p, case["limbs"], case["rows"], gen)
        s["w"] = rng.normal(0.0, 0.02, (case["rows"], case["cols"]))
        if kind == "masked":
            s["mask"] = (rng.random(n // 2) < 0.7).astype(np.int32)
    elif kind == "scores":
        s["x"] = _ciphertexts(p, case["limbs"], case["cols"], gen)
        s["y"] = _ciphertexts(p, case["limbs"], case["cols"], gen)
        s["gk"], s["rk"] = p.galois([256 * i for i in range(1, max(2, case["rows"]))]), p.relin()
    elif kind == "gelu":
        zs = [rng.uniform(-19.5, 12.5, n // 2) for _ in range(case["members"])]
        s["x"], s["rk"] = _encrypted(p, zs, case["limbs"], seed), p.relin()
    elif kind == "boot":
        zs = [rng.uniform(-1, 1, n // 2) for _ in range(case["members"])]
        s["x"], s["rk"], s["boot"] = _encrypted(p, zs, 4, seed), p.relin(), p.boot()
        if case["shared"]:
            s["keys"] = p.shared(case["members"])
        else:
            s["gk"] = p.galois(p.boot().rotation_steps())
    return s


def run(s):
    case, p = s["case"], s["party"]
    kind, ctx, ev = case["kind"], p.ctx, p.ev
    if kind == "pipeline":
        ct = s["x"].copy()
        ctx.ntt_forward(ct.data_ptr(), 2, case["limbs"], 0)
        ev.rotate_vector_inplace(ct, 1, s["gk"])
        ev.multiply_plain_inplace(ct, s["pt"])
        ev.rescale_to_next_inplace(ct)
        ctx.ntt_inverse(ct.data_ptr(), 2, case["limbs"] - 1, 0)
        return words(ct)
    if kind == "client":
        pt = p.enc.encode(s["z"], p.scale, 1)
        ct = s["encryptor"].encrypt(pt, s["seed"])
        ev.mod_switch_to_inplace(ct, ctx.chain(case["limbs"]))
        return words(ct), p.enc.decode(p.dec.decrypt(ct))
    if kind == "ntt":
        forward = s["x"].clone()
        ctx.ntt_forward(forward.data_ptr(), case["polys"], case["limbs"], 0)
        inverse = s["x"].clone()
        ctx.ntt_inverse(inverse.data_ptr(), case["polys"], case["limbs"], 0)
        return forward, inverse
    if kind == "keyswitch":
        ct = s["x"][0].copy()
        if case["op"] == "multiply":
            ev.multiply_inplace(ct, s["x"][1])
            ev.relinearize_inplace(ct, s["rk"])
            ev.rescale_to_next_inplace(ct)
        elif case["op"] == "sum":
            ev.hoisting_inplace(ct, s["gk"], s["steps"])
        else:
            ev.rotate_vector_inplace(ct, s["steps"][0], s["gk"])
        return words(ct)
    if kind == "matmul":
        out = shm.ct_pt_matrix_mul_wo_pre(s["x"], s["w"], case["rows"], case["cols"], case["rows"], ctx)
    elif kind == "masked":
        out = shm.ct_pt_matrix_mul_wo_pre_w_mask(s["x"], s["w"], s["mask"], case["rows"], case["cols"], case["rows"],
                                                 ctx)
    elif kind == "scores":
        out = shm.ct_ct_matrix_mul_colpacking(s["x"], s["y"], s["gk"], s["rk"], ctx, case["cols"], case["rows"],
                                              case["cols"], case["rows"], 256)
    elif kind == "gelu":
        out = [x.copy() for x in s["x"]]
        ev.evaluate_chebyshev_inplace(out, GELU, -19.5, 12.5, s["rk"])
    elif case["shared"]:
        out = shm.bootstrap_shared_a_s2c_first(s["boot"], s["keys"], s["x"], s["rk"])
    else:
        out = s["boot"].bootstrap_s2c_first(s["x"], s["gk"], s["rk"])
    return [words(ct) for ct in out]


def _butterflies(limbs, log_n):
    """Operations of transforms of `limbs` limbs: one product and two sums a butterfly."""
    return 3.0 * limbs * (log_n << (log_n - 1))


def work(case):
    """Bytes: inputs, keys and outputs once. Operations: modular products and sums."""
    kind, log_n = case["kind"], case["log_n"]
    bits, n_special = CHAINS[case["chain"]]
    n, n_data, limb = 1 << log_n, len(bits) - n_special, 8.0 * (1 << log_n)
    dnum = n_data // n_special

    def switch(limbs):
        """(key bytes, operations) of one key switch of one polynomial at `limbs` primes."""
        digits, ext = -(-limbs // n_special), limbs + n_special
        ops = _butterflies(limbs + digits * ext + 2 * n_special + 2 * limbs, log_n)
        ops += 2.0 * n * (digits * ext * (n_special + 2) + 2 * limbs * n_special)
        return 2.0 * digits * ext * limb, ops

    if kind == "pipeline":
        q = case["limbs"]
        key, ops = switch(q)
        return {"bytes": (2 * q + q + 2 * (q - 1)) * limb + key, "flops": ops + _butterflies(8 * q, log_n)}
    if kind == "client":
        q = case["limbs"]
        return {"bytes": (2 * (n_data + n_special) + 2 * q) * limb + 8.0 * (case["slots"] + n // 2),
                "flops": _butterflies(4 * (n_data + n_special) + q, log_n)}
    if kind == "ntt":
        limbs = case["polys"] * case["limbs"]
        return {"bytes": 4 * limbs * limb, "flops": _butterflies(2 * limbs, log_n)}
    if kind == "keyswitch":
        q = case["limbs"]
        key, ops = switch(q)
        if case["op"] == "multiply":
            return {"bytes": (4 * q + 2 * (q - 1)) * limb + key, "flops": ops + _butterflies(2 * q, log_n) + 8.0 * q * n}
        return {"bytes": 4 * q * limb + case["steps"] * key, "flops": ops}
    if kind in ("matmul", "masked"):
        q, r, c = case["limbs"], case["rows"], case["cols"]
        ops = 4.0 * r * c * q * n + _butterflies(2 * c * q, log_n)
        if kind == "masked":
            ops += _butterflies(r * c * q, log_n)
        return {"bytes": 2 * (r * q + c * (q - 1)) * limb + 8.0 * r * c, "flops": ops}
    if kind == "scores":
        q, c, r = case["limbs"], case["cols"], case["rows"]
        key, ops = switch(q)
        return {"bytes": (4 * c * q + 2 * r * (q - 1)) * limb + r * key,
                "flops": ops * (c * (r - 1) + r) + 8.0 * c * r * q * n + _butterflies(2 * r * q, log_n)}
    if kind == "gelu":
        q, m = case["limbs"], case["members"]
        key, ops = switch(q - 3)
        return {"bytes": m * (2 * q + 2 * (q - 6)) * limb + key, "flops": 10.0 * m * (ops + _butterflies(2 * q, log_n))}
    # bootstrapping: the keys of 38 rotations and the conjugation, diagonals, in- and outputs
    m, out = case["members"], n_data - 13
    per_key = dnum * (n_data + n_special) * limb * ((m + 1) if case["shared"] else 2)
    rotation_keys, mid = 39, n_data - 6
    _, ops = switch(n_data)
    _, product = switch(mid)
    rotations = 38.0 * (ops * (1 if case["shared"] else m))
    return {"bytes": rotation_keys * per_key + m * 2 * (4 + out) * limb + 15 * 6 * n_data * limb / 2,
            "flops": rotations / 2 + 2 * m * 18.0 * (product + _butterflies(2 * mid, log_n))}


def exact(case, seed):
    """A client's round trip gives back the message; every other output is whole numbers."""
    if case["kind"] != "client":
        return None
    z = np.zeros(1 << (case["log_n"] - 1))
    z[:case["slots"]] = np.random.default_rng(seed).uniform(-1, 1, case["slots"])
    return None, z
