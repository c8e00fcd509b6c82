"""What a program that uses this engine has it do, as cases that can be timed: transforms, products, rotations, encryption,
decryption and encrypted Krum, through pyCAHEL (what Lancelot's Python calls) and through the C-ABI on torch tensors (what a
C++ host or a server with buffers of its own calls).

The sizes are those of BASELINE.json's configurations, of Lancelot's own chain ([60, 40, 40, 60] at N = 2^16) and of the
range between: degrees 2^12 to 2^16, 1 to 24 data limbs, 1 to 8 special primes, primes of 30 to 60 bits, levels in the
middle of a chain (a last digit that is not full).  Polynomials are [poly][limb][coefficient] words; a limb is 8 N bytes.
"""
import collections
import math

import numpy as np
import torch

import lancelot_amd  # noqa: F401  (registers the native module as pyCAHEL)
import pyCAHEL as cahel
from lancelot_amd import capi, krum

KEY_SEED = 2025     # keys and context are the program's, whatever the inputs


def listed():
    return [
        # the smallest call there is: one ciphertext at N = 2^12 with the three small primes that 128-bit security
        # leaves there.  Latency of one launch.
        {"name": "ntt_forward_n4096", "op": "ntt", "log_n": 12, "first": 36, "mid": 36, "limbs": 3, "polys": 2, "inverse": False},
        # batched transform of one ciphertext at the benchmark shape
        {"name": "ntt_inverse_n65536_24", "op": "ntt", "log_n": 16, "first": 50, "mid": 50, "limbs": 24, "polys": 2, "inverse": True},
        # multiply, relinearise, rescale as three pyCAHEL calls at N = 2^14, 4 + 1 primes
        {"name": "multiply_n16384_4", "op": "multiply", "log_n": 14, "first": 50, "mid": 50, "special": 50, "size_q": 4,
         "size_p": 1, "limbs": 4, "log_scale": 40},
        # the usual chain of a CKKS program (60-bit first and special primes, 40-bit scaling primes), two levels down: the
        # last of its digits holds one limb of three
        {"name": "multiply_n32768_10_of_12", "op": "multiply", "log_n": 15, "first": 60, "mid": 40, "special": 60, "size_q": 12,
         "size_p": 3, "limbs": 10, "log_scale": 36},
        # BASELINE.json configs[2], one product at a time as the reference's evaluator calls it
        {"name": "multiply_n65536_24", "op": "multiply", "log_n": 16, "first": 50, "mid": 50, "special": 50, "size_q": 24,
         "size_p": 8, "limbs": 24, "log_scale": 40},
        # the same product for a server that has eight independent ones in hand
        {"name": "multiply_batch8_n65536_24", "op": "multiply_batch", "log_n": 16, "first": 50, "mid": 50, "special": 50,
         "size_q": 24, "size_p": 8, "limbs": 24, "items": 8},
        # one keyed rotation of its rotate-and-sum
        {"name": "rotate_n65536_24", "op": "rotate", "log_n": 16, "first": 50, "mid": 50, "special": 50, "size_q": 24,
         "size_p": 8, "limbs": 24, "log_scale": 40, "step": 1},
        # the same slot sum in hoisted rounds: one round of seven rotations
        {"name": "hoist_n65536_24_7steps", "op": "hoist", "log_n": 16, "first": 50, "mid": 50, "special": 50, "size_q": 24,
         "size_p": 8, "limbs": 24, "log_scale": 40, "steps": 7},
        # one chunk of a client's update, encoded and encrypted on Lancelot's chain from host values
        {"name": "encrypt_n65536_3", "op": "encrypt", "log_n": 16, "first": 60, "mid": 40, "special": 60, "size_q": 3,
         "size_p": 1, "limbs": 3, "log_scale": 40, "values": 32768},
        # one result of Lancelot's chain after its rescale, decrypted and decoded to host values
        {"name": "decrypt_n65536_2", "op": "decrypt", "log_n": 16, "first": 60, "mid": 40, "special": 60, "size_q": 3,
         "size_p": 1, "limbs": 2, "log_scale": 40, "values": 32768},
        # the distance of one pair of clients, call for call as Lancelot's driver computes it (two chunks a client, every
        # operand encoded and encrypted, one pyCAHEL call per operation)
        {"name": "krum_pair_n65536_2chunks", "op": "krum_pair", "log_n": 16, "params": 62006},
        # a whole encrypted Krum round with the masked sum of the updates at its end
        {"name": "krum_round_10x62006", "op": "krum_round", "log_n": 16, "clients": 10, "params": 62006, "aggregate": True},
    ]


# ---- drawn cases ------------------------------------------------------------------------------------------------------

def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _chain(rng):
    """(first, mid, special) prime sizes: all of one size below or above 50 bits, or the usual 60 / smaller / 60."""
    kind = rng.randrange(4)
    if kind == 0:
        return 50, 50, 50
    if kind == 1:
        b = rng.randrange(34, 50)
        return b, b, b
    if kind == 2:
        b = rng.randrange(51, 61)
        return b, b, b
    return 60, rng.randrange(35, 51), 60


def _level(rng, most=24):
    """(size_q, size_p, limbs): a chain of whole digits and a level of it."""
    size_p = _log_int(rng, 1, 8)
    digits = _log_int(rng, 1, max(1, min(most // size_p, 8)))
    size_q = max(2, digits * size_p)
    return size_q, size_p, rng.randrange(2, size_q + 1)


def draw(rng):
    op = rng.choice(["ntt", "multiply", "multiply", "multiply_batch", "rotate", "hoist", "encrypt", "decrypt", "krum_pair",
                     "krum_round"])
    log_n = rng.randrange(12, 17)
    if op == "ntt":
        first, mid, _ = _chain(rng)
        return {"op": op, "log_n": log_n, "first": first, "mid": mid, "limbs": _log_int(rng, 1, 24), "polys": rng.randrange(1, 5),
                "inverse": rng.random() < 0.5}
    if op == "krum_pair":
        log_n = rng.randrange(13, 17)
        return {"op": op, "log_n": log_n, "params": _log_int(rng, 1000, 2 << (log_n - 1))}
    if op == "krum_round":
        log_n = rng.randrange(13, 17)
        return {"op": op, "log_n": log_n, "clients": rng.randrange(3, 11), "params": _log_int(rng, 1000, min(62006, 2 << (log_n - 1))),
                "aggregate": rng.random() < 0.5}
    first, mid, special = _chain(rng)
    size_q, size_p, limbs = _level(rng)
    case = {"op": op, "log_n": log_n, "first": first, "mid": mid, "special": special, "size_q": size_q, "size_p": size_p,
            "limbs": limbs}
    if op == "multiply_batch":
        # up to eight products at the benchmark shape, more of smaller ones
        return dict(case, items=_log_int(rng, 1, min(32, max(1, (8 * 24 << 16) // (limbs << log_n)))))
    case["log_scale"] = min(40, mid - 4)
    if op == "rotate":
        return dict(case, step=rng.randrange(1, 1 << (log_n - 2)) * rng.choice([1, -1]))
    if op == "hoist":
        return dict(case, steps=rng.randrange(2, 8))
    if op in ("encrypt", "decrypt"):
        return dict(case, values=_log_int(rng, 256, 1 << (log_n - 1)))
    return case


# ---- what a program holds before the call -----------------------------------------------------------------------------

Session = collections.namedtuple("Session", "context sk pk rlk glk moduli")
_sessions = collections.OrderedDict()


def _kept(key, make):
    """A program makes its context and keys once and runs many inputs on them; the last two sets are kept."""
    if key not in _sessions:
        while len(_sessions) >= 2:
            _sessions.popitem(last=False)
        _sessions[key] = make()
    _sessions.move_to_end(key)
    return _sessions[key]


def _session(log_n, bits, size_p, steps=(), relin=True):
    def make():
        n = 1 << log_n
        parms = cahel.params(cahel.scheme_type.ckks)
        parms.set_poly_modulus_degree(n)
        moduli = cahel.coeff_modulus_create(n, bits)
        parms.set_coeff_modulus(moduli)
        parms.set_special_modulus_size(size_p)
        parms.set_galois_elts(cahel.get_elts_from_steps(list(steps) or [1], n))
        context = cahel.context(parms, True, cahel.sec_level_type.none)
        context.set_seed(KEY_SEED)
        sk = cahel.secret_key(parms)
        sk.gen_secretkey(context)
        pk = cahel.public_key(context)
        sk.gen_publickey(context, pk)
        rlk = glk = None
        if size_p and relin:
            rlk = cahel.relin_key(context)
            sk.gen_relinkey(context, rlk)
        if size_p and steps:
            glk = cahel.galois_key(context)
            sk.create_galois_keys(context, glk)
        return Session(context, sk, pk, rlk, glk, [m.value() for m in moduli])
    return _kept(("session", log_n, tuple(bits), size_p, tuple(steps), relin), make)


def _krum_state(case):
    """The driver's context and keys; a pair by itself takes the reference's plan (hoisting of 1..15, then doublings)."""
    def make():
        if case["op"] == "krum_pair":
            return krum.gpu_init(krum.KrumConfig(log_n=case["log_n"], seed=KEY_SEED, hoisting_radix=0, batched=False, lanes=0))
        return krum.gpu_init(krum.KrumConfig(log_n=case["log_n"], seed=KEY_SEED))
    return _kept(("krum", case["op"], case["log_n"]), make)


def _bits(case):
    return [case["first"]] + [case["mid"]] * (case["size_q"] - 1) + [case["special"]] * case["size_p"]


def _hoist_steps(case):
    return list(range(1, case["steps"] + 1))


def _uniform(case, moduli, shape, generator):
    """Uniform residues on the GPU, limb i below moduli[i]: what ciphertext words look like."""
    out = torch.empty(shape, dtype=torch.int64, device="cuda")
    for i in range(shape[-2]):
        out[..., i, :] = torch.randint(0, moduli[i], shape[:-2] + shape[-1:], dtype=torch.int64, device="cuda", generator=generator)
    return out


def prepare(case, seed):
    op, n = case["op"], 1 << case["log_n"]
    rng = np.random.default_rng(seed)
    if op == "ntt":
        s = _session(case["log_n"], [case["first"]] + [case["mid"]] * (case["limbs"] - 1), 0, relin=False)
        generator = torch.Generator(device="cuda")
        generator.manual_seed(seed)
        return {"op": op, "case": case, "h": s.context.he_handle(), "keep": s,
                "data": _uniform(case, s.moduli, (case["polys"], case["limbs"], n), generator)}
    if op in ("krum_pair", "krum_round"):
        state = _krum_state(case)
        clients = case.get("clients", 2)
        # flattened updates of a small network, Gaussian; the last fifth of the clients Byzantine (scaled up)
        updates = [rng.normal(0.0, 0.01, case["params"]).astype(np.float32) for _ in range(clients)]
        if op == "krum_round":
            for k in range(clients - clients // 5, clients):
                updates[k] = updates[k] * 10
        state.context.set_seed(seed)
        st = {"op": op, "case": case, "state": state, "updates": updates}
        if op == "krum_pair":
            st["chunks"] = krum.split_updates(updates, state.slots)
        return st
    if op == "multiply_batch":
        s = _session(case["log_n"], _bits(case), case["size_p"])
        h, L, items = s.context.he_handle(), case["limbs"], case["items"]
        generator = torch.Generator(device="cuda")
        generator.manual_seed(seed)
        words = capi.lib().he_multiply_relin_rescale_batch_workspace_words(h, L, items)
        return {"op": op, "case": case, "h": h, "keep": s, "L": L,
                "evk": capi.evk_array([s.rlk.digit_ptr(d) for d in range(-(-L // case["size_p"]))]),
                "a": _uniform(case, s.moduli, (items, 2, L, n), generator),
                "b": _uniform(case, s.moduli, (items, 2, L, n), generator),
                "out": torch.empty((items, 2, L - 1, n), dtype=torch.int64, device="cuda"),
                "ws": torch.empty(words, dtype=torch.int64, device="cuda")}
    steps = [case["step"]] if op == "rotate" else _hoist_steps(case) if op == "hoist" else []
    s = _session(case["log_n"], _bits(case), case["size_p"], steps, relin=op == "multiply")
    ctx, scale = s.context, 2.0 ** case["log_scale"]
    ctx.set_seed(seed)
    encoder = cahel.ckks_encoder(ctx)
    chain = 1 + case["size_q"] - case["limbs"]
    st = {"op": op, "case": case, "s": s, "encoder": encoder, "scale": scale, "chain": chain}

    def fresh():
        # slots uniform in [-1, 1]: what BASELINE.json's configurations encrypt
        values = rng.uniform(-1.0, 1.0, case.get("values", n // 2))
        return s.pk.encrypt_asymmetric(ctx, encoder.encode_to(ctx, values, chain, scale))

    if op == "encrypt":
        st["values"] = rng.uniform(-1.0, 1.0, case["values"])
    else:
        st["ct1"] = fresh()
        if op == "multiply":
            st["ct2"] = fresh()
    return st


# ---- one pass ---------------------------------------------------------------------------------------------------------

class _DeviceWords:
    """A ciphertext's words as a device array that torch can look at without a copy; keeps the ciphertext alive."""

    def __init__(self, ct, n):
        self.ct = ct
        self.__cuda_array_interface__ = {"shape": (ct.size(), ct.coeff_modulus_size(), n), "typestr": "<i8",
                                         "data": (ct.data_ptr(), False), "version": 2}


def _words(ct, n):
    return torch.as_tensor(_DeviceWords(ct, n), device="cuda")


def _pair(st):
    """GPU_compute_pair_distance of lancelot-main-GPU/utils/byzantine_fl.py:173-321, call for call."""
    state, (msg1, msg2) = st["state"], st["chunks"]
    ctx, enc, pk, scale = state.context, state.encoder, state.pk, state.config.scale
    acc, tmp = None, cahel.ciphertext(ctx)
    for x1, x2 in zip(msg1, msg2):
        ct1 = pk.encrypt_asymmetric(ctx, enc.encode(ctx, x1, scale))
        ct2 = pk.encrypt_asymmetric(ctx, enc.encode(ctx, x2, scale))
        cahel.sub(ctx, ct2, ct1, tmp)
        cahel.square_inplace(ctx, tmp)
        if acc is None:
            acc, tmp = tmp, cahel.ciphertext(ctx)
        else:
            cahel.add_inplace(ctx, acc, tmp)
    cahel.relinearize_inplace(ctx, acc, state.rlk)
    cahel.rescale_to_next_inplace(ctx, acc)
    acc.set_scale(scale)
    cahel.add_inplace(ctx, acc, cahel.hoisting(ctx, acc, state.glk, list(range(1, 16))))
    rot = cahel.ciphertext(ctx)
    for k in range(4, int(math.log2(state.slots))):
        cahel.rotate_vector(ctx, acc, 2 ** k, state.glk, rot)
        cahel.add_inplace(ctx, acc, rot)
    return acc


def run(st):
    op, case = st["op"], st["case"]
    if op == "ntt":
        transform = capi.lib().he_ntt_inverse if case["inverse"] else capi.lib().he_ntt_forward
        capi.check(transform(st["h"], st["data"].data_ptr(), case["polys"], case["limbs"], case["limbs"], 0, case["limbs"], 0, None))
        return st["data"]
    if op == "multiply_batch":
        capi.check(capi.lib().he_multiply_relin_rescale_batch(st["h"], st["L"], case["items"], st["a"].data_ptr(), st["b"].data_ptr(),
                                                              st["evk"], st["out"].data_ptr(), st["ws"].data_ptr(), None))
        return st["out"]
    n = 1 << case["log_n"]
    if op == "krum_pair":
        return _words(_pair(st), n)
    if op == "krum_round":
        if case["aggregate"]:
            chosen, weights, _ = krum.gpu_krum_aggregate(st["updates"], state=st["state"])
            return {"chosen": chosen, "weights": weights}
        chosen, distances, _ = krum.gpu_krum(st["updates"], state=st["state"])
        return {"chosen": chosen, "distances": distances}
    s = st["s"]
    ctx = s.context
    if op == "multiply":
        product = cahel.ciphertext(ctx)
        cahel.multiply(ctx, st["ct1"], st["ct2"], product)
        cahel.relinearize_inplace(ctx, product, s.rlk)
        cahel.rescale_to_next_inplace(ctx, product)
        return _words(product, n)
    if op == "rotate":
        rotated = cahel.ciphertext(ctx)
        cahel.rotate_vector(ctx, st["ct1"], case["step"], s.glk, rotated)
        return _words(rotated, n)
    if op == "hoist":
        return _words(cahel.hoisting(ctx, st["ct1"], s.glk, _hoist_steps(case)), n)
    if op == "encrypt":
        return _words(s.pk.encrypt_asymmetric(ctx, st["encoder"].encode_to(ctx, st["values"], st["chain"], st["scale"])), n)
    if op == "decrypt":
        return st["encoder"].decode_array(ctx, s.sk.decrypt(ctx, st["ct1"]))
    raise ValueError(op)


# ---- what a pass cannot do without ------------------------------------------------------------------------------------

def _transforms(n, limbs):
    """Operations of `limbs` transforms: a butterfly is a modular product (a multiply-add), an addition, a subtraction."""
    return limbs * 4 * (n // 2) * int(math.log2(n))


def _key_switch(n, L, K, steps=1):
    """(limbs of key read, operations) of ModUp, `steps` inner products and one ModDown of two polynomials."""
    beta = -(-L // K)
    ops = _transforms(n, L + beta * (L + K) - L + 2 * K + 2 * L)
    sizes = [min(K, L - d * K) for d in range(beta)]
    ops += 2 * n * (sum(k * (L + K - k) for k in sizes) + 2 * K * L)     # base conversions
    ops += steps * 2 * n * 2 * beta * (L + K)                            # products with the keys
    return steps * 2 * beta * (L + K), ops


def work(case):
    op, n = case["op"], 1 << case["log_n"]
    limb = 8 * n
    if op == "ntt":
        limbs = case["polys"] * case["limbs"]
        return {"bytes": 2 * limbs * limb, "flops": _transforms(n, limbs)}
    if op in ("krum_pair", "krum_round"):
        clients = case.get("clients", 2)
        chunks = -(-case["params"] // (n // 2))
        pairs = clients * (clients - 1) // 2
        log_slots = case["log_n"] - 1
        # slots in and out of the encoder (a product and two additions a butterfly, complex), transform of the limbs,
        # u pk + e of two polynomials over the four primes
        encrypt = 10 * (n // 4) * log_slots + _transforms(n, 3 + 12 + 6) + 2 * 2 * 4 * n
        key, relin = _key_switch(n, 3, 1)
        # one key switch per doubling is the least that the slot sum's arithmetic allows without more keys
        rot_key, rot = _key_switch(n, 2, 1)
        pair = chunks * (2 + 6) * 3 * n + relin + log_slots * rot
        flops = clients * chunks * encrypt + pairs * pair
        moved = clients * case["params"] * 4 + (key + log_slots * rot_key + 2 * 4) * limb
        if op == "krum_pair":
            moved += 4 * limb
        elif case["aggregate"]:
            moved += 8 * case["params"]
            flops += clients * chunks * 8 * 3 * n + chunks * _transforms(n, 3)
        else:
            moved += 8 * clients * clients
            flops += pairs * _transforms(n, 2)
        return {"bytes": moved, "flops": flops}
    L, K = case["limbs"], case["size_p"]
    if op == "encrypt":
        return {"bytes": 8 * case["values"] + (2 * (L + K) + 2 * L) * limb,
                "flops": 10 * (n // 4) * (case["log_n"] - 1) + _transforms(n, L + 3 * (L + K) + 2 * K + 2 * L) + 2 * 2 * (L + K) * n}
    if op == "decrypt":
        return {"bytes": (2 * L + L) * limb + 8 * case["values"],
                "flops": 10 * (n // 4) * (case["log_n"] - 1) + _transforms(n, 2 * L) + 2 * L * n + L * L * n}
    if op == "rotate":
        key, ops = _key_switch(n, L, K)
        return {"bytes": (4 * L + key) * limb, "flops": ops}
    if op == "hoist":
        key, ops = _key_switch(n, L, K, case["steps"])
        return {"bytes": (4 * L + key) * limb, "flops": ops}
    # multiply, multiply_batch: two operands in, one out, the key once for the call
    items = case.get("items", 1)
    key, ops = _key_switch(n, L, K)
    rescale = _transforms(n, 2)
    return {"bytes": (items * (4 * L + 2 * (L - 1)) + key) * limb, "flops": items * (ops + rescale + 2 * 4 * L * n)}


def tolerance(case):
    # Residues are integers: every correct implementation gives the same words.
    if case["op"] == "decrypt":
        # slots in double precision, after 2^15 terms of a Fourier transform in double precision
        return {"rel": 1e-10}
    if case["op"] == "krum_round":
        # decoded values of approximate arithmetic: the rounding of the rescale and the noise of the key switches, which
        # depend on the order of the rotations (scale 2^40, distances to 7e-6 of the float64 closed form)
        return {"rel": 2e-5}
    return "exact"
