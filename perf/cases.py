"""The calls a program that uses this library makes, as measurable cases.

Every case goes through the public Python binding (``tfhe_amd``), which is a thin
layer over the C ABI:

* ``gate``  a batch of independent gate bootstraps (``GateContext.eval_batch``);
* ``func``  a batch of programmable bootstraps with an arbitrary table
  (``GateContext.eval_func``);
* ``cbs_lut``  circuit bootstrapping of the bits of some bytes, the conversion to
  evaluation form, one 8-bit table lookup per byte and the switch back to the
  level-0 key (``CbsContext.cbs_batch`` ... ``keyswitch_batch``);
* ``aes_ctr``  AES-128 CTR transciphering of public ciphertext blocks
  (``CbsContext.aes_ctr_transcipher``);
* ``aes_dec``  homomorphic AES-128 decryption of public ciphertext blocks with
  T-table rounds (``CbsContext.aes_decrypt``).

The parameter sets (``form``) are the ones the library offers: ``exact`` (the
default: two-limb PBS, lookup keys), ``fast`` (one-product two-bit PBS, linear keys;
what the bench's headline runs) and ``htss`` (HomTrace + SchemeSwitch conversion).

A program makes its context and keys once and calls it for as long as it runs, so
contexts are made on first use and shared by the cases of one form; what depends on
the seed (ciphertexts, tables, counters) is made anew by ``prepare``.
"""
import math
import os
import random
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "gpu-circuitbootstrapping-aestransciphering_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import tfhe_amd  # noqa: E402

KEY_SEED = 21
AES_KEY = bytes(range(16))  # the FIPS-197 C.1 key
MAX_GATES = 4096
MAX_BLOCKS = 64
GATES = {"NAND": tfhe_amd.NAND, "AND": tfhe_amd.AND, "OR": tfhe_amd.OR, "NOR": tfhe_amd.NOR, "XOR": tfhe_amd.XOR,
         "XNOR": tfhe_amd.XNOR}
FORMS = {"exact": {},
         "fast": {"pbs_approx": 1, "pbs_multibit": 3, "pfks_linear": 1, "ks_linear": 1},
         "htss": {"lwe_to_rgsw": 1}}


def listed():
    return [
        # the latency of one gate: what an interactive circuit waits for at every level
        {"name": "gate_nand_1", "kind": "gate", "gate": "NAND", "batch": 1},
        # one level of a small circuit (an adder's or comparator's parallel gates), ragged
        {"name": "gate_xor_61", "kind": "gate", "gate": "XOR", "batch": 61},
        # throughput of independent gates: the gate benchmark's batch
        {"name": "gate_nand_4096", "kind": "gate", "gate": "NAND", "batch": 4096},
        # an arbitrary function of 3-bit messages on a batch (two bootstraps each)
        {"name": "gate_func_1000", "kind": "func", "batch": 1000, "msgs": 8},
        # 256 LWE bits to RGSW, 32 byte lookups, key switch: the circuit-bootstrap benchmark,
        # in the default parameter set and in the fastest
        {"name": "cbs_lut_32_exact", "kind": "cbs_lut", "form": "exact", "nbytes": 32, "out_bits": 8},
        {"name": "cbs_lut_32_fast", "kind": "cbs_lut", "form": "fast", "nbytes": 32, "out_bits": 8},
        # AES-128 CTR transciphering: one block (latency, the captured graph a serving loop
        # replays), an uneven batch, a large one
        {"name": "aes_ctr_1_fast", "kind": "aes_ctr", "form": "fast", "blocks": 1, "mode": "graph"},
        {"name": "aes_ctr_17_fast", "kind": "aes_ctr", "form": "fast", "blocks": 17, "mode": "batch"},
        {"name": "aes_ctr_64_fast", "kind": "aes_ctr", "form": "fast", "blocks": 64, "mode": "batch"},
        # the default parameter set: exact products, lookup keys
        {"name": "aes_ctr_1_exact", "kind": "aes_ctr", "form": "exact", "blocks": 1, "mode": "batch"},
        # decryption of public ciphertext with T-table rounds (the other direction), uneven
        {"name": "aes_dec_5_fast", "kind": "aes_dec", "form": "fast", "blocks": 5},
        # the trace-based conversion with its small keys
        {"name": "aes_ctr_2_htss", "kind": "aes_ctr", "form": "htss", "blocks": 2, "mode": "batch"},
    ]


def _log_int(rng, lo, hi):
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng: random.Random):
    kind = rng.choice(["gate", "gate", "func", "cbs_lut", "cbs_lut", "aes_ctr", "aes_ctr", "aes_dec"])
    if kind == "gate":
        return {"kind": kind, "gate": rng.choice(sorted(GATES)), "batch": _log_int(rng, 1, MAX_GATES)}
    if kind == "func":
        return {"kind": kind, "batch": _log_int(rng, 1, 1024), "msgs": rng.choice([4, 8])}
    form = rng.choice(["exact", "fast", "fast", "htss"])
    if kind == "cbs_lut":
        return {"kind": kind, "form": form, "nbytes": _log_int(rng, 1, 280), "out_bits": rng.choice([8, 8, 5, 1])}
    if kind == "aes_dec":
        return {"kind": kind, "form": "fast", "blocks": _log_int(rng, 1, 24)}
    return {"kind": kind, "form": form, "blocks": _log_int(rng, 1, MAX_BLOCKS if form == "fast" else 12),
            "mode": rng.choice(["batch", "batch", "graph"])}


# ------------------------------------------------------------------ contexts and keys
_contexts = {}


def _gate_context():
    if "gate" not in _contexts:
        ctx = tfhe_amd.GateContext(max_batch=MAX_GATES)
        sk = tfhe_amd.lwe_keygen(ctx.p.n, KEY_SEED)
        ctx.bt_keygen(sk, KEY_SEED)
        _contexts["gate"] = (ctx, torch.from_numpy(sk).to("cuda"))
    return _contexts["gate"]


def _cbs_context(form, ttable=False):
    # a program that decrypts with T-table rounds keeps its own context for them
    name = (form, ttable)
    if name not in _contexts:
        params = tfhe_amd.cbs_params(**FORMS[form])
        ctx = tfhe_amd.CbsContext(max_blocks=MAX_BLOCKS if form == "fast" and not ttable else 24, params=params)
        sk = tfhe_amd.lwe_keygen(params.n, KEY_SEED)
        ctx.keygen(sk, KEY_SEED)
        ctx.set_round_keys(tfhe_amd.aes_encrypt_key_bits(sk, KEY_SEED + 1, AES_KEY))
        if ttable:
            ctx.set_dec_round_keys(tfhe_amd.aes_encrypt_dec_key_bits(sk, KEY_SEED + 1, AES_KEY))
            ctx.set_round_form(1)
        _contexts[name] = (ctx, torch.from_numpy(sk).to("cuda"))
    return _contexts[name]


def _encrypt(msgs, delta, sk, gen, modulus_bits=32):
    """LWE encryptions [len][n + 1] (int32 words) of msgs * delta over Z_2^modulus_bits under the
    binary key sk, noise sigma 2^-15 of the modulus (at least one unit)."""
    n = sk.numel()
    mask = (1 << modulus_bits) - 1
    a = torch.randint(0, 1 << modulus_bits, (msgs.numel(), n), dtype=torch.int64, device="cuda", generator=gen)
    e = torch.randn(msgs.numel(), device="cuda", dtype=torch.float64, generator=gen)
    e = torch.round(e * float(max(1.0, 2.0 ** (modulus_bits - 15)))).to(torch.int64)
    b = (a * sk.to(torch.int64)).sum(1) + msgs.to(torch.int64) * delta + e
    words = torch.cat([a, b.unsqueeze(1)], 1) & mask
    return torch.where(words >= 1 << 31, words - (1 << 32), words).to(torch.int32).contiguous()


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["kind"]
    state = {"case": case}
    if kind in ("gate", "func"):
        ctx, sk = _gate_context()
        batch = case["batch"]
        state["ctx"] = ctx
        state["out"] = torch.empty((batch, ctx.p.n + 1), dtype=torch.int32, device="cuda")
        if kind == "gate":
            bits = torch.randint(0, 2, (2, batch), device="cuda", generator=gen)
            state["gate"] = GATES[case["gate"]]
            state["ct1"] = _encrypt(bits[0], 1 << 30, sk, gen)
            state["ct2"] = _encrypt(bits[1], 1 << 30, sk, gen)
        else:
            q, p = tfhe_amd.FUNC_Q, case["msgs"]
            msgs = torch.randint(0, p, (batch,), device="cuda", generator=gen)
            values = np.random.default_rng(seed).integers(0, p, p)
            state["q"] = q
            state["lut"] = np.repeat(values * (q // p), q // p).astype(np.uint32)
            # messages in the middle of their slices of Z_q
            state["ct"] = _encrypt(msgs * (q // p) + q // (2 * p), 1, sk, gen, modulus_bits=10)
        return state
    if kind == "cbs_lut":
        ctx, sk = _cbs_context(case["form"])
        nbytes, out_bits, p = case["nbytes"], case["out_bits"], ctx.p
        bits = torch.randint(0, 2, (8 * nbytes,), device="cuda", generator=gen)
        state["ctx"] = ctx
        state["ct"] = _encrypt(bits, 1 << 31, sk, gen)
        table = torch.randint(0, 2, (p.N,), device="cuda", generator=gen)  # bit j of T[x] at 8 x + j
        state["table"] = torch.where(table > 0, -(1 << 31), 0).to(torch.int32)
        state["rgsw"] = torch.empty((8 * nbytes, 4, 2, p.N), dtype=torch.int32, device="cuda")
        state["rgsw_f"] = torch.empty((8 * nbytes, 8, 1024, 2), dtype=torch.float64, device="cuda")
        state["bits"] = torch.empty((out_bits * nbytes, p.N + 1), dtype=torch.int32, device="cuda")
        state["out"] = torch.empty((out_bits * nbytes, p.n + 1), dtype=torch.int32, device="cuda")
        return state
    ctx, _ = _cbs_context(case["form"], ttable=kind == "aes_dec")
    rng = np.random.default_rng(seed)
    blocks = case["blocks"]
    state["ctx"] = ctx
    state["cipher"] = [rng.bytes(16) for _ in range(blocks)]
    nonce = rng.bytes(12)
    state["ctr"] = [nonce + int(k).to_bytes(4, "big") for k in range(blocks)]
    state["out"] = torch.empty((blocks, 128, ctx.p.n + 1), dtype=torch.int32, device="cuda")
    return state


def run(state):
    kind, ctx, out = state["case"]["kind"], state["ctx"], state["out"]
    if kind == "gate":
        ctx.eval_batch(state["gate"], state["ct1"], state["ct2"], out)
        return out
    if kind == "func":
        ctx.eval_func(state["ct"], state["q"], state["lut"], out)
        return out
    if kind == "cbs_lut":
        nbytes, out_bits = state["case"]["nbytes"], state["case"]["out_bits"]
        ctx.cbs_batch(state["ct"], state["rgsw"])
        ctx.rgsw_to_fourier(state["rgsw"], 8 * nbytes, state["rgsw_f"])
        ctx.lut8(state["rgsw_f"], nbytes, state["table"], 0, out_bits, state["bits"])
        ctx.keyswitch_batch(state["bits"], out_bits * nbytes, out)
        return {"rgsw": state["rgsw"], "lut": state["bits"], "out": out}
    if kind == "aes_dec":
        ctx.aes_decrypt(state["cipher"], out)
        return out
    ctx.aes_ctr_transcipher(state["ctr"], state["cipher"], out, mode=state["case"]["mode"])
    return out


# ------------------------------------------------------------------ what a pass cannot do without
def _fft(points):
    return 5 * points * math.log2(points)


# one external product: forward transforms, products (8 per complex multiply-add), inverses
_GATE_PBS = 636 * (8 * _fft(512) + 8 * 4 * 3 * 512)
_PBS = {"exact": 636 * (12 * _fft(1024) + 8 * 2 * 2 * 8 * 1024),  # two limbs per torus-64 word
        "fast": 318 * (10 * _fft(1024) + 3 * 8 * 2 * 8 * 1024),   # two key bits per step
        "htss": 636 * (12 * _fft(1024) + 8 * 2 * 2 * 8 * 1024)}
_LUT = 8 * (6 * _fft(1024) + 8 * 2 * 4 * 1024)
_HTSS = 2 * 12 * (9 * _fft(1024) + 5 * 2 * 2 * 8 * 1024)
# keys read once: BSK as the words its generator writes, conversion key, key-switching key
_BSK = {"exact": 636 * 8 * 2 * 2048 * 8, "fast": 318 * 3 * 8 * 2 * 2048 * 8, "htss": 636 * 8 * 2 * 2048 * 8}
_CONV = {"exact": 2 * 2049 * 8 * 15 * 4096 * 4, "fast": 2 * 2049 * 8 * 4096 * 5, "htss": 12 * 5 * 2 * 2048 * 8}
_KSK = {"exact": 2048 * 8 * 4 * 637 * 4, "fast": 2048 * 8 * 637 * 4, "htss": 2048 * 8 * 4 * 637 * 4}


def work(case):
    """Bytes: the keys, inputs and outputs once.  Operations: FFT and product FLOPs of the
    bootstraps plus the key switches' additions or (linear keys) 8-bit products."""
    kind = case["kind"]
    row = 637 * 4
    if kind in ("gate", "func"):
        boots = case["batch"] * (1 if kind == "gate" else 2)
        keys = 636 * 6 * 2 * 1024 * 4 + 1024 * 8 * 4 * 637 * 4
        rows = case["batch"] * (3 if kind == "gate" else 2)
        return {"bytes": keys + rows * row, "flops": boots * (_GATE_PBS + 1024 * 8 * 637)}
    form = case["form"]
    conv = {"exact": 4 * 16392 * 4096, "fast": 4 * 16392 * 4096 * 5 * 2, "htss": _HTSS}[form]
    ks = 16384 * 637 * (8 if form == "fast" else 1)
    keys = _BSK[form] + _CONV[form] + _KSK[form]
    if kind == "cbs_lut":
        bits, outs = 8 * case["nbytes"], case["out_bits"] * case["nbytes"]
        return {"bytes": keys + bits * (row + 4 * 2 * 2048 * 4) + outs * (row + 2049 * 4) + 2048 * 4,
                "flops": bits * (_PBS[form] + conv) + outs * ks + case["nbytes"] * _LUT}
    bits = 1280 * case["blocks"]
    luts = 16 * case["blocks"] * (10 if kind == "aes_ctr" else 37)  # T-table rounds: four tables per byte
    return {"bytes": keys + 11 * 128 * row + case["blocks"] * (32 + 128 * row),
            "flops": bits * (_PBS[form] + conv + ks) + luts * _LUT}


def exact(case, seed):
    """Every output is a torus word (an integer), compared as it is."""
    return None
