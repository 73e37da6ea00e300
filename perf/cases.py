"""The calls that a user of the library makes, over the range in which they are made, as cases that can be timed and compared.

  listed()             named cases: the smallest, the ordinary and the largest calls of every path
  draw(rng)            one more case of the same ranges
  prepare(case, seed)  what a program holds before the call: contexts, keys, weights, inputs - all functions of the seed
  run(state)           one pass through the package's public entry points; its outputs
  work(case)           the bytes and operations that no implementation can do without
  tolerance(case)      every output is an exact integer or the nearest double of one

Kinds of case (field "kind"):
  ntt      Context_23.FromNTTInplace of one batch of limbs and ToNTTInplace of another
  hybrid   the textbook hybrid key switch (one polynomial)
  mult     Scheme_23.mult_23 of two ciphertexts and the rescale that follows every product
  rotate   Scheme_23.leftRotate_23 of one ciphertext
  level    EncodingMatrix.EvalLevel: one baby-step / giant-step level of the slot <-> coefficient transforms, with its rescale
  ppmm     PCMM_Scheme.PPMM: plaintext matrix times MLWE samples, the weights read in every call
  layer    one linear layer on ciphertexts: decomposition into samples, PPMM, packing of the product rows
  client   encode, encrypt, decrypt, decode of one vector of coefficients
"""
import numpy as np
import torch

from ckks_llm_amd import (Ciphertext, Context_23, DeviceBuffer, EncodingMatrix, MLWESecretKey, PCMM_Context, PCMM_Scheme, Plaintext,
                          PlaintextT, Scheme_23, SecretKey)
from ckks_llm_amd.params import CFG1_Q, CFG2_Q, CFG3_P, REF_PARAMS

N1 = 128                                   # coefficients of an MLWE sample: the 128 tokens of a layer
LAYER_PART = 512                           # samples per ciphertext at N = 2^16


def listed():
    return [
        # ---- transforms: what every other path is made of, and a call of its own for a user who moves between the domains ----
        # a small ring with a short chain, sixteen ciphertexts: launch-bound
        dict(name="ntt_n4096_4x32", kind="ntt", logN=12, bits=36, mods=4, polys=32),
        # one ciphertext at the top level of the 24-prime chain
        dict(name="ntt_n65536_one_ciphertext", kind="ntt", logN=16, bits=36, mods=24, polys=2),
        # a batch of 32 ciphertexts of that chain (the benchmark's shape)
        dict(name="ntt_n65536_32_ciphertexts", kind="ntt", logN=16, bits=36, mods=24, polys=64),
        # the 12 primes of 49 bits of the logN = 15 parameter set, an odd number of polynomials
        dict(name="ntt_n32768_49bit_12x9", kind="ntt", logN=15, bits=49, mods=12, polys=9),
        # ---- key switching ----
        # 24 + 6 primes, four digits (the benchmark's shape)
        dict(name="hybrid_n65536_24q_6p", kind="hybrid", logN=16, q=24, p=6, level=23),
        # product of two ciphertexts at the top of the logN = 16 set: the largest key, 60-bit auxiliary primes
        dict(name="mult_n65536_level27", kind="mult", logN=16, level=27),
        # the same on the smallest parameter set: a chain of short launches
        dict(name="mult_n8192_level4", kind="mult", logN=13, level=4),
        # a rotation half way down the logN = 15 chain: a digit that the level cuts
        dict(name="rotate_n32768_level6", kind="rotate", logN=15, level=6, rot=37),
        # a level of the slot <-> coefficient transforms: eight hoisted rotations, four baby steps, 31 diagonals
        dict(name="level_n32768_g8_b4", kind="level", logN=15, level=11, g=8, b=4),
        # ---- plaintext matrix x ciphertext ----
        # the projection of a 768-wide layer over 12 primes (the benchmark's shape)
        dict(name="ppmm_768x768_12_primes", kind="ppmm", logN=16, bits=36, M=768, K=768, mods=12),
        # a whole 768 -> 768 layer on the logN = 16 parameter set with its own 49-bit ring-pack primes and 46-bit plaintext entries
        dict(name="layer_768x768_49bit", kind="layer", bits=49, M=768, K=768),
        # ---- the client's side ----
        dict(name="client_n16384_level9", kind="client", logN=14, level=9),
    ]


def _log(rng, lo, hi):
    """An integer of lo .. hi, even over its logarithm."""
    return min(hi, max(lo, int(round(2.0 ** rng.uniform(np.log2(lo), np.log2(hi))))))


def draw(rng):
    known = [{k: v for k, v in c.items() if k != "name"} for c in listed()]
    while True:
        case = _draw(rng)
        if case not in known:
            return case


def _draw(rng):
    kind = rng.choice(["ntt", "ntt", "ntt", "ntt", "hybrid", "mult", "mult", "rotate", "level", "ppmm", "layer", "client"])
    if kind == "ntt":
        logN, bits = rng.randint(12, 16), rng.choice([36, 36, 49, 60])
        mods = rng.randint(1, {36: 24, 49: 28, 60: 8}[bits])
        return dict(kind=kind, logN=logN, bits=bits, mods=mods, polys=_log(rng, 1, 64))
    if kind == "hybrid":
        logN, p = rng.randint(12, 16), rng.randint(2, 6)
        q = rng.randint(max(4, p), 4 * p)
        return dict(kind=kind, logN=logN, q=q, p=p, level=rng.randint(1, q - 1))
    logN = rng.randint(13, 16)
    L = len(REF_PARAMS[logN]["q"]) - 1
    if kind == "mult":
        return dict(kind=kind, logN=logN, level=rng.randint(1, L))
    if kind == "rotate":
        return dict(kind=kind, logN=logN, level=rng.randint(1, L), rot=rng.randint(1, (1 << (logN - 1)) - 1))
    if kind == "level":
        return dict(kind=kind, logN=logN, level=rng.randint(1, L), g=rng.choice([5, 8, 16]), b=rng.randint(2, 4))
    if kind == "ppmm":
        return dict(kind=kind, logN=rng.randint(13, 16), bits=36, M=_log(rng, 1, 768), K=_log(rng, 8, 768), mods=rng.randint(2, 12))
    if kind == "layer":
        return dict(kind=kind, bits=rng.choice([36, 49]), M=64 * _log(rng, 1, 24), K=64 * _log(rng, 1, 24))
    return dict(kind=kind, logN=logN, level=rng.randint(1, L))


# ---------------------------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------------------------

class _OnDevice:
    """The memory of a DeviceBuffer as the array that torch can look at."""

    def __init__(self, buf, shape, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (buf.ptr, False), "version": 2}


def _view(buf, *shape, typestr="<i8"):
    return torch.as_tensor(_OnDevice(buf, shape, typestr), device="cuda")


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _key(seed):
    """32 bytes of key material of the seed, for the streams that the library expands on the device."""
    return np.random.default_rng(int(seed)).bytes(32)


def _uniform(gen, out, primes):
    """Residues as a ciphertext, a key or a transformed plaintext holds them: out[..., j, :] uniform in [0, primes[j])."""
    for j, q in enumerate(primes):
        out[..., j, :] = torch.randint(0, q, out[..., j, :].shape, generator=gen, dtype=torch.int64, device="cuda")
    return out


def _buffer(words):
    return DeviceBuffer(8 * int(words))


def _uniform_buffer(gen, primes, *polys_and_n):
    """A DeviceBuffer of uniform residues [polys ...][primes][n]."""
    shape = (*polys_and_n[:-1], len(primes), polys_and_n[-1])
    buf = _buffer(np.prod(shape))
    _uniform(gen, _view(buf, *shape), primes)
    return buf


def _random_ciphertext(gen, ctx, level):
    ct = Ciphertext(ctx.N, ctx.L, level, ctx.slots, float(1 << 40))
    _uniform(gen, _view(ct.cipher_device, 2, ctx.L + 1, ctx.N), ctx.qVec)
    return ct


def _limbs(ct, ctx, level):
    """The limbs 0 .. level of both polynomials of a ciphertext: all that a ciphertext at that level holds."""
    return _view(ct.cipher_device, 2, ctx.L + 1, ctx.N)[:, : level + 1]


def _set(logN):
    return Context_23(logN, logN - 1, 192)


def _parts(total, most):
    """total as a sum of powers of two of at most `most`, the largest first: the samples that each ciphertext of a layer carries."""
    got, n = [], most
    while total:
        while n > total:
            n //= 2
        got.append(n)
        total -= n
    return got


def _ntt_primes(case):
    if case["logN"] == 12 and case["bits"] == 36 and case["mods"] <= len(CFG1_Q):
        return CFG1_Q[: case["mods"]]
    return {36: CFG2_Q, 49: REF_PARAMS[16]["q"], 60: REF_PARAMS[16]["t"]}[case["bits"]][: case["mods"]]


def _prepare_ntt(case, seed):
    primes, N = _ntt_primes(case), 1 << case["logN"]
    gen = _generator(seed)
    shape = (case["polys"], len(primes), N)
    s = dict(ctx=Context_23(case["logN"], [], primes))
    for name in ("evaluations", "coefficients"):
        s[name] = _uniform(gen, torch.empty(shape, dtype=torch.int64, device="cuda"), primes)
    return s


def _prepare_hybrid(case, seed):
    q, p = CFG2_Q[: case["q"]], CFG3_P[: case["p"]]
    ctx = Context_23(case["logN"], p, q)
    gen, N = _generator(seed), ctx.N
    digits = -(-len(q) // len(p))
    return dict(ctx=ctx, inp=_uniform_buffer(gen, q, N), evk=_uniform_buffer(gen, p + q, 2, digits, N), out=_buffer(2 * len(q) * N),
                scratch=_buffer((digits + 2) * (len(p) + len(q)) * N))


def _prepare_mult(case, seed):
    ctx = _set(case["logN"])
    scheme, sk = Scheme_23(ctx, key=_key(seed)), SecretKey(ctx, key=_key(seed + 1), nonce=1)
    scheme.addMultKey_23(sk)
    gen = _generator(seed)
    return dict(ctx=ctx, scheme=scheme, x=_random_ciphertext(gen, ctx, case["level"]), y=_random_ciphertext(gen, ctx, case["level"]),
                res=Ciphertext(ctx.N, ctx.L, case["level"], ctx.slots, 1.0))


def _prepare_rotate(case, seed):
    ctx = _set(case["logN"])
    scheme, sk = Scheme_23(ctx, key=_key(seed)), SecretKey(ctx, key=_key(seed + 1), nonce=1)
    scheme.addLeftRotKey_23(sk, case["rot"])
    return dict(ctx=ctx, scheme=scheme, x=_random_ciphertext(_generator(seed), ctx, case["level"]),
                res=Ciphertext(ctx.N, ctx.L, case["level"], ctx.slots, 1.0))


def _prepare_level(case, seed):
    ctx, g, b = _set(case["logN"]), case["g"], case["b"]
    scheme, sk = Scheme_23(ctx, key=_key(seed)), SecretKey(ctx, key=_key(seed + 1), nonce=1)
    rot_in, rot_out = list(range(g)), [g * i for i in range(b)]
    for r in sorted(set(rot_in + rot_out) - {0}):
        scheme.addLeftRotKey_23(sk, r)
    gen = _generator(seed)
    diagonals = []
    for _ in range(b * g):
        pt = PlaintextT(ctx.N, ctx.t_num, float(1 << 40))
        _uniform(gen, _view(pt.mx_device, ctx.t_num, ctx.N), ctx.tVec)
        diagonals.append(pt)
    return dict(ctx=ctx, matrix=EncodingMatrix(scheme), diagonals=diagonals, rot_in=rot_in, rot_out=rot_out,
                ct=_random_ciphertext(gen, ctx, case["level"]))


def _weights(seed, M, K):
    return DeviceBuffer.from_numpy(np.random.default_rng(int(seed)).normal(0, 0.02, (M, K)).astype(np.float32))


def _prepare_ppmm(case, seed):
    primes = CFG2_Q[: case["mods"]]
    ctx = Context_23(case["logN"], [], primes)
    rank = ctx.N // N1
    words = (rank + 1) * N1
    samples = _uniform(_generator(seed), torch.empty((case["K"], len(primes), words), dtype=torch.int64, device="cuda"), primes)
    return dict(ctx=ctx, scheme=PCMM_Scheme(PCMM_Context(N1, rank, [], primes, ctx)), W=_weights(seed, case["M"], case["K"]),
                samples=list(samples), out=torch.zeros((case["M"], len(primes), words), dtype=torch.int64, device="cuda"))


def _prepare_layer(case, seed):
    if case["bits"] == 36:
        # one special prime and two moduli below 2^39, activations at 2^33, plaintext entries of 26 bits of fraction
        ctx, in_scale, scaler = Context_23(16, CFG3_P[:1], CFG2_Q[:2]), float(1 << 33), float(1 << 26)
        ctx.h_weight = 192
    else:
        # the parameter set's own precision of 2^49 on both sides: the scaler is then q1
        ctx = _set(16)
        in_scale, scaler = float(ctx.precision), float(ctx.qVec[1])
    rank = ctx.N // N1
    p_pack, q_pack = ctx.pVec[-1:], ctx.qVec[:2]
    pc = PCMM_Context(N1, rank, p_pack, q_pack, ctx)
    ps, sk = PCMM_Scheme(pc, key=_key(seed)), SecretKey(ctx, key=_key(seed + 1), nonce=1)
    mlwe_sk = MLWESecretKey(N1, pc.ringpack_pq_count - 1, rank)
    ps.convertMLWESKfromRLWESK(mlwe_sk, sk)
    ps.addRepakcingKey(mlwe_sk, sk)
    gen, words = _generator(seed), (rank + 1) * N1
    M, K = case["M"], case["K"]
    s = dict(ctx=ctx, ps=ps, M=M, K=K, scaler=scaler, parts_in=_parts(K, LAYER_PART), parts_out=_parts(M, LAYER_PART), W=_weights(seed, M, K),
             product=_buffer(M * 2 * words), embed=_buffer((rank + 1) * 2 * ctx.N), mult=_buffer(4 * ctx.N))
    s["x"] = [_random_ciphertext(gen, ctx, 1) for _ in s["parts_in"]]
    s["y"] = [Ciphertext(ctx.N, ctx.L, 0, ctx.slots, 1.0) for _ in s["parts_out"]]
    s["rows"] = [s["product"].ptr + 8 * m * 2 * words for m in range(M)]
    if case["bits"] == 36:
        pc.weights_static(s["W"])                      # a layer's own weights, as the Bert class declares them
    else:
        s["samples"] = [_buffer(2 * words) for _ in range(K)]
    return s


def _prepare_client(case, seed):
    ctx = _set(case["logN"])
    scheme, sk = Scheme_23(ctx, key=_key(seed)), SecretKey(ctx, key=_key(seed + 1), nonce=1)
    scheme.addEncKey(sk)
    level = case["level"]
    values = torch.empty(ctx.N, dtype=torch.float64, device="cuda").normal_(0.0, 1.0, generator=_generator(seed))
    return dict(ctx=ctx, scheme=scheme, sk=sk, values=values, msg=Plaintext(ctx.N, ctx.L, level, ctx.slots, ctx.precision >> 8),
                ct=Ciphertext(ctx.N, ctx.L, level, ctx.slots, 1.0), dec=Plaintext(ctx.N, ctx.L, level, ctx.slots, 1.0),
                got=torch.zeros(ctx.N, dtype=torch.float64, device="cuda"))


_PREPARE = {"ntt": _prepare_ntt, "hybrid": _prepare_hybrid, "mult": _prepare_mult, "rotate": _prepare_rotate, "level": _prepare_level,
            "ppmm": _prepare_ppmm, "layer": _prepare_layer, "client": _prepare_client}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, seed)
    state["case"] = case
    return state


# ---------------------------------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------------------------------

def _run_ntt(s, case):
    polys, mods = case["polys"], case["mods"]
    s["ctx"].FromNTTInplace(s["evaluations"], 0, 0, polys, mods, mods)
    s["ctx"].ToNTTInplace(s["coefficients"], 0, 0, polys, mods, mods)
    return s["evaluations"], s["coefficients"]


def _run_hybrid(s, case):
    s["ctx"].hybrid_keyswitch(s["out"], s["inp"], s["evk"], case["level"], s["scratch"])
    return _view(s["out"], 2, case["q"], s["ctx"].N)[:, : case["level"] + 1]


def _run_mult(s, case):
    s["scheme"].mult_23(s["res"], s["x"], s["y"])
    s["scheme"].rescaleAndEqual(s["res"])
    return _limbs(s["res"], s["ctx"], case["level"] - 1)


def _run_rotate(s, case):
    s["scheme"].leftRotate_23(s["res"], s["x"], case["rot"])
    return _limbs(s["res"], s["ctx"], case["level"])


def _run_level(s, case):
    ct = s["ct"]
    ct.l, ct.scale = case["level"], float(1 << 40)     # the pass before took a level
    s["matrix"].EvalLevel(s["diagonals"], ct, s["rot_in"], s["rot_out"], case["b"], case["g"], case["b"] * case["g"] - 1)
    return _limbs(ct, s["ctx"], case["level"] - 1)


def _run_ppmm(s, case):
    s["scheme"].PPMM(s["W"], s["samples"], s["out"], case["M"], case["K"], N1, case["K"], case["mods"], float(1 << 26))
    return s["out"]


def _run_layer(s, case):
    ps, ctx, M, K = s["ps"], s["ctx"], s["M"], s["K"]
    if case["bits"] == 36:
        ps.packed_begin(K, 2)
        at = 0
        for ct, n in zip(s["x"], s["parts_in"]):
            ps.rlweCipherDecompose_packed(ct.cipher_device, n, at, 1)
            at += n
        ps.PPMM_packed(s["W"], s["product"], M, s["scaler"])
    else:
        at = 0
        for ct, n in zip(s["x"], s["parts_in"]):
            ps.rlweCipherDecompose(ct.cipher_device, s["samples"], n, at, 1)
            at += n
        ps.PPMM(s["W"], s["samples"], s["product"], M, K, N1, K, 2, s["scaler"])
    at = 0
    for ct, n in zip(s["y"], s["parts_out"]):
        ps.mlweCipherPacking(ct.cipher_device, s["rows"], n, at, ps.repackingKeys, s["embed"], s["mult"])
        ct.l = 0
        at += n
    return [_limbs(ct, ctx, 0) for ct in s["y"]]


def _run_client(s, case):
    ctx, scheme = s["ctx"], s["scheme"]
    ctx.encode_coeffs(s["values"], s["msg"])
    scheme.encryptMsg(s["ct"], s["msg"])
    scheme.decryptMsg(s["dec"], s["sk"], s["ct"])
    ctx.decode_coeffs(s["dec"], s["got"])
    level = case["level"]
    return {"ciphertext": _limbs(s["ct"], ctx, level), "plaintext": _view(s["dec"].mx_device, ctx.L + 1, ctx.N)[: level + 1], "values": s["got"]}


_RUN = {"ntt": _run_ntt, "hybrid": _run_hybrid, "mult": _run_mult, "rotate": _run_rotate, "level": _run_level, "ppmm": _run_ppmm,
        "layer": _run_layer, "client": _run_client}


def run(state):
    case = state["case"]
    return _RUN[case["kind"]](state, case)


# ---------------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without: every input and key once, every output once; a modular butterfly is one product, one sum and
# one difference, a modular multiply-add two operations
# ---------------------------------------------------------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "ppmm":
        words = (1 << case["logN"]) + N1
        M, K, mods = case["M"], case["K"], case["mods"]
        return {"bytes": 8 * words * mods * (M + K) + 4 * M * K, "flops": 2 * M * K * words * mods}
    if kind == "layer":
        N, M, K = 1 << 16, case["M"], case["K"]
        rank, outs = N // N1, len(_parts(M, LAYER_PART))
        limbs = 4 * len(_parts(K, LAYER_PART)) + 4 * rank + 2 * outs                   # ciphertexts in, repacking keys, ciphertexts out
        mults = M * K * (N + N1) * 2 + outs * rank * 4 * N
        return {"bytes": 8 * N * limbs + 4 * M * K, "flops": 2 * mults + 3 * (N // 2) * 16 * 2 * rank * outs}
    logN = case["logN"]
    N = 1 << logN
    butterflies = 3 * (N // 2) * logN                                                  # of one limb
    if kind == "ntt":
        limbs = 2 * case["polys"] * case["mods"]
        return {"bytes": 16 * N * limbs, "flops": butterflies * limbs}
    l1 = case["level"] + 1
    if kind == "client":
        # values in, public key, secret, ciphertext out, plaintext out, values out
        return {"bytes": 16 * N + 8 * N * (2 * l1 + l1 + 2 * l1 + l1), "flops": butterflies * 5 * l1 + 2 * N * (5 * l1 + l1 * l1)}
    if kind == "hybrid":
        K, all_primes = case["p"], case["p"] + l1
        digits = -(-l1 // K)
        transforms = l1 + digits * all_primes - l1 + 2 * all_primes + 2 * l1
        products = l1 * (all_primes - min(K, l1)) + 2 * digits * all_primes + 2 * K * l1
        return {"bytes": 8 * N * (l1 + 2 * digits * all_primes + 2 * l1), "flops": butterflies * transforms + 2 * N * products}
    r = REF_PARAMS[logN]
    K, T, gamma = len(r["p"]), len(r["t"]), r["gamma"]
    digits, blocks = -(-l1 // K), -(-(K + l1) // gamma)
    key = 2 * digits * blocks * T
    transforms = l1 + digits * T + 2 * blocks * T + 2 * l1
    products = l1 * T + key + 2 * (K + l1) * T + 2 * K * l1
    if kind == "mult":
        # two ciphertexts in, one a level lower out; the tensor product before the switch and the transforms of the rescale behind it
        return {"bytes": 8 * N * (4 * l1 + key + 2 * (l1 - 1)), "flops": butterflies * (transforms + 2 + 2 * (l1 - 1)) + 2 * N * (products + 4 * l1)}
    if kind == "rotate":
        return {"bytes": 8 * N * (4 * l1 + key), "flops": butterflies * transforms + 2 * N * products}
    g, b = case["g"], case["b"]
    limbs = 2 * l1 + (g - 1 + b - 1) * key + (b * g - 1) * T + 2 * (l1 - 1)
    products = (g - 1 + b - 1) * key + (b * g - 1) * 2 * blocks * T + b * (l1 * T + 2 * (K + l1) * T + 2 * K * l1)
    transforms = b * (digits * T + 2 * blocks * T)
    return {"bytes": 8 * N * limbs, "flops": butterflies * transforms + 2 * N * products}


def tolerance(case):
    # residues are canonical representatives and decoded values the nearest doubles of exact quotients: one right answer
    return "exact"
