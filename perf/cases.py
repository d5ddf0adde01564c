"""Performance cases of the CKKS engine: the calls a user of the package makes.

Every case is one call (or the short sequence a program writes at that place)
through the public entry points of nexus_amd, at the rings and modulus chains
the package is used with: the 2^13 matrix-product chains, the 2^15
bootstrapping chain, the 2^16 chain of the evaluator programs (one special
prime) and the 2^16 chain of the encrypted BERT-base layer (eight special
primes).  Contexts, keys, bootstrappers, weights and masks are what a program
keeps; ciphertexts and message vectors are new for every seed.

Outputs are ciphertext residues: whole numbers, defined word for word by the
arithmetic, so every comparison is exact.
"""
import math

import numpy as np
import torch

import nexus_amd as nx
from nexus_amd import mm

# name: (log2 N, data and special primes' bits, special primes, Hamming weight, scale)
CHAINS = {
    "matmul": (13, [60, 40, 60], 1, 0, 2.0 ** 40),
    "matmul4": (13, [60, 40, 40, 60], 1, 0, 2.0 ** 40),
    "server": (14, [58] + [40] * 8 + [58], 1, 0, 2.0 ** 40),
    "boot": (15, [51] + [46] * 16 + [51] * 14 + [51], 1, 192, 2.0 ** 46),
    "eval": (16, [58] + [40] * 18 + [58], 1, 0, 2.0 ** 40),
    "bert": (16, [51] + [46] * 19 + [51] * 14 + [51] * 8, 8, 192, 2.0 ** 46),
}
EVAL_STEPS = [-1024] + [-(1 << i) for i in range(4, 9)] + [1 << i for i in range(10)]  # softmax and LayerNorm
TOKEN = 256  # slots of one token in a token-group ciphertext
MIX_PERIOD = 64  # features of one attention head


def listed():
    return [
        # one multiplication of two ciphertexts on the smallest ring in use:
        # latency and launches count
        {"name": "product_n8192", "work": "product", "chain": "matmul4", "limbs": 3},
        # a fresh message vector times a ciphertext at the evaluators' top level
        {"name": "plain_n65536", "work": "plain", "chain": "eval", "limbs": 19, "count": 32768},
        # matrix product of a plaintext matrix with one packed ciphertext: its
        # expansion into 8192 ciphertexts and ten output columns of 768 terms
        {"name": "matmul_n8192", "work": "matmul", "chain": "matmul", "inner": 768, "cols": 10},
        # GELU of one ciphertext of 32768 activations, one call per operation
        {"name": "gelu_n65536", "work": "gelu", "chain": "eval", "count": 1},
        # one sparse bootstrap (2^13 slots) with one special prime
        {"name": "bootstrap_n32768", "work": "bootstrap", "chain": "boot", "log_slots": 13, "count": 1},
        # a linear layer's outputs refreshed together: dense bootstraps in lockstep
        {"name": "bootstrap_many_n65536", "work": "bootstrap", "chain": "bert", "log_slots": 15, "count": 4},
        # the attention's query-key products of one ciphertext, relinearised and rescaled
        {"name": "products_n65536", "work": "products", "chain": "bert", "limbs": 20, "count": 64, "fused": True},
        # the token rotations of the three key ciphertexts, hoisted
        {"name": "rotations_n65536", "work": "rotations", "chain": "bert", "limbs": 20, "inputs": 3, "steps": 15},
        # rotation sums of the attention's compaction: sixteen inputs a sum
        {"name": "rotation_sums_n65536", "work": "rotation_sums", "chain": "bert", "limbs": 19, "groups": 6,
         "size": 16},
        # the attention's expansion: 127 rotated probability ciphertexts to the
        # 64 features of each head, through one-hot periodic masks
        {"name": "mask_mix_n65536", "work": "mask_mix", "chain": "bert", "limbs": 20, "inputs": 127, "outputs": 64},
        # the multiply-accumulates of one CoeffToSlot level and their rescales
        {"name": "linear_n65536", "work": "linear", "chain": "bert", "limbs": 34, "babies": 16, "giants": 8},
        # the whole encrypted BERT-base layer over one set of 128 tokens
        {"name": "bert_layer_n65536", "work": "bert", "chain": "bert", "tokens": 128},
    ]


def _spread(rng, lo, hi):
    """a whole number in [lo, hi], spread over its logarithm"""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    work = rng.choice(["product", "product", "plain", "matmul", "gelu", "softmax", "layer_norm", "bootstrap",
                       "products", "products", "rotations", "rotations", "rotation_sums", "rotation_sums",
                       "mask_mix", "linear"])
    if work == "product":
        chain = rng.choice(["matmul4", "server", "boot", "eval", "bert"])
        return {"work": work, "chain": chain, "limbs": rng.randint(2, _data_primes(chain))}
    if work == "plain":
        chain = rng.choice(["matmul4", "server", "boot", "eval", "bert"])
        return {"work": work, "chain": chain, "limbs": rng.randint(2, _data_primes(chain)),
                "count": _spread(rng, 1, 1 << (CHAINS[chain][0] - 1))}
    if work == "matmul":
        inner = _spread(rng, 64, 1024)
        return {"work": work, "chain": "matmul", "inner": inner, "cols": rng.randint(1, 8192 // inner)}
    if work == "gelu":
        return {"work": work, "chain": "eval", "count": rng.randint(2, 6)}
    if work == "softmax":
        return {"work": work, "chain": "eval", "length": 1 << rng.randint(4, 8), "rows": rng.randint(1, 64)}
    if work == "layer_norm":
        return {"work": work, "chain": "eval", "rows": rng.randint(1, 16)}
    if work == "bootstrap":
        if rng.random() < 0.5:
            return {"work": work, "chain": "boot", "log_slots": rng.randint(11, 14), "count": rng.randint(1, 3)}
        return {"work": work, "chain": "bert", "log_slots": rng.choice([12, 15]), "count": rng.randint(1, 7)}
    if work == "products":
        return {"work": work, "chain": "bert", "limbs": rng.randint(2, 34), "count": _spread(rng, 1, 48),
                "fused": rng.random() < 0.5}
    if work == "rotations":
        inputs = _spread(rng, 1, 6)
        return {"work": work, "chain": "bert", "limbs": rng.randint(1, 34), "inputs": inputs,
                "steps": _spread(rng, 1, min(16, 60 // inputs))}
    if work == "rotation_sums":
        return {"work": work, "chain": "bert", "limbs": rng.randint(1, 26), "groups": _spread(rng, 1, 8),
                "size": _spread(rng, 1, 16)}
    if work == "mask_mix":
        return {"work": work, "chain": "bert", "limbs": rng.randint(1, 24), "inputs": rng.randint(16, 127),
                "outputs": rng.randint(1, 64)}
    return {"work": work, "chain": "bert", "limbs": rng.randint(2, 34), "babies": _spread(rng, 2, 32),
            "giants": _spread(rng, 1, 8)}


# ---------------------------------------------------------------- what a program keeps
class _Session:
    """One context with its keys and the objects a program builds on them once."""

    def __init__(self, chain):
        logn, bits, special, h, self.scale = CHAINS[chain]
        self.ctx = nx.Context(logn, bits, hamming_weight=h, special_primes=special)
        self.sk = nx.SecretKey(self.ctx, seed=1)
        self.rk = nx.KSwitchKeys(self.ctx).generate_relin(self.sk, seed=2)
        self.gk = nx.KSwitchKeys(self.ctx)
        self.elements = set()
        self.made = {}

    def need(self, elements):
        new = sorted(set(elements) - self.elements)
        if new:
            self.gk.generate_galois(self.sk, new, seed=3 + len(self.elements))
            self.elements.update(new)

    def need_steps(self, steps):
        self.need([self.ctx.elt_from_step(s) for s in steps if s])

    def keep(self, key, make):
        if key not in self.made:
            self.made[key] = make()
        return self.made[key]

    def evaluator(self):
        return self.keep("evaluator", lambda: nx.CKKSEvaluator(self.ctx, self.rk, self.gk, self.scale, self.sk))

    def encrypt(self, values, limbs, seed, scale=None):
        pt = nx.encode(self.ctx, values, scale or self.scale, self.ctx.L + 1 - limbs)
        return nx.encrypt(self.ctx, self.sk, pt, seed=seed)


_open = {}


def _session(chain):
    """the session of `chain`; only one is open at a time (keys take GPU memory)"""
    if chain not in _open:
        _open.clear()
        _open[chain] = _Session(chain)
    return _open[chain]


def _data_primes(chain):
    return len(CHAINS[chain][1]) - CHAINS[chain][2]


def _rotation_steps(count):
    return [TOKEN * (i + 1) for i in range(count)]


def _mask_index(inputs, outputs):
    """output t takes offset p = t - d of the input rotated by d"""
    index = np.full((outputs, inputs), -1, dtype=np.int32)
    for t in range(outputs):
        for k in range(inputs):
            p = t - (k - (inputs // 2))
            if 0 <= p < MIX_PERIOD:
                index[t, k] = p
    index[:, 0] = np.where((index >= 0).any(axis=1), index[:, 0], 0)  # every output has a term
    return index


def prepare(case, seed):
    s = _session(case["chain"])
    ctx, work = s.ctx, case["work"]
    slots = ctx.slot_count
    rng = np.random.default_rng(seed)
    base = (seed % (1 << 24)) * 4096 + 1  # encryption randomness: other seeds, other ciphertexts
    st = {"case": case, "s": s}

    def fresh(count, limbs, lo=-1.0, hi=1.0):
        # ciphertexts of messages in [lo, hi]; one message, randomised by encryption
        v = rng.uniform(lo, hi, slots)
        return [s.encrypt(np.roll(v, i), limbs, base + i) for i in range(count)]

    if work == "product":
        st["a"], st["b"] = fresh(2, case["limbs"])
    elif work == "plain":
        st["a"] = fresh(1, case["limbs"])[0]
        st["v"] = rng.uniform(-1, 1, case["count"])
    elif work == "matmul":
        s.need(mm.reference_elts(ctx.n, 13))
        x = np.round(rng.uniform(-1, 1, (4096, case["inner"])), 4)
        y = np.round(rng.uniform(-1, 1, ctx.n), 4)
        st["rows"] = [nx.encode(ctx, x[:, i], s.scale) for i in range(case["inner"])]
        st["a"] = mm.compress(ctx, s.sk, y, 1e10, seed=base)
    elif work == "gelu":
        s.evaluator()
        v = np.clip(rng.normal(0, 1, slots), -5, 5)
        st["x"] = [s.encrypt(np.roll(v, i), ctx.L, base + i) for i in range(case["count"])]
    elif work == "softmax":
        s.need_steps(EVAL_STEPS)
        s.evaluator()
        n = case["length"]  # a row of scores, then as many empty slots
        v = np.zeros(slots)
        for r in range(case["rows"]):
            row = rng.normal(0, 3, n)
            v[2 * n * r: 2 * n * r + n] = np.clip(row - row.max(), -10, 0)
        st["x"] = [s.encrypt(v, ctx.L, base)]
    elif work == "layer_norm":
        s.need_steps(EVAL_STEPS)
        s.evaluator()
        v = np.zeros(slots)
        for r in range(case["rows"]):
            v[2048 * r: 2048 * r + 768] = rng.normal(0, 1, 768) * math.sqrt(30.0)
        st["x"] = [s.encrypt(v, ctx.L, base)]
    elif work == "bootstrap":
        logn = CHAINS[case["chain"]][0]
        s.need_steps(nx.boot_plan_steps(logn - 1, case["log_slots"], 25))
        if 0 in nx.boot_plan_steps(logn - 1, case["log_slots"], 25):
            s.need([2 * ctx.n - 1])  # conjugation
        log_slots = case["log_slots"]
        st["bt"] = s.keep(("boot", log_slots), lambda: nx.Bootstrapper(s.evaluator(), log_slots=log_slots))
        st["x"] = []
        for i in range(case["count"]):
            v = rng.uniform(-1, 1, 1 << log_slots)
            st["x"].append(s.encrypt(np.tile(v, slots >> log_slots), 1, base + i))
    elif work == "products":
        c = fresh(2 * case["count"], case["limbs"])
        st["a"], st["b"] = c[: case["count"]], c[case["count"]:]
    elif work == "rotations":
        st["steps"] = _rotation_steps(case["steps"])
        s.need_steps(st["steps"])
        st["x"] = fresh(case["inputs"], case["limbs"])
    elif work == "rotation_sums":
        steps = list(range(case["size"]))  # the first term of a sum is not rotated
        s.need_steps(steps)
        c = fresh(case["groups"] * case["size"], case["limbs"])
        st["x"] = [c[g * case["size"]:(g + 1) * case["size"]] for g in range(case["groups"])]
        st["steps"] = [steps] * case["groups"]
    elif work == "mask_mix":
        limbs = case["limbs"]
        st["w"] = s.keep(("masks", limbs), lambda: nx.PeriodicPlaintexts(ctx, np.eye(MIX_PERIOD), s.scale,
                                                                         ctx.L + 1 - limbs))
        st["index"] = _mask_index(case["inputs"], case["outputs"])
        st["x"] = fresh(case["inputs"], limbs)
    elif work == "linear":
        limbs, K, G = case["limbs"], case["babies"], case["giants"]

        def diagonals():
            w = np.random.default_rng(7).uniform(-1, 1, slots)
            return [[nx.encode(ctx, np.roll(w, g * K + k), s.scale, ctx.L + 1 - limbs) for k in range(K)]
                    for g in range(G)]
        st["w"] = s.keep(("diagonals", limbs, K, G), diagonals)
        st["x"] = fresh(K, limbs)
    elif work == "bert":
        def layer():
            s.need_steps(nx.bert_rotation_steps(slots))
            boot = nx.boot_plan_steps(15, 15, 25)
            s.need_steps(boot)
            s.need([2 * ctx.n - 1])
            bt = nx.Bootstrapper(s.evaluator())
            r = np.random.default_rng(42)
            w = {k: r.normal(0, 0.02, shape) for k, shape in
                 (("wq", (768, 768)), ("wk", (768, 768)), ("wv", (768, 768)), ("wo", (768, 768)),
                  ("w1", (768, 3072)), ("w2", (3072, 768)))}
            return nx.BertLayer(bt, w)
        st["layer"] = s.keep("layer", layer)
        rows = np.zeros((128, 768))
        rows[: case["tokens"]] = rng.normal(0, 1, (case["tokens"], 768))
        st["x"] = [s.encrypt(v, 2, base + i) for i, v in enumerate(nx.bert_pack(rows, slots))]
    else:
        raise ValueError(work)
    ctx.synchronize()
    return st


# ---------------------------------------------------------------- the calls
class _Residues:
    """a ciphertext's residues in device memory, as an array torch can view"""

    def __init__(self, ct):
        self.ct = ct  # the memory lives as long as the view
        i = ct.info()
        self.__cuda_array_interface__ = {"shape": (i["size"], i["limbs"], ct.ctx.n), "typestr": "<i8",
                                         "data": (ct.device_data()[0], False), "version": 2}


def _words(cts):
    return [torch.as_tensor(_Residues(c), device="cuda") for c in cts]


def run(st):
    case, s = st["case"], st["s"]
    ctx, work = s.ctx, case["work"]
    if work == "product":
        return _words([nx.rescale_to_next(nx.relinearize(nx.multiply(st["a"], st["b"]), s.rk))])
    if work == "plain":
        pt = nx.encode(ctx, st["v"], s.scale, st["a"].chain_index)
        return _words([nx.rescale_to_next(nx.multiply_plain(st["a"], pt))])
    if work == "matmul":
        return _words(mm.accumulate(st["rows"], [mm.expand(st["a"], ctx.n, s.gk)], case["cols"]))
    if work == "gelu":
        ev = s.evaluator()
        return _words([ev.gelu(st["x"][0])] if case["count"] == 1 else ev.gelu_many(st["x"]))
    if work == "softmax":
        return _words([s.evaluator().softmax(st["x"][0], case["length"])])
    if work == "layer_norm":
        return _words([s.evaluator().layer_norm(st["x"][0], 1024)])
    if work == "bootstrap":
        return _words([st["bt"].bootstrap(st["x"][0])] if case["count"] == 1 else st["bt"].bootstrap_many(st["x"]))
    if work == "products":
        return _words(nx.multiply_relin_rescale_many(st["a"], st["b"], s.rk, fused=case["fused"]))
    if work == "rotations":
        if case["inputs"] == 1:
            out = [nx.rotate_hoisted(st["x"][0], st["steps"], s.gk)]
        else:
            out = nx.rotate_hoisted_many(st["x"], st["steps"], s.gk)
        return [_words(o) for o in out]
    if work == "rotation_sums":
        return _words(nx.rotate_sum_many(st["x"], st["steps"], s.gk))
    if work == "mask_mix":
        return _words(nx.multiply_periodic_mix(st["x"], st["w"], st["index"]))
    if work == "linear":
        return _words(nx.rescale_to_next_many(nx.multiply_plain_accumulate_multi(st["x"], st["w"])))
    return _words(st["layer"].forward(st["x"], case["tokens"]))


# ---------------------------------------------------------------- what a pass cannot do without
class _Count:
    """bytes of inputs, keys, weights and outputs (each once) and modular
    products and additions"""

    def __init__(self, chain):
        logn, bits, self.alpha, _, _ = CHAINS[chain]
        self.n, self.logn, self.L = 1 << logn, logn, len(bits) - self.alpha
        self.bytes = self.flops = 0.0

    def polys(self, count, limbs):
        self.bytes += 8.0 * self.n * count * limbs
        return self

    def key(self, limbs, count=1):
        # the half of a key that is not derived from its seeds
        self.bytes += 8.0 * self.n * count * self._digits(limbs) * (limbs + self.alpha)
        return self

    def _digits(self, limbs):
        return -(-limbs // self.alpha)

    def transforms(self, limbs):
        self.flops += 3.0 * self.n / 2 * self.logn * limbs
        return self

    def point(self, ops):
        self.flops += float(self.n) * ops
        return self

    def modup(self, limbs, count=1):
        for _ in range(count):
            d, out = self._digits(limbs), limbs + self.alpha
            self.transforms(limbs + d * out - limbs).point(2.0 * self.alpha * (d * out - limbs))
        return self

    def moddown(self, limbs, count=1):
        for _ in range(count):
            self.transforms(2 * (limbs + self.alpha)).point(2.0 * 2 * limbs * (self.alpha + 1))
        return self

    def inner(self, limbs, count=1):
        return self.point(4.0 * count * self._digits(limbs) * (limbs + self.alpha))

    def switch(self, limbs, count=1):
        return self.modup(limbs, count).inner(limbs, count).moddown(limbs, count)

    def rescale(self, limbs, count=1):
        return self.transforms(2.0 * count * limbs).point(4.0 * count * limbs)


# Key switches (relinearisations and rotations) of the programs by the limbs they
# run at, as their operation sequences define them.
GELU = {2: 2, 3: 2, 4: 4, 5: 2, 6: 2, 7: 2, 8: 4, 9: 2, 10: 2, 11: 2, 12: 4, 13: 2, 14: 2, 15: 2, 16: 6, 17: 4,
        18: 3, 19: 1}
SOFTMAX = {4: 1, 6: 1, 7: 2, 8: 2, 9: 2, 10: 1, 12: 1, 13: 1, 14: 1, 15: 1, 16: 1, 17: 1, 18: 1, 19: 1}  # + the sums
LAYER_NORM = {2: 1, 4: 2, 5: 1, 6: 2, 7: 1, 8: 1, 9: 1, 10: 2, 11: 1, 12: 2, 13: 1, 14: 2, 15: 1, 16: 2, 18: 10, 19: 2}
SLOT_MAPS = {"boot": {17: 1, 18: 11, 19: 10, 20: 10, 29: 10, 30: 10, 31: 12},
             "bert": {21: 11, 22: 14, 23: 14, 31: 1, 32: 14, 33: 14, 34: 11}}
EVAL_MOD = {"boot": {21: 1, 22: 1, 23: 3, 24: 4, 25: 2, 26: 4, 27: 2, 28: 1},
            "bert": {24: 1, 25: 1, 26: 3, 27: 4, 28: 2, 29: 4, 30: 2, 31: 1}}
BERT_REST = {2: 1248, 3: 6, 4: 3, 5: 10, 6: 8, 7: 10, 8: 23, 9: 20, 10: 2, 11: 10, 12: 8, 13: 10, 14: 8, 15: 10,
             16: 8, 17: 10, 18: 16, 19: 1162, 20: 1548}
BERT_BOOTSTRAPS = 18


def _switches(c, table, times, keys):
    for limbs, count in table.items():
        c.switch(limbs, count * times).rescale(limbs, count * times).key(limbs, min(count, keys))


def _bootstraps(c, case, count):
    dense = case.get("log_slots", 15) == c.logn - 1
    _switches(c, SLOT_MAPS[case["chain"]], count, 14)
    _switches(c, EVAL_MOD[case["chain"]], count * (2 if dense else 1), 1)


def work(case):
    c, w = _Count(case["chain"]), case["work"]
    l = case.get("limbs", c.L)
    if w == "product":
        c.polys(4, l).polys(2, l - 1).key(l).switch(l).rescale(l).point(6 * l)
    elif w == "plain":
        c.polys(2, l).polys(2, l - 1).rescale(l).transforms(l).point(2 * l)
        c.bytes += 8.0 * case["count"]
    elif w == "matmul":
        c.polys(case["inner"], 2).polys(2, 2).polys(2 * case["cols"], 2).key(2, 13)
        c.switch(2, c.n - 1).point(4.0 * case["inner"] * case["cols"] * 2)
    elif w == "gelu":
        k = case["count"]
        c.polys(2 * k, c.L).polys(2 * k, 1)
        _switches(c, GELU, k, 1)
    elif w == "softmax":
        c.polys(2, c.L).polys(2, 3)
        _switches(c, SOFTMAX, 1, 1)
        _switches(c, {11: int(math.log2(case["length"]))}, 1, 8)
    elif w == "layer_norm":
        c.polys(2, c.L).polys(2, 1)
        _switches(c, LAYER_NORM, 1, 10)
    elif w == "bootstrap":
        c.polys(2 * case["count"], 1).polys(2 * case["count"], c.L - 14)
        _bootstraps(c, case, case["count"])
    elif w == "bert":
        c.polys(2 * 3, 2).polys(2 * 3, 2)
        _bootstraps(c, case, BERT_BOOTSTRAPS)
        _switches(c, BERT_REST, 1, 64)
    elif w == "products":
        k = case["count"]
        c.polys(4 * k, l).polys(2 * k, l - 1).key(l).switch(l, k).rescale(l, k).point(6.0 * l * k)
    elif w == "rotations":
        b, r = case["inputs"], case["steps"]
        c.polys(2 * b, l).polys(2 * b * r, l).key(l, r).modup(l, b).inner(l, b * r).moddown(l, b * r)
    elif w == "rotation_sums":
        g, k = case["groups"], case["size"]
        c.polys(2 * g * k, l).polys(2 * g, l).key(l, k - 1).modup(l, g * (k - 1)).inner(l, g * (k - 1)).moddown(l, g)
    elif w == "mask_mix":
        terms = int((_mask_index(case["inputs"], case["outputs"]) >= 0).sum())
        c.polys(2 * (case["inputs"] + case["outputs"]), l).point(4.0 * terms * l)
    elif w == "linear":
        k, g = case["babies"], case["giants"]
        c.polys(2 * k + k * g, l).polys(2 * g, l - 1).point(4.0 * k * g * l).rescale(l, g)
    return {"bytes": c.bytes, "flops": c.flops}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """Outputs are whole numbers, compared word for word: no floating-point value to be off from."""
    return None
