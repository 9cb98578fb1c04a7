"""Timed cases of the RNS-CKKS engine: one pass of each public entry point a user's program calls, from
one small ciphertext to batches that fill the GPU.

A case names a modulus chain (ring dimension, scaling-prime size), a kind of work and its sizes.
Residues and keys are uniform modulo each prime, which is how ciphertexts, keys and encoded diagonals
look to the engine. Buffers are torch tensors handed over by address; a program's contexts are
created once per chain and kept, as a user's program keeps them.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "fideslib-fork_amd"))

import fides_hip as fh  # noqa: E402

# (log2 N, scaling-prime bits) -> (Q towers, special primes, dnum). 2^16 with 50-bit scaling is the
# production chain of the benchmark, 2^13 the small test chain, 2^16 with 59-bit scaling the chain of
# the bootstrap (every prime on the integer NTT path); 2^14 and 2^15 lie between them.
CHAINS = {(13, 50): (4, 2, 2), (14, 50): (8, 4, 2), (15, 50): (14, 4, 4), (16, 50): (25, 9, 3), (16, 59): (25, 9, 3)}

_contexts = {}


def _context(case):
    key = (case["log_n"], case["bits"])
    if key not in _contexts:
        towers, special, dnum = CHAINS[key]
        _contexts[key] = fh.Context(case["log_n"], towers, special, dnum, scale_bits=case["bits"])
    return _contexts[key]


class Buffer:
    """A torch tensor in the place of the binding's device array."""

    def __init__(self, tensor):
        self.tensor, self.shape, self.words, self.ptr = tensor, tuple(tensor.shape), tensor.numel(), tensor.data_ptr()

    def addr(self, word_offset=0):
        return self.ptr + 8 * word_offset


class State:
    """What a program holds: a context, buffers, keys. Keys and batches go back with it."""

    def __init__(self, case, seed):
        self.case, self.ctx = case, _context(case)
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)
        self.keys, self.batch = {}, None

    def __del__(self):
        try:
            for k in self.keys.values():
                k.free()
            if self.batch is not None:
                self.batch.free()
        except Exception:
            pass

    def empty(self, limbs):
        return Buffer(torch.empty((limbs, self.ctx.N), dtype=torch.int64, device="cuda"))

    def uniform(self, ids, copies=1):
        """copies polynomials of uniform residues modulo the primes ids, back to back."""
        q = torch.tensor([int(self.ctx.moduli[i]) for i in ids], dtype=torch.int64, device="cuda").view(1, -1, 1)
        t = torch.empty((copies, len(ids), self.ctx.N), dtype=torch.int64, device="cuda")
        step = max(1, (1 << 25) // (len(ids) * self.ctx.N))  # the draw and its remainder in pieces
        for i in range(0, copies, step):
            part = t[i:i + step]
            part.random_(0, 1 << 62, generator=self.gen)
            part.remainder_(q)
        return Buffer(t.view(copies * len(ids), self.ctx.N))

    def ct(self, level, copies=1):
        return self.uniform(list(range(level + 1)), 2 * copies)

    def key(self, name):
        if name not in self.keys:
            c = self.ctx
            buf = self.uniform(list(range(c.L1 + c.K)), 2 * c.dnum)
            torch.cuda.synchronize()  # the context copies the key on a stream of its own
            self.keys[name] = c.key_from_device(buf)
        return self.keys[name]


# ---------------------------------------------------------------------------------------------- cases


def listed():
    return [
        # one multiplication, Rescale and rotation of a single small ciphertext: the shortest calls, where launches count
        {"name": "chain_n13", "kind": "chain", "log_n": 13, "bits": 50, "level": 3},
        # the same chain part of the way down an odd modulus chain, its last digit partly filled
        {"name": "chain_n15_level9", "kind": "chain", "log_n": 15, "bits": 50, "level": 9},
        # one rotation at the top of the production chain: what a program issues one call at a time
        {"name": "rotate_n16", "kind": "rotate", "log_n": 16, "bits": 50, "level": 24, "count": 1, "steps": 1},
        # the headline workload: 64 ciphertexts rotated by steps drawn from 16 keyed ones
        {"name": "rotate_n16_batch64", "kind": "rotate", "log_n": 16, "bits": 50, "level": 24, "count": 64, "steps": 16},
        # one product with relinearization and Rescale at the top of the chain
        {"name": "mult_n16", "kind": "mult", "log_n": 16, "bits": 50, "level": 24, "count": 1},
        # the paired products (real and imaginary parts) of a bootstrap's sine evaluation, in its 59-bit chain,
        # with the weighted sum that follows them
        {"name": "mult_n16_59bit_pair", "kind": "mult", "log_n": 16, "bits": 59, "level": 15, "count": 2},
        # forward and inverse transforms over a whole batch of ciphertexts
        {"name": "ntt_n16_batch64", "kind": "ntt", "log_n": 16, "bits": 50, "level": 24, "count": 128},
        # one tick of a server: rotations, products and sums at levels all over the chain, planned and run as one batch
        {"name": "stream_n16_128", "kind": "stream", "log_n": 16, "bits": 50, "count": 128, "steps": 16, "order": 7},
        # one matrix-vector product as the bootstrap makes it: 63 diagonals, giant steps side by side
        {"name": "lt_n16_flat63", "kind": "lt", "log_n": 16, "bits": 50, "level": 20, "rows": 63, "baby": 16, "count": 1, "flat": True},
        # the same matrix applied to a batch of ciphertexts
        {"name": "lt_n16_batch16", "kind": "lt", "log_n": 16, "bits": 50, "level": 20, "rows": 64, "baby": 8, "count": 16, "flat": False},
        # the sum of 256 slots by a radix-4 fold
        {"name": "sum_n16_256", "kind": "sum", "log_n": 16, "bits": 50, "level": 24, "size": 256, "radix": 4},
        # full-slot plaintexts encoded from host values
        {"name": "encode_n16_16", "kind": "encode", "log_n": 16, "bits": 50, "level": 24, "slots": 32768, "count": 16},
    ]


def _between(rng, low, high):
    """A whole number, evenly spread over its logarithm."""
    return min(high, int(math.exp(rng.uniform(math.log(low), math.log(high + 1)))))


def draw(rng):
    kind = rng.choice(["chain", "rotate", "rotate", "mult", "mult", "ntt", "stream", "lt", "sum", "encode"])
    log_n = rng.choice([13, 14, 15, 16, 16])
    bits = rng.choice([50, 59]) if log_n == 16 and kind in ("chain", "rotate", "mult", "ntt") else 50
    top = CHAINS[(log_n, bits)][0] - 1
    case = {"kind": kind, "log_n": log_n, "bits": bits}
    if kind != "stream":
        case["level"] = rng.randint(2, top)
    if kind == "rotate":
        case.update(count=_between(rng, 1, 64), steps=rng.randint(1, 16))
    elif kind == "mult":
        case.update(count=_between(rng, 1, 32))
    elif kind == "ntt":
        case.update(count=_between(rng, 1, 128))
    elif kind == "stream":
        case.update(count=_between(rng, 3, 128), steps=rng.randint(1, 16), order=rng.randrange(1 << 20))
    elif kind == "lt":
        flat = rng.random() < 0.5
        case.update(rows=_between(rng, 3, 64), baby=rng.choice([2, 4, 5, 7, 8, 11, 16]), count=1 if flat else _between(rng, 1, 16), flat=flat)
    elif kind == "sum":
        case.update(size=_between(rng, 2, 256), radix=rng.choice([2, 4, 8]))
    elif kind == "encode":
        case.update(slots=1 << rng.randint(3, log_n - 1), count=_between(rng, 1, 16))
    return case


def _ops(case):
    """The server tick's operations: (kind, level, step) each, 40% rotations, 40% products, 20% sums."""
    rng = np.random.default_rng(case["order"])
    top = CHAINS[(case["log_n"], case["bits"])][0] - 1
    return [(("rotate", "mult", "add")[int(rng.choice(3, p=[0.4, 0.4, 0.2]))], int(rng.integers(1, top + 1)), int(rng.integers(case["steps"])))
            for _ in range(case["count"])]


def _step(i):
    return 3 if i == 15 else 1 << i


def prepare(case, seed):
    s = State(case, seed)
    c, kind = s.ctx, case["kind"]
    lq = case.get("level", 0) + 1
    if kind == "chain":
        s.a, s.b = s.ct(lq - 1), s.ct(lq - 1)
        s.relin, s.rot, s.galois = s.key("relin"), s.key("rot"), c.galois_index(1)
        s.prod, s.scaled, s.out = s.empty(2 * lq), s.empty(2 * lq - 2), s.empty(2 * lq - 2)
    elif kind == "rotate":
        s.a, s.out = s.ct(lq - 1, case["count"]), s.empty(2 * lq * case["count"])
        order = np.random.default_rng(seed).integers(0, case["steps"], case["count"])
        steps = [_step(int(i)) % (c.N // 2) or 1 for i in order]
        s.rot, s.galois = [s.key(r) for r in steps], [c.galois_index(r) for r in steps]
    elif kind == "mult":
        n = case["count"]
        s.a, s.b, s.relin = s.ct(lq - 1, n), s.ct(lq - 1, n), s.key("relin")
        s.prod, s.scaled, s.out = s.empty(2 * lq * n), s.empty((2 * lq - 2) * n), s.empty(2 * lq - 2)
        s.weights = np.random.default_rng(seed).integers(1, 1 << 40, (min(n, 8), lq - 1)).astype(np.uint64)
    elif kind == "ntt":
        s.ids = list(range(lq))
        s.a, s.b = s.uniform(s.ids, case["count"] // 2 + 1), s.uniform(s.ids, case["count"] // 2 + 1)
    elif kind == "stream":
        s.ops, s.batch, s.relin = [], fh.Batch(c), s.key("relin")
        s.out = s.empty(sum(2 * lvl + (0 if what == "mult" else 2) for what, lvl, _ in _ops(case)))
        at = 0
        for what, lvl, step in _ops(case):
            r = _step(step) % (c.N // 2) or 1
            rot, y = (s.key(r), None) if what == "rotate" else (None, s.ct(lvl))
            s.ops.append((what, lvl, rot, c.galois_index(r), s.ct(lvl), y, s.out.addr(at * c.N)))
            at += 2 * lvl + (0 if what == "mult" else 2)
    elif kind == "lt":
        rows, baby, n = case["rows"], case["baby"], case["count"]
        s.a, s.out = s.ct(lq - 1, n), s.empty(2 * lq * n)
        s.diags = s.uniform(list(range(lq)) + [c.L1 + k for k in range(c.K)], rows)
        s.baby = [None] + [s.key(i) for i in range(1, baby)]
        s.baby_galois = [c.galois_index(i) for i in range(baby)]
        giants = range(1, -(-rows // baby)) if case["flat"] else range(1, 2)
        s.giant = [s.key(j * baby) for j in giants]
        s.giant_galois = [c.galois_index(j * baby) for j in giants]
    elif kind == "sum":
        s.a, s.out = s.ct(lq - 1), s.empty(2 * lq)
        steps = c.accumulate_indices(case["radix"], 1, case["size"])
        s.rot, s.galois = [s.key(r) for r in steps], [c.galois_index(r) for r in steps]
    elif kind == "encode":
        rng = np.random.default_rng(seed)
        s.values = rng.uniform(-1, 1, (case["count"], case["slots"])) + 1j * rng.uniform(-1, 1, (case["count"], case["slots"]))
        s.ids, s.out = list(range(lq)), s.empty(lq * case["count"])
    torch.cuda.synchronize()  # inputs are complete before the context's stream reads them
    return s


def run(s):
    case, c = s.case, s.ctx
    kind, level = case["kind"], case.get("level", 0)
    if kind == "chain":
        c.eval_mult(s.a, s.b, level, s.relin, s.prod)
        c.rescale(s.prod, level, 2, s.scaled)
        c.eval_rotate(s.scaled, level - 1, s.rot, s.galois, s.out)
        return [s.prod.tensor, s.scaled.tensor, s.out.tensor]
    if kind == "rotate":
        if case["count"] == 1:
            c.eval_rotate(s.a, level, s.rot[0], s.galois[0], s.out)
        else:
            c.rotate_batch(s.a, case["count"], level, s.rot, s.galois, s.out)
        return s.out.tensor
    if kind == "mult":
        n, limbs = case["count"], level + 1
        if n == 1:
            c.eval_mult(s.a, s.b, level, s.relin, s.prod)
        else:
            c.eval_mult_many(n, s.a, s.b, level, s.relin, s.prod)
        for i in range(0, 2 * n, 8):  # a Rescale call takes up to 8 components
            k = min(8, 2 * n - i)
            c.rescale(Buffer(s.prod.tensor[i * limbs:(i + k) * limbs]), level, k, Buffer(s.scaled.tensor[i * level:(i + k) * level]))
        if n == 1:
            return [s.prod.tensor, s.scaled.tensor]
        terms = [Buffer(s.scaled.tensor[2 * i * level:(2 * i + 2) * level]) for i in range(min(n, 8))]
        c.linear_wsum(terms, [level] * len(terms), s.weights, level, 2, s.out)
        return [s.prod.tensor, s.scaled.tensor, s.out.tensor]
    if kind == "ntt":
        c.ntt_forward(s.a, s.ids, num_polys=case["count"] // 2 + 1)
        c.ntt_inverse(s.b, s.ids, num_polys=case["count"] // 2 + 1)
        return [s.a.tensor, s.b.tensor]
    if kind == "stream":
        b = s.batch
        b.reset()
        for what, lvl, rot, galois, x, y, out in s.ops:
            if what == "rotate":
                b.rotate(x.ptr, lvl, rot, galois, out)
            elif what == "mult":
                b.mult(x.ptr, y.ptr, lvl, s.relin, True, out)
            else:
                b.add(x.ptr, y.ptr, lvl, 2, out)
        b.finalize()
        b.run()
        return s.out.tensor
    if kind == "lt":
        baby = case["baby"]
        if case["flat"]:
            c.linear_transform_flat(s.a, level, case["rows"], baby, 1, s.diags, s.baby, s.baby_galois, s.out, giant_keys=s.giant,
                                    giant_galois=s.giant_galois)
        elif case["count"] == 1:
            c.linear_transform(s.a, level, case["rows"], baby, 1, s.diags, s.baby, s.baby_galois, s.out, giant_key=s.giant[0],
                               giant_galois=s.giant_galois[0])
        else:
            c.linear_transform_batch(s.a, case["count"], level, case["rows"], baby, 1, s.diags, s.baby, s.baby_galois, s.out,
                                     giant_key=s.giant[0], giant_galois=s.giant_galois[0])
        return s.out.tensor
    if kind == "sum":
        c.accumulate_sum(s.a, level, case["radix"], 1, case["size"], s.rot, s.galois, s.out)
        return s.out.tensor
    if kind == "encode":
        c.encode_slots(s.values, 2.0 ** 50, s.ids, s.out)
        return s.out.tensor
    raise ValueError(kind)


def exact(case, seed):
    """None: every output is residues, whole numbers that have to be equal bit for bit."""
    return None


def work(case):
    """Bytes of one pass: inputs, keys and diagonals read once, results written once. The work is
    modular integer arithmetic, for which there is no rate of floating operations."""
    towers, special, dnum = CHAINS[(case["log_n"], case["bits"])]
    alpha = -(-towers // dnum)
    limb = 8 << case["log_n"]

    def key(level):  # the limbs of one key that a key switch at this level reads
        return 2 * (-(-(level + 1) // alpha)) * (level + 1 + special)

    kind, level, n = case["kind"], case.get("level", 0), case.get("count", 1)
    lq = level + 1
    if kind == "chain":
        limbs = 4 * lq + key(level) + 2 * lq + 2 * level + key(level - 1) + 2 * level
    elif kind == "rotate":
        limbs = 4 * lq * n + min(n, case["steps"]) * key(level)
    elif kind == "mult":
        limbs = n * (4 * lq + 2 * lq + 2 * level) + key(level) + (2 * level if n > 1 else 0)
    elif kind == "ntt":
        limbs = 4 * lq * (n // 2 + 1)
    elif kind == "stream":
        limbs, keys = 0, {}
        for what, lvl, step in _ops(case):
            limbs += {"rotate": 4 * lvl + 4, "mult": 6 * lvl + 4, "add": 6 * lvl + 6}[what]
            if what != "add":
                k = step if what == "rotate" else "relin"
                keys[k] = max(keys.get(k, 0), key(lvl))
        limbs += sum(keys.values())
    elif kind == "lt":
        giants = -(-case["rows"] // case["baby"]) - 1 if case["flat"] else 1
        limbs = 4 * lq * n + (case["baby"] - 1 + giants) * key(level) + case["rows"] * (lq + special)
    elif kind == "sum":
        rotations, s = 0, 1
        while s < case["size"]:
            rotations += sum(1 for i in range(1, case["radix"]) if i * s < case["size"])
            s *= case["radix"]
        limbs = 4 * lq + rotations * key(level)
    else:
        return {"bytes": float(16 * case["slots"] * n + limb * lq * n), "flops": 0.0}
    return {"bytes": float(limb * limbs), "flops": 0.0}
