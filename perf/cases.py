"""What the framework's speed is measured on: the calls a program makes, through
the public classes of qsketch_amd, over the range of sizes and options they take.

Kinds of case (every size is a number of keys unless it says otherwise):

  window   a tumbling window: clear the sketch, insert the window's keys, read
           the estimates of the distinct keys (19 of 20 of them: the same
           number for every seed; blocking calls)
  batch    the next batch of a running stream: insert it into a sketch that
           already holds a history, look its keys up (stream-ordered calls)
  lookup   a serving sketch answers a skewed stream of lookups
  multi    many independent sketches updated by one captured launch, then read
  learned  a window through the learned form (network, exact table, sketch)
  train    a short training run of the learned form's network
  sf       the next batch of a sketch with split counters, then its lookups

Key streams: Zipf(alpha) over 2^log2u keys, or uniform 32-bit keys when alpha is
0; 64-bit keys carry a noisy log-rank in their upper bits (the learned form's
workload).  Sketches are sized by the library's own rule at its default load
factor; high pools by the rule of the multi-sketch workload (n / 256, at least
1024) unless a case says otherwise.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import qsketch_amd as q

# training constants: the library's defaults, learning rate of its pipeline
LR, BETA1, BETA2, EPS = 2e-3, 0.9, 0.999, 1e-8
HID = 64  # inputs and hidden units of the network
# the learned form's router admits keys whose noisy log-rank is at most this
HEAVY_LOG_RANK = 15


def listed():
    return [
        # the smallest window a program reads out: latency and launches
        dict(name="window_1500", kind="window", n=1500, alpha=1.0, log2u=10, key_bytes=4, n_high=1024),
        # an odd-sized batch into a running sketch, no host wait in between
        dict(name="batch_65537", kind="batch", n=65537, alpha=1.0, log2u=18, history=1 << 22, n_high=1 << 16),
        # the CPU reference path's configuration: an ordinary window
        dict(name="window_2e22", kind="window", n=1 << 22, alpha=1.0, log2u=18, key_bytes=4, n_high=1 << 14),
        # an odd-sized ordinary window of little skew
        dict(name="window_10000019", kind="window", n=10000019, alpha=0.8, log2u=24, key_bytes=4, n_high=1 << 16),
        # 64-bit keys, as a flow or user id
        dict(name="window_2e25_u64", kind="window", n=(1 << 25) - 39, alpha=1.1, log2u=24, key_bytes=8, n_high=1 << 17),
        # no skew at all: nearly every key is new
        dict(name="window_2e27_uniform", kind="window", n=1 << 27, alpha=0.0, log2u=32, key_bytes=4, n_high=1 << 18),
        # the benchmark's workload
        dict(name="window_2e28_zipf", kind="window", n=1 << 28, alpha=1.1, log2u=26, key_bytes=4, n_high=1 << 18),
        # lookups alone, hot keys repeated as a service sees them
        dict(name="lookup_12582917", kind="lookup", n=12582917, alpha=1.1, log2u=24, history=1 << 26, n_high=1 << 18),
        # hundreds of streams of very different lengths and skews at once
        dict(name="multi_512", kind="multi", streams=512, log2max=20),
        # the learned form's window
        dict(name="learned_2e25", kind="learned", n=1 << 25, alpha=1.1, log2u=24, table_log2=19),
        # the learned form's training loop
        dict(name="train_4096x8", kind="train", n=4096, steps=8),
        # split counters: a large skewed batch
        dict(name="sf_2e26", kind="sf", n=1 << 26, alpha=1.1, log2u=24, times=3),
    ]


def _log_int(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi], odd half of the time."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return min(hi, v | 1) if rng.random() < 0.5 else v


def _universe(n):
    """Key universes between about n / 8 and 2 n, within 2^10 .. 2^24."""
    return max(10, min(24, n.bit_length() - 1))


def draw(rng):
    kind = rng.choice(["window", "window", "window", "batch", "lookup", "multi", "learned", "train", "sf"])
    alpha = rng.choice([0.0, 0.8, 1.0, 1.1, 1.5])
    if kind == "window":
        n = _log_int(rng, 1 << 10, 1 << 27)
        kb = 8 if n <= (1 << 25) and alpha and rng.random() < 0.3 else 4
        log2u = min(24, max(10, _universe(n) - rng.randrange(3)))
        return dict(kind=kind, n=n, alpha=alpha, log2u=log2u if alpha else 32, key_bytes=kb, n_high=max(1024, n // 128))
    if kind == "batch":
        n = _log_int(rng, 1 << 10, 1 << 20)
        log2u = rng.choice([18, 20])  # a long run links every key's bucket in the end
        return dict(kind=kind, n=n, alpha=alpha or 0.8, log2u=log2u, history=1 << 22, n_high=(1 << log2u) + 1024)
    if kind == "lookup":
        n = _log_int(rng, 1 << 10, 1 << 25)
        return dict(kind=kind, n=n, alpha=alpha or 0.8, log2u=24, history=1 << 24, n_high=1 << 17)
    if kind == "multi":
        return dict(kind=kind, streams=_log_int(rng, 8, 512), log2max=rng.randrange(14, 21))
    if kind == "learned":
        return dict(kind=kind, n=_log_int(rng, 1 << 16, 1 << 25), alpha=1.1, log2u=24, table_log2=19)
    if kind == "train":
        return dict(kind=kind, n=_log_int(rng, 256, 16384), steps=rng.randrange(4, 13))
    return dict(kind=kind, n=_log_int(rng, 1 << 12, 1 << 26), alpha=alpha, log2u=24 if alpha else 32,
                times=rng.choice([2, 3, 4]))


# -- inputs ---------------------------------------------------------------------
@functools.lru_cache(maxsize=96)
def _zipf(alpha, log2u):
    return q.Zipf(alpha, 1 << log2u)


def _keys(case, n, seed):
    if case.get("key_bytes", 4) == 8:
        return _zipf(case["alpha"], case["log2u"]).keys_u64_noisy(seed=seed, n=n)
    if case["alpha"] == 0:
        return q.uniform_u32(seed=seed, n=n)
    return _zipf(case["alpha"], case["log2u"]).keys_u32(seed=seed, n=n)


def _sketch(case, n):
    return q.Sketch_GPU_Sub_Warp_Level(q.number_of_buckets(n), 8, case["n_high"], 32,
                                       key_bytes=case.get("key_bytes", 4), rng_seed=1)


def _int32(n):
    return torch.empty(n, dtype=torch.int32, device="cuda")


def _reads(case):
    return max(1, int(0.95 * _distinct(case["n"], case["alpha"], case["log2u"])))


def _seen(case, keys):
    """The distinct keys a window's program reads back."""
    u = torch.unique(keys)
    m = _reads(case)
    return u[:m].contiguous() if u.numel() >= m else u.repeat(-(-m // u.numel()))[:m].contiguous()


def prepare(case, seed):
    kind, seed = case["kind"], int(seed) + 1
    if kind == "train":
        return _prepare_train(case, seed)
    if kind == "multi":
        return _prepare_multi(case, seed)
    n = case["n"]
    if kind == "learned":
        keys = _zipf(case["alpha"], case["log2u"]).keys_u64_noisy(seed=seed, n=n)
        L = q.LearnedSketch(q.make_params(q.number_of_buckets(n), max(1024, n // 256), key_bytes=8),
                            table_log2=case["table_log2"])
        L.set_params(_router_weights())
        L.threshold = 31.0 - HEAVY_LOG_RANK
        seen = _seen(case, keys)
        return dict(kind=kind, sketch=L, keys=keys, seen=seen, counts=_int32(seen.numel()))
    keys = _keys(case, n, seed)
    if kind == "sf":
        sk = q.Sketch_GPU_SF_Host_Sub_Warp(q.number_of_buckets(n), 8, case["times"], rng_seed=1)
        seen = _seen(case, keys)
        return dict(kind=kind, sketch=sk, keys=keys, seen=seen, counts=_int32(seen.numel()))
    if kind == "window":
        seen = _seen(case, keys)
        return dict(kind=kind, sketch=_sketch(case, n), keys=keys, seen=seen, counts=_int32(seen.numel()))
    # a sketch with a history, of the same stream
    sk = _sketch(case, case["history"])
    sk.insert(_keys(case, case["history"], seed + 1000003))
    return dict(kind=kind, sketch=sk, keys=keys, n=n, counts=_int32(n))


def _stream_lengths(case):
    """Per stream: a length spread over the logarithm of [2^10, 2^log2max] and a skew."""
    rs = np.random.default_rng(case["streams"])
    lengths = np.rint(2.0 ** rs.uniform(10, case["log2max"], case["streams"])).astype(np.int64)
    return lengths, np.round(rs.uniform(0.7, 1.3, case["streams"]), 1)


def _prepare_multi(case, seed):
    lengths, alphas = _stream_lengths(case)
    ns = len(lengths)
    offs = np.zeros(ns + 1, np.uint64)
    offs[1:] = np.cumsum(lengths)
    keys = _int32(int(offs[-1]))
    for i in range(ns):
        a, b = int(offs[i]), int(offs[i + 1])
        _zipf(float(alphas[i]), 16).keys_u32(seed=seed * 100003 + i, n=b - a, out=keys[a:b])
    sketches = q.SketchSet([q.make_params(q.number_of_buckets(int(m)), max(1024, int(m) // 128), rng_seed=i + 1)
                            for i, m in enumerate(lengths)])
    # the keys of every stream's last quarter are read back
    latest = torch.cat([keys[int(b) - int(m) // 4:int(b)] for b, m in zip(offs[1:], lengths)])
    d_read = torch.from_numpy(np.concatenate([[0], np.cumsum(lengths // 4)])).cuda()
    d_offs = torch.from_numpy(offs.view(np.int64).copy()).cuda()
    graph = sketches.capture_insert(keys, offs, d_offs)
    return dict(kind="multi", sketch=sketches, graph=graph, keys=keys, d_offs=d_offs, latest=latest, d_read=d_read,
                n=latest.numel(), counts=_int32(latest.numel()))


def _router_weights():
    """A network that reads the noisy log-rank v in key bits 48..52 and scores
    31 - v; its other units carry ordinary weights that the output ignores."""
    rs = np.random.default_rng(5)
    w1, w2 = (rs.uniform(-0.125, 0.125, (HID, HID)) for _ in range(2))
    b1, b2, w3 = np.zeros(HID), np.zeros(HID), np.zeros(HID)
    for j in range(5):
        w1[j], w2[j] = 0, 0
        w1[j, 48 + j], w2[j, j], w3[j] = 1, 1, -(2.0 ** j)
    return np.concatenate([w1.ravel(), b1, w2.ravel(), b2, w3, [31.0]]).astype(np.float32)


def _train_inputs(case, seed):
    """(keys, targets, weights) on the host: per step, pairs of a key with a
    noisy log-rank in its upper bits and log2(1 + its count)."""
    rs = np.random.default_rng(seed)
    shape = (case["steps"], case["n"])
    rank = np.exp2(rs.uniform(0, 24, shape))
    field = np.clip(np.rint(np.log2(rank) + rs.normal(0, 1.5, shape)), 0, 31).astype(np.int64)
    keys = (field << 48) | rs.integers(0, 1 << 48, shape)
    targets = np.log2(1.0 + np.floor(2.0 ** 24 / rank ** 1.1)).astype(np.float32)
    bound = 1 / math.sqrt(HID)
    w = [rs.uniform(-bound, bound, HID * HID), np.zeros(HID), rs.uniform(-bound, bound, HID * HID), np.zeros(HID),
         rs.uniform(-bound, bound, HID), np.zeros(1)]
    return keys, targets, np.concatenate(w).astype(np.float32)


def _prepare_train(case, seed):
    keys, targets, weights = _train_inputs(case, seed)
    L = q.LearnedSketch(q.make_params(1021, 1024, key_bytes=8), table_log2=12)
    return dict(kind="train", sketch=L, weights=weights, keys=[torch.from_numpy(k).cuda() for k in keys],
                targets=[torch.from_numpy(t).cuda() for t in targets])


# -- one pass ---------------------------------------------------------------------
def run(s):
    kind, sk = s["kind"], s["sketch"]
    if kind in ("window", "learned"):
        sk.clear()
        sk.insert(s["keys"])
        return sk.search(s["seen"], counts=s["counts"])
    if kind == "batch":
        sk.insert_async(s["keys"], s["n"])
        sk.search_async(s["keys"], s["n"], s["counts"])
        return s["counts"]
    if kind == "lookup":
        return sk.search(s["keys"], counts=s["counts"])
    if kind == "multi":
        sk.clear()
        s["graph"].launch()
        sk.search_async(s["latest"], s["d_read"], s["n"], s["counts"])
        return s["counts"]
    if kind == "sf":
        sk.insert(s["keys"])
        return sk.search(s["seen"], counts=s["counts"])
    # train: from the given weights, one Adam step per batch; the trained weights
    sk.set_params(s["weights"])
    for k, t in zip(s["keys"], s["targets"]):
        sk.step(k, t, lr=LR, want_loss=False)
    return sk.get_params()


# -- what a pass cannot do without ----------------------------------------------------
def _distinct(n, alpha, log2u):
    """Expected distinct keys of n draws (64 groups of ranks to a factor of two)."""
    u = 2.0 ** log2u
    if alpha == 0:
        return u * -math.expm1(-n / u)
    edges = np.unique(np.floor(np.exp2(np.linspace(0, log2u, 64 * log2u + 1))))
    mid, width = (edges[:-1] + edges[1:]) / 2, np.diff(edges)
    mid[width == 1] = edges[:-1][width == 1]
    p = mid ** -alpha
    p /= (p * width).sum()
    return float((width * -np.expm1(-n * p)).sum())


def work(case):
    kind = case["kind"]
    if kind == "train":
        macs = 3 * (2 * HID * HID + HID)  # forward, to the inputs, to the weights
        return {"bytes": case["steps"] * case["n"] * 12 + case["steps"] * 16 * 8385, "flops": 2.0 * macs * case["n"] * case["steps"]}
    if kind == "multi":
        lengths, alphas = _stream_lengths(case)
        d = sum(_distinct(int(m), float(al), 16) for m, al in zip(lengths, alphas))
        n, n_high = float(lengths.sum()), float(np.maximum(1024, lengths // 128).sum())
        return {"bytes": 24 * n + 128 * n_high + 4 * n + 64 * d + 2 * n + 32 * d, "flops": 0}
    n, kb = case["n"], 8 if kind == "learned" else case.get("key_bytes", 4)
    d = _distinct(n, case["alpha"], case["log2u"])
    reads = 0.95 * d
    if kind == "lookup":  # each key, each distinct bucket once, each estimate
        return {"bytes": (kb + 4) * n + 32 * d, "flops": 0}
    if kind == "batch":  # insert: each key and bucket; lookup: each key, bucket and estimate
        return {"bytes": 2 * kb * n + 4 * n + 96 * d, "flops": 0}
    if kind == "sf":  # three splits and three counters of a key, read and written; 32-byte rows read back
        return {"bytes": kb * n + d * 3 * (case["times"] + 2) * 4 + (kb + 36) * reads, "flops": 0}
    # clear: the table written; insert: each key, each touched bucket read and
    # written; search: each distinct key, its bucket and its estimate
    bytes_ = 32 * 0.75 * n + 128 * case.get("n_high", max(1024, n // 256)) + kb * n + 64 * d + (kb + 36) * reads
    return {"bytes": bytes_, "flops": 2.0 * (2 * HID * HID + HID) * n if kind == "learned" else 0}


# -- the same in 64 bits ------------------------------------------------------------
def exact(case, seed):
    """The trained weights.  (Every other kind returns whole numbers.)"""
    if case["kind"] != "train":
        return None
    keys, targets, w = _train_inputs(case, int(seed) + 1)
    p = torch.from_numpy(w).double()
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    cut = [HID * HID, HID, HID * HID, HID, HID, 1]

    def bf16(x):  # the network's own precision of weights and activations
        return x.to(torch.bfloat16).double()

    for t in range(case["steps"]):
        x = torch.from_numpy(((keys[t][:, None] >> np.arange(HID)) & 1).astype(np.float64))
        w1, b1, w2, b2, w3, b3 = p.split(cut)
        w1, w2, w3 = bf16(w1).view(HID, HID), bf16(w2).view(HID, HID), bf16(w3)
        z1 = x @ w1.T + b1
        h1 = bf16(z1.relu())
        z2 = h1 @ w2.T + b2
        h2 = bf16(z2.relu())
        dy = (h2 @ w3 + b3 - torch.from_numpy(targets[t]).double()) / case["n"]
        d2 = dy[:, None] * w3 * (z2 > 0)
        d1 = (d2 @ w2) * (z1 > 0)
        g = torch.cat([(d1.T @ x).reshape(-1), d1.sum(0), (d2.T @ h1).reshape(-1), d2.sum(0), dy @ h2, dy.sum()[None]])
        m = BETA1 * m + (1 - BETA1) * g
        v = BETA2 * v + (1 - BETA2) * g * g
        p = p - LR * (m / (1 - BETA1 ** (t + 1))) / ((v / (1 - BETA2 ** (t + 1))).sqrt() + EPS)
    return p.numpy()
