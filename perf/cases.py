"""Performance cases of the partitioned join: what a program that uses this
package has it do, through its public calls, from lookups of a few thousand
rows to the 64M x 256M join.

A case is one of four kinds of call:
- "join": an equi-join of a build and a probe table.  `api` is the call the
  program makes: "sync" (partitioned_join: output allocated and pair count
  waited for in the call), "async" (partitioned_join_async into an output and a
  workspace that the program keeps) or "noalloc" (partitioned_join_noalloc,
  small joins in a serving loop).  Keys are int32 or int64 (`key_bytes`),
  unique on the build side or each repeated `dup` times; probes draw build keys
  uniformly (`theta` 0) or by a Zipf law, a share `match` of them has a partner;
  `payload` adds an int32 payload column on both sides; `unique` declares the
  build keys unique in the plan; `dense` keys are ids 0..n-1, others spread
  over the whole key range.
- "gather": payload columns fetched by a join's pairs.
- "partition": the phase calls (combined histogram, pass one, pass two).
- "plan": the learned planner's steps for a join (key sketch, model, exact counts
  of the heavy-key candidates).
"""
import math

import torch

import partitioned_join_amd as pj
from partitioned_join_amd import planner

_FIELDS = ("kind", "api", "key_bytes", "n_build", "n_probe", "match", "theta", "dup", "unique", "payload", "dense")


def _join(name, api, key_bytes, n_build, n_probe, match, theta=0.0, dup=1, unique=False, payload=False, dense=False):
    return {"name": name, "kind": "join", "api": api, "key_bytes": key_bytes, "n_build": n_build, "n_probe": n_probe,
            "match": match, "theta": theta, "dup": dup, "unique": unique, "payload": payload, "dense": dense}


def listed():
    return [
        # a small dimension table looked up once: launches and latency are all of it
        _join("lookup_4k_16k", "sync", 4, 4000, 16000, 1.0, dense=True),
        # one of many uneven int64 joins of a serving loop that allocates nothing
        _join("i64_zipf_120k_500k", "noalloc", 8, 120011, 500009, 1.0, theta=0.9),
        # the reference benchmark's small configuration: 1M unique keys, every probe matches
        _join("join_1m_4m", "sync", 4, 1 << 20, 1 << 22, 1.0, dense=True),
        # an ordinary fact-to-dimension join of ragged sizes, mildly skewed, some keys without a partner
        _join("ragged_3m_41m", "async", 4, 2999999, 41000003, 0.7, theta=0.8),
        # the headline workload: 64M unique int32 keys, 256M probes, half of them match
        _join("join_64m_256m", "async", 4, 1 << 26, 1 << 28, 0.5, unique=True, dense=True),
        # the skewed workload: Zipf(1.0) probes of 16M keys
        _join("zipf_16m_256m", "async", 4, 1 << 24, 1 << 28, 1.0, theta=1.0, unique=True, dense=True),
        # 64-bit surrogate keys
        _join("i64_16m_64m", "async", 8, 1 << 24, 1 << 26, 0.5),
        # the payload columns of the reference's -V runs, both tables
        _join("payload_20m_90m", "sync", 4, 20000003, 90000001, 0.8, unique=True, payload=True),
        # a many-to-many join: every build key four times, four pairs a match
        _join("dup_12m_24m", "async", 4, 12000000, 24000000, 0.5, dup=4),
        # the columns of a finished join: an 8-byte build column and a 4-byte probe column
        {"name": "gather_10m_40m", "kind": "gather", "n_build": 10000000, "n_probe": 40000000},
        # the partitioning phases on their own, 7 + 6 bits
        {"name": "partition_40m", "kind": "partition", "key_bytes": 4, "n_build": 40000001, "bits1": 7, "bits2": 6},
        # planning the skewed join with the learned planner
        {"name": "plan_16m_256m", "kind": "plan", "key_bytes": 4, "n_build": 1 << 24, "n_probe": 1 << 28, "theta": 1.0},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["join", "gather", "partition", "plan"], [8, 1, 1, 1])[0]
    if kind == "gather":
        nb = _log_uniform(rng, 1e4, 1 << 25)
        return {"kind": kind, "n_build": nb, "n_probe": min(1 << 27, int(nb * rng.uniform(1, 8)))}
    if kind == "partition":
        n, kb = _log_uniform(rng, 1e5, 1 << 27), rng.choice([4, 4, 8])
        b = max(2, min(15, int(math.log2(n / 1024.0))))
        return {"kind": kind, "key_bytes": kb, "n_build": n // (kb // 4), "bits1": (b + 1) // 2, "bits2": b // 2}
    kb = rng.choice([4, 4, 8])
    nb = _log_uniform(rng, 1e3, (1 << 26) // (kb // 4) ** 2)
    ns = min(int(nb * math.exp(rng.uniform(0.0, math.log(16.0)))), (1 << 28) // (kb // 4) ** 2)
    theta = round(rng.uniform(0.3, 1.5), 2) if rng.random() < 0.5 else 0.0
    if kind == "plan":
        return {"kind": kind, "key_bytes": kb, "n_build": nb, "n_probe": ns, "theta": theta}
    dup = rng.choice([1, 1, 1, 2, 5])
    nb -= nb % dup
    ns = min(ns, (1 << 28) // dup)
    small = (nb + ns) * kb * 4 < 96 << 20
    api = rng.choice(["sync", "noalloc"] if small and dup == 1 else ["sync", "async"] if dup == 1 else ["async"])
    c = _join(None, api, kb, nb, ns, round(rng.uniform(0.1, 1.0), 2), theta, dup, dup == 1 and rng.random() < 0.5,
              rng.random() < 0.25, rng.random() < 0.5)
    return {k: c[k] for k in _FIELDS}


# --------------------------------------------------------------------------- inputs
def _keys_of(ids, key_bytes, dense):
    """Keys of the ids (distinct for distinct ids): the ids themselves, or
    spread over the whole key range by multiplications with odd numbers."""
    if key_bytes == 4:
        return (ids if dense else ids * 0x9E3779B1).to(torch.int32)
    if dense:
        return ids.clone()
    k = (ids + 1) * -0x61C8864680B583EB
    k ^= k >> 29
    return k * -0x40A7B892E31B1A47


def _tables(case, gen):
    """Build and probe keys, in no order."""
    nb, ns, dup = case["n_build"], case["n_probe"], case.get("dup", 1)
    kb, dense, match, theta = case["key_bytes"], case.get("dense", False), case.get("match", 1.0), case.get("theta", 0.0)
    dev = gen.device
    nk = nb // dup  # distinct build keys
    build = torch.randperm(nb, generator=gen, device=dev)
    if dup > 1:
        build %= nk
    if theta > 0:
        # in whole numbers: a parallel sum of floats would differ from run to run
        weight = torch.arange(1, nk + 1, dtype=torch.float64, device=dev).pow_(-theta).mul_(2.0 ** 36)
        cdf = weight.to(torch.int64).clamp_(min=1).cumsum_(0)
        u = torch.randint(0, int(cdf[-1].item()), (ns,), generator=gen, device=dev)
        probe = torch.searchsorted(cdf, u, right=True)
        del weight, cdf, u
        probe = torch.randperm(nk, generator=gen, device=dev)[probe]
    else:
        probe = torch.randint(0, nk, (ns,), generator=gen, device=dev)
    misses = ns - _matches(case)
    if misses > 0:  # so many rows, anywhere, take ids that no build row has
        probe[torch.randperm(ns, generator=gen, device=dev)[:misses]] += nk
    return _keys_of(build, kb, dense), _keys_of(probe, kb, dense)


def _matches(case):
    """Probe rows with a partner: their number is exact, so a case's pair count is the same for every seed."""
    return int(round(case["n_probe"] * case.get("match", 1.0)))


def _pairs(case):
    return _matches(case) * case["dup"]


def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    kind = case["kind"]
    if kind == "gather":
        # pairs in a join's order: partition by partition of the key's low bits, each probe row once
        nb, ns = case["n_build"], case["n_probe"]
        row_of = torch.randperm(nb, generator=gen, device=dev)
        key = torch.randint(0, nb, (ns,), generator=gen, device=dev)
        parts = 1 << max(1, min(15, int(math.log2(max(2.0, nb / 2048.0)))))
        order = torch.sort((key % parts).to(torch.int16), stable=True).indices
        pairs = torch.stack([row_of[key[order]].to(torch.int32), order.to(torch.int32)], 1).contiguous()
        bcol = torch.randint(-1 << 62, 1 << 62, (nb,), generator=gen, device=dev)
        pcol = torch.randint(-1 << 31, 1 << 31, (ns,), generator=gen, device=dev).to(torch.int32)
        return {"case": case, "pairs": pairs, "bcol": bcol, "pcol": pcol}
    if kind == "partition":
        keys = torch.randint(-1 << 31, 1 << 31, (case["n_build"],), generator=gen, device=dev)
        keys = keys.to(torch.int32) if case["key_bytes"] == 4 else keys * 0x9E3779B1
        return {"case": case, "keys": keys}
    build, probe = _tables(case, gen)
    state = {"case": case, "build": build, "probe": probe}
    if kind == "plan":
        state["weights"] = planner.load_weights(device=dev)
        return state
    nb, ns = case["n_build"], case["n_probe"]
    state["bpay"] = state["ppay"] = state["plan"] = None
    if case["payload"]:
        state["bpay"] = torch.randint(-1 << 31, 1 << 31, (nb,), generator=gen, device=dev).to(torch.int32)
        state["ppay"] = torch.randint(-1 << 31, 1 << 31, (ns,), generator=gen, device=dev).to(torch.int32)
    if case["unique"]:
        state["plan"] = pj.plan_default(nb, ns, case["key_bytes"])
        state["plan"].unique_build_keys = 1
    if case["api"] != "sync":
        room = ns * case["dup"]  # every probe row may match
        state["out"] = torch.empty((room, 2), dtype=torch.int32, device=dev)
        state["count"] = torch.zeros(1, dtype=torch.int64, device=dev)
    if case["api"] == "async":
        state["ws"] = torch.empty(pj.workspace_size(nb, ns, case["key_bytes"], state["plan"]), dtype=torch.uint8,
                                  device=dev)
    return state


# --------------------------------------------------------------------------- passes
class _Pairs(dict):
    """The pairs that a join left in its output buffer.  A join's pairs are a
    set: the package leaves their order open and two runs order them
    differently.  Looked up, they come sorted, so that two joins of the same
    tables can be compared pair by pair."""

    def __getitem__(self, key):
        pairs, count = dict.__getitem__(self, key)
        n = pairs.shape[0] if count is None else min(int(count.item()), pairs.shape[0])
        return torch.sort(pairs[:n].contiguous().view(torch.int64).view(-1)).values


class _Partitions(dict):
    """Tuples grouped into partitions at their offsets: {name: (tuples,
    offsets, key bytes)}.  Within a partition the order is open; looked up,
    each partition's tuples come sorted."""

    def __getitem__(self, key):
        tuples, offsets, key_bytes = dict.__getitem__(self, key)
        sizes = (offsets[1:] - offsets[:-1]).to(torch.int64)
        part = torch.repeat_interleave(torch.arange(sizes.numel(), device=sizes.device), sizes)
        if key_bytes == 4:
            minor = tuples.contiguous().view(torch.int64).view(-1)
        else:  # the payloads are row ids: distinct
            minor = pj.tuple_payloads(tuples, 8).to(torch.int64)
        order = torch.sort(minor, stable=True).indices
        order = order[torch.sort(part[order], stable=True).indices]
        return tuples[order]


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "join":
        if case["api"] == "sync":
            pairs = pj.partitioned_join(state["build"], state["probe"], state["bpay"], state["ppay"],
                                        plan=state["plan"])
            return _Pairs(pairs=(pairs, None))
        if case["api"] == "async":
            count = pj.partitioned_join_async(state["build"], state["probe"], state["out"], state["bpay"],
                                              state["ppay"], plan=state["plan"], workspace=state["ws"])
            return [_Pairs(pairs=(state["out"], count)), count]
        pj.partitioned_join_noalloc(state["build"], state["probe"], state["out"], state["count"], state["bpay"],
                                    state["ppay"], plan=state["plan"])
        return [_Pairs(pairs=(state["out"], state["count"])), state["count"]]
    if kind == "gather":
        return list(pj.gather(state["pairs"], state["bcol"], state["pcol"]))
    if kind == "partition":
        kb, b1, b2 = case["key_bytes"], case["bits1"], case["bits2"]
        fine, coarse = pj.combined_histogram_pass(state["keys"], b1 + b2, b2)
        t1, o1 = pj.partition_input_tables_pass_one(state["keys"], None, b1, b2)
        t2, o2 = pj.partition_input_tables_pass_two(t1, kb, b1, b2, o1)
        return [fine, coarse, o1, o2, _Partitions(one=(t1, o1, kb), two=(t2, o2, kb))]
    features, candidates, seen = planner.sketch(state["build"], state["probe"])
    logits = planner.forward(state["weights"], features.view(1, -1))
    counts = planner.candidate_counts(state["probe"], candidates, seen)
    return [features, logits, candidates, seen, counts]


# --------------------------------------------------------------------------- 64-bit values
def _murmur3(words):
    """MurmurHash3_x86_32 (seed 0) of keys given as 32-bit words, in int64 tensors."""
    rot = lambda x, r: ((x << r) | (x >> (32 - r))) & 0xFFFFFFFF
    mul = lambda x, c: ((x * (c & 0xFFFF)) + (((x * (c >> 16)) & 0xFFFF) << 16)) & 0xFFFFFFFF
    h = torch.zeros_like(words[0])
    for w in words:
        h = (mul(rot(h ^ mul(rot(mul(w, 0xCC9E2D51), 15), 0x1B873593), 13), 5) + 0xE6546B64) & 0xFFFFFFFF
    h = h ^ (4 * len(words))
    h = mul(h ^ (h >> 16), 0x85EBCA6B)
    h = mul(h ^ (h >> 13), 0xC2B2AE35)
    return h ^ (h >> 16)


def exact(case, seed):
    """The planner's features and logits in 64 bits.  Every other output is
    whole numbers (row ids, payloads, counts, offsets): nothing is rounded."""
    if case["kind"] != "plan":
        return None
    state = prepare(case, seed)
    n, nb, kb = case["n_probe"], case["n_build"], case["key_bytes"]
    j = torch.arange(4096, dtype=torch.int64, device=state["probe"].device)
    sample = state["probe"][((2 * j + 1) * n) // 8192].to(torch.int64)
    words = [sample & 0xFFFFFFFF] + ([(sample >> 32) & 0xFFFFFFFF] if kb == 8 else [])
    bins = torch.bincount(_murmur3(words) & 1023, minlength=1024).to(torch.float64)
    runs = torch.unique(sample, return_counts=True)[1].to(torch.float64)
    size = [math.log2(nb + 1.0) / 32, math.log2(n + 1.0) / 32, math.log2((n + 1.0) / (nb + 1.0)) / 8, kb / 8,
            runs.max().item() / 4096, (runs * runs).sum().item() / 4096 ** 2]
    x = torch.cat([torch.sort(bins, descending=True).values / 4096,
                   torch.tensor(size, dtype=torch.float64, device=bins.device)])
    w, h, at = state["weights"].double(), x, 0
    for rows, cols in ((1030, 256), (256, 256), (256, 81)):
        h = h @ w[at:at + rows * cols].view(rows, cols) + w[at + rows * cols:at + rows * cols + cols]
        at += rows * cols + cols
        if cols != 81:
            h = torch.relu(h)
    return [x, h.view(1, -1), None, None, None]


def work(case):
    """Bytes that one pass cannot do without: each column read once, each
    output written once.  The operations are a few integers per row."""
    kind = case["kind"]
    if kind == "gather":
        return {"bytes": case["n_probe"] * (8 + 8 + 4 + 8 + 4), "flops": 0}
    if kind == "partition":
        n, kb = case["n_build"], case["key_bytes"]
        return {"bytes": n * (kb + 2 * (8 if kb == 4 else 16)), "flops": 0}
    n = case["n_build"] + case["n_probe"]
    if kind == "plan":  # the probe column, whose heavy keys are counted
        return {"bytes": case["n_probe"] * case["key_bytes"], "flops": 0}
    row = case["key_bytes"] + (4 if case["payload"] else 0)
    return {"bytes": n * row + 8 * _pairs(case), "flops": 0}
