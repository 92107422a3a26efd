"""Performance cases: what a decode server has the expert cache do, through its public entry
points, over the range of shapes it meets.

Kinds of case (`kind`):

  decode    `ExpertSlotCache.refresh` of every layer over a window of decode steps, captured
            in one HIP graph as a serving engine captures its decode steps; the experts' slabs
            are in pinned host memory. Each pass copies the window's routing in and replays.
  eager     the same calls made from Python one by one, for an engine that runs without graphs.
  policy    the policy step alone through the C entry points, one graph of a model's layers:
            `expert_cache_manage`, or `expert_cache_manage_remap` where slot ids are wanted.
  fused     `expert_cache_fused`: the policy step with both block alignments, for decode
            batches and for prefill chunks.

Routing is the package's synthetic trace (Zipf popularity with temporal locality, or
group-limited); states are warmed over the trace's first steps, so passes run at the
steady-state hit rate. Passes walk on through the trace and start it again at its end.
"""
from __future__ import annotations

import ctypes
import functools
import os
import sys
from types import SimpleNamespace

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "vllm-expert-cache_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from vllm_expert_cache import _lib, traces  # noqa: E402
from vllm_expert_cache.cache import ExpertSlotCache  # noqa: E402

DEV = "cuda:0"
DECAY = 64  # the package's default LFU halving period

# int8 experts with fp32 per-channel scales: w13 [1536, 2048], w2 [2048, 768]
_W8A8 = {"w13": 1536 * 2048, "w2": 2048 * 768, "s13": 1536 * 4, "s2": 2048 * 4}
# bf16 experts of 352 MB: w13 [28672, 4096], w2 [4096, 14336]
_BF16_BIG = {"w13": 28672 * 4096 * 2, "w2": 4096 * 14336 * 2, "s13": 0, "s2": 0}


def _decode(name, experts, slots, tokens, top_k=8, layers=4, steps=8, windows=24, warm=96,
            lru=False, id64=False, zipf=1.1, keep=0.6, kind="decode", **slabs):
    return {"name": name, "kind": kind, "experts": experts, "slots": slots, "tokens": tokens,
            "top_k": top_k, "layers": layers, "steps": steps, "windows": windows, "warm": warm,
            "lru": lru, "id64": id64, "zipf": zipf, "keep": keep, "groups": 0, "pad": 0,
            **slabs}


def _policy(name, experts, slots, tokens, top_k, layers=48, windows=64, warm=64, lru=False,
            id64=False, remap=True, groups=0, pad=0, zipf=1.1, keep=0.6):
    return {"name": name, "kind": "policy", "experts": experts, "slots": slots,
            "tokens": tokens, "top_k": top_k, "layers": layers, "steps": 1, "windows": windows,
            "warm": warm, "lru": lru, "id64": id64 and remap, "remap": remap, "groups": groups,
            "pad": pad, "zipf": zipf, "keep": keep}


def _fused(name, experts, slots, tokens, top_k, block, layers, windows, warm=32, groups=0,
           pad=0, zipf=1.1, keep=0.6):
    return {"name": name, "kind": "fused", "experts": experts, "slots": slots,
            "tokens": tokens, "top_k": top_k, "block": block, "layers": layers, "steps": 1,
            "windows": windows, "warm": warm, "lru": True, "id64": False, "groups": groups,
            "pad": pad, "zipf": zipf, "keep": keep}


def listed():
    return [
        # single-user decode of a 128-expert int8 model, half its experts resident
        _decode("decode-1", 128, 64, 1, **_W8A8),
        # the same with three quarters resident: few copies, the chain of launches shows
        _decode("decode-1-s96", 128, 96, 1, **_W8A8),
        # four users at once, int64 routing ids (torch.topk's own type), LRU
        _decode("decode-4", 128, 48, 4, steps=4, lru=True, id64=True, **_W8A8),
        # few very large bf16 experts, top-2, half resident: one copy takes milliseconds
        _decode("decode-1-e8-bf16", 8, 4, 1, top_k=2, layers=1, steps=12, windows=1, warm=16,
                zipf=0.0, keep=0.5, **_BF16_BIG),
        # an engine without graphs: every layer's refresh is called from Python
        _decode("eager-1", 128, 96, 1, steps=1, windows=192, kind="eager", **_W8A8),
        # the policy step of 48 layers: single-user decode
        _policy("policy-8", 128, 64, 1, 8),
        # 512 experts at 257 slots and 50 ids, LRU, the policy alone: odd slots, ragged ids
        _policy("policy-50-e512", 512, 257, 5, 10, lru=True, remap=False),
        # 16 users on 256 experts with group-limited routing, int64 ids, padded batch
        _policy("policy-128-e256", 256, 192, 15, 8, id64=True, groups=8, pad=8),
        # policy and block alignment: single-user decode
        _fused("fused-8", 128, 64, 1, 8, 16, layers=48, windows=64),
        # a batch of 64 sequences on 256 experts (padded from 60), half resident
        _fused("fused-512-e256", 256, 128, 60, 8, 16, layers=16, windows=16, groups=8, pad=32),
        # a prefill chunk of 2048 tokens
        _fused("fused-16384", 128, 64, 2048, 8, 64, layers=4, windows=4),
    ]


def _log(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def draw(rng):
    case = _drawn(rng)
    del case["name"]
    return case


def _drawn(rng):
    kind = rng.choice(["decode", "decode", "decode", "eager", "policy", "policy", "fused",
                       "fused", "fused"])
    common = {"zipf": round(rng.uniform(0.7, 1.3), 2), "keep": round(rng.uniform(0.3, 0.8), 2)}
    if kind == "fused":
        experts = _log(rng, 8, 512)
        top_k = rng.randint(1, min(8, experts))
        tokens = _log(rng, 1, 8192)
        groups = 8 if experts % 8 == 0 and experts >= 64 and rng.random() < 0.5 else 0
        return _fused("", experts, max(1, round(experts * rng.uniform(0.2, 0.9))), tokens,
                      top_k, rng.choice([8, 16, 16, 32, 64, 128]),
                      layers=48 if tokens <= 16 else 16 if tokens <= 128 else 4,
                      windows=64 if tokens <= 16 else 16 if tokens <= 128 else 2,
                      groups=groups, pad=rng.choice([0, 0, rng.randint(1, 40)]), **common)
    if kind == "policy":
        experts = _log(rng, 8, 1024)
        top_k = rng.randint(1, min(10, max(1, experts // 4)))
        slots = max(top_k, round(experts * rng.uniform(0.2, 0.9)))
        tokens = _log(rng, 1, max(1, slots // top_k))
        return _policy("", experts, slots, tokens, top_k, lru=rng.random() < 0.5,
                       id64=rng.random() < 0.5, remap=rng.random() < 0.7,
                       pad=rng.randint(0, max(0, min(24, slots - tokens * top_k))), **common)
    # slabs of 16-byte multiples, 2 MB to 352 MB of experts a layer, in up to 2.4 GB
    layers = 4 if kind != "eager" else rng.randint(1, 4)
    experts = _log(rng, 8, 256)
    top_k = rng.randint(1, min(8, max(1, experts // 4)))
    total = _log(rng, 1 << 16, min(48 << 20, int(2.4e9) // (experts * layers)))
    w13 = max(16, int(total * 2 / 3) // 16 * 16)
    w2 = max(16, (total - w13) // 16 * 16)
    scales = rng.random() < 0.6
    slots = max(top_k, round(experts * rng.uniform(0.3, 0.9)))
    tokens = min(_log(rng, 1, 8), slots // top_k)
    # a window moves at most half the 352 MB case's bytes
    steps = 1 if kind == "eager" else max(1, min(8, int(1.5e9) // (tokens * top_k * layers *
                                                                   (w13 + w2))))
    return _decode("", experts, slots, tokens, top_k, layers=layers, steps=steps,
                   windows=max(1, 192 // steps), lru=rng.random() < 0.5,
                   id64=rng.random() < 0.5, kind=kind, w13=w13, w2=w2,
                   s13=64 * rng.randint(1, 128) if scales else 0,
                   s2=64 * rng.randint(1, 128) if scales else 0, **common)


# ---- inputs ------------------------------------------------------------------------------

def _mk(case):
    return case["tokens"] * case["top_k"] + case["pad"]


def _routing(case, seed, layers, steps):
    """[steps, layers, mk] int32 routing ids; the last `pad` ids of a step are -1, as a padded
    batch has them."""
    out = np.full((steps, layers, _mk(case)), -1, np.int32)
    for l in range(layers):
        w = traces.Workload("case", case["experts"], case["top_k"], case["tokens"], layers,
                            steps, (case["slots"],), (),
                            "grouped" if case["groups"] else "locality", zipf_s=case["zipf"],
                            keep=case["keep"], groups=case["groups"],
                            topk_groups=case["groups"] // 2, seed0=1000 * seed)
        out[:, l, :case["tokens"] * case["top_k"]] = traces.routing(w, l)
    return out


def _ids(case, seed):
    """(warm-up routing, windows of routing) on the device."""
    # a prefill chunk needs no trace of chunks to warm the cache: decode steps do
    wide = case["kind"] == "fused" and case["tokens"] > 64
    warm_case = dict(case, tokens=8, pad=0) if wide else case
    n = case["steps"] * case["windows"]
    if wide:
        warm = _routing(warm_case, seed, case["layers"], case["warm"])
        rest = _routing(case, seed, case["layers"], n)
    else:
        both = _routing(case, seed, case["layers"], case["warm"] + n)
        warm, rest = both[:case["warm"]], both[case["warm"]:]
    dt = torch.int64 if case["id64"] else torch.int32
    rest = rest.reshape(case["windows"], case["steps"], case["layers"], -1)
    return (torch.as_tensor(warm, device=DEV).to(dt), torch.as_tensor(rest, device=DEV).to(dt))


def _pinned(experts, nbytes, dtype, gen):
    """One expert tensor [experts, n] in pinned host memory, random content."""
    size = torch.empty((), dtype=dtype).element_size()
    host = torch.empty((experts, nbytes // size), dtype=dtype, pin_memory=True)
    step = max(1, (256 << 20) // nbytes)
    for e in range(0, experts, step):
        rows = host[e:e + step]
        if dtype == torch.float32:
            rows.copy_(torch.rand(rows.shape, device=DEV, generator=gen))
        else:
            rows.copy_(torch.randint(-128, 128, rows.shape, dtype=dtype, device=DEV,
                                     generator=gen))
    return host


def _caches(case, seed):
    """One armed cache a layer, over pinned expert tensors."""
    os.environ["EXPERT_CACHE_POLICY"] = "lru" if case["lru"] else "lfu"
    os.environ["EXPERT_CACHE_DECAY"] = str(DECAY)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    made = []
    for _ in range(case["layers"]):
        owner = SimpleNamespace()
        for name, key, dtype in (("w13_weight", "w13", torch.int8),
                                 ("w2_weight", "w2", torch.int8),
                                 ("w13_weight_scale", "s13", torch.float32),
                                 ("w2_weight_scale", "s2", torch.float32)):
            if case[key]:
                setattr(owner, name, _pinned(case["experts"], case[key], dtype, gen))
        names = list(vars(owner))
        cache = ExpertSlotCache(owner, names, case["experts"], case["slots"], DEV,
                                required=names[:2])
        for slot in cache.slots.values():
            slot.zero_()  # a slot that no expert has reached yet compares equal
        made.append(cache)
    return made


class _Rows:
    """Policy state of all layers: one row a layer, each row on a 256-byte boundary."""

    FIELDS = ("table", "map_cold", "slot_expert", "slot_stamp", "routed", "step", "miss",
              "n_miss")

    def __init__(self, layers, experts, slots):
        self.table = self.rows(layers, experts, torch.int32, -1)
        self.map_cold = self.rows(layers, experts, torch.int32, 0)
        self.map_cold.copy_(torch.arange(experts, device=DEV).expand(layers, -1))
        self.slot_expert = self.rows(layers, slots, torch.int32, -1)
        self.slot_stamp = self.rows(layers, slots, torch.int64, 0)
        self.routed = self.rows(layers, experts, torch.uint8, 0)
        self.step = self.rows(layers, 1, torch.int64, 0)
        self.miss = self.rows(layers, 2 * slots, torch.int32, 0)
        self.n_miss = self.rows(layers, 1, torch.int32, 0)

    @staticmethod
    def rows(layers, n, dtype, fill):
        wide = -(-n // 256) * 256
        return torch.full((layers, wide), fill, dtype=dtype, device=DEV)[:, :n]

    def args(self, l):
        return [_row(getattr(self, f), l) for f in self.FIELDS]


def _row(t, l):
    return ctypes.c_void_p(t[l].data_ptr())


def _align_lengths(mk, experts, block):
    """Buffer lengths of one align output, as vLLM's wrapper allocates them."""
    length = mk + experts * (block - 1)
    if mk < experts:
        length = min(mk * block, length)
    return length, -(-length // block)


def _capture(launch):
    """`launch()` in a HIP graph, on the capture's own stream."""
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        result = launch()
    return graph, result


def _step_layers(caches, ids):
    """One decode step: every layer's refresh, slot ids out."""
    return [c.refresh(i) for c, i in zip(caches, ids)]


def prepare(case, seed):
    warm, windows = _ids(case, seed)
    s = SimpleNamespace(case=case, windows=windows, at=0, graph=None, out=None)
    if case["kind"] in ("decode", "eager"):
        s.caches = _caches(case, seed)
        for step in warm:
            _step_layers(s.caches, step)
        if case["kind"] != "eager":
            s.ids = windows[0].clone()
            s.graph, s.out = _capture(lambda: torch.stack(
                [o for step in s.ids for o in _step_layers(s.caches, step)]))
        s.state = {"%d.%s" % (l, f): getattr(c, f) for l, c in enumerate(s.caches)
                   for f in _Rows.FIELDS}
        s.state.update({"%d.%s" % (l, n): t for l, c in enumerate(s.caches)
                        for n, t in c.slots.items()})
    else:
        layers, experts, slots = case["layers"], case["experts"], case["slots"]
        st = s.rows = _Rows(layers, experts, slots)
        s.ids = windows[0, 0].clone()
        s.state = {f: getattr(st, f) for f in _Rows.FIELDS}
        if case["kind"] == "fused":
            mk = _mk(case)
            length, blocks = _align_lengths(mk, experts, case["block"])
            for side in ("hot", "cold"):
                for f, n in (("sorted", length), ("eids", blocks), ("npad", 1)):
                    s.state[f + "_" + side] = _Rows.rows(layers, n, torch.int32, -7)
            for step in warm:
                _launch_policy(case, st, step, None)
            s.graph, _ = _capture(lambda: _launch_fused(case, st, s.ids, s.state))
        else:
            if case["remap"]:
                s.state["out"] = torch.full_like(s.ids, -7)
            for step in warm:
                _launch_policy(case, st, step, s.state.get("out"))
            s.graph, _ = _capture(lambda: _launch_policy(case, st, s.ids, s.state.get("out")))
    return s


def _launch_policy(case, st, ids, out):
    """The policy step of every layer, with the slot ids where `out` is given."""
    lib, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    experts, slots, mk = case["experts"], case["slots"], ids.shape[1]
    head = (mk, experts, slots, min(experts, mk), slots)
    lru_or_lfu = (0 if case["lru"] else 1, DECAY)
    for l in range(case["layers"]):
        if out is None:
            rc = lib.expert_cache_manage(_row(ids, l), *head, *st.args(l), *lru_or_lfu, stream)
        else:
            rc = lib.expert_cache_manage_remap(_row(ids, l), ids.element_size(), *head,
                                               *st.args(l), *lru_or_lfu, _row(out, l), stream)
        if rc:
            raise RuntimeError("policy step failed rc=%d" % rc)


def _launch_fused(case, st, ids, state):
    """The policy step and both alignments of every layer."""
    lib, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    experts, slots, mk = case["experts"], case["slots"], ids.shape[1]
    length, blocks = _align_lengths(mk, experts, case["block"])
    for l in range(case["layers"]):
        rc = lib.expert_cache_fused(
            _row(ids, l), mk, experts, slots, min(experts, mk), slots, *st.args(l),
            case["block"], length, blocks,
            *[_row(state[f + "_" + side], l) for side in ("hot", "cold")
              for f in ("sorted", "eids", "npad")], stream)
        if rc:
            raise RuntimeError("fused step failed rc=%d" % rc)


def run(s):
    ids = s.windows[s.at % len(s.windows)]
    s.at += 1
    if s.case["kind"] == "eager":
        outs = [o for step in ids for o in _step_layers(s.caches, step)]
        return outs, s.state
    s.ids.copy_(ids.view(s.ids.shape))
    s.graph.replay()
    return s.out, s.state


# ---- what a pass cannot do without -------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _inserts(key):
    """Mean inserts a layer-step at the steady state: the policy over one layer's trace of
    another seed, in plain Python."""
    case = dict(key)
    steps = min(256, case["warm"] + case["steps"] * case["windows"])
    if case["kind"] == "fused" and case["tokens"] > 64:
        steps = 8
    ids = _routing(case, 7, 1, steps)[:, 0]
    slots, resident, stamp, total, counted = case["slots"], {}, {}, 0, 0
    for t, row in enumerate(ids, 1):
        routed = sorted(set(int(e) for e in row if e >= 0))
        for e in routed:
            if e in resident:
                stamp[e] = t if case["lru"] else stamp[e] + 1
        new = [e for e in routed if e not in resident]
        if new and not case["lru"] and t % DECAY == 0:
            stamp = {e: v >> 1 for e, v in stamp.items()}
        n = 0
        hold = set(routed)
        victims = sorted((x for x in resident if x not in hold),
                         key=lambda x: (stamp[x], resident[x]))
        for e in new:
            if len(resident) < slots:
                slot = len(resident)
            elif victims:
                victim = victims.pop(0)
                slot = resident.pop(victim)
                del stamp[victim]
            else:
                break
            resident[e], stamp[e], n = slot, t if case["lru"] else 1, n + 1
        if t > len(ids) // 2:
            total, counted = total + n, counted + 1
    return total / max(1, counted)


def work(case):
    """Routing ids read, the policy state read and written, slot ids or alignments written,
    and every inserted expert read from the host and written to its slot."""
    mk, experts, slots = _mk(case), case["experts"], case["slots"]
    wide = 8 if case["id64"] else 4
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    inserts = _inserts(key)
    # table, slot_expert and slot_stamp read; stamps and flags written; a few words an insert
    one = wide * mk + 4 * experts + 12 * slots + 8 + experts + 8 * slots + 24 * inserts + 12
    if case["kind"] == "fused":
        length, blocks = _align_lengths(mk, experts, case["block"])
        one += 2 * (4 * length + 4 * blocks + 4)
    elif case["kind"] != "policy" or case["remap"]:
        one += wide * mk
    if "w13" in case:
        one += 2 * inserts * (case["w13"] + case["w2"] + case["s13"] + case["s2"])
    n = case["layers"] * case["steps"]
    return {"bytes": float(one * n), "flops": 0.0}


def tolerance(case):
    """Routing ids, slots, counts and copied bytes: whole values, the same in every correct
    implementation."""
    return "exact"


def exact(case, seed):
    """Nothing is a computed floating-point number here: the outputs are whole values and
    copied bytes, compared as they are."""
    return None
