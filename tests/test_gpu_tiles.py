"""Sizes at the edges of the policy step's and the alignments' work split, against the oracle.

The policy step gives every expert and slot a thread of a workgroup of 1, 2, 4, 8 or 16
waves, finds few victims one by one and many by sorting each wave's keys, and orders stamps by
32-bit keys where they fit. The fused call runs in one workgroup up to 1024 ids and, above, in
a workgroup per 1024 ids after the policy step. Whole values, so every comparison is exact.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

import gpu_util as gu
import oracle
from test_gpu_fuzz import _device_state
from test_gpu_remap_fused import _fused_call, _outs
from test_oracle import align_lengths

pytestmark = pytest.mark.gpu


def _check_state(st, ref, tag):
    for name in ("table", "map_cold", "slot_expert", "slot_stamp", "routed", "step", "miss",
                 "n_miss"):
        got, want = getattr(st, name)[0].cpu().numpy(), getattr(ref, name)
        assert np.array_equal(got, want), f"{tag}: {name} at {gu.first_diff(got, want)}"


def _step(st, ref, ids, mi, policy, decay, id64, tag):
    dt = torch.int64 if id64 else torch.int32
    d_ids = torch.as_tensor(ids, device=gu.DEV).to(dt)
    out = torch.full_like(d_ids, -9)
    rc = gu.manage_call(gu.lib(), st, 0, gu.ptr(d_ids), len(ids), st.E, mi, policy, decay,
                        gu.ptr(out), 8 if id64 else 4)
    assert rc == 0 and ref.manage(ids, st.E, mi, policy, decay) == 0
    torch.cuda.synchronize()
    _check_state(st, ref, tag)
    assert np.array_equal(out.cpu().numpy(), oracle.remap(ids, ref.table)), tag


@pytest.mark.parametrize("E,S", [(63, 64), (64, 65), (65, 3), (128, 129), (129, 128), (200, 256),
                                 (257, 257), (512, 100), (513, 513), (900, 1024), (1024, 1000),
                                 (1025, 1024), (2050, 40)])
@pytest.mark.parametrize("policy", [0, 1])
def test_policy_step_at_every_width(E, S, policy):
    """Few inserts (1 .. 9 misses a step, across the line between the two victim searches) and
    many, with few distinct stamps so that keys tie up to the slot, and ids past one and past
    four of the workgroup's passes."""
    rng = np.random.default_rng(E * 7 + S)
    nhot = min(S, E)
    hot, slots = rng.choice(E, nhot, replace=False), rng.choice(S, nhot, replace=False)
    st, ref = _device_state(E, S, S, hot, slots, rng.integers(0, 5, size=S))
    for t, misses in enumerate([0, 1, 2, 5, 6, 8, 9, 40, E, 1]):
        table = ref.table
        cold, warm = np.nonzero(table < 0)[0], np.nonzero(table >= 0)[0]
        ids = np.concatenate([rng.permutation(cold)[:misses], rng.permutation(warm)[:3], [-1, E]])
        ids = rng.permutation(ids).astype(np.int32)
        if t == 4:
            ids = np.resize(ids, 5 * 1024 + 3)
        _step(st, ref, ids, S, policy, 3, t % 2 == 1, f"E={E} S={S} policy={policy} step {t}")


@pytest.mark.parametrize("E,S", [(8, 4), (64, 40), (128, 64), (500, 200), (1100, 300)])
@pytest.mark.parametrize("policy", [0, 1])
def test_more_experts_routed_than_slots(E, S, policy):
    """Misses with few or no slots to evict: the slots' experts are all routed, or all but one
    or two, while several or most of the others miss."""
    rng = np.random.default_rng(E)
    st, ref = _device_state(E, S, S, rng.choice(E, S, replace=False), rng.permutation(S),
                            rng.integers(0, 5, size=S))
    for t, (kept, missing) in enumerate([(S, 1), (S, 4), (S, E), (S - 1, 2), (S - 2, E), (S, E)]):
        cold, warm = np.nonzero(ref.table < 0)[0], np.nonzero(ref.table >= 0)[0]
        ids = np.concatenate([rng.permutation(warm)[:kept], rng.permutation(cold)[:missing]])
        _step(st, ref, rng.permutation(ids).astype(np.int32), S, policy, 2, t % 2 == 1,
              f"E={E} S={S} policy={policy} step {t}")


@pytest.mark.parametrize("S,bits", [(40, 26), (100, 25), (200, 24), (500, 23), (1000, 22)])
@pytest.mark.parametrize("policy", [0, 1])
@pytest.mark.parametrize("misses", [3, 30])
def test_stamps_at_the_edge_of_the_short_keys(S, bits, policy, misses):
    """Stamps on both sides of the largest that has a 32-bit key (`bits` bits above the slot),
    counted from zero under LFU and back from the step under LRU, beside empty slots."""
    E = min(1024, S + 60)
    rng = np.random.default_rng(S + policy)
    hot, slots = rng.choice(E, S - 4, replace=False), rng.choice(S, S - 4, replace=False)
    top = 1 << bits
    for far in (False, True):
        edge = np.arange(top - 12, top + 4 if far else top - 6)
        stamps = rng.choice(np.concatenate([[0, 1, 2], edge]), size=S)
        if policy == 0:
            stamps = np.where(stamps > 2, (1 << 40) - stamps, stamps * (1 << 39) if far else 0)
        st, ref = _device_state(E, S, S, hot, slots, stamps)
        st.step[0] = 1 << 40
        ref.step[:] = 1 << 40
        for t in range(3):
            cold = np.nonzero(ref.table < 0)[0]
            ids = rng.permutation(cold)[:misses].astype(np.int32)
            _step(st, ref, ids, S, policy, 0, False, f"S={S} policy={policy} far={far} step {t}")


@pytest.mark.parametrize("mk", [1, 64, 65, 255, 256, 257, 1023, 1024, 1025, 2048, 2051, 5000])
@pytest.mark.parametrize("E,S,bs", [(7, 3, 1), (128, 64, 16), (200, 257, 12), (1024, 1024, 64)])
def test_fused_at_the_workgroups_edges(mk, E, S, bs):
    """From one id to several workgroups' ids, with padding and out-of-range ids and a few
    popular experts; the ids start on a 16-byte boundary and 4 bytes past one."""
    rng = np.random.default_rng(mk + E)
    L, NB = align_lengths(mk, E, bs)
    st, ref = gu.Layers(1, E, S), oracle.State(E, S)
    for t in range(3):
        ids = rng.integers(-2, E + 2, size=mk).astype(np.int32)
        ids[rng.random(mk) < 0.3] = rng.integers(0, min(E, 4))
        outs = _outs(L, NB)
        d_ids = torch.zeros(mk + 1, dtype=torch.int32, device=gu.DEV)
        d_ids = d_ids[1:] if t == 1 else d_ids[:mk]
        d_ids.copy_(torch.as_tensor(ids))
        assert _fused_call(gu.lib(), st, d_ids, mk, bs, L, NB, outs) == 0
        rc, want = ref.fused(ids, min(E, mk), S, bs, L, NB)
        assert rc == 0
        torch.cuda.synchronize()
        for k, v in want.items():
            assert np.array_equal(outs[k].cpu().numpy(), v), (t, k)
        _check_state(st, ref, f"mk={mk} step {t}")


@pytest.mark.parametrize("E,S", [(8, 4), (64, 64), (200, 130), (256, 256), (257, 100)])
@pytest.mark.parametrize("chunks", [1, 7, 32, 128, 300])
@pytest.mark.parametrize("id64", [False, True])
def test_refresh_matches_policy_step_and_gather(E, S, chunks, id64, monkeypatch):
    """One-launch refreshes (one workgroup, fewer than the tiles, the most) and two-launch ones
    beside the separate calls on a twin, over steps with no, some and all slots replaced and
    pending prefetches to settle; state, slot ids and slot bytes after every step."""
    from types import SimpleNamespace

    from vllm_expert_cache.cache import ExpertSlotCache

    monkeypatch.setenv("EXPERT_CACHE_CHUNKS", str(chunks))
    rng = np.random.default_rng(E + S + chunks)
    sizes = [4096 * 3 + 16, 48, 8192 * 2, 16, 64, 32, 80]  # seven: a second gather call
    owner = SimpleNamespace(**{f"w{i}": gu.pinned(E * n).view(E, n)
                               for i, n in enumerate(sizes)})
    for t in vars(owner).values():
        gu.fill_random(t.view(-1), int(rng.integers(1 << 30)))
    one, two = (ExpertSlotCache(owner, list(vars(owner)), E, S, gu.DEV) for _ in range(2))
    for c in (one, two):
        c.policy, c.decay = 1, 3
        for t in c.slots.values():
            t.zero_()
    two._layer_plan = lambda: (None, None)  # the separate calls
    dt = torch.int64 if id64 else torch.int32
    for t in range(12):
        k = int(rng.choice([1, 2, max(1, S // 2), S, E]))
        ids = rng.permutation(E)[:k]
        ids = torch.as_tensor(np.resize(ids, max(k, 3)), device=gu.DEV).to(dt)
        ids[rng.integers(0, ids.numel())] = -1
        if t % 4 == 3:
            for c in (one, two):
                c.prefetch(ids[:min(S, ids.numel())].roll(1) + 1)
                c.join()
        if t == 6:
            for c in (one, two):
                c.policy = 0
        outs = [c.refresh(ids) for c in (one, two)]
        torch.cuda.synchronize()
        assert torch.equal(*outs), t
        assert int(one.arrived) == 0
        for f in ("table", "map_cold", "slot_expert", "slot_stamp", "routed", "step", "miss",
                  "n_miss"):
            assert torch.equal(getattr(one, f), getattr(two, f)), (t, f)
        for n in one.names:
            assert torch.equal(one.slots[n], two.slots[n]), (t, n)


@pytest.mark.parametrize("E,S", [(60, 64), (128, 100), (256, 256), (200, 90)])
@pytest.mark.parametrize("chunks,lanes", [(32, 1), (16, 2), (3, 5)])
@pytest.mark.parametrize("id64", [False, True])
def test_refresh_with_more_ids_than_threads(E, S, chunks, lanes, id64, monkeypatch):
    """The one launch's four waves over several hundred to a few thousand ids, on a 16-byte
    boundary and one id past it, on grids of one and of several lanes, beside the separate
    calls on a twin: a cold start, steps whose experts are all resident, new experts, ids
    that cover every expert, and no ids."""
    from types import SimpleNamespace

    from vllm_expert_cache.cache import ExpertSlotCache

    monkeypatch.setenv("EXPERT_CACHE_CHUNKS", str(chunks))
    monkeypatch.setenv("EXPERT_CACHE_LANES", str(lanes))
    rng = np.random.default_rng(E + S + chunks)
    owner = SimpleNamespace(a=gu.pinned(E * 12304).view(E, 12304),
                            b=gu.pinned(E * 80).view(E, 80))
    for t in vars(owner).values():
        gu.fill_random(t.view(-1), int(rng.integers(1 << 30)))
    one, two = (ExpertSlotCache(owner, list(vars(owner)), E, S, gu.DEV) for _ in range(2))
    for c in (one, two):
        c.policy, c.decay = 1, 2
        for t in c.slots.values():
            t.zero_()
    two._layer_plan = lambda: (None, None)  # the separate calls
    dt = torch.int64 if id64 else torch.int32
    for t, mk in enumerate([257, 300, 300, 1000, 1025, 2600, 3001, 4096, 0, 700]):
        if t in (2, 4):
            some = np.nonzero(one.table.cpu().numpy() >= 0)[0]  # resident: nothing to insert
        else:
            some = rng.permutation(E)[:E if t == 6 else min(E, S // 2 + 1)]
        ids = rng.choice(some, mk)
        ids[:2] = [-1, E + 3][:mk]
        buf = torch.zeros(mk + 4, device=gu.DEV, dtype=dt)
        ids_dev = buf[t % 2:t % 2 + mk]
        ids_dev.copy_(torch.as_tensor(rng.permutation(ids)))
        outs = [c.refresh(ids_dev) for c in (one, two)]
        torch.cuda.synchronize()
        assert torch.equal(*outs), t
        assert int(one.arrived) == 0
        for f in ("table", "map_cold", "slot_expert", "slot_stamp", "routed", "step", "miss",
                  "n_miss"):
            assert torch.equal(getattr(one, f), getattr(two, f)), (t, f)
        for n in one.names:
            assert torch.equal(one.slots[n], two.slots[n]), (t, n)


def test_refresh_in_a_graph():
    """Captured refreshes of two layers, replayed with the eager twin's steps between."""
    from types import SimpleNamespace

    from vllm_expert_cache.cache import ExpertSlotCache

    E, S, k = 96, 40, 12
    rng = np.random.default_rng(9)
    owner = SimpleNamespace(w=gu.pinned(E * 4112).view(E, 4112))
    gu.fill_random(owner.w.view(-1), 1)
    caches = [ExpertSlotCache(owner, ["w"], E, S, gu.DEV) for _ in range(4)]
    for c in caches:
        c.slots["w"].zero_()
    ids = torch.zeros(2, k, dtype=torch.int32, device=gu.DEV)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        outs = [c.refresh(i) for c, i in zip(caches[:2], ids)]
    for t in range(10):
        ids.copy_(torch.as_tensor(np.stack([rng.permutation(E)[:k] for _ in range(2)])))
        graph.replay()
        want = [c.refresh(i) for c, i in zip(caches[2:], ids)]
        torch.cuda.synchronize()
        for l in range(2):
            assert torch.equal(outs[l], want[l]), (t, l)
            for f in ("table", "slot_expert", "slot_stamp", "step", "n_miss"):
                assert torch.equal(getattr(caches[l], f), getattr(caches[l + 2], f)), (t, l, f)
            assert torch.equal(caches[l].slots["w"], caches[l + 2].slots["w"]), (t, l)


@pytest.mark.parametrize("id64", [False, True])
def test_refresh_in_place(id64):
    """Slot ids written over the routing ids, beside a twin that gets a buffer of its own."""
    from types import SimpleNamespace

    from vllm_expert_cache.cache import ExpertSlotCache

    E, S, k = 128, 48, 24
    rng = np.random.default_rng(5)
    owner = SimpleNamespace(w=gu.pinned(E * 8208).view(E, 8208))
    gu.fill_random(owner.w.view(-1), 2)
    one, two = (ExpertSlotCache(owner, ["w"], E, S, gu.DEV) for _ in range(2))
    for c in (one, two):
        c.slots["w"].zero_()
    one._plan()
    for t in range(12):
        ids = torch.as_tensor(rng.integers(-1, E, size=k if t % 3 else 4), device=gu.DEV)
        ids = ids.to(torch.int64 if id64 else torch.int32)
        want = two.refresh(ids)
        assert gu.lib().expert_cache_refresh(one._layer_at, ids.data_ptr(), ids.element_size(),
                                             ids.numel(), ids.data_ptr(), gu.stream()) == 0
        torch.cuda.synchronize()
        assert torch.equal(ids, want) and int(one.arrived) == 0, t
        for f in ("table", "slot_expert", "slot_stamp", "routed", "step", "miss", "n_miss"):
            assert torch.equal(getattr(one, f), getattr(two, f)), (t, f)
        assert torch.equal(one.slots["w"], two.slots["w"]), t


def _prefetch_step(st, ref, pred, budget, tag):
    """expert_cache_prefetch into the layer's own miss list, against the oracle's."""
    d = torch.as_tensor(pred, device=gu.DEV)
    assert gu.lib().expert_cache_prefetch(
        gu.ptr(d), len(pred), st.E, st.S, budget, st.row("table", 0), st.row("map_cold", 0),
        st.row("slot_expert", 0), st.row("slot_stamp", 0), st.row("routed", 0),
        st.row("miss", 0), st.row("n_miss", 0), gu.stream()) == 0
    assert ref.prefetch(pred, budget) == 0
    torch.cuda.synchronize()
    _check_state(st, ref, tag + " (prefetch)")


@pytest.mark.parametrize("E,S", [(64, 40), (128, 100), (256, 200), (512, 300), (1024, 900),
                                 (1300, 1000)])
@pytest.mark.parametrize("kind", ["one high", "half high", "all high", "spread", "one old",
                                  "half old", "past 43 bits"])
@pytest.mark.parametrize("policy", [0, 1])
def test_stamps_far_apart(E, S, kind, policy):
    """Evictable slots without a 32-bit key: above all keys (they are victims only where too
    few others are), below them (the keys start again from the smallest stamp), too few keys
    within reach of the smallest, and stamps that have none at all. Few and many victims, in
    the policy step and the prefetch step."""
    rng = np.random.default_rng(E + S + len(kind))
    for t, misses in enumerate([1, 3, 30, min(100, E - S)]):
        near, step = rng.integers(1, 50, size=S), 1 << 20
        stamps, pick = near.copy(), rng.permutation(S)
        if kind == "one high":
            stamps[pick[0]] += 1 << 40
        elif kind == "half high":
            stamps[pick[::2]] += 1 << 40
        elif kind == "all high":
            stamps += 1 << 40
        elif kind == "spread":
            stamps = (1 + pick) << 27
        elif kind == "past 43 bits":
            stamps[pick[:3]] = [1 << 43, 1 << 62, -5]
        else:  # stamps a long way back from the step
            step = (1 << 40) + 100
            stamps = near + (1 << 40)
            old = pick[:1] if kind == "one old" else pick[::2]
            stamps[old] = near[old]
        experts = rng.choice(E, S, replace=False)
        st, ref = _device_state(E, S, S, experts, rng.permutation(S), stamps)
        st.step[0] = step
        ref.step[:] = step
        for n in range(3):
            cold = np.nonzero(ref.table < 0)[0]
            ids = rng.permutation(cold)[:misses].astype(np.int32)
            tag = f"E={E} S={S} {kind} policy={policy} misses={misses} step {n}"
            if t % 2 == n % 2:
                _prefetch_step(st, ref, rng.permutation(cold)[:misses].astype(np.int32), S, tag)
            _step(st, ref, ids, S, policy, 0, False, tag)
