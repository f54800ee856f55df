"""The C++ host binding of the hip backend's per-call store and gather
(csrc/nkv_host.cpp), on the host: its checks restate the reference
validators (nanovllm/layers/paged_kv/base.py:75-151, restated in Python as
nanokv.paged_kv.base.check_store_inputs / check_gather_inputs), so every
input is held to the same outcome in both, the same ValueError message or
none, over the reference's own bad-input cases and more; and the binding
refuses to run before it is bound, and reports its build id."""
from __future__ import annotations

import os
from unittest.mock import patch

import pytest
import torch

from nanokv import _lib
from nanokv import build as nkv_build
from nanokv.paged_kv.base import check_gather_inputs, check_store_inputs


@pytest.fixture(scope="module")
def host():
    return _lib.load_host()


def _outcome(fn, *args):
    try:
        fn(*args)
    except ValueError as exc:
        return str(exc)
    return None


def store_inputs():
    key = torch.arange(3 * 2 * 4, dtype=torch.float32).reshape(3, 2, 4)
    return key, key + 100, torch.full((3, 4, 2, 4), -1.0), torch.full((3, 4, 2, 4), -1.0), \
        torch.tensor([0, 5, -1], dtype=torch.int32)


def store_cases():
    key, value, kc, vc, slots = store_inputs()
    yield "valid", (key, value, kc, vc, slots)
    yield "short key", (key[:2], value, kc, vc, slots)
    yield "2-d key", (key[0], value[0], kc, vc, slots)
    yield "narrow cache", (key, value, kc[:, :, :1], vc, slots)
    yield "cache dims", (key, value, kc[0], vc[0], slots)
    yield "cache head_dim", (key, value, kc[..., :2], vc[..., :2], slots)
    yield "int64 slots", (key, value, kc, vc, slots.to(torch.int64))
    yield "2-d slots", (key, value, kc, vc, slots.view(3, 1))
    yield "transposed", (key.transpose(1, 2), value.transpose(1, 2), kc, vc, slots)
    yield "value dtype", (key, value.to(torch.float16), kc, vc, slots)
    yield "cache dtype", (key, value, kc.double(), vc.double(), slots)
    yield "slot count", (key, value, kc, vc, slots[:2])
    yield "strided slots", (key, value, kc, vc, torch.tensor([0, 9, 5, 9, -1, 9], dtype=torch.int32)[::2])
    for bad in (12, -2):
        yield f"slot {bad}", (key, value, kc, vc, torch.tensor([0, bad, -1], dtype=torch.int32))
    empty = torch.empty(0, 2, 4)
    yield "empty", (empty, empty.clone(), kc, vc, torch.empty(0, dtype=torch.int32))


def gather_cases():
    cache = torch.zeros(3, 4, 2, 4)
    table = torch.tensor([2, 0], dtype=torch.int32)
    yield "valid", (cache, table, 6)
    yield "zero length", (cache, table, 0)
    yield "negative", (cache, table, -1)
    yield "int64 table", (cache, table.to(torch.int64), 6)
    yield "2-d table", (cache, table.view(1, 2), 6)
    yield "short table", (cache, table[:1], 6)
    yield "block 3", (cache, torch.tensor([3, 0], dtype=torch.int32), 6)
    yield "block -1", (cache, torch.tensor([-1, 0], dtype=torch.int32), 6)
    yield "tail not inspected", (cache, torch.tensor([2, 0, -1], dtype=torch.int32), 6)
    yield "3-d cache", (cache[0], table, 2)
    yield "strided cache", (cache.transpose(2, 3), table, 6)
    yield "strided table", (cache, torch.tensor([2, 9, 0, 9], dtype=torch.int32)[::2], 6)


@pytest.mark.parametrize("name,args", list(store_cases()), ids=[n for n, _ in store_cases()])
def test_store_checks_match_the_validator(host, name, args):
    expected = _outcome(check_store_inputs, *args)
    assert _outcome(host.check_store, *args) == expected
    # after the checks, host tensors are refused before any launch
    if expected is None:
        with pytest.raises(ValueError, match="ROCm"):
            host.store(*args, 0)


@pytest.mark.parametrize("name,args", list(gather_cases()), ids=[n for n, _ in gather_cases()])
def test_gather_checks_match_the_validator(host, name, args):
    expected = _outcome(check_gather_inputs, *args)
    assert _outcome(host.check_gather, *args) == expected
    if expected is None:
        with pytest.raises(ValueError, match="ROCm"):
            host.gather(*args, 0)


def test_index_validation_flag_is_read_per_call(host):
    """Device-resident indexes are value-checked only under the flag (host
    tensors always); the binding reads the flag as the validator does."""
    key, value, kc, vc, _ = store_inputs()
    bad = torch.tensor([0, 12, -1], dtype=torch.int32)
    with patch.dict(os.environ, {"NANOVLLM_PAGED_KV_VALIDATE_INDICES": "0"}):
        # host tensors: checked whatever the flag says
        assert "slot outside" in _outcome(host.check_store, key, value, kc, vc, bad)


def test_build_id_matches_the_sources_and_torch(host):
    assert host.build_id() == nkv_build.host_build_id()


def test_graph_buffers_collect_dead_cycles_before_a_capture():
    """Allocating a decode graph's buffers frees what only reference cycles
    hold (a dead CUDAGraph collected during the capture that follows would
    end the process)."""
    import weakref

    from nanokv.packing import DecodeGraphBuffers

    class Holder:
        pass

    holder = Holder()
    holder.self = holder
    dead = weakref.ref(holder)
    del holder
    DecodeGraphBuffers.allocate("cpu", 2, 3)
    assert dead() is None


def test_graph_buffers_leave_the_whole_heap_alone():
    """Only capture_graph pays for a full collection."""
    import gc

    from nanokv.packing import DecodeGraphBuffers

    full = []

    def watch(phase, info):
        if phase == "start" and info["generation"] == 2:
            full.append(info)

    gc.disable()
    gc.callbacks.append(watch)
    try:
        DecodeGraphBuffers.allocate("cpu", 2, 3)
    finally:
        gc.callbacks.remove(watch)
        gc.enable()
    assert not full


@pytest.mark.parametrize("collector_on", [True, False])
@pytest.mark.parametrize("fails", [False, True])
def test_capture_graph_keeps_the_collector_out(monkeypatch, collector_on, fails):
    """Dead cycles of any age are freed before the capture starts, the
    collector is off until the last capture under way has ended, also when
    one raises, and is then as it was."""
    import gc
    import weakref
    from contextlib import contextmanager

    from nanokv import packing

    class Holder:
        pass

    old = Holder()
    old.self = old
    gc.collect()  # now of the oldest generation
    dead = weakref.ref(old)
    del old
    seen = []

    @contextmanager
    def capture(graph, **options):
        seen.append((graph, options, dead() is None, gc.isenabled()))
        yield
        seen.append(gc.isenabled())

    monkeypatch.setattr(torch.cuda, "graph", capture)
    (gc.enable if collector_on else gc.disable)()
    try:
        try:
            with packing.capture_graph("outer", pool=3):
                with packing.capture_graph("inner"):
                    pass
                assert not gc.isenabled()
                if fails:
                    raise RuntimeError("captured work failed")
        except RuntimeError:
            assert fails
        assert gc.isenabled() == collector_on
    finally:
        gc.enable()
    assert seen[:3] == [("outer", {"pool": 3}, True, False), ("inner", {}, True, False), False]
    assert seen[3:] == ([] if fails else [False])


def test_attention_calls_the_binding_leaves_to_the_general_path():
    """Host tensors, and calls any check of the general path looks into, are
    not taken by the binding's attention entries: they return None, and the
    backend's own checks answer."""
    import torch

    from nanokv import _lib

    host = _lib.load_host()
    q = torch.zeros((2, 4, 128), dtype=torch.bfloat16)
    cache = torch.zeros((3, 16, 2, 128), dtype=torch.bfloat16)
    tables = torch.zeros((2, 1), dtype=torch.int32)
    cu = torch.tensor([0, 1, 2], dtype=torch.int32)
    plan = torch.zeros((1030, 4), dtype=torch.int32)
    assert host.decode(q, cache, cache, tables, cu, plan, cu, 2, 0.1, None, 0) is None
    assert host.prefill(q, cache, cache, tables, cu, cu, None, 0.1, None, 0) is None
    rows = torch.zeros((2, 2, 128), dtype=torch.bfloat16)
    assert host.varlen(q, rows, rows, cu, cu, 1, 0.1, 0) is None


@pytest.mark.parametrize("total,error", [(-1, ValueError), ("many", ValueError), ([3], TypeError)])
def test_prefill_refuses_a_bad_context_total_before_the_binding(host, monkeypatch, total, error):
    """The binding does not read total_context_tokens; what the general path
    refuses there never reaches it."""
    from nanokv.paged_kv import hip_backend

    backend = hip_backend.HIPPagedKVBackend()
    backend._load()

    class Taken:
        prefill = staticmethod(lambda *args: "taken")

    monkeypatch.setattr(hip_backend, "_HOST", Taken)
    q = torch.zeros((3, 4, 128), dtype=torch.bfloat16)
    cache = torch.zeros((3, 16, 2, 128), dtype=torch.bfloat16)
    tables = torch.zeros((2, 1), dtype=torch.int32)
    cu = torch.tensor([0, 1, 3], dtype=torch.int32)
    args = (q, cache, cache, tables, cu, cu, 0.1)
    assert backend.paged_attention_prefill(*args, total_context_tokens=3) == "taken"
    with pytest.raises(error):
        backend.paged_attention_prefill(*args, total_context_tokens=total)
